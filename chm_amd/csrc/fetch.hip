// Upwind fetch (CHM fetchr, src/modules/fetchr.cpp:28-120) on the GPU.
//
// A face's steps along the upwind azimuth each need the face whose centroid is
// nearest to a point (triangulation.cpp:170-178: a CGAL k = 1 kd-tree query).
// Centroids are bucketed once into a uniform grid (about two per cell) and laid
// out cell by cell, row by row, faces ascending inside a cell, so a run of cells
// of one row is one run of memory.  A query scans the three rows of cells around
// its point, then square rings of cells, on each side only the cells that can
// still hold something nearer than the best so far, and stops when the next ring
// lies farther than the best distance.  The result is the exact nearest centroid
// under the squared distance dx*dx + dy*dy (ties to the lower face index),
// identical to a brute-force scan.  Queries outside the grid (upwind of the
// domain edge) start at the first ring that reaches the grid.
//
// A step only asks whether the nearest face rises above the sight line (or
// shelters the distance), so each cell also keeps bounds of what the nearest face
// of a point in it can be: most steps are decided by the bounds alone, and only
// the others search.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/pbsm3d_fetch.h"
#include "kernels.hpp"

namespace pb {
namespace {

struct CentroidGrid {
    double xmin, ymin, h, inv_h;
    int64_t nx, ny;
    const int32_t* start;  // [nx*ny + 1] first slot of each cell (cell = cy * nx + cx)
    const int32_t* face;   // [F] face ids by cell, ascending inside a cell
    const double2* xy;     // [F] centroids in slot order
};

__device__ __forceinline__ void take(const CentroidGrid& g, int32_t s, double2 c, double qx, double qy, double& best,
                                     int32_t& bs) {
    const double dx = qx - c.x;
    const double dy = qy - c.y;
    const double d2 = dx * dx + dy * dy;
    if (d2 < best || (d2 == best && bs >= 0 && g.face[s] < g.face[bs])) {
        best = d2;
        bs = s;
    }
}

// slots [a, b) against the best so far, kRun loads in flight
constexpr int kRun = 4;
__device__ __forceinline__ void scan_slots(const CentroidGrid& g, int32_t a, int32_t b, double qx, double qy,
                                           double& best, int32_t& bs) {
    for (; a < b; a += kRun) {
        double2 c[kRun];
#pragma unroll
        for (int k = 0; k < kRun; ++k) c[k] = g.xy[min(a + k, b - 1)];
#pragma unroll
        for (int k = 0; k < kRun; ++k)
            if (a + k < b) take(g, a + k, c[k], qx, qy, best, bs);
    }
}

// cells [lo, hi] along x in row cy (or along y in column cx) that may hold a
// centroid within sqrt(best) of q, given the perpendicular gap `gap`
__device__ __forceinline__ void span(double best, double gap, double q, double origin, double h, int64_t lo,
                                     int64_t hi, int64_t& a, int64_t& b) {
    a = lo;
    b = hi;
    if (best < INFINITY) {
        const double w2 = best - gap * gap;
        if (w2 < 0) {
            a = 1;
            b = 0;
            return;
        }
        const double w = sqrt(w2) * (1 + 1e-12) + 1e-9;
        a = max(lo, (int64_t)floor((q - w - origin) / h));
        b = min(hi, (int64_t)floor((q + w - origin) / h));
    }
}

// the cell index of q along one axis, bounded so that a point far outside stays representable
__device__ __forceinline__ int64_t cell_of(double q, double origin, double inv_h) {
    const double lim = (double)((int64_t)1 << 40);
    return (int64_t)fmin(fmax(floor((q - origin) * inv_h), -lim), lim);
}

// slot of the centroid nearest to q, -1 where q is not finite
__device__ int32_t nearest_slot(const CentroidGrid& g, double qx, double qy) {
    if (!isfinite(qx) || !isfinite(qy)) return -1;
    const int64_t ix = cell_of(qx, g.xmin, g.inv_h), iy = cell_of(qy, g.ymin, g.inv_h);
    const int64_t r0 = max(max((int64_t)0, max(-ix, ix - (g.nx - 1))), max(-iy, iy - (g.ny - 1)));
    const int64_t rmax = max(max(ix, g.nx - 1 - ix), max(iy, g.ny - 1 - iy));
    double best = INFINITY;
    int32_t bs = -1;
    // The 3 x 3 cells around q, or around the grid cell nearest to it: rings 0 and 1 of a point in
    // the grid, and a first bound for one outside (without it the first ring that reaches the grid
    // is scanned whole).  A row
    // is one run of slots, and the bounds of the three runs load together.
    const int64_t jx = min(max(ix, (int64_t)0), g.nx - 1), jy = min(max(iy, (int64_t)0), g.ny - 1);
    const int64_t xa = max((int64_t)0, jx - 1), xb = min(g.nx - 1, jx + 1) + 1;
    int32_t lo[3], hi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int64_t row = jy + (k == 0 ? 0 : k == 1 ? -1 : 1);
        const bool in = row >= 0 && row < g.ny;
        const int64_t at = (in ? row : jy) * g.nx;
        lo[k] = g.start[at + xa];
        hi[k] = in ? g.start[at + xb] : lo[k];
    }
    scan_slots(g, lo[0], hi[0], qx, qy, best, bs);
    const double y0 = g.ymin + jy * g.h;
    const double below = fmax(0.0, qy - y0 - 1e-6 * (1.0 + g.h)), above = fmax(0.0, y0 + g.h - qy - 1e-6 * (1.0 + g.h));
    if (below * below <= best) scan_slots(g, lo[1], hi[1], qx, qy, best, bs);
    if (above * above <= best) scan_slots(g, lo[2], hi[2], qx, qy, best, bs);
    int64_t r = r0;
    if (r0 == 0) {
        // what is left lies beyond the block's edges; the margin covers the rounding of the cell index
        const double x0 = g.xmin + jx * g.h;
        const double edge = fmin(fmin(qx - x0, x0 + g.h - qx), fmin(qy - y0, y0 + g.h - qy));
        const double lb = g.h + edge - 1e-6 * (1.0 + g.h);
        if (bs >= 0 && lb > 0 && best <= lb * lb) return bs;
        r = 2;
    }
    for (; r <= rmax; ++r) {
        int64_t a, b;
        // rows iy - r and iy + r (corners included)
        for (int side = 0; side < 2; ++side) {
            const int64_t cyr = side == 0 ? iy - r : iy + r;
            if (cyr < 0 || cyr >= g.ny) continue;
            const double y0 = g.ymin + cyr * g.h;
            const double gap = side == 0 ? fmax(0.0, qy - (y0 + g.h)) : fmax(0.0, y0 - qy);
            span(best, gap, qx, g.xmin, g.h, max((int64_t)0, ix - r), min(g.nx - 1, ix + r), a, b);
            if (a <= b) scan_slots(g, g.start[cyr * g.nx + a], g.start[cyr * g.nx + b + 1], qx, qy, best, bs);
        }
        // columns ix - r and ix + r (corners excluded)
        for (int side = 0; side < 2; ++side) {
            const int64_t cxr = side == 0 ? ix - r : ix + r;
            if (cxr < 0 || cxr >= g.nx) continue;
            const double x0 = g.xmin + cxr * g.h;
            const double gap = side == 0 ? fmax(0.0, qx - (x0 + g.h)) : fmax(0.0, x0 - qx);
            span(best, gap, qy, g.ymin, g.h, max((int64_t)0, iy - r + 1), min(g.ny - 1, iy + r - 1), a, b);
            for (int64_t c = a; c <= b; ++c)
                scan_slots(g, g.start[c * g.nx + cxr], g.start[c * g.nx + cxr + 1], qx, qy, best, bs);
        }
        // every cell of ring r + 1 or beyond lies at least r * h from q (q is inside
        // cell (ix, iy)); the margin covers the rounding of the cell index
        if (bs >= 0) {
            const double lb = r * g.h - 1e-6 * (1.0 + g.h);
            if (lb > 0 && best <= lb * lb) break;
        }
    }
    return bs;
}

// What a step needs of a slot's face: the height of its top and the distance its canopy shelters
// (0 without vegetation), fetchr.cpp:86-104, expression order kept.
__global__ void __launch_bounds__(kBlock) k_slot_terrain(int64_t F, const int32_t* __restrict__ face,
                                                         const double* __restrict__ cx, const double* __restrict__ cy,
                                                         const double* __restrict__ cz,
                                                         const double* __restrict__ canopy, double2* __restrict__ xy,
                                                         double* __restrict__ top, double* __restrict__ shelter) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= F) return;
    const int32_t f = face[s];
    xy[s] = make_double2(cx[f], cy[f]);
    double Z_CanTop = 0;
    if (canopy) Z_CanTop = canopy[f];
    top[s] = cz[f] + Z_CanTop;
    if (!shelter) return;
    const double z0_1 = 0.12 * Z_CanTop;
    const double z0_2 = 0.001;
    const double n = 1.0 / 0.8;
    const double h = 5;
    shelter[s] = pow(((33.33333333 * h - 25. * z0_2) / (log(z0_1 / z0_2) * z0_2)), n) * z0_2;
}

// Bounds of each cell: the lowest and highest top, and the longest shelter, of the faces that can
// be nearest to a point in the cell.  With a centroid in the cell itself the nearest one is within
// sqrt(2) h, so at most 2 cells away; with one among the 8 around it, within 2 sqrt(2) h: 3 cells
// away (both with slack for the rounding of the cell index).  A sparser cell, or one with a NaN
// top in reach, gets bounds that decide nothing.
__global__ void __launch_bounds__(kBlock) k_cell_bounds(CentroidGrid g, const double* __restrict__ top,
                                                        const double* __restrict__ shelter,
                                                        float2* __restrict__ range, float* __restrict__ reach) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.nx * g.ny) return;
    const int64_t ix = c % g.nx, iy = c / g.nx;
    int ring = 4;
    if (g.start[c + 1] > g.start[c])
        ring = 2;
    else
        for (int64_t y = max((int64_t)0, iy - 1); y <= min(g.ny - 1, iy + 1); ++y)
            if (g.start[y * g.nx + min(g.nx - 1, ix + 1) + 1] > g.start[y * g.nx + max((int64_t)0, ix - 1)]) ring = 3;
    double lo = INFINITY, hi = -INFINITY, sh = 0;
    bool known = ring < 4;
    for (int64_t y = max((int64_t)0, iy - ring); known && y <= min(g.ny - 1, iy + ring); ++y) {
        const int32_t a = g.start[y * g.nx + max((int64_t)0, ix - ring)];
        const int32_t b = g.start[y * g.nx + min(g.nx - 1, ix + ring) + 1];
        for (int32_t s = a; s < b; ++s) {
            const double t = top[s];
            known = known && t == t;
            lo = fmin(lo, t);
            hi = fmax(hi, t);
            if (shelter) sh = fmax(sh, shelter[s]);  // a NaN shelters nothing
        }
    }
    range[c] = known ? make_float2(__double2float_rd(lo), __double2float_ru(hi)) : make_float2(-INFINITY, INFINITY);
    if (reach) reach[c] = known ? __double2float_ru(sh) : INFINITY;
}

struct FetchArgs {
    int64_t F;
    int steps;
    double max_distance, I;
    const double *cx, *cy, *cz;
    const double* canopy;  // null: no vegetation, or ignored
    const double *top, *shelter;
    const float2* range;
    const float* reach;
    const double* vw_dir;
    double* fetch;
};

// One step of fetchr::run (fetchr.cpp:55-118, expression order kept): the face's own values and
// the step's query point.
struct Sight {
    double x, y, z, sb, cb;
    // point_from_bearing_UTM (coordinates.cpp:60-71)
    __device__ __forceinline__ void look(const FetchArgs& a, int64_t i, double wind_dir) {
        const double DegreesToRadians = M_PI / 180.0;
        const double bearing = wind_dir * DegreesToRadians;
        sb = sin(bearing);
        cb = cos(bearing);
        x = a.cx[i];
        y = a.cy[i];
        z = a.cz[i];
    }
    __device__ __forceinline__ double qx(double distance) const {
        const double dist_x = distance * sb;
        return x + dist_x;
    }
    __device__ __forceinline__ double qy(double distance) const {
        const double dist_y = distance * cb;
        return y + dist_y;
    }
};

enum Step { kMiss, kHit, kUnknown };

// what the bounds of the query point's cell say
__device__ __forceinline__ Step step_by_bounds(const CentroidGrid& g, const FetchArgs& a, const Sight& f,
                                               double distance) {
    const int64_t ix = cell_of(f.qx(distance), g.xmin, g.inv_h), iy = cell_of(f.qy(distance), g.ymin, g.inv_h);
    if (ix < 0 || ix >= g.nx || iy < 0 || iy >= g.ny) return kUnknown;
    const float2 zr = a.range[iy * g.nx + ix];
    const float sh = a.reach ? a.reach[iy * g.nx + ix] : 0.0f;
    const double Z_core = f.z + distance * a.I;
    if ((double)zr.x >= Z_core) return kHit;
    return (double)zr.y < Z_core && distance >= (double)sh ? kMiss : kUnknown;
}

__device__ __forceinline__ bool step_by_search(const CentroidGrid& g, const FetchArgs& a, double qx, double qy,
                                               double Z_core, double distance) {
    const int32_t s = nearest_slot(g, qx, qy);
    return s >= 0 && (a.top[s] >= Z_core || (a.shelter && distance < a.shelter[s]));
}

// Few faces: 16 lanes share a face, each with a step of its own, and the first step that hits is
// the answer.  The chains of dependent loads (cell, bounds, search) are the bound there, and side
// by side a face's steps take one chain's time.
constexpr int kLanes = 16;
__global__ void __launch_bounds__(kBlock) k_fetch_lanes(CentroidGrid g, FetchArgs a) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t i = t / kLanes;
    const int lane = (int)(t % kLanes);
    if (i >= a.F) return;  // the lanes of a face leave together
    const double size_of_step = a.max_distance / a.steps;
    double out = a.max_distance;
    const double wind_dir = a.vw_dir[i];
    const bool canopy = a.canopy && a.canopy[i] > 1;
    if (canopy || !isfinite(wind_dir)) {  // the latter: no upwind point to search from (-9999 is finite)
        if (lane == 0) a.fetch[i] = canopy ? 0 : out;
        return;
    }
    Sight f;
    f.look(a, i, wind_dir);
    for (int j0 = 1; j0 <= a.steps; j0 += kLanes) {
        const int j = j0 + lane;
        const double distance = j * size_of_step;
        bool hit = false;
        if (j <= a.steps) {
            const Step st = step_by_bounds(g, a, f, distance);
            hit = st == kHit || (st == kUnknown && step_by_search(g, a, f.qx(distance), f.qy(distance),
                                                                  f.z + distance * a.I, distance));
        }
        const uint64_t group =
            (__ballot(hit) >> ((threadIdx.x & 63) / kLanes * kLanes)) & (((uint64_t)1 << kLanes) - 1);
        if (group) {
            out = (j0 + __ffsll((unsigned long long)group) - 1) * size_of_step;
            break;
        }
    }
    if (lane == 0) a.fetch[i] = out;
}

// Many faces: a workgroup takes kBlock faces and up to kChunk steps at a time.  Each thread decides
// its face's steps by the bounds up to the first sure hit and queues the undecided ones in LDS;
// then all threads search for the queue's entries, so that the searches, which bound the kernel and
// which only some faces need at any one step, run on full waves.  Entries past a hit already
// found are skipped.
constexpr int kChunk = 10;
__global__ void __launch_bounds__(kBlock) k_fetch_queue(CentroidGrid g, FetchArgs a) {
    __shared__ Sight face[kBlock];
    __shared__ int first[kBlock];  // first step known to hit
    __shared__ uint16_t queue[kBlock * kChunk];
    __shared__ int count, open;
    const int tid = threadIdx.x;
    const int64_t i = (int64_t)blockIdx.x * kBlock + tid;
    const double size_of_step = a.max_distance / a.steps;
    const int none = a.steps + 1;
    bool canopy = false, search = false;
    Sight f{};
    if (i < a.F) {
        const double wind_dir = a.vw_dir[i];
        canopy = a.canopy && a.canopy[i] > 1;
        search = !canopy && isfinite(wind_dir);  // not finite: no upwind point (-9999 is finite)
        if (search) f.look(a, i, wind_dir);
    }
    face[tid] = f;
    first[tid] = none;
    for (int j0 = 1; j0 <= a.steps; j0 += kChunk) {
        if (tid == 0) count = open = 0;
        __syncthreads();
        const int end = min(a.steps, j0 + kChunk - 1);
        bool going = search && first[tid] == none;
        if (going) open = 1;
        for (int j = j0; j <= end; ++j) {
            const Step st = going ? step_by_bounds(g, a, f, j * size_of_step) : kMiss;
            const uint64_t want = __ballot(st == kUnknown);
            int at = 0;
            if (want && (tid & 63) == 0) at = atomicAdd(&count, __popcll(want));
            at = __shfl(at, 0);
            if (st == kUnknown)
                queue[at + __popcll(want & (((uint64_t)1 << (tid & 63)) - 1))] = (uint16_t)(tid * kChunk + (j - j0));
            if (st == kHit) {
                first[tid] = j;
                going = false;
            }
        }
        __syncthreads();
        if (!open) break;  // every face has its answer
        for (int q = tid; q < count; q += kBlock) {
            const int e = queue[q], k = e / kChunk, j = j0 + e % kChunk;
            if (j >= first[k]) continue;
            const double distance = j * size_of_step;
            const Sight& s = face[k];
            if (step_by_search(g, a, s.qx(distance), s.qy(distance), s.z + distance * a.I, distance))
                atomicMin(&first[k], j);
        }
        __syncthreads();
    }
    if (i < a.F) a.fetch[i] = canopy ? 0 : first[tid] < none ? first[tid] * size_of_step : a.max_distance;
}

__global__ void __launch_bounds__(kBlock) k_nearest(CentroidGrid g, int64_t n, const double* __restrict__ qx,
                                                    const double* __restrict__ qy, int32_t* __restrict__ idx) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int32_t s = nearest_slot(g, qx[k], qy[k]);
    idx[k] = s < 0 ? -1 : g.face[s];
}

// Where the two kernels meet (us per call without / with canopy, lanes against queue): 13,000
// faces 32 / 32 against 129 / 106, 200,000 faces 122 / 131 against 202 / 139, 400,000 faces 208 / 235
// against 216 / 180, 1,000,000 faces 444 / 535 against 265 / 241 (one thread per face that searched
// at every step and scanned the first ring outside the grid whole: 190 us at 13,000 faces, 1,665 us
// at 1,000,000).
constexpr int64_t kFetchQueueFaces = 400000;

}  // namespace
}  // namespace pb

using namespace pb;

struct pbsm3d_fetch_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    int64_t F = 0;
    pbsm3d_fetch_config cfg{};
    DevBuf<double> cx, cy, cz, canopy, stage_in, stage_out;
    DevBuf<double> top, shelter;  // by slot (k_slot_terrain)
    DevBuf<double2> xy;
    DevBuf<float2> range;  // by cell (k_cell_bounds)
    DevBuf<float> reach;
    DevBuf<int32_t> start, face;
    double xmin = 0, ymin = 0, h = 1;
    int64_t nx = 1, ny = 1;
    bool has_canopy = false;
    std::string err;
    ~pbsm3d_fetch_ctx() {
        if (stream) (void)hipStreamDestroy(stream);
    }
    bool veg() const { return cfg.incl_veg && has_canopy; }
    CentroidGrid grid() const { return CentroidGrid{xmin, ymin, h, 1.0 / h, nx, ny, start.p, face.p, xy.p}; }
};

namespace {
std::string g_fetch_err;  // last creation error (no context to hold it)

template <typename Fn>
int fetch_guard(pbsm3d_fetch_ctx* c, Fn&& fn) {
    try {
        fn();
        return PBSM3D_OK;
    } catch (const Error& e) {
        if (c) c->err = e.what();
        g_fetch_err = e.what();
        return e.code;
    } catch (const std::exception& e) {
        if (c) c->err = e.what();
        g_fetch_err = e.what();
        return PBSM3D_EINVAL;
    }
}
}  // namespace

extern "C" {

void pbsm3d_fetch_config_default(pbsm3d_fetch_config* c) {
    std::memset(c, 0, sizeof(*c));
    c->steps = 10;
    c->incl_veg = 1;
    c->max_distance = 1000.0;
    c->I = 0.06;
}

int pbsm3d_fetch_create(pbsm3d_fetch_ctx** out, int device, int64_t F, const double* x, const double* y,
                        const double* z, const double* canopy, const pbsm3d_fetch_config* cfg) {
    if (!out || F <= 0 || F > INT32_MAX || !x || !y || !z || !cfg) {
        g_fetch_err = "invalid argument";
        return PBSM3D_EINVAL;
    }
    if (cfg->steps < 1 || !(cfg->max_distance > 0)) {
        g_fetch_err = "steps must be >= 1 and max_distance > 0";
        return PBSM3D_EINVAL;
    }
    *out = nullptr;
    auto* c = new pbsm3d_fetch_ctx();
    const int rc = fetch_guard(c, [&] {
        c->device = device;
        c->F = F;
        c->cfg = *cfg;
        PB_HIP(hipSetDevice(device));
        PB_HIP(hipStreamCreate(&c->stream));
        hipStream_t s = c->stream;
        // uniform grid of about two centroids per cell
        double xmin = x[0], xmax = x[0], ymin = y[0], ymax = y[0];
        for (int64_t i = 0; i < F; ++i) {
            if (!std::isfinite(x[i]) || !std::isfinite(y[i])) throw Error(PBSM3D_EINVAL, "non-finite centroid");
            xmin = std::min(xmin, x[i]);
            xmax = std::max(xmax, x[i]);
            ymin = std::min(ymin, y[i]);
            ymax = std::max(ymax, y[i]);
        }
        const double ext = std::max(xmax - xmin, ymax - ymin);
        double h = std::sqrt(std::max((xmax - xmin) * (ymax - ymin), 1e-300) * 2.0 / (double)F);
        if (!(h > 0) || h < ext * 1e-6) h = std::max(ext / std::sqrt((double)F), 1e-3);
        const int64_t nx = (int64_t)std::floor((xmax - xmin) / h) + 1;
        const int64_t ny = (int64_t)std::floor((ymax - ymin) / h) + 1;
        if (nx * ny > 8 * F + 64) throw Error(PBSM3D_EINVAL, "degenerate centroid extent");
        std::vector<int32_t> cell(F), start(nx * ny + 1, 0), face(F);
        for (int64_t i = 0; i < F; ++i) {
            const int64_t ix = std::min(nx - 1, (int64_t)std::floor((x[i] - xmin) / h));
            const int64_t iy = std::min(ny - 1, (int64_t)std::floor((y[i] - ymin) / h));
            cell[i] = (int32_t)(iy * nx + ix);
            start[cell[i] + 1]++;
        }
        for (int64_t k = 0; k < nx * ny; ++k) start[k + 1] += start[k];
        std::vector<int32_t> fill(start.begin(), start.end() - 1);
        for (int64_t i = 0; i < F; ++i) face[fill[cell[i]]++] = (int32_t)i;
        c->xmin = xmin;
        c->ymin = ymin;
        c->h = h;
        c->nx = nx;
        c->ny = ny;
        auto up = [&](DevBuf<double>& d, const double* hsrc) {
            d.alloc(F);
            PB_HIP(hipMemcpyAsync(d.p, hsrc, F * sizeof(double), hipMemcpyHostToDevice, s));
        };
        up(c->cx, x);
        up(c->cy, y);
        up(c->cz, z);
        c->has_canopy = canopy != nullptr;
        if (canopy) up(c->canopy, canopy);
        c->start.alloc(nx * ny + 1);
        c->face.alloc(F);
        PB_HIP(hipMemcpyAsync(c->start.p, start.data(), start.size() * sizeof(int32_t), hipMemcpyHostToDevice, s));
        PB_HIP(hipMemcpyAsync(c->face.p, face.data(), F * sizeof(int32_t), hipMemcpyHostToDevice, s));
        c->stage_in.alloc(F);
        c->stage_out.alloc(F);
        const bool veg = c->veg();
        c->xy.alloc(F);
        c->top.alloc(F);
        c->range.alloc(nx * ny);
        if (veg) {
            c->shelter.alloc(F);
            c->reach.alloc(nx * ny);
        }
        hipLaunchKernelGGL(k_slot_terrain, dim3(grid_for(F)), dim3(kBlock), 0, s, F, c->face.p, c->cx.p, c->cy.p,
                           c->cz.p, veg ? c->canopy.p : nullptr, c->xy.p, c->top.p, c->shelter.p);
        hipLaunchKernelGGL(k_cell_bounds, dim3(grid_for(nx * ny)), dim3(kBlock), 0, s, c->grid(), c->top.p,
                           c->shelter.p, c->range.p, c->reach.p);
        PB_HIP(hipGetLastError());
        PB_HIP(hipStreamSynchronize(s));
    });
    if (rc != PBSM3D_OK) {
        delete c;
        return rc;
    }
    *out = c;
    return PBSM3D_OK;
}

int pbsm3d_fetch_run(pbsm3d_fetch_ctx* c, const double* vw_dir, double* fetch, int on_device) {
    if (!c || !vw_dir || !fetch) return PBSM3D_EINVAL;
    return fetch_guard(c, [&] {
        PB_HIP(hipSetDevice(c->device));
        hipStream_t s = c->stream;
        const double* din = vw_dir;
        double* dout = fetch;
        if (!on_device) {
            PB_HIP(hipMemcpyAsync(c->stage_in.p, vw_dir, c->F * sizeof(double), hipMemcpyHostToDevice, s));
            din = c->stage_in.p;
            dout = c->stage_out.p;
        }
        const FetchArgs a{c->F,    c->cfg.steps, c->cfg.max_distance, c->cfg.I,  c->cx.p,    c->cy.p,
                          c->cz.p, c->veg() ? c->canopy.p : nullptr,   c->top.p,  c->shelter.p, c->range.p,
                          c->reach.p, din, dout};
        if (c->F < kFetchQueueFaces)
            hipLaunchKernelGGL(k_fetch_lanes, dim3(grid_for(c->F * kLanes)), dim3(kBlock), 0, s, c->grid(), a);
        else
            hipLaunchKernelGGL(k_fetch_queue, dim3(grid_for(c->F)), dim3(kBlock), 0, s, c->grid(), a);
        PB_HIP(hipGetLastError());
        if (!on_device) PB_HIP(hipMemcpyAsync(fetch, dout, c->F * sizeof(double), hipMemcpyDeviceToHost, s));
        PB_HIP(hipStreamSynchronize(s));
    });
}

int pbsm3d_fetch_nearest(pbsm3d_fetch_ctx* c, int64_t n, const double* qx, const double* qy, int32_t* idx) {
    if (!c || n < 0 || (n > 0 && (!qx || !qy || !idx))) return PBSM3D_EINVAL;
    if (n == 0) return PBSM3D_OK;
    return fetch_guard(c, [&] {
        PB_HIP(hipSetDevice(c->device));
        hipStream_t s = c->stream;
        DevBuf<double> dqx, dqy;
        DevBuf<int32_t> di;
        dqx.alloc(n);
        dqy.alloc(n);
        di.alloc(n);
        PB_HIP(hipMemcpyAsync(dqx.p, qx, n * sizeof(double), hipMemcpyHostToDevice, s));
        PB_HIP(hipMemcpyAsync(dqy.p, qy, n * sizeof(double), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(k_nearest, dim3(grid_for(n)), dim3(kBlock), 0, s, c->grid(), n, dqx.p, dqy.p, di.p);
        PB_HIP(hipGetLastError());
        PB_HIP(hipMemcpyAsync(idx, di.p, n * sizeof(int32_t), hipMemcpyDeviceToHost, s));
        PB_HIP(hipStreamSynchronize(s));
    });
}

void pbsm3d_fetch_destroy(pbsm3d_fetch_ctx* c) { delete c; }

const char* pbsm3d_fetch_last_error(const pbsm3d_fetch_ctx* c) { return c ? c->err.c_str() : g_fetch_err.c_str(); }

}  // extern "C"
