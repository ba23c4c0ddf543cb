// Vertical wind scaling (CHM scale_wind_vert, domain mode) on the GPU.
//
// Two passes over the faces: k_point_scale applies the log / exponential
// profiles of scale_wind_vert::point_scale (scale_wind_vert.cpp:56-155) to
// every face; k_smooth then gives each face the thin-plate-spline value of its
// (at most three) neighbours' point-scaled winds at its own centroid
// (scale_wind_vert.cpp:199-233, TPSpline.cpp:39-180): an (n+1) x (n+1) system
// per face, solved in registers by Gaussian elimination with partial pivoting --
// once per context, for the weights of the neighbours (k_weights), as it depends
// on the mesh alone.
// E1 (the reference takes GSL's gsl_sf_expint_E1) is evaluated from
// Abramowitz & Stegun: the power series 5.1.11 for x <= 1 and the continued
// fraction 5.1.22 by Lentz's method above.
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>

#include "../../include/pbsm3d_wind.h"
#include "kernels.hpp"

namespace pb {
namespace {

constexpr double kEulerGamma = 0.57721566490153286061;

__device__ double expint_e1(double x) {
    if (!(x > 0)) return x == 0 ? INFINITY : NAN;
    if (x <= 1.0) {
        double sum = 0, term = 1;
        for (int k = 1; k < 60; ++k) {
            term *= -x / k;
            const double add = term / k;
            sum += add;
            if (fabs(add) < 1e-18 * fabs(sum)) break;
        }
        return -kEulerGamma - log(x) - sum;
    }
    const double tiny = 1e-300;
    double b = x + 1.0, c = 1.0 / tiny, d = 1.0 / b, h = d;
    for (int i = 1; i < 1000; ++i) {
        const double an = -(double)i * i;
        b += 2.0;
        d = 1.0 / (an * d + b);
        c = b + an / c;
        const double del = c * d;
        h *= del;
        if (fabs(del - 1.0) < 1e-16) break;
    }
    return h * exp(-x);
}

__device__ __forceinline__ double log_scale_wind(double u, double Z_in, double Z_out, double snowdepthavg,
                                                 double z0) {
    const double Z0_SNOW = z0;
    u = u * log((Z_out - (snowdepthavg + Z0_SNOW)) / Z0_SNOW) / log((Z_in - (snowdepthavg + Z0_SNOW)) / Z0_SNOW);
    return u;
}

__device__ __forceinline__ double exp_scale_wind(double u, double Z_in, double Z_out, double alpha) {
    u = u * exp(alpha * (Z_out / Z_in - 1));
    return u;
}

struct WindArgs {
    int64_t F;
    int ignore_canopy;
    double z0;
    const double *canopy, *lai;  // null: no vegetation
    const double *U_R, *snowdepthavg;
    double* out;
};

__global__ void __launch_bounds__(kBlock) k_point_scale(WindArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.F) return;
    const double U_R = a.U_R[i];
    const double Z_R = 50.0;  // Atmosphere::Z_U_R
    double Z_CanTop = 0;
    if (!a.ignore_canopy && a.canopy) Z_CanTop = a.canopy[i];
    const double Z_CanBot = Z_CanTop / 2.0;
    double snowdepthavg = a.snowdepthavg ? a.snowdepthavg[i] : 0.0;
    if (chm_missing(snowdepthavg)) snowdepthavg = 0.0;
    const double Z_2m_above_srf = snowdepthavg + 2.0;
    if (Z_2m_above_srf >= Z_R) {
        a.out[i] = U_R;
        return;
    }
    double U_2m_above_srf;
    if (!a.ignore_canopy && (Z_CanTop > 0.0) && (Z_2m_above_srf < Z_CanTop)) {
        const double alpha = a.lai[i];
        if (snowdepthavg < Z_CanTop) {
            const double U_CanTop = log_scale_wind(U_R, Z_R, Z_CanTop, snowdepthavg, a.z0);
            const double U_CanBot = exp_scale_wind(U_CanTop, Z_CanTop, Z_CanBot, alpha);
            if (Z_2m_above_srf < Z_CanBot)
                U_2m_above_srf = log_scale_wind(U_CanBot, Z_CanBot, Z_2m_above_srf, snowdepthavg, a.z0);
            else
                U_2m_above_srf = exp_scale_wind(U_CanTop, Z_CanTop, Z_2m_above_srf, alpha);
        } else {
            U_2m_above_srf = log_scale_wind(U_R, Z_R, Z_2m_above_srf, snowdepthavg, a.z0);
        }
    } else {
        U_2m_above_srf = log_scale_wind(U_R, Z_R, Z_2m_above_srf, snowdepthavg, a.z0);
    }
    a.out[i] = fmax(0.1, U_2m_above_srf);
}

__device__ __forceinline__ double tps_basis(double sx, double sy, double ex, double ey) {
    const double c = 0.577215, weight = 0.01;  // TPSpline.cpp:196-201
    const double xdiff = sx - ex, ydiff = sy - ey;
    double dij = sqrt(xdiff * xdiff + ydiff * ydiff);
    dij = (dij * weight / 2.0) * (dij * weight / 2.0);
    return -(log(dij) + c + expint_e1(dij));
}

__global__ void k_clear_flag(double* flag) { *flag = 0.0; }

// The neighbours of face i (nb[j], -1 where there is none), the centroids of those that exist in
// slot order, and their count.  neigh[i * sf + j * sj] is neighbour j of face i (sf = 1, sj = F:
// the context's j-major copy; sf = 3, sj = 1: the ABI's face-major array).  CHECKED: the indices
// come straight from the caller's device memory, unvalidated: one outside [-1, F) counts as no
// neighbour and sets *bad = 1.
template <bool CHECKED>
__device__ __forceinline__ int tps_sites(int64_t F, int64_t i, const int32_t* neigh, int64_t sf, int64_t sj,
                                         const double* cx, const double* cy, int32_t nb[3], double sx[3],
                                         double sy[3], double* bad) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        nb[j] = neigh[i * sf + j * sj];
        if (CHECKED && (nb[j] < -1 || nb[j] >= F)) {
            *bad = 1.0;
            nb[j] = -1;
        }
        sx[j] = cx[nb[j] < 0 ? i : nb[j]];
        sy[j] = cy[nb[j] < 0 ? i : nb[j]];
    }
    // the existing ones to the front, without an index that only the lane knows: such an array
    // lies in scratch memory
    const bool h0 = nb[0] >= 0, h1 = nb[1] >= 0, h2 = nb[2] >= 0;
    if (!h1) {
        sx[1] = sx[2];
        sy[1] = sy[2];
    }
    if (!h0) {
        sx[0] = sx[1];
        sy[0] = sy[1];
        sx[1] = sx[2];
        sy[1] = sy[2];
    }
    return h0 + h1 + h2;
}

// The spline's value at (x, y) is linear in the sites' winds, and both the system and the basis
// depend on the mesh alone.  It reproduces constants, so the weights add up to one and the
// value is p1 + w2 (p2 - p1) + w3 (p3 - p1) over the sites in order; this form keeps the
// weights' rounding off the common part of the winds.  w[0] = w2 and w[1] = w3: the values for a
// unit wind at that site, from the (N + 1) x (N + 1) system by Gaussian elimination with partial
// pivoting, unrolled so that the system stays in registers.
template <int N>
__device__ __forceinline__ void tps_weights_of(const double sx[3], const double sy[3], double x, double y, double w[2]) {
    constexpr int M = N + 1, Q = N - 1;  // unknowns, right-hand sides
    double A[M][M + Q];
#pragma unroll
    for (int r = 0; r < M; ++r)
#pragma unroll
        for (int cc = 0; cc < M + Q; ++cc)
            A[r][cc] = cc >= M ? (r == cc - M + 1 ? 1.0 : 0.0) : cc == 0 ? (r < N ? 1.0 : 0.0) : r == N ? 1.0 : 0.0;
#pragma unroll
    for (int r = 0; r < N; ++r)
#pragma unroll
        for (int j = r + 1; j < N; ++j) {
            const double xdiff = sx[r] - sx[j], ydiff = sy[r] - sy[j];
            if (xdiff == 0. && ydiff == 0.) continue;
            const double Rd = tps_basis(sx[r], sy[r], sx[j], sy[j]);
            A[r][j + 1] = Rd;
            A[j][r + 1] = Rd;
        }
#pragma unroll
    for (int k = 0; k < M; ++k) {
        int p = k;
        double big = fabs(A[k][k]);
#pragma unroll
        for (int r = k + 1; r < M; ++r)
            if (fabs(A[r][k]) > big) {
                big = fabs(A[r][k]);
                p = r;
            }
#pragma unroll
        for (int r = k + 1; r < M; ++r)
#pragma unroll
            for (int cc = k; cc < M + Q; ++cc) {
                const double t = A[k][cc], u = A[r][cc];
                A[k][cc] = p == r ? u : t;
                A[r][cc] = p == r ? t : u;
            }
#pragma unroll
        for (int r = k + 1; r < M; ++r) {
            const double f = A[r][k] / A[k][k];
#pragma unroll
            for (int cc = k + 1; cc < M + Q; ++cc) A[r][cc] -= f * A[k][cc];
        }
    }
    double c[Q][M];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = M - 1; k >= 0; --k) {
            double s = A[k][M + q];
#pragma unroll
            for (int cc = k + 1; cc < M; ++cc) s -= A[k][cc] * c[q][cc];
            c[q][k] = s / A[k][k];
        }
#pragma unroll
    for (int q = 0; q < Q; ++q) w[q] = c[q][0];
#pragma unroll
    for (int r = 1; r < M; ++r) {
        const double b = tps_basis(sx[r - 1], sy[r - 1], x, y);
#pragma unroll
        for (int q = 0; q < Q; ++q) w[q] = w[q] + c[q][r] * b;
    }
}
// w[0] and w[1] of n sites (0 where there is no such site)
__device__ __forceinline__ void tps_weights(int n, const double sx[3], const double sy[3], double x, double y,
                                            double w[2]) {
    w[0] = w[1] = 0;
    if (n == 3) tps_weights_of<3>(sx, sy, x, y, w);
    if (n == 2) tps_weights_of<2>(sx, sy, x, y, w);
    // The value is the site's wind plus 0 times its basis, which is NaN (the floor) at the site itself.
    if (n == 1) w[0] = 0 * tps_basis(sx[0], sy[0], x, y);
}

// The smoothed wind of a face whose neighbours have the winds a, b and c; where there is none
// (nb[j] < 0), it is the face's own.
__device__ __forceinline__ double smoothed(const int32_t nb[3], double a, double b, double c, double w2, double w3) {
    const bool h0 = nb[0] >= 0, h1 = nb[1] >= 0, h2 = nb[2] >= 0;
    const double p1 = h0 ? a : h1 ? b : c;
    const double d2 = h0 ? (h1 ? b - p1 : h2 ? c - p1 : 0.0) : (h1 && h2 ? c - p1 : 0.0);
    const double d3 = h0 && h1 && h2 ? c - p1 : 0.0;
    double z = p1 + (w2 * d2 + w3 * d3);
    // an infinite neighbour makes NaN, and so the floor, as solving the system with it does
    if ((h0 || h1 || h2) && isinf(z)) z = NAN;
    return fmax(0.1, z);
}

// Smoothing from the caller's own geometry arrays (pbsm3d_wind_run_noalloc, which keeps nothing
// between calls): the weights are formed on every call.  A whole call on 399,968 faces takes 109 us,
// 100 of them launches, the wait and the flag's copy; 154 us with one right-hand side (the winds)
// and 182 with the weights' two when the system lay in scratch memory.
__global__ void __launch_bounds__(kBlock) k_smooth_checked(int64_t F, const int32_t* __restrict__ neigh,
                                                           const double* __restrict__ cx,
                                                           const double* __restrict__ cy,
                                                           const double* __restrict__ pt, double* __restrict__ out,
                                                           double* __restrict__ bad) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F) return;
    int32_t nb[3];
    double sx[3], sy[3], p[3], w[2];
    const int n = tps_sites<true>(F, i, neigh, 3, 1, cx, cy, nb, sx, sy, bad);
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] = pt[nb[j] < 0 ? i : nb[j]];
    tps_weights(n, sx, sy, cx[i], cy[i], w);
    out[i] = smoothed(nb, p[0], p[1], p[2], w[0], w[1]);
}

// The weights of every face: w[i] = w2, w[F + i] = w3.
__global__ void __launch_bounds__(kBlock) k_weights(int64_t F, const int32_t* __restrict__ neigh,
                                                    const double* __restrict__ cx, const double* __restrict__ cy,
                                                    double* __restrict__ w) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F) return;
    int32_t nb[3];
    double sx[3], sy[3], v[2];
    const int n = tps_sites<false>(F, i, neigh, 1, F, cx, cy, nb, sx, sy, nullptr);
    tps_weights(n, sx, sy, cx[i], cy[i], v);
    w[i] = v[0];
    w[F + i] = v[1];
}

// Smoothing with the context's weights: three gathers and two products per face, bound by
// the gathers (12 B of indices, 16 B of weights, 24 B gathered, 8 B out per face).  Solving the
// spline per call took six E1 series per face: 999,968 faces, both kernels, 262 us, now 32 us.
__global__ void __launch_bounds__(kBlock) k_smooth(int64_t F, const int32_t* __restrict__ neigh,
                                                   const double* __restrict__ w, const double* __restrict__ pt,
                                                   double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= F) return;
    int32_t nb[3];
    double p[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) nb[j] = neigh[i + j * F];
    const double w2 = w[i], w3 = w[F + i];
#pragma unroll
    for (int j = 0; j < 3; ++j) p[j] = pt[nb[j] < 0 ? i : nb[j]];
    out[i] = smoothed(nb, p[0], p[1], p[2], w2, w3);
}

}  // namespace
}  // namespace pb

using namespace pb;

struct pbsm3d_wind_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    int64_t F = 0;
    pbsm3d_wind_config cfg{};
    DevBuf<int32_t> neigh;  // j-major [j*F + i]
    DevBuf<double> cx, cy, canopy, lai, stage_u, stage_sd, stage_out, point, weights;  // weights: [2F] of k_smooth
    bool veg = false;
    std::string err;
    ~pbsm3d_wind_ctx() {
        if (stream) (void)hipStreamDestroy(stream);
    }
};

// Scratch of pbsm3d_wind_run_noalloc, which allocates nothing: the point-scaled wind of
// every face (the smoothing kernel reads the neighbours' values back) and, after it, one
// flag word for out-of-range neighbour indices.  32 MiB per GPU for the rest of the
// process.  Calls that overlap on one GPU share it and race.
static __device__ __align__(256) double scratch[PBSM3D_WIND_NOALLOC_MAX_FACES + 32];

namespace {
std::string g_wind_err;

// The device address of `scratch` on `device` (current), looked up once per device: each
// GPU holds its own copy at its own address, and the host-side name is not that address.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double* g_scratch_ptr[kMaxDevices] = {};

double* noalloc_scratch(int device) {
    if (device < 0 || device >= kMaxDevices) throw Error(PBSM3D_EINVAL, "device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        PB_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[device] = static_cast<double*>(p);
    }
    return g_scratch_ptr[device];
}

template <typename Fn>
int wind_guard(pbsm3d_wind_ctx* c, Fn&& fn) {
    try {
        fn();
        return PBSM3D_OK;
    } catch (const Error& e) {
        if (c) c->err = e.what();
        g_wind_err = e.what();
        return e.code;
    } catch (const std::exception& e) {
        if (c) c->err = e.what();
        g_wind_err = e.what();
        return PBSM3D_EINVAL;
    }
}
}  // namespace

extern "C" {

void pbsm3d_wind_config_default(pbsm3d_wind_config* c) {
    std::memset(c, 0, sizeof(*c));
    c->ignore_canopy = 0;
    c->smooth = 1;
    c->z0_snow = 0.01;
}

int pbsm3d_wind_create(pbsm3d_wind_ctx** out, int device, int64_t F, const int32_t* neigh, const double* x,
                       const double* y, const double* canopy, const double* lai, const pbsm3d_wind_config* cfg) {
    if (!out || F <= 0 || F > INT32_MAX || !neigh || !x || !y || !cfg || !(cfg->z0_snow > 0)) {
        g_wind_err = "invalid argument";
        return PBSM3D_EINVAL;
    }
    if (canopy && !lai && !cfg->ignore_canopy) {
        g_wind_err = "LAI is required with canopy heights (scale_wind_vert.cpp:110)";
        return PBSM3D_EINVAL;
    }
    for (int64_t k = 0; k < 3 * F; ++k)
        if (neigh[k] < -1 || neigh[k] >= F) {
            g_wind_err = "neighbour index out of range";
            return PBSM3D_EINVAL;
        }
    *out = nullptr;
    auto* c = new pbsm3d_wind_ctx();
    const int rc = wind_guard(c, [&] {
        c->device = device;
        c->F = F;
        c->cfg = *cfg;
        PB_HIP(hipSetDevice(device));
        PB_HIP(hipStreamCreate(&c->stream));
        hipStream_t s = c->stream;
        std::vector<int32_t> nj(3 * F);
        for (int64_t i = 0; i < F; ++i)
            for (int j = 0; j < 3; ++j) nj[j * F + i] = neigh[3 * i + j];
        c->neigh.alloc(3 * F);
        PB_HIP(hipMemcpyAsync(c->neigh.p, nj.data(), 3 * F * sizeof(int32_t), hipMemcpyHostToDevice, s));
        auto up = [&](DevBuf<double>& d, const double* h) {
            d.alloc(F);
            PB_HIP(hipMemcpyAsync(d.p, h, F * sizeof(double), hipMemcpyHostToDevice, s));
        };
        up(c->cx, x);
        up(c->cy, y);
        c->veg = canopy != nullptr;
        if (canopy) up(c->canopy, canopy);
        if (lai) up(c->lai, lai);
        for (DevBuf<double>* b : {&c->stage_u, &c->stage_sd, &c->stage_out, &c->point}) b->alloc(F);
        if (cfg->smooth) {
            c->weights.alloc(2 * F);
            hipLaunchKernelGGL(k_weights, dim3(grid_for(F)), dim3(kBlock), 0, s, F, c->neigh.p, c->cx.p, c->cy.p,
                               c->weights.p);
            PB_HIP(hipGetLastError());
        }
        PB_HIP(hipStreamSynchronize(s));
    });
    if (rc != PBSM3D_OK) {
        delete c;
        return rc;
    }
    *out = c;
    return PBSM3D_OK;
}

int pbsm3d_wind_run(pbsm3d_wind_ctx* c, const double* U_R, const double* snowdepthavg, double* U2, int on_device) {
    if (!c || !U_R || !U2) return PBSM3D_EINVAL;
    return wind_guard(c, [&] {
        PB_HIP(hipSetDevice(c->device));
        hipStream_t s = c->stream;
        const int64_t F = c->F;
        const double* du = U_R;
        const double* dsd = snowdepthavg;
        double* dout = U2;
        if (!on_device) {
            PB_HIP(hipMemcpyAsync(c->stage_u.p, U_R, F * sizeof(double), hipMemcpyHostToDevice, s));
            du = c->stage_u.p;
            if (snowdepthavg) {
                PB_HIP(hipMemcpyAsync(c->stage_sd.p, snowdepthavg, F * sizeof(double), hipMemcpyHostToDevice, s));
                dsd = c->stage_sd.p;
            }
            dout = c->stage_out.p;
        }
        WindArgs a{F, c->cfg.ignore_canopy, c->cfg.z0_snow, c->veg ? c->canopy.p : nullptr, c->lai.p, du, dsd,
                   c->cfg.smooth ? c->point.p : dout};
        hipLaunchKernelGGL(k_point_scale, dim3(grid_for(F)), dim3(kBlock), 0, s, a);
        if (c->cfg.smooth)
            hipLaunchKernelGGL(k_smooth, dim3(grid_for(F)), dim3(kBlock), 0, s, F, c->neigh.p, c->weights.p,
                               c->point.p, dout);
        PB_HIP(hipGetLastError());
        if (!on_device) PB_HIP(hipMemcpyAsync(U2, dout, F * sizeof(double), hipMemcpyDeviceToHost, s));
        PB_HIP(hipStreamSynchronize(s));
    });
}

int pbsm3d_wind_run_noalloc(int device, int64_t F, const int32_t* neigh, const double* x, const double* y,
                            const double* canopy, const double* lai, const pbsm3d_wind_config* cfg, const double* U_R,
                            const double* snowdepthavg, double* U2) {
    if (F <= 0 || !neigh || !x || !y || !cfg || !U_R || !U2 || !(cfg->z0_snow > 0)) {
        g_wind_err = "invalid argument";
        return PBSM3D_EINVAL;
    }
    if (F > PBSM3D_WIND_NOALLOC_MAX_FACES) {
        g_wind_err = "pbsm3d_wind_run_noalloc: " + std::to_string(F) + " faces exceed the scratch of " +
                     std::to_string((long long)PBSM3D_WIND_NOALLOC_MAX_FACES) + " faces";
        return PBSM3D_EINVAL;
    }
    if (canopy && !lai && !cfg->ignore_canopy) {
        g_wind_err = "LAI is required with canopy heights (scale_wind_vert.cpp:110)";
        return PBSM3D_EINVAL;
    }
    return wind_guard(nullptr, [&] {
        PB_HIP(hipSetDevice(device));
        double* scr = noalloc_scratch(device);  // [max faces] point-scaled winds, then the flag word
        double* bad = scr + PBSM3D_WIND_NOALLOC_MAX_FACES;
        hipStream_t s = nullptr;  // the device's null stream: creating a stream is left to the caller's set-up
        hipLaunchKernelGGL(k_clear_flag, dim3(1), dim3(1), 0, s, bad);
        WindArgs a{F, cfg->ignore_canopy, cfg->z0_snow, canopy, lai, U_R, snowdepthavg, cfg->smooth ? scr : U2};
        hipLaunchKernelGGL(k_point_scale, dim3(grid_for(F)), dim3(kBlock), 0, s, a);
        if (cfg->smooth)
            hipLaunchKernelGGL(k_smooth_checked, dim3(grid_for(F)), dim3(kBlock), 0, s, F, neigh, x, y, scr, U2, bad);
        PB_HIP(hipGetLastError());
        PB_HIP(hipStreamSynchronize(s));
        double flag = 0;
        PB_HIP(hipMemcpy(&flag, bad, sizeof(double), hipMemcpyDeviceToHost));
        if (flag != 0.0) throw Error(PBSM3D_EINVAL, "neighbour index out of range");
    });
}

void pbsm3d_wind_destroy(pbsm3d_wind_ctx* c) { delete c; }

const char* pbsm3d_wind_last_error(const pbsm3d_wind_ctx* c) { return c ? c->err.c_str() : g_wind_err.c_str(); }

}  // extern "C"
