// GMRES(m) with classical Gram-Schmidt and a conditional second pass (the
// DGKS test ||w_after|| < ||w_before|| / sqrt(2)), as iterated classical
// Gram-Schmidt does.  The basis lives in HBM, its vectors unscaled with their
// factors beside them; each Arnoldi step is
//   z = M^-1 w_j ; u = A z ; h = V^T u (one batched pass) ;
//   w_{j+1} = s_j u - V h (one pass, fused norm)
// The Hessenberg column, its Givens rotations and the least-squares solve stay
// on the device; the host reads only the residual estimate of the step before
// the one it queues, so the stream does not wait for it (a 5,000 x 5 system
// spent 78 us per step with a synchronisation in each, of which the kernels
// took 55).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <vector>

#include "krylov.hpp"

namespace pb {
namespace {

constexpr int kVecBlocks = 512;  // two workgroups per CU

inline int reduce_blocks(int64_t n) {
    int64_t b = (n + kBlock - 1) / kBlock;
    if (b > kReduceBlocks) b = kReduceBlocks;
    return (int)(b < 1 ? 1 : b);
}

// workgroups of a kernel that takes four rows per thread
inline int reduce_blocks4(int64_t n) { return reduce_blocks((n + 3) / 4); }

}  // namespace

void wait_slot(hipStream_t s, const HostSlot* slot, uint64_t seq) {
    const volatile uint64_t* at = &slot->seq;
    for (uint32_t spin = 1; *at != seq; ++spin) {
        if (spin % 4096 == 0) {  // a stream that failed, or ended without the report, never writes it
            const hipError_t e = hipStreamQuery(s);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();  // no error of the launches that follow
            } else if (*at != seq) {
                PB_HIP(e);
                throw Error(PBSM3D_EHIP, "a kernel ended without its report");
            }
        }
        __builtin_ia32_pause();
    }
    std::atomic_thread_fence(std::memory_order_acquire);
}

template <typename T>
void GmresWork<T>::ensure(int64_t n_, int m_) {
    if (n == n_ && m == m_ && V.p) return;
    n = n_;
    m = m_;
    ld = (n + 63) / 64 * 64;
    V.alloc((size_t)(m + 1) * ld);
    z.alloc(n);
    u.alloc(n);
    // residual partials: one per block of kBlock rows, or ceil(F / kBlock) * L <= n / kBlock + L
    // for the launches that run layer by layer (L <= 64)
    const size_t spmv_blocks = (size_t)((n + kBlock - 1) / kBlock) + 64;
    size_t pbytes = (size_t)kReduceBlocks * (m + 2);
    if (pbytes < spmv_blocks) pbytes = spmv_blocks;
    partial.alloc(pbytes);
    ss.alloc(kReduceBlocks);
    dsc.alloc(GmresSc::kDoubles);
    slot.alloc(4);
    for (int k = 0; k < 4; ++k) slot.p[k].seq = 0;
    seq = 0;
    PB_HIP(hipHostGetDevicePointer((void**)&dslot, slot.p, 0));
}

// How far the last known residual must lie above the target for the host to queue another Arnoldi
// step before the estimate of the one in flight: a step rarely gains more, and one queued past
// the end is work for nothing.
constexpr double kAhead = 30.0;

template <typename T>
int gmres_cycle(hipStream_t s, GmresWork<T>& w, const CsrOp<T>& A, const PcFn<T>& M, const T* r0, double beta,
                double stop_abs, int max_steps, T* out, double* resid_est) {
    const int64_t n = A.n, ld = w.ld;
    const int nblk = reduce_blocks4(n);
    T* V = w.V.p;
    const GmresSc sc = GmresSc::of(w.dsc.p);
    if (max_steps > w.m) max_steps = w.m;

    scale_host<T>(s, n, r0, 1.0 / beta, V);
    gmres_start(s, sc, beta);
    const uint64_t seq0 = w.seq;
    auto queue = [&](int j) {
        T* vj = V + (size_t)j * ld;
        T* vj1 = V + (size_t)(j + 1) * ld;
        if (M) {
            ProfScope ps(A.prof, s, PBSM3D_K_PRECOND);
            M(s, vj, w.z.p);
        }
        {
            ProfScope ps(A.prof, s,
                         A.prof_class >= 0 ? A.prof_class : sizeof(T) == 8 ? PBSM3D_K_SPMV64 : PBSM3D_K_SPMV32);
            op_spmv<T>(s, A, M ? w.z.p : vj, vj1);
        }
        ProfScope ps(A.prof, s, PBSM3D_K_ORTHO);
        mdot<T>(s, n, V, ld, j + 1, vj1, w.partial.p, nblk);
        gmres_h(s, sc, w.partial.p, nblk, j, 0);
        gs_update<T>(s, n, V, ld, j + 1, sc.coef, sc.scal + j, vj1, w.ss.p, nblk);
        if (w.passes > 1) {
            gmres_gate(s, sc, w.ss.p, nblk);
            mdot<T>(s, n, V, ld, j + 1, vj1, w.partial.p, nblk, sc.gate);
            gmres_h(s, sc, w.partial.p, nblk, j, 1);
            gs_update<T>(s, n, V, ld, j + 1, sc.coef, nullptr, vj1, w.ss.p, nblk, sc.gate);
        }
        gmres_step(s, sc, w.ss.p, nblk, j, w.dslot + (j & 1), ++w.seq);
        PB_HIP(hipGetLastError());
    };
    double res = beta;
    int queued = 0, known = 0;
    while (known < max_steps) {
        if (queued < max_steps && (queued == known || (queued == known + 1 && res > kAhead * stop_abs))) {
            queue(queued++);
            continue;
        }
        const HostSlot& sl = w.slot.p[known & 1];
        wait_slot(s, &sl, seq0 + known + 1);
        ++known;
        res = sl.v[0];
        if (res <= stop_abs || sl.v[1] == 0.0) break;
    }
    gmres_y(s, sc, known);
    combine<T>(s, n, V, ld, known, sc.coef, M ? w.u.p : out);
    if (M) {
        ProfScope ps(A.prof, s, PBSM3D_K_PRECOND);
        M(s, w.u.p, out);
    }
    *resid_est = res;
    return known;
}

namespace {
// A start whose residual exceeds ||b|| (that of x0 = 0) is dropped: x is reset
// to zero and the caller recomputes the residual.  Records ||r0|| / ||b||.  The
// margin keeps x0 = 0 itself, whose ||r0|| and ||b|| differ only by the order of
// their two reductions, from counting as a fallback.
bool drop_worse_start(hipStream_t s, SolveInfo& info, double beta, double nb, double* x, int64_t n) {
    info.resid0 = beta / nb;
    if (!(info.resid0 > 1.0 + 1e-12)) return false;
    PB_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, s));
    info.cold_fallback = true;
    return true;
}

// The norms below are queued with the number of their report, and read by norm_report.
template <typename T>
uint64_t queue_residual(hipStream_t s, GmresWork<T>& w, const CsrOp<double>& A, const double* x, const double* b,
                        double* r) {
    int nblk = 0;
    {
        ProfScope ps(A.prof, s, PBSM3D_K_RESIDUAL);
        nblk = op_residual(s, A, x, b, r, w.partial.p);
    }
    report_sum(s, w.partial.p, nblk, w.dslot + 2, ++w.seq);
    return w.seq;
}

template <typename T>
uint64_t queue_norm(hipStream_t s, GmresWork<T>& w, int64_t n, const double* v) {
    const int nblk = reduce_blocks4(n);
    mdot<double>(s, n, nullptr, 0, 0, v, w.partial.p, nblk);
    report_sum(s, w.partial.p, nblk, w.dslot + 3, ++w.seq);
    return w.seq;
}

template <typename T>
double norm_report(hipStream_t s, GmresWork<T>& w, int slot, uint64_t seq) {
    PB_HIP(hipGetLastError());
    wait_slot(s, w.slot.p + slot, seq);
    return std::sqrt(w.slot.p[slot].v[0]);
}

template <typename T>
double residual_norm(hipStream_t s, GmresWork<T>& w, const CsrOp<double>& A, const double* x, const double* b,
                     double* r) {
    return norm_report(s, w, 2, queue_residual(s, w, A, x, b, r));
}

template <typename T>
double norm_of(hipStream_t s, GmresWork<T>& w, int64_t n, const double* v) {
    return norm_report(s, w, 3, queue_norm(s, w, n, v));
}

// ||b|| and the start's residual: one wait for both.  False where b is zero; x is zero then.
template <typename T>
bool start_norms(hipStream_t s, GmresWork<T>& w, const CsrOp<double>& A, double* x, const double* b, double* r,
                 SolveInfo& info, double& nb, double& beta) {
    const uint64_t qb = queue_norm(s, w, A.n, b), qr = queue_residual(s, w, A, x, b, r);
    nb = norm_report(s, w, 3, qb);
    beta = norm_report(s, w, 2, qr);
    if (nb != 0.0) return true;
    PB_HIP(hipMemsetAsync(x, 0, sizeof(double) * A.n, s));
    info.converged = true;
    return false;
}
}  // namespace

namespace {
// One cycle on Ahat with the Neumann polynomial: x += (D~ + U)^-1 q(Ahat) y, where y minimises
// ||rhat - Ahat q(Ahat) y||, rhat = D~ (D~ + L)^-1 r; sp.work[0] keeps the x before.  *spent receives
// the operator applications of its steps.  False when the polynomial overflowed (x is unchanged).
bool split_cycle(hipStream_t s, GmresWork<double>& w, const SplitCycles& sp, const double* r, double beta,
                 double stop_rel, int max_steps, double* x, int* spent) {
    const CsrOp<double>& A = sp.Ahat;
    const int64_t n = A.n;
    double *r1 = sp.work[0], *rh = sp.work[1], *y = sp.work[2];
    scale_host<double>(s, n, r, 1.0 / beta, r1);
    split_op<double>(1, s, *A.co, A.F, A.L, *A.split, r1, rh, A.mode);
    const double bh = norm_of(s, w, n, rh);
    *spent = 0;
    if (!(bh > 0)) return false;
    PcFn<double> q;  // degree 1: q = 1
    if (sp.degree > 1)
        q = [&](hipStream_t st, const double* v, double* z) {
            // Horner: y0 = v, then y <- v + y - Ahat y, alternating between two vectors so that the
            // last lands in z
            const double* from = v;
            for (int k = 1; k < sp.degree; ++k) {
                double* to = (sp.degree - 1 - k) % 2 == 0 ? z : y;
                split_neumann(st, *A.co, A.F, A.L, *A.split, v, from, to, A.mode);
                from = to;
            }
        };
    double est = 0;
    *spent = sp.degree * gmres_cycle<double>(s, w, A, q, rh, bh, stop_rel * bh, max_steps, r1, &est);
    if (!std::isfinite(est)) return false;
    split_op<double>(2, s, *A.co, A.F, A.L, *A.split, r1, y, A.mode);
    axpy_f64_keep(s, n, beta, y, x, r1);
    return true;
}
}  // namespace

SolveInfo gmres_solve(hipStream_t s, GmresWork<double>& w, const CsrOp<double>& A, const PcFn<double>& M,
                      const double* b, double* x, double* r, int m, int maxit, double tol, SplitCycles split) {
    SolveInfo info;
    w.ensure(A.n, m);
    double nb = 0, beta = 0;
    if (!start_norms(s, w, A, x, b, r, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, A.n)) beta = residual_norm(s, w, A, x, b, r);
    // The split cycles need no SpMV, and take `degree` operator applications per basis vector: a
    // cycle reaches degree times as far for the same basis traffic, and restarts forget the slow
    // modes that much less often.  Suspension solve, GMRES(30), mean of three to five forcings, ms, plain
    // against split: 5,000 faces x 5 layers 1.05 and 0.82, 50,000 x 10 3.95 and 2.25, 125,000 x 7 5.30
    // and 2.98, 200,000 x 9 11.6 and 6.3, 999,968 x 10 171 and 62.
    // The split residual's norm stands for ||b - A x||; their reductions lie close together.  The long
    // polynomial reaches a residual with more of the error left in the slow modes than plain cycles
    // leave there: at 999,968 faces x 10 layers, 18 forcings, the concentration's relative error
    // (2-norm, against a solve to 2e-13) was 3.7e-7 rms and 8.2e-7 at most after plain cycles, 7.3e-7
    // and 3.1e-6 with 0.8 of the target, 2.8e-7 and 1.2e-6 with 0.2, 1.0e-7 and 4.3e-7 with 0.15 for
    // one to three steps more (60 ms a solve, 55 with 0.8, 214 with plain cycles).
    const double aim = split.degree > 4 ? 0.15 : 0.8;
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            break;
        }
        if (info.iters >= maxit) break;
        if (split.degree > maxit - info.iters) split.degree = 0;
        if (split.degree > 0) {
            int spent = 0;
            const double before = beta;
            const bool moved = split_cycle(s, w, split, r, beta, aim * tol * nb / beta,
                                           (maxit - info.iters) / split.degree, x, &spent);
            info.iters += spent;
            info.cycles += 1;
            if (moved) beta = residual_norm(s, w, A, x, b, r);
            // a spectrum the polynomial does not suit: plain cycles from here, and from the x before
            // where the residual did not fall
            if (!moved || !(beta < 0.5 * before)) split.degree = 0;
            if (moved && !(beta < before)) {
                copy_f64(s, A.n, split.work[0], x);
                beta = residual_norm(s, w, A, x, b, r);
            }
            continue;
        }
        double est = 0;
        info.iters += gmres_cycle<double>(s, w, A, M, r, beta, tol * nb, maxit - info.iters, r, &est);
        axpy_f64(s, A.n, 1.0, r, x);
        info.cycles += 1;
        beta = residual_norm(s, w, A, x, b, r);
    }
    return info;
}

SolveInfo mixed_solve(hipStream_t s, GmresWork<float>& w, const CsrOp<double>& A64, const CsrOp<float>& A32,
                      const PcFn<float>& M32, const double* b, double* x, double* r, float* r32, float* d32, int m,
                      int maxit, double tol, double inner_rtol) {
    SolveInfo info;
    w.ensure(A64.n, m);
    double nb = 0, beta = 0;
    if (!start_norms(s, w, A64, x, b, r, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, A64.n)) beta = residual_norm(s, w, A64, x, b, r);
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            break;
        }
        if (info.iters >= maxit) break;
        // inner FP32 cycle on the normalised FP64 residual
        scale_f64_to_f32_host(s, A64.n, r, 1.0 / beta, r32);
        double est = 0;
        double stop = 0.5 * tol * nb / beta;
        if (stop < inner_rtol) stop = inner_rtol;
        const int steps = gmres_cycle<float>(s, w, A32, M32, r32, 1.0, stop, maxit - info.iters, d32, &est);
        axpy_f32_into_f64(s, A64.n, beta, d32, x);
        info.iters += steps;
        info.cycles += 1;
        info.refinements += 1;
        beta = residual_norm(s, w, A64, x, b, r);
    }
    return info;
}

// ---------------------------------------------------------------------------
// BiCGStab
// ---------------------------------------------------------------------------
template <typename T>
void BicgWork<T>::ensure(int64_t n_) {
    if (n == n_ && r.p) return;
    n = n_;
    for (DevBuf<T>* b : {&r, &rh, &p, &v, &s, &t, &ph, &sh}) b->alloc(n);
    // two partial sums per block of the fused SpMV + dot launches, or of the vector kernels
    partial.alloc(std::max<size_t>(4 * (size_t)kReduceBlocks, 2 * (size_t)pos_spmv_dots_max_blocks(n)));
    dsc.alloc(SC_COUNT);
    ss_partial.alloc(kReduceBlocks);
    xr_partial.alloc(2 * (size_t)kReduceBlocks);
    slot.alloc(2);
    slot.p[0].seq = slot.p[1].seq = 0;
    seq = 0;
    PB_HIP(hipHostGetDevicePointer((void**)&dslot, slot.p, 0));
}

namespace {
// y = A x with the partial sums (w.y, y.y) of each block (two per block); returns the block count
// (stop: the split operator's launches return at entry once *stop != 0)
template <typename T>
int64_t spmv_dots(hipStream_t s, const CsrOp<T>& A, const T* x, T* y, const T* w, double* partial, int nblk,
                  const double* stop) {
    if (A.split) return split_apply_dots<T>(s, *A.co, A.F, A.L, *A.split, x, y, w, partial, A.mode, stop);
    if (A.pos) return pos_spmv_dots<T>(s, A.variant, *A.co, A.F, A.L, *A.pos, x, y, w, partial);
    op_spmv<T>(s, A, x, y);
    mdot<T>(s, A.n, w, 0, 1, y, partial, nblk);
    return nblk;
}

// One BiCGStab run on A x = b from the x given; stops when ||r|| <= stop_abs,
// on a breakdown (the caller restarts from the true residual) or after maxit
// iterations; returns the iterations.  alpha, omega, rho and the stop test live
// on the device, and the host queues iteration k+1 before it waits for the
// scalars of iteration k, so the device never idles on the host round trip;
// after the stop every kernel of the queued iteration returns at entry (x and r
// keep the values of the stopping iteration).
// An empty M means no preconditioner (the operator already carries it, as the
// split operator does).  stop_rel: stop_abs is relative to the starting ||r||.
template <typename T>
int bicg_run(hipStream_t s, BicgWork<T>& w, const CsrOp<T>& A, const PcFn<T>& M, const T* b, T* x, bool x_zero,
             double stop_abs, int maxit, double* res_out, bool stop_rel = false, double restart_eps = 0.0,
             int* restarts = nullptr) {
    const int64_t n = A.n;
    const int nblk = reduce_blocks(n);
    // The s and x/r kernels: every workgroup first sums the operator's dot partials itself,
    // so they run as few workgroups as fill the chip (grid-stride over the vectors).
    const int nvec = std::min(nblk, kVecBlocks);
    const int spmv_id = A.prof_class >= 0 ? A.prof_class : (sizeof(T) == 8 ? PBSM3D_K_SPMV64 : PBSM3D_K_SPMV32);
    const bool pc = static_cast<bool>(M);
    T* ph = pc ? w.ph.p : w.p.p;  // the preconditioned search directions
    T* sh = pc ? w.sh.p : w.s.p;
    double* sc = w.dsc.p;
    // r = b - A x, rh = r, (rh.r, r.r)
    if (x_zero) {
        PB_HIP(hipMemcpyAsync(w.r.p, b, n * sizeof(T), hipMemcpyDeviceToDevice, s));
    } else {
        {
            ProfScope ps(A.prof, s, spmv_id);
            op_spmv<T>(s, A, x, w.v.p);
        }
        axpy_dots<T>(s, n, 1.0, w.v.p, b, w.r.p, nullptr, w.partial.p, nblk);
    }
    PB_HIP(hipMemcpyAsync(w.rh.p, w.r.p, n * sizeof(T), hipMemcpyDeviceToDevice, s));
    mdot<T>(s, n, w.rh.p, 0, 1, w.r.p, w.partial.p, nblk);
    bicg_stage(s, w.partial.p, nblk, 2, 0, sc, 0.0, w.dslot, ++w.seq, 0.0);
    PB_HIP(hipGetLastError());
    wait_slot(s, w.slot.p, w.seq);
    double rr = std::sqrt(w.slot.p[0].v[SC_RR]);
    const uint64_t seq0 = w.seq;
    *res_out = rr;
    if (stop_rel) stop_abs *= rr;
    if (rr <= stop_abs) return 0;
    const double* stop = sc + SC_STOP;
    auto iterate = [&](int it) {
        if (it == 1) {
            PB_HIP(hipMemcpyAsync(w.p.p, w.r.p, n * sizeof(T), hipMemcpyDeviceToDevice, s));
        } else {
            ProfScope ps(A.prof, s, PBSM3D_K_ORTHO);
            bicg_p_dev<T>(s, n, w.r.p, w.v.p, sc, w.p.p, w.rh.p);
        }
        if (pc) {
            ProfScope ps(A.prof, s, PBSM3D_K_PRECOND);
            M(s, w.p.p, w.ph.p);
        }
        int64_t nb = 0;
        {
            ProfScope ps(A.prof, s, spmv_id);
            nb = spmv_dots<T>(s, A, ph, w.v.p, w.rh.p, w.partial.p, nblk, stop);  // v = A ph; rh.v, v.v
        }
        {
            ProfScope ps(A.prof, s, PBSM3D_K_ORTHO);
            bicg_s_dev<T>(s, n, w.v.p, w.r.p, sc, w.s.p, w.ss_partial.p, nvec, w.partial.p, nb);  // alpha, s, s.s
        }
        if (pc) {
            ProfScope ps(A.prof, s, PBSM3D_K_PRECOND);
            M(s, w.s.p, w.sh.p);
        }
        {
            ProfScope ps(A.prof, s, spmv_id);
            nb = spmv_dots<T>(s, A, sh, w.t.p, w.s.p, w.partial.p, nblk, stop);  // t = A sh; s.t, t.t
        }
        {
            ProfScope ps(A.prof, s, PBSM3D_K_ORTHO);
            // omega, x, r, (rh.r, r.r)
            bicg_xr_dev<T>(s, n, ph, sh, w.s.p, w.t.p, w.rh.p, sc, x, w.r.p, w.xr_partial.p, nvec, w.partial.p, nb,
                           w.ss_partial.p, nvec);
            // rho, rr, the stop test, and the scalars into host slot it % 2 (no copy launch)
            bicg_stage(s, w.xr_partial.p, nvec, 2, 1, sc, stop_abs, w.dslot + (it & 1), ++w.seq, restart_eps);
        }
        PB_HIP(hipGetLastError());
    };
    if (maxit <= 0) return 0;
    iterate(1);
    for (int it = 1;; ++it) {
        if (it < maxit) iterate(it + 1);
        wait_slot(s, w.slot.p + (it & 1), seq0 + it);
        const double* hk = w.slot.p[it & 1].v;
        rr = std::sqrt(hk[SC_RR]);
        *res_out = rr;
        if (hk[SC_STOP] != 0.0 || it >= maxit) {
            if (restarts) *restarts += (int)hk[SC_NRESTART];
            return it;
        }
    }
}
}  // namespace

SolveInfo bicgstab_solve(hipStream_t s, BicgWork<double>& w, GmresWork<double>& gw, const CsrOp<double>& A,
                         const PcFn<double>& M, const double* b, double* x, int maxit, double tol) {
    SolveInfo info;
    w.ensure(A.n);
    GmresWork<double>& dummy = gw;
    double nb = 0, beta = 0;
    if (!start_norms(s, dummy, A, x, b, w.r.p, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, A.n)) beta = residual_norm(s, dummy, A, x, b, w.r.p);
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            break;
        }
        if (info.iters >= maxit) break;
        double est = 0;
        info.iters += bicg_run<double>(s, w, A, M, b, x, false, 0.9 * tol * nb, maxit - info.iters, &est);
        info.cycles += 1;
        beta = residual_norm(s, dummy, A, x, b, w.r.p);
    }
    return info;
}

namespace {
void scale_into(hipStream_t s, int64_t n, const double* r, double a, double* out) { scale_host<double>(s, n, r, a, out); }
void scale_into(hipStream_t s, int64_t n, const double* r, double a, float* out) { scale_f64_to_f32_host(s, n, r, a, out); }
void add_into(hipStream_t s, int64_t n, double a, const double* d, double* x) { axpy_f64(s, n, a, d, x); }
void add_into(hipStream_t s, int64_t n, double a, const float* d, double* x) { axpy_f32_into_f64(s, n, a, d, x); }
}  // namespace

template <typename T>
SolveInfo bicgstab_split(hipStream_t s, BicgWork<T>& w, GmresWork<T>& gw, const CsrOp<double>& A64,
                         const CsrOp<T>& Ahat, const double* b, double* x, double* r, T* work1, T* work2, T* work3,
                         int maxit, double tol, double inner_rtol, double inner_rtol_cold, const CoarseFn& coarse,
                         double restart_eps32) {
    SolveInfo info;
    const int64_t n = A64.n;
    w.ensure(n);
    double nb = 0, beta = 0;
    if (!start_norms(s, gw, A64, x, b, r, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, n)) {
        beta = residual_norm(s, gw, A64, x, b, r);
        if (inner_rtol_cold > 0) inner_rtol = inner_rtol_cold;  // the start is x0 = 0 after all
    }
    const int pclass = Ahat.prof_class >= 0 ? Ahat.prof_class : PBSM3D_K_PRECOND;
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            break;
        }
        if (info.iters >= maxit) break;
        if (coarse) {
            coarse(s, r, x);
            beta = residual_norm(s, gw, A64, x, b, r);
            if (info.cycles == 0) info.resid_coarse = beta / nb;
            info.resid = beta / nb;
            if (info.resid <= tol) {
                info.converged = true;
                break;
            }
        }
        scale_into(s, n, r, 1.0 / beta, work1);  // r / ||r||
        {
            ProfScope ps(Ahat.prof, s, pclass);
            split_op<T>(1, s, *Ahat.co, Ahat.F, Ahat.L, *Ahat.split, work1, work2, Ahat.mode);  // rhat
        }
        PB_HIP(hipMemsetAsync(work3, 0, n * sizeof(T), s));
        double stop = 0.5 * tol * nb / beta;
        if (stop < inner_rtol) stop = inner_rtol;
        double est = 0;
        info.iters += bicg_run<T>(s, w, Ahat, PcFn<T>(), work2, work3, true, stop, maxit - info.iters, &est, true,
                                  sizeof(T) == 4 ? restart_eps32 : 0.0, &info.restarts);
        {
            ProfScope ps(Ahat.prof, s, pclass);
            split_op<T>(2, s, *Ahat.co, Ahat.F, Ahat.L, *Ahat.split, work3, work1, Ahat.mode);  // d = (D~+U)^-1 dhat
        }
        add_into(s, n, beta, work1, x);
        info.cycles += 1;
        info.refinements += 1;
        beta = residual_norm(s, gw, A64, x, b, r);
    }
    return info;
}

template SolveInfo bicgstab_split<double>(hipStream_t, BicgWork<double>&, GmresWork<double>&, const CsrOp<double>&,
                                          const CsrOp<double>&, const double*, double*, double*, double*, double*,
                                          double*, int, double, double, double, const CoarseFn&, double);
template SolveInfo bicgstab_split<float>(hipStream_t, BicgWork<float>&, GmresWork<float>&, const CsrOp<double>&,
                                         const CsrOp<float>&, const double*, double*, double*, float*, float*, float*,
                                         int, double, double, double, const CoarseFn&, double);

void CgWork::ensure(int64_t n_) {
    if (n == n_ && p.p) return;
    n = n_;
    for (DevBuf<double>* v : {&rh, &p, &pw, &q, &xh}) v->alloc(n);
    work.alloc(n + 1);
    zero_tail(work, n);
    dots.alloc(2 * (size_t)pos_spmv_dots_max_blocks(n));
    partial.alloc(kVecBlocks);
    sc.alloc(CG_COUNT);
    slot.alloc(2);
    slot.p[0].seq = slot.p[1].seq = seq = 0;
    PB_HIP(hipHostGetDevicePointer((void**)&dslot, slot.p, 0));
}

SolveInfo cg_split(hipStream_t s, CgWork& w, GmresWork<double>& gw, const CsrOp<double>& A, const CsrOp<double>& Ahat,
                   const double* b, double* x, double* r, int maxit, double tol) {
    SolveInfo info;
    const int64_t n = A.n;
    w.ensure(n);
    double nb = 0, beta = 0;
    if (!start_norms(s, gw, A, x, b, r, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, n)) beta = residual_norm(s, gw, A, x, b, r);
    const double* dinv = Ahat.split->dinv.p;
    double* sc = w.sc.p;
    const int nvec = std::min(reduce_blocks(n), kVecBlocks);
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            return info;
        }
        const int most = maxit - info.iters;
        if (most <= 0) return info;
        scale_host<double>(s, n, r, 1.0 / beta, w.work.p);
        split_op<double>(1, s, *Ahat.co, Ahat.F, Ahat.L, *Ahat.split, w.work.p, w.rh.p, Ahat.mode);
        cg_start(s, n, w.rh.p, dinv, w.xh.p, w.p.p, w.pw.p, sc, w.partial.p, nvec);
        // sqrt(rho), the residual's norm under M^-1, stands for ||b - A x||: their reductions lie
        // within a factor of two of each other.  0.3 leaves a residual no larger than the
        // BiCGStab and GMRES solves left (1 to 2e-9 at 1e-8), for one iteration more than 0.5.
        const double rel = 0.3 * tol * nb / beta, stop2 = rel * rel;
        const uint64_t seq0 = w.seq;
        auto iterate = [&](int it) {
            const int64_t nd = split_apply_dots<double>(s, *Ahat.co, Ahat.F, Ahat.L, *Ahat.split, w.p.p, w.q.p, w.pw.p,
                                                        w.dots.p, Ahat.mode, sc + CG_STOP);
            cg_xr(s, n, it, w.p.p, w.q.p, dinv, w.xh.p, w.rh.p, sc, w.dots.p, nd, w.partial.p, nvec);
            cg_p(s, n, it, w.rh.p, dinv, w.p.p, w.pw.p, sc, stop2, w.partial.p, nvec, w.dslot + (it & 1), ++w.seq);
            PB_HIP(hipGetLastError());
        };
        double stop = 0;
        iterate(1);
        for (int it = 1;; ++it) {
            if (it < most) iterate(it + 1);
            wait_slot(s, w.slot.p + (it & 1), seq0 + it);
            stop = w.slot.p[it & 1].v[1];
            if (stop != 0.0 || it >= most) {
                info.iters += it;
                break;
            }
        }
        if (stop == 2.0) {  // x keeps what the runs before gained
            info.breakdown = std::isfinite(info.resid);  // else the start or b is at fault
            return info;
        }
        split_op<double>(2, s, *Ahat.co, Ahat.F, Ahat.L, *Ahat.split, w.xh.p, w.work.p, Ahat.mode);
        axpy_f64(s, n, beta, w.work.p, x);
        info.cycles += 1;
        const double before = beta;
        beta = residual_norm(s, gw, A, x, b, r);
        if (!(beta < 0.5 * before)) {
            info.resid = beta / nb;
            info.converged = info.resid <= tol;
            return info;
        }
    }
}

SolveInfo bicgstab_mixed(hipStream_t s, BicgWork<float>& w, GmresWork<float>& gw, const CsrOp<double>& A64,
                         const CsrOp<float>& A32, const PcFn<float>& M32, const double* b, double* x, double* r,
                         float* r32, float* d32, int maxit, double tol, double inner_rtol, double restart_eps32) {
    SolveInfo info;
    w.ensure(A64.n);
    double nb = 0, beta = 0;
    if (!start_norms(s, gw, A64, x, b, r, info, nb, beta)) return info;
    if (drop_worse_start(s, info, beta, nb, x, A64.n)) beta = residual_norm(s, gw, A64, x, b, r);
    while (true) {
        info.resid = beta / nb;
        if (info.resid <= tol) {
            info.converged = true;
            break;
        }
        if (info.iters >= maxit) break;
        scale_f64_to_f32_host(s, A64.n, r, 1.0 / beta, r32);
        PB_HIP(hipMemsetAsync(d32, 0, A64.n * sizeof(float), s));
        double stop = 0.5 * tol * nb / beta;
        if (stop < inner_rtol) stop = inner_rtol;
        double est = 0;
        info.iters += bicg_run<float>(s, w, A32, M32, r32, d32, true, stop, maxit - info.iters, &est, false,
                                      restart_eps32, &info.restarts);
        axpy_f32_into_f64(s, A64.n, beta, d32, x);
        info.cycles += 1;
        info.refinements += 1;
        beta = residual_norm(s, gw, A64, x, b, r);
    }
    return info;
}

template struct BicgWork<double>;
template struct BicgWork<float>;
template struct GmresWork<double>;
template struct GmresWork<float>;
template int gmres_cycle<double>(hipStream_t, GmresWork<double>&, const CsrOp<double>&, const PcFn<double>&,
                                 const double*, double, double, int, double*, double*);
template int gmres_cycle<float>(hipStream_t, GmresWork<float>&, const CsrOp<float>&, const PcFn<float>&, const float*,
                                double, double, int, float*, double*);

}  // namespace pb
