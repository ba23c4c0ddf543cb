// Per-face network of the learned warm start: 16 -> 128 -> 128 -> 128 -> 11,
// ReLU, BF16 operands with FP32 accumulation on the matrix cores
// (gfx950's v_mfma_f32_16x16x32_bf16), trained on the GPU by its own forward
// and backward kernels with Adam.
//
// For a layer with weights W [out x in], activations A and pre-activations Z [samples x features]
//   forward   Z = A_in W^T + b,   A_out = relu(Z)
//   backward  dW = dZ^T A_in,     db = colsum(dZ),   dZ_in = (dZ W) * [Z_in > 0]
// Inference (k_mlp_infer) carries a wave's samples through all layers in registers; training
// (k_mlp_train) runs forward and backward of a 64-sample tile in one workgroup and keeps the
// weight gradients in its accumulators; k_gemm_bf16 is the layer-by-layer forward that the
// fused inference is checked against.  MFMA operand layout of v_mfma_f32_16x16x32_bf16
// (A: row = lane%16, k = 8*(lane/16)+j, j < 8; B: col = lane%16, same k;
// C: col = lane%16, row = 4*(lane/16)+j, j < 4).
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "mlp.hpp"

namespace pb {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 64, TN = 64, TK = 32;

// 8 consecutive BF16 values (16 bytes, 16-byte aligned) as an MFMA operand fragment
__device__ __forceinline__ bf16x8 frag8(const uint16_t* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}

__device__ __forceinline__ uint16_t to_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;  // NaN
    u += 0x7fffu + ((u >> 16) & 1u);                    // round to nearest even
    return (uint16_t)(u >> 16);
}

// C [M x N] = A [M x K] B^T + bias, B [N x K] (k contiguous in both)
struct GemmArgs {
    int M, N, K;
    const uint16_t* A;
    const uint16_t* B;
    const float* bias;  // per output column, the accumulators' start
    float* C;           // fp32 output, may be null
    uint16_t* Cb;       // bf16 copy of relu(C), may be null
};

// One 16-byte chunk of a 64 x 32 operand tile into LDS T[64][TK + 8] (T[row][k]): 8 k of one
// row.  rows: the matrix's row count (M or N); r0 / k0: the tile origin.
__device__ __forceinline__ void stage_chunk(const uint16_t* __restrict__ X, int ld, int rows, int r0, int k0, int tid,
                                            uint16_t (*T)[TK + 8]) {
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    const int r = tid >> 2, c = (tid & 3) * 8;  // 64 rows x 4 chunks
    const int gr = r0 + r, gk = k0 + c;
    u16x8 v = {0, 0, 0, 0, 0, 0, 0, 0};
    if (gr < rows && gk < ld) v = *reinterpret_cast<const u16x8*>(X + (size_t)gr * ld + gk);  // ld is 16 or 128
    *reinterpret_cast<u16x8*>(&T[r][c]) = v;
}

// 64x32 A and B tiles of BF16 in LDS; each of the four wavefronts owns a 32x32 quarter of the
// 64x64 output tile, i.e. 2x2 MFMA blocks, one 16-byte LDS read per lane and fragment.
__global__ void __launch_bounds__(256) k_gemm_bf16(GemmArgs g) {
    __shared__ __align__(16) uint16_t As[TM][TK + 8];
    __shared__ __align__(16) uint16_t Bs[TN][TK + 8];
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 acc[2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int col = n0 + wn + b * 16 + (lane & 15);
        const float start = col < g.N ? g.bias[col] : 0.f;
#pragma unroll
        for (int a = 0; a < 2; ++a) acc[a][b] = f32x4{start, start, start, start};
    }
    for (int k0 = 0; k0 < g.K; k0 += TK) {
        stage_chunk(g.A, g.K, g.M, m0, k0, tid, As);
        stage_chunk(g.B, g.K, g.N, n0, k0, tid, Bs);
        __syncthreads();
#pragma unroll
        for (int tm = 0; tm < 2; ++tm) {
            const bf16x8 a = frag8(&As[wm + tm * 16 + (lane & 15)][8 * (lane >> 4)]);
#pragma unroll
            for (int tn = 0; tn < 2; ++tn) {
                const bf16x8 b = frag8(&Bs[wn + tn * 16 + (lane & 15)][8 * (lane >> 4)]);
                acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[tm][tn], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 2; ++tn)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int row = m0 + wm + tm * 16 + 4 * (lane >> 4) + j;
                const int col = n0 + wn + tn * 16 + (lane & 15);
                if (row >= g.M || col >= g.N) continue;
                const float v = acc[tm][tn][j];
                if (g.C) g.C[(size_t)row * g.N + col] = v;
                if (g.Cb) g.Cb[(size_t)row * g.N + col] = to_bf16(fmaxf(v, 0.f));
            }
}

// x (rows x 16, f32) -> normalised bf16 rows
__global__ void k_prep_inputs(int64_t n, const float* __restrict__ X, const float* __restrict__ mu,
                              const float* __restrict__ sd, uint16_t* __restrict__ Xb) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * MlpDims::IN) return;
    const int c = (int)(t % MlpDims::IN);
    Xb[t] = to_bf16((X[t] - mu[c]) / sd[c]);
}

// BF16 copies of one layer's weights W [dout x din]: as they are, and transposed
__global__ void k_pack_weights(int din, int dout, const float* __restrict__ W, uint16_t* __restrict__ Wb,
                               uint16_t* __restrict__ WbT) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= din * dout) return;
    const uint16_t v = to_bf16(W[t]);
    Wb[t] = v;
    WbT[(t % din) * dout + t / din] = v;
}

// de-normalise network outputs (OUTP wide) into OUT-wide rows
__global__ void k_denorm(int64_t n, const float* __restrict__ Yp, const float* __restrict__ mu,
                         const float* __restrict__ sd, float* __restrict__ Y) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * MlpDims::OUT) return;
    const int64_t r = t / MlpDims::OUT;
    const int c = (int)(t % MlpDims::OUT);
    Y[t] = Yp[r * MlpDims::OUTP + c] * sd[c] + mu[c];
}

// Inference of the whole network in one launch, activations in registers.
//
// A wave owns 64 samples and carries them through all four layers by itself: the weights are
// the MFMA's A operand and the activations its B operand, so a product leaves four consecutive
// output features of one sample in a lane (C: column = sample = lane % 16, rows 4 (lane / 16)
// + j).  The weight rows of two 16-row blocks are permuted so that a lane's 2 x 4 results are
// the eight features 32 kk + 8 (lane / 16) .. + 7 -- the B operand of the next layer's k-step
// kk, in natural k order -- so a layer's output feeds the next layer's MFMAs after bias, ReLU
// and BF16 packing without touching LDS, and there is no barrier between layers.  LDS holds
// only the weights, laid out once per workgroup in the order the lanes read them (one
// conflict-free 16-byte load per lane and fragment, each used for four MFMAs).
//
// Bound: the matrix cores (304 MFMAs of 16x16x32 per 64 samples against 76 16-byte LDS reads
// per lane) and the packing between layers.  999,968 samples: 581 -> 100 us (127 -> 737 TFLOP/s;
// before, each 64-sample workgroup tile re-read the 74 KB of weights through the vector cache,
// and its activations crossed LDS with a barrier per layer).
// The bias is the accumulator's start and k runs in increasing order, as in k_gemm_bf16, so
// the output equals the layer-by-layer forward bit for bit.
constexpr int kInferCols = 64;      // samples per wave and tile
constexpr int kInferThreads = 512;  // eight waves, one workgroup per CU (78 KB of weights)
constexpr int kFrags[5] = {0, 8, 40, 72, 76};  // first weight fragment of each layer

struct InferArgs {
    int64_t n;
    const float* X;        // [n x IN] raw features
    const uint16_t* W[4];  // BF16 [dout x din]
    const float* b[4];
    const float* norm;     // x_mean[IN], x_std[IN], y_mean[OUT], y_std[OUT]
    float* Y;              // [n x OUT] raw outputs
    int x16;               // X is 16-byte aligned
};

// one hidden layer of a wave's 64 samples: in[ks][cb] / out[kk][cb] are B operands (k-step,
// 16-sample block); wf: the layer's fragments in LDS, block rb's k-step ks at rb * KS + ks
template <int KS>
__device__ __forceinline__ void infer_hidden(const bf16x8 (&in)[KS][4], bf16x8 (&out)[4][4],
                                             const uint16_t* __restrict__ wf, const float* __restrict__ bias,
                                             int lane) {
    const int q = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        f32x4 acc[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f32x4 bq = *reinterpret_cast<const f32x4*>(&bias[32 * kk + 8 * q + 4 * h]);
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[h][cb] = bq;
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const bf16x8 w = frag8(wf + (((2 * kk + h) * KS + ks) * 64 + lane) * 8);
#pragma unroll
                for (int cb = 0; cb < 4; ++cb)
                    acc[h][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, in[ks][cb], acc[h][cb], 0, 0, 0);
            }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) out[kk][cb][4 * h + j] = (__bf16)fmaxf(acc[h][cb][j], 0.f);
        // keeps the scheduler from starting the next block pair's accumulators and weight
        // reads early, which spilled 328 of the 256 registers
        __builtin_amdgcn_sched_barrier(0);
    }
}

__global__ void __launch_bounds__(kInferThreads) k_mlp_infer(InferArgs p) {
    constexpr int H = MlpDims::H, IN = MlpDims::IN, OUT = MlpDims::OUT, OUTP = MlpDims::OUTP;
    __shared__ __align__(16) uint16_t wf[kFrags[4] * 64 * 8];
    __shared__ __align__(16) float bias[3 * H + OUTP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < kFrags[4] * 64; e += kInferThreads) {
        const int f = e >> 6, r = e & 15, q = (e >> 4) & 3;
        const int l = f < kFrags[1] ? 0 : f < kFrags[2] ? 1 : f < kFrags[3] ? 2 : 3;
        const int g = f - kFrags[l], ks = l == 0 ? 0 : g & 3, rb = l == 0 ? g : g >> 2;
        const int row = l < 3 ? 32 * (rb >> 1) + 8 * (r >> 2) + 4 * (rb & 1) + (r & 3) : r;
        const int K = l == 0 ? IN : H, col = 32 * ks + 8 * q;
        bf16x8 v = {};
        if (col < K) v = frag8(p.W[l] + row * K + col);  // K = 16: the upper half of the k-step is zero
        *reinterpret_cast<bf16x8*>(&wf[e * 8]) = v;
    }
    for (int e = tid; e < 3 * H + OUTP; e += kInferThreads) bias[e] = p.b[e / H][e % H];
    __syncthreads();
    const int r = lane & 15, q = lane >> 4;
    float xmu[8], xsd[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        xmu[j] = q < 2 ? p.norm[8 * q + j] : 0.f;
        xsd[j] = q < 2 ? p.norm[IN + 8 * q + j] : 1.f;
    }
    float ymu[4], ysd[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int o = min(4 * q + j, OUT - 1);
        ymu[j] = p.norm[2 * IN + o];
        ysd[j] = p.norm[2 * IN + OUT + o];
    }
    const int64_t ntiles = (p.n + kInferCols - 1) / kInferCols;
    for (int64_t tile = blockIdx.x + (int64_t)gridDim.x * wave; tile < ntiles;
         tile += (int64_t)gridDim.x * (kInferThreads / 64)) {
        const int64_t s0 = tile * kInferCols;
        bf16x8 x[1][4], a[4][4], c[4][4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int64_t g = s0 + 16 * cb + r;
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = xmu[j];
            if (q < 2 && g < p.n) {
                const float* src = p.X + g * IN + 8 * q;
                if (p.x16) {
                    const f32x4 lo = *reinterpret_cast<const f32x4*>(src);
                    const f32x4 hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = lo[j], v[4 + j] = hi[j];
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j) v[j] = src[j];
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) x[0][cb][j] = (__bf16)((v[j] - xmu[j]) / xsd[j]);
        }
        infer_hidden<1>(x, a, wf, bias, lane);
        infer_hidden<4>(a, c, wf + kFrags[1] * 512, bias + H, lane);
        infer_hidden<4>(c, a, wf + kFrags[2] * 512, bias + 2 * H, lane);
        f32x4 acc[4];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) acc[cb] = *reinterpret_cast<const f32x4*>(&bias[3 * H + 4 * q]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const bf16x8 w = frag8(wf + ((kFrags[3] + ks) * 64 + lane) * 8);
#pragma unroll
            for (int cb = 0; cb < 4; ++cb)
                acc[cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a[ks][cb], acc[cb], 0, 0, 0);
        }
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const int64_t g = s0 + 16 * cb + r;
            if (g < p.n) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (4 * q + j < OUT) p.Y[g * OUT + 4 * q + j] = acc[cb][j] * ysd[j] + ymu[j];
            }
        }
    }
}

// Row t of a training batch: a counter hash of the batch key, modulo the sample count.
__device__ __forceinline__ int64_t sample_row(uint64_t key, int64_t t, int64_t n) {
    uint64_t z = key + (uint64_t)t * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (int64_t)(z % (uint64_t)n);
}

// Forward, loss and backward of a training batch in one launch.
//
// A workgroup of eight waves takes tiles of 64 samples; wave w owns the 16 hidden features
// 16 w .. + 15 of every layer.  Its weight fragments (W for the forward products, W^T for the
// backward ones) and its rows of every weight gradient stay in registers for all of the
// workgroup's tiles (the latter as MFMA accumulators), so per tile only activations and
// back-propagated gradients pass through LDS: once as [sample][feature], the B operand of the
// next product, and once as [feature][sample], the operands of dW = dZ^T A (k = samples).  A
// bias gradient is the product of dZ^T with a vector of ones.  The ReLU masks stay in the
// registers of the lane that computed them.  Each workgroup writes its gradients to a slab of
// its own; k_mlp_update adds the slabs in a fixed order, so results do not depend on
// scheduling.
//
// Bound: LDS reads and the nine barriers of a tile (a tile's 900 MFMAs take about 3 us on a
// CU), then the slabs (149 KB per workgroup).  A batch of 8,192 took 215 us in 29 launches
// (11 GEMMs of 13 us, split-K and column sums, one launch per elementwise step); it takes
// 27.7 us here and 7.0 us in k_mlp_update.
constexpr int kTrainCols = 64;
constexpr int kTrainThreads = 512;
constexpr int kLs = MlpDims::H + 8;      // LDS row stride (BF16) of [sample][128 features]
constexpr int kLt = kTrainCols + 8;      // of [feature][64 samples]
constexpr int kLx = MlpDims::IN + 8;     // of [sample][16 features]
// flat parameters: W1 b1 W2 b2 W3 b3 W4 b4
constexpr int kOffW[4] = {0, 2176, 18688, 35200}, kOffB[4] = {2048, 18560, 35072, 37248};
constexpr int kParams = 37264;

struct TrainArgs {
    int64_t n;        // samples of the batch
    int64_t total;    // > 0: batch row t is sample_row(key, t, total) of X / Y; 0: row t itself
    uint64_t key;
    const float *X, *Y;
    const float* norm;
    const uint16_t *W[4], *WT[4];  // BF16 [dout x din] and [din x dout]
    const float* b[4];
    float* slab;   // [gridDim.x][kParams]
    double* loss;  // [gridDim.x] summed squared error
};

__device__ __forceinline__ uint16_t bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// four consecutive features of one sample to both layouts
__device__ __forceinline__ void put4(const float (&v)[4], uint16_t* __restrict__ s, uint16_t* __restrict__ t) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    u16x4 u;
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = bf16_bits(v[j]);
    if (s) *reinterpret_cast<u16x4*>(s) = u;
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j * kLt] = u[j];
}

__global__ void __launch_bounds__(kTrainThreads) k_mlp_train(TrainArgs p) {
    constexpr int H = MlpDims::H, IN = MlpDims::IN, OUT = MlpDims::OUT, OUTP = MlpDims::OUTP;
    constexpr int T = kTrainCols;
    __shared__ __align__(16) uint16_t xs[T * kLx], xt[IN * kLt];
    __shared__ __align__(16) uint16_t as[2][T * kLs];   // activations / gradients by sample, in turn
    __shared__ __align__(16) uint16_t at[3][H * kLt];   // activations of the hidden layers by feature
    __shared__ __align__(16) uint16_t dt[2][H * kLt];   // gradients by feature, in turn
    __shared__ __align__(16) uint16_t ds4[T * kLx], dt4[OUTP * kLt];
    __shared__ __align__(16) float bias[3 * H + OUTP];
    __shared__ int64_t src[T];
    __shared__ double s_loss[4];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, q = lane >> 4;
    const int f0 = 16 * w + 4 * q;  // the lane's first output feature
    const bf16x8 zero8 = {};
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; ++j) ones[j] = (__bf16)1.0f;
    // weight fragments of this wave (rows 16 w .. of W, and of W^T)
    const bf16x8 w1 = q < 2 ? frag8(p.W[0] + (16 * w + r) * IN + 8 * q) : zero8;
    const bf16x8 t4 = q < 2 ? frag8(p.WT[3] + (16 * w + r) * OUTP + 8 * q) : zero8;
    bf16x8 w2[4], w3[4], t2[4], t3[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int o = (16 * w + r) * H + 32 * ks + 8 * q;
        w2[ks] = frag8(p.W[1] + o);
        w3[ks] = frag8(p.W[2] + o);
        t2[ks] = frag8(p.WT[1] + o);
        t3[ks] = frag8(p.WT[2] + o);
    }
    for (int e = tid; e < 3 * H + OUTP; e += kTrainThreads) bias[e] = p.b[e / H][e % H];
    auto bias_of = [&](int l) { return *reinterpret_cast<const f32x4*>(&bias[l * H + (l < 3 ? f0 : 4 * q)]); };
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
    f32x4 g1 = zero4, g2[8], g3[8], g4 = zero4, gb1 = zero4, gb2 = zero4, gb3 = zero4, gb4 = zero4;
#pragma unroll
    for (int c = 0; c < 8; ++c) g2[c] = g3[c] = zero4;
    double se = 0.0;

    // Z = W A + b of 16 features x 64 samples; relu to both layouts; the mask Z > 0, bit 4 cb + j
    auto forward = [&](const bf16x8 (&wk)[4], f32x4 bias, const uint16_t* in, uint16_t* os, uint16_t* ot) {
        uint32_t mask = 0;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            f32x4 acc = bias;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk[ks], frag8(in + (16 * cb + r) * kLs + 32 * ks + 8 * q),
                                                              acc, 0, 0, 0);
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                mask |= (acc[j] > 0.f ? 1u : 0u) << (4 * cb + j);
                v[j] = fmaxf(acc[j], 0.f);
            }
            put4(v, os + (16 * cb + r) * kLs + f0, ot + f0 * kLt + 16 * cb + r);
        }
        return mask;
    };
    // dZ_in = (W^T dZ) masked, to both layouts (os may be null)
    auto backward = [&](const bf16x8 (&tk)[4], uint32_t mask, const uint16_t* in, uint16_t* os, uint16_t* ot) {
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            f32x4 acc = zero4;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tk[ks], frag8(in + (16 * cb + r) * kLs + 32 * ks + 8 * q),
                                                              acc, 0, 0, 0);
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (mask >> (4 * cb + j)) & 1u ? acc[j] : 0.f;
            put4(v, os ? os + (16 * cb + r) * kLs + f0 : nullptr, ot + f0 * kLt + 16 * cb + r);
        }
        __builtin_amdgcn_sched_barrier(0);  // keeps the next phase's operand reads out of this one's registers
    };
    // rows 16 w .. of dW += dZ^T A over the tile's samples, and of db
    auto weight_grad = [&](const uint16_t* dz, const uint16_t* a, f32x4 (&g)[8], f32x4& gb) {
#pragma unroll
        for (int ks = 0; ks < T / 32; ++ks) {
            const bf16x8 d = frag8(dz + (16 * w + r) * kLt + 32 * ks + 8 * q);
            gb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, ones, gb, 0, 0, 0);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                g[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, frag8(a + (16 * c + r) * kLt + 32 * ks + 8 * q), g[c],
                                                               0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    const int64_t ntiles = (p.n + T - 1) / T;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        if (tid < T) {
            const int64_t row = tile * T + tid;
            src[tid] = row >= p.n ? -1 : p.total > 0 ? sample_row(p.key, row, p.total) : row;
        }
        __syncthreads();  // the previous tile's readers are done, src is there
        for (int e = tid; e < T * IN; e += kTrainThreads) {
            const int s = e / IN, c = e % IN;
            const int64_t g = src[s];
            const uint16_t v = g >= 0 ? bf16_bits((p.X[g * IN + c] - p.norm[c]) / p.norm[IN + c]) : (uint16_t)0;
            xs[s * kLx + c] = v;
            xt[c * kLt + s] = v;
        }
        __syncthreads();
        // ---- forward
        uint32_t m1 = 0;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const bf16x8 x = q < 2 ? frag8(xs + (16 * cb + r) * kLx + 8 * q) : zero8;
            const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, x, bias_of(0), 0, 0, 0);
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                m1 |= (acc[j] > 0.f ? 1u : 0u) << (4 * cb + j);
                v[j] = fmaxf(acc[j], 0.f);
            }
            put4(v, as[0] + (16 * cb + r) * kLs + f0, at[0] + f0 * kLt + 16 * cb + r);
        }
        __syncthreads();
        const uint32_t m2 = forward(w2, bias_of(1), as[0], as[1], at[1]);
        __syncthreads();
        const uint32_t m3 = forward(w3, bias_of(2), as[1], as[0], at[2]);
        __syncthreads();
        // ---- output layer, loss and its gradient: waves 0 .. 3, 16 samples each
        if (w < 4) {
            const int s = 16 * w + r;
            const int64_t g = src[s];
            f32x4 acc = bias_of(3);
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag8(p.W[3] + r * H + 32 * ks + 8 * q),
                                                              frag8(as[0] + s * kLs + 32 * ks + 8 * q), acc, 0, 0, 0);
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int o = 4 * q + j;
                v[j] = 0.f;
                if (o < OUT && g >= 0) {
                    const float y = (p.Y[g * OUT + o] - p.norm[2 * IN + o]) / p.norm[2 * IN + OUT + o];
                    const float d = acc[j] - y;
                    se = fma((double)d, (double)d, se);
                    v[j] = 2.f * d / (float)(p.n * OUT);
                }
            }
            put4(v, ds4 + s * kLx + 4 * q, dt4 + 4 * q * kLt + s);
        }
        __syncthreads();
        // ---- backward
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const bf16x8 d = q < 2 ? frag8(ds4 + (16 * cb + r) * kLx + 8 * q) : zero8;
            const f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(t4, d, zero4, 0, 0, 0);
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = (m3 >> (4 * cb + j)) & 1u ? acc[j] : 0.f;
            put4(v, as[1] + (16 * cb + r) * kLs + f0, dt[0] + f0 * kLt + 16 * cb + r);
        }
#pragma unroll
        for (int ks = 0; ks < T / 32; ++ks) {
            const bf16x8 d = frag8(dt4 + r * kLt + 32 * ks + 8 * q);
            g4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, frag8(at[2] + (16 * w + r) * kLt + 32 * ks + 8 * q), g4, 0, 0,
                                                         0);
            gb4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, ones, gb4, 0, 0, 0);
        }
        __syncthreads();
        backward(t3, m2, as[1], as[0], dt[1]);
        weight_grad(dt[0], at[1], g3, gb3);
        __syncthreads();
        backward(t2, m1, as[0], nullptr, dt[0]);
        weight_grad(dt[1], at[0], g2, gb2);
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < T / 32; ++ks) {
            const bf16x8 d = frag8(dt[0] + (16 * w + r) * kLt + 32 * ks + 8 * q);
            g1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, frag8(xt + r * kLt + 32 * ks + 8 * q), g1, 0, 0, 0);
            gb1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, ones, gb1, 0, 0, 0);
        }
        __syncthreads();  // src and xs are rewritten next
    }
    // ---- this workgroup's slab
    float* sl = p.slab + (size_t)blockIdx.x * kParams;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sl[kOffW[0] + (f0 + j) * IN + r] = g1[j];
        sl[kOffW[3] + (4 * q + j) * H + 16 * w + r] = g4[j];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            sl[kOffW[1] + (f0 + j) * H + 16 * c + r] = g2[c][j];
            sl[kOffW[2] + (f0 + j) * H + 16 * c + r] = g3[c][j];
        }
        if (r == 0) {
            sl[kOffB[0] + f0 + j] = gb1[j];
            sl[kOffB[1] + f0 + j] = gb2[j];
            sl[kOffB[2] + f0 + j] = gb3[j];
            if (w == 0) sl[kOffB[3] + 4 * q + j] = gb4[j];
        }
    }
    if (w < 4) {
        se = wave_sum(se);
        if (lane == 0) s_loss[w] = se;
    }
    __syncthreads();
    if (tid == 0) p.loss[blockIdx.x] = s_loss[0] + s_loss[1] + s_loss[2] + s_loss[3];
}

// Sums the slabs of a batch in a fixed order (eight interleaved groups, then the groups in
// order), and steps Adam with the sums or writes them out (ADAM = false).  Eight threads per
// parameter keep enough loads in flight to read the slabs at memory rate.
struct UpdateArgs {
    const float* slab;
    int nslab;
    const double* loss;
    double loss_scale;
    double* loss_acc;  // += loss_scale * (sum of loss[])
    float *p[8], *m[8], *v[8], *g[8];  // W1 b1 W2 b2 W3 b3 W4 b4
    uint16_t *pb[4], *pbT[4];          // BF16 weights and their transposes
    int off[9];
    float lr, c1, c2;
};
constexpr int kUpdCols = 32, kUpdGroups = 8;
template <bool ADAM>
__global__ void __launch_bounds__(kUpdCols* kUpdGroups) k_mlp_update(UpdateArgs a) {
    __shared__ float red[kUpdGroups][kUpdCols];
    const int col = threadIdx.x % kUpdCols, grp = threadIdx.x / kUpdCols;
    const int t = blockIdx.x * kUpdCols + col;
    float acc = 0.f;
    if (t < kParams) {
        int s = grp;
        for (; s + 7 * kUpdGroups < a.nslab; s += 8 * kUpdGroups) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = a.slab[(size_t)(s + u * kUpdGroups) * kParams + t];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += v[u];
        }
        for (; s < a.nslab; s += kUpdGroups) acc += a.slab[(size_t)s * kParams + t];
    }
    red[grp][col] = acc;
    __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        double e = 0;
        for (int k = threadIdx.x; k < a.nslab; k += 64) e += a.loss[k];
        e = wave_sum(e);
        if (threadIdx.x == 0) *a.loss_acc += e * a.loss_scale;
    }
    if (grp != 0 || t >= kParams) return;
    float gt = red[0][col];
#pragma unroll
    for (int k = 1; k < kUpdGroups; ++k) gt += red[k][col];
    int seg = 0;
#pragma unroll
    for (int j = 1; j < 8; ++j) seg += t >= a.off[j] ? 1 : 0;
    const int i = t - a.off[seg];
    if constexpr (ADAM) {
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        const float mt = b1 * a.m[seg][i] + (1.f - b1) * gt;
        const float vt = b2 * a.v[seg][i] + (1.f - b2) * gt * gt;
        a.m[seg][i] = mt;
        a.v[seg][i] = vt;
        const float pt = a.p[seg][i] - a.lr * (mt / a.c1) / (sqrtf(vt / a.c2) + eps);
        a.p[seg][i] = pt;
        if ((seg & 1) == 0) {
            const int l = seg >> 1, din = l == 0 ? MlpDims::IN : MlpDims::H, dout = l == 3 ? MlpDims::OUTP : MlpDims::H;
            const uint16_t v = to_bf16(pt);
            a.pb[l][i] = v;
            a.pbT[l][(i % din) * dout + i / din] = v;
        }
    } else {
        a.g[seg][i] = gt;
    }
}

unsigned g1(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace

// layer l: W[l] is [dout(l) x din(l)] row-major
int MlpDims::din(int l) { return l == 0 ? IN : H; }
int MlpDims::dout(int l) { return l == 3 ? OUTP : H; }

Mlp::Mlp(int device_, uint64_t seed) : device(device_) {
    PB_HIP(hipSetDevice(device));
    PB_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    std::mt19937_64 rng(seed);
    std::normal_distribution<double> nd(0.0, 1.0);
    for (int l = 0; l < 4; ++l) {
        const int di = MlpDims::din(l), dn = MlpDims::dout(l);
        std::vector<float> w((size_t)di * dn), b(dn, 0.f);
        const double sc = std::sqrt(2.0 / di);  // He initialisation
        for (int o = 0; o < dn; ++o)
            for (int i = 0; i < di; ++i) w[(size_t)o * di + i] = (l == 3 && o >= MlpDims::OUT) ? 0.f : (float)(nd(rng) * sc);
        W[l].alloc(w.size());
        Wb[l].alloc(w.size());
        WbT[l].alloc(w.size());
        bvec[l].alloc(dn);
        gW[l].alloc(w.size());
        gb[l].alloc(dn);
        mW[l].alloc(w.size());
        vW[l].alloc(w.size());
        mb[l].alloc(dn);
        vb[l].alloc(dn);
        PB_HIP(hipMemcpyAsync(W[l].p, w.data(), w.size() * 4, hipMemcpyHostToDevice, stream));
        PB_HIP(hipMemcpyAsync(bvec[l].p, b.data(), b.size() * 4, hipMemcpyHostToDevice, stream));
        for (auto* d : {&mW[l], &vW[l]}) PB_HIP(hipMemsetAsync(d->p, 0, d->bytes(), stream));
        for (auto* d : {&mb[l], &vb[l]}) PB_HIP(hipMemsetAsync(d->p, 0, d->bytes(), stream));
        hipLaunchKernelGGL(k_pack_weights, dim3(g1(w.size())), dim3(256), 0, stream, di, dn, W[l].p, Wb[l].p, WbT[l].p);
    }
    norm.alloc(2 * MlpDims::IN + 2 * MlpDims::OUT);
    std::vector<float> nrm(norm.n, 0.f);
    for (int c = 0; c < MlpDims::IN; ++c) nrm[MlpDims::IN + c] = 1.f;
    for (int c = 0; c < MlpDims::OUT; ++c) nrm[2 * MlpDims::IN + MlpDims::OUT + c] = 1.f;
    PB_HIP(hipMemcpyAsync(norm.p, nrm.data(), nrm.size() * 4, hipMemcpyHostToDevice, stream));
    loss_dev.alloc(1);
    int cus = 0;
    PB_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
    max_blocks = cus > 0 ? cus : 256;  // one workgroup (eight waves) of either fused kernel per CU
    PB_HIP(hipStreamSynchronize(stream));
}

Mlp::~Mlp() {
    if (stream) (void)hipStreamDestroy(stream);
}

void Mlp::ensure(int64_t n) {
    if (n <= cap) return;
    cap = n;
    Xb.alloc(n * MlpDims::IN);
    for (int l = 0; l < 3; ++l) Ab[l].alloc(n * MlpDims::H);
    Yp.alloc(n * MlpDims::OUTP);
}

const float* Mlp::xmu() const { return norm.p; }
const float* Mlp::xsd() const { return norm.p + MlpDims::IN; }
const float* Mlp::ymu() const { return norm.p + 2 * MlpDims::IN; }
const float* Mlp::ysd() const { return norm.p + 2 * MlpDims::IN + MlpDims::OUT; }

void Mlp::forward_prepared(int64_t n, hipStream_t s) {
    const uint16_t* in = Xb.p;
    for (int l = 0; l < 4; ++l) {
        GemmArgs g{};
        g.M = (int)n;
        g.N = MlpDims::dout(l);
        g.K = MlpDims::din(l);
        g.A = in;
        g.B = Wb[l].p;
        g.bias = bvec[l].p;
        if (l < 3)
            in = g.Cb = Ab[l].p;
        else
            g.C = Yp.p;
        hipLaunchKernelGGL(k_gemm_bf16, dim3((g.N + TN - 1) / TN, (g.M + TM - 1) / TM), dim3(256), 0, s, g);
    }
}

void Mlp::batch_pass(const float* X, const float* Y, int64_t n, int64_t total, uint64_t key, bool adam, float lr) {
    const int64_t tiles = (n + kTrainCols - 1) / kTrainCols;
    const int blocks = (int)std::min<int64_t>(tiles, max_blocks);
    if (slab.n < (size_t)blocks * kParams) {
        slab.alloc((size_t)blocks * kParams);
        loss_part.alloc(blocks);
    }
    TrainArgs a{};
    a.n = n;
    a.total = total;
    a.key = key;
    a.X = X;
    a.Y = Y;
    a.norm = norm.p;
    UpdateArgs u{};
    u.off[0] = 0;
    for (int l = 0; l < 4; ++l) {
        a.W[l] = u.pb[l] = Wb[l].p;
        a.WT[l] = u.pbT[l] = WbT[l].p;
        a.b[l] = bvec[l].p;
        const int kw = 2 * l, kb = 2 * l + 1;
        u.p[kw] = W[l].p, u.m[kw] = mW[l].p, u.v[kw] = vW[l].p, u.g[kw] = gW[l].p;
        u.p[kb] = bvec[l].p, u.m[kb] = mb[l].p, u.v[kb] = vb[l].p, u.g[kb] = gb[l].p;
        u.off[kw + 1] = u.off[kw] + MlpDims::din(l) * MlpDims::dout(l);
        u.off[kb + 1] = u.off[kb] + MlpDims::dout(l);
    }
    a.slab = slab.p;
    a.loss = loss_part.p;
    u.slab = slab.p;
    u.nslab = blocks;
    u.loss = loss_part.p;
    u.loss_scale = 1.0 / (double)(n * MlpDims::OUT);
    u.loss_acc = loss_dev.p;
    hipLaunchKernelGGL(k_mlp_train, dim3(blocks), dim3(kTrainThreads), 0, stream, a);
    const dim3 ug((kParams + kUpdCols - 1) / kUpdCols), ub(kUpdCols * kUpdGroups);
    if (adam) {
        ++t_adam;
        u.lr = lr;
        u.c1 = 1.f - std::pow(0.9f, (float)t_adam);
        u.c2 = 1.f - std::pow(0.999f, (float)t_adam);
        hipLaunchKernelGGL(k_mlp_update<true>, ug, ub, 0, stream, u);
    } else {
        hipLaunchKernelGGL(k_mlp_update<false>, ug, ub, 0, stream, u);
    }
    PB_HIP(hipGetLastError());
}

double Mlp::train(const float* X, const float* Y, int64_t n, int epochs, int batch, float lr, uint64_t seed) {
    const int64_t per_epoch = (n + batch - 1) / batch;
    double loss = 0;
    for (int e = 0; e < epochs; ++e) {
        PB_HIP(hipMemsetAsync(loss_dev.p, 0, sizeof(double), stream));
        for (int64_t b = 0; b < per_epoch; ++b) {
            const uint64_t key = seed * 0x9E3779B97F4A7C15ull + (uint64_t)(e * per_epoch + b) * 0xD1B54A32D192ED03ull;
            batch_pass(X, Y, batch, n, key, true, lr);
        }
        double acc = 0;
        PB_HIP(hipMemcpyAsync(&acc, loss_dev.p, sizeof(double), hipMemcpyDeviceToHost, stream));
        PB_HIP(hipStreamSynchronize(stream));
        loss = acc / (double)per_epoch;
    }
    PB_HIP(hipStreamSynchronize(stream));
    return loss;
}

void Mlp::predict_fused(const float* X, float* Y, int64_t n, hipStream_t s) {
    InferArgs a;
    a.n = n;
    a.X = X;
    for (int l = 0; l < 4; ++l) {
        a.W[l] = Wb[l].p;
        a.b[l] = bvec[l].p;
    }
    a.norm = norm.p;
    a.Y = Y;
    a.x16 = ((uintptr_t)X & 15) == 0;
    const int64_t tiles = (n + kInferCols - 1) / kInferCols;
    const unsigned grid = (unsigned)std::min<int64_t>(tiles, max_blocks);
    hipLaunchKernelGGL(k_mlp_infer, dim3(grid), dim3(kInferThreads), 0, s, a);
    PB_HIP(hipGetLastError());
}

// layer by layer on the caller's stream, chunked so that the workspace stays bounded
void Mlp::predict_layers(const float* X, float* Y, int64_t n, hipStream_t s) {
    const int64_t chunk = 1 << 20;
    for (int64_t o = 0; o < n; o += chunk) {
        const int64_t m = std::min(chunk, n - o);
        ensure(m);
        hipLaunchKernelGGL(k_prep_inputs, dim3(g1(m * MlpDims::IN)), dim3(256), 0, s, m, X + o * MlpDims::IN, xmu(),
                           xsd(), Xb.p);
        forward_prepared(m, s);
        hipLaunchKernelGGL(k_denorm, dim3(g1(m * MlpDims::OUT)), dim3(256), 0, s, m, Yp.p, ymu(), ysd(),
                           Y + o * MlpDims::OUT);
    }
}

int64_t Mlp::param_count() {
    int64_t c = 0;
    for (int l = 0; l < 4; ++l) c += (int64_t)MlpDims::din(l) * MlpDims::dout(l) + MlpDims::dout(l);
    return c;
}

void Mlp::get_params(float* host, bool grads) {
    int64_t o = 0;
    for (int l = 0; l < 4; ++l) {
        const int64_t nw = (int64_t)MlpDims::din(l) * MlpDims::dout(l), nb = MlpDims::dout(l);
        PB_HIP(hipMemcpyAsync(host + o, grads ? gW[l].p : W[l].p, nw * 4, hipMemcpyDeviceToHost, stream));
        o += nw;
        PB_HIP(hipMemcpyAsync(host + o, grads ? gb[l].p : bvec[l].p, nb * 4, hipMemcpyDeviceToHost, stream));
        o += nb;
    }
    PB_HIP(hipStreamSynchronize(stream));
}

void Mlp::set_params(const float* host) {
    int64_t o = 0;
    for (int l = 0; l < 4; ++l) {
        const int64_t nw = (int64_t)MlpDims::din(l) * MlpDims::dout(l), nb = MlpDims::dout(l);
        PB_HIP(hipMemcpyAsync(W[l].p, host + o, nw * 4, hipMemcpyHostToDevice, stream));
        o += nw;
        PB_HIP(hipMemcpyAsync(bvec[l].p, host + o, nb * 4, hipMemcpyHostToDevice, stream));
        o += nb;
        hipLaunchKernelGGL(k_pack_weights, dim3(g1(nw)), dim3(256), 0, stream, MlpDims::din(l), MlpDims::dout(l), W[l].p,
                           Wb[l].p, WbT[l].p);
    }
    PB_HIP(hipStreamSynchronize(stream));
}

void Mlp::set_normalization(const float* host) {
    PB_HIP(hipMemcpyAsync(norm.p, host, norm.bytes(), hipMemcpyHostToDevice, stream));
    PB_HIP(hipStreamSynchronize(stream));
}

double Mlp::gradients(const float* Xh, const float* Yh, int64_t n, float* grads_host) {
    DevBuf<float> X, Y;
    X.alloc(n * MlpDims::IN);
    Y.alloc(n * MlpDims::OUT);
    PB_HIP(hipMemcpyAsync(X.p, Xh, X.bytes(), hipMemcpyHostToDevice, stream));
    PB_HIP(hipMemcpyAsync(Y.p, Yh, Y.bytes(), hipMemcpyHostToDevice, stream));
    PB_HIP(hipMemsetAsync(loss_dev.p, 0, sizeof(double), stream));
    batch_pass(X.p, Y.p, n, 0, 0, false, 0.f);
    double loss = 0;
    PB_HIP(hipMemcpyAsync(&loss, loss_dev.p, sizeof(double), hipMemcpyDeviceToHost, stream));
    PB_HIP(hipStreamSynchronize(stream));
    if (grads_host) get_params(grads_host, true);
    return loss;
}

}  // namespace pb
