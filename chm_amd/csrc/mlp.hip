// Per-face network of the learned warm start: 16 -> 128 -> 128 -> 128 -> 11,
// ReLU, BF16 operands with FP32 accumulation on the matrix cores
// (gfx950's v_mfma_f32_16x16x32_bf16), trained on the GPU by its own forward
// and backward kernels with Adam.
//
// For a layer with weights W [out x in], activations A and pre-activations Z [samples x features]
//   forward   Z = A_in W^T + b,   A_out = relu(Z)
//   backward  dW = dZ^T A_in,     db = colsum(dZ),   dZ_in = (dZ W) * [Z_in > 0]
// Inference (k_mlp_infer) carries a wave's samples through all layers in registers; training
// (k_mlp_train) runs forward and backward of a 64-sample tile in one workgroup, k_mlp_wgrad forms
// the weight and bias gradients of the batch and k_mlp_update steps Adam; k_gemm_bf16 is the
// layer-by-layer forward that the fused inference is checked against.  Every sum has a fixed
// order of its own, whatever the grid: a layer's bias is added to the finished product, a weight
// gradient is the sum of row slabs (wgrad_split) in order, a bias gradient that of row blocks.  MFMA operand layout of v_mfma_f32_16x16x32_bf16
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
    const float* bias;  // per output column, added to the finished product
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
    f32x4 acc[2][2] = {};
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
                const float v = acc[tm][tn][j] + g.bias[col];
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
// k runs in increasing order and the bias is added to the finished product, as in k_gemm_bf16,
// so the output equals the layer-by-layer forward bit for bit.
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
        f32x4 acc[2][4] = {}, bq[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) bq[h] = *reinterpret_cast<const f32x4*>(&bias[32 * kk + 8 * q + 4 * h]);
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
                for (int j = 0; j < 4; ++j) out[kk][cb][4 * h + j] = (__bf16)fmaxf(acc[h][cb][j] + bq[h][j], 0.f);
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
        f32x4 acc[4] = {};
        const f32x4 bq = *reinterpret_cast<const f32x4*>(&bias[3 * H + 4 * q]);
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
                    if (4 * q + j < OUT) p.Y[g * OUT + 4 * q + j] = (acc[cb][j] + bq[j]) * ysd[j] + ymu[j];
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

// A training batch, in three launches.
//
// k_mlp_train: forward, loss and backward.  A workgroup of eight waves takes tiles of 64 samples;
// wave w owns the 16 hidden features 16 w .. + 15 of every layer.  Its weight fragments (W for the
// forward products, W^T for the backward ones) stay in registers for all of the workgroup's
// tiles; activations and back-propagated gradients pass through LDS twice: as [sample][feature],
// the B operand of the next product, and as [feature][sample], from where they leave for the
// tile's block in memory (TileAt) while the next product runs.  The ReLU masks stay in the
// registers of the lane that computed them.
// k_mlp_wgrad: dW = dZ^T A over the rows of one slab, a 32 x 32 block of the output per wave; its
// operands are read in the MFMA lane layout straight from the tiles' blocks (k = samples).
// k_mlp_update: the slabs and the bias gradients' partial sums added in order, then Adam.
//
// Bound: k_mlp_train by the arrival of its weight fragments (a third of its time) and the
// LDS reads and barriers of a tile, the other two by the latency of their loads (13 MB of tiles
// and 2.4 MB of slabs at a batch of 8,192 stay in the caches).  A batch of 8,192 took 215 us in 29
// launches (11 GEMMs of 13 us, split-K and column sums, one launch per elementwise step); these
// three take 20.3 + 8.1 + 4.5 us with the same bits.
constexpr int kTrainCols = 64;
constexpr int kTrainThreads = 512;
constexpr int kLs = MlpDims::H + 8;      // LDS row stride (BF16) of [sample][128 features]
constexpr int kLt = kTrainCols + 8;      // of [feature][64 samples]
constexpr int kLx = MlpDims::IN + 8;     // of [sample][16 features]
constexpr int kWeights = 36864, kBiases = 400;
constexpr int kOffW[4] = {0, 2048, 18432, 34816};  // a layer's weights in a slab
constexpr int kMaxSlabs = 64;            // row ranges of the weight gradients
constexpr int kMaxBiasBlocks = 512;      // row blocks of the bias gradients

// Where a tile's [feature][64 samples] blocks lie in its 64 x 800 values
struct TileAt {
    static constexpr int H64 = MlpDims::H * kTrainCols, IN64 = MlpDims::IN * kTrainCols;
    static constexpr int x = 0, d4 = IN64;                             // inputs, output gradients
    static constexpr int a(int l) { return 2 * IN64 + l * H64; }       // activations of hidden layer l
    static constexpr int d(int l) { return 2 * IN64 + (3 + l) * H64; }  // gradients of its pre-activations
    static constexpr int size = 2 * IN64 + 6 * H64;
};

struct TrainArgs {
    int64_t n;        // samples of the batch
    int64_t total;    // > 0: batch row t is sample_row(key, t, total) of X / Y; 0: row t itself
    uint64_t key;
    const float *X, *Y;
    const float* norm;
    const uint16_t *W[4], *WT[4];  // BF16 [dout x din] and [din x dout]
    const float* b[4];
    uint16_t* tiles;  // [ceil(n / 64)][TileAt::size]
    float* loss;      // [ceil(n / 16)] summed squared error of 16 rows
    float* bias;      // [ceil(n / 64)][kBiases]: the tiles' bias gradients (null: k_mlp_wgrad forms them)
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

// rows x 64 samples from LDS to a tile's block, the samples from `live` on as zeros
__device__ __forceinline__ void store_block(const uint16_t* __restrict__ t, int rows, int live,
                                            uint16_t* __restrict__ out, int tid) {
    typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
    for (int e = tid; e < rows * 8; e += kTrainThreads) {
        u16x8 v = *reinterpret_cast<const u16x8*>(t + (e >> 3) * kLt + 8 * (e & 7));
        if (live < kTrainCols) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = 8 * (e & 7) + j < live ? v[j] : (uint16_t)0;
        }
        *reinterpret_cast<u16x8*>(out + e * 8) = v;
    }
}

__device__ __forceinline__ float bf16_low(uint32_t two) { return __uint_as_float(two << 16); }
__device__ __forceinline__ float bf16_high(uint32_t two) { return __uint_as_float(two & 0xffff0000u); }

// Bias gradients of a tile's 128 hidden features from LDS: the sum of the even rows and that of the odd
// rows, a thread each (threads 0 .. 255).
__device__ __forceinline__ void tile_bias(const uint16_t* __restrict__ t, float* __restrict__ out, int tid) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const int c = tid >> 1, odd = tid & 1;
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < kTrainCols / 8; ++u) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(t + c * kLt + 8 * u);
#pragma unroll
        for (int j = 0; j < 4; ++j) s += odd ? bf16_high(v[j]) : bf16_low(v[j]);
    }
    s += __shfl_xor(s, 1);
    if (!odd) out[c] = s;
}
// Those of the 16 outputs: sixteen sums of every sixteenth row, added in order (256 threads).
__device__ __forceinline__ void tile_bias_out(const uint16_t* __restrict__ t, float* __restrict__ out, int tid) {
    const int c = tid >> 4, k = tid & 15;
    float s = 0.f, sum = 0.f;
#pragma unroll
    for (int u = 0; u < kTrainCols / 16; ++u) s += bf16_low(t[c * kLt + k + 16 * u]);
#pragma unroll
    for (int j = 0; j < 16; ++j) sum += __shfl(s, (tid & 48) + j);
    if (k == 0) out[c] = sum;
}

__global__ void __launch_bounds__(kTrainThreads) k_mlp_train(TrainArgs p) {
    constexpr int H = MlpDims::H, IN = MlpDims::IN, OUT = MlpDims::OUT, OUTP = MlpDims::OUTP;
    constexpr int T = kTrainCols;
    __shared__ __align__(16) uint16_t xs[T * kLx], xt[IN * kLt];
    __shared__ __align__(16) uint16_t as[2][T * kLs];  // activations / gradients by sample, in turn
    __shared__ __align__(16) uint16_t ft[2][H * kLt];  // the same by feature, in turn
    __shared__ __align__(16) uint16_t ds4[T * kLx], dt4[OUTP * kLt];
    __shared__ __align__(16) float bias[3 * H + OUTP];
    __shared__ int64_t src[T];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, q = lane >> 4;
    const int f0 = 16 * w + 4 * q;  // the lane's first output feature
    const bf16x8 zero8 = {};
    // Loads in the order of their use, so that a phase waits for no later one's: the first tile's
    // rows, then the weight fragments (147 KB per workgroup).
    const float xmu = p.norm[tid % IN], xsd = p.norm[IN + tid % IN];  // of the input column the thread stages
    float ymu[4], ysd[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int o = min(4 * q + j, OUT - 1);
        ymu[j] = p.norm[2 * IN + o];
        ysd[j] = p.norm[2 * IN + OUT + o];
    }
    if (tid < 3 * H + OUTP) {
        const float* b = tid < H ? p.b[0] : tid < 2 * H ? p.b[1] : tid < 3 * H ? p.b[2] : p.b[3];
        bias[tid] = b[tid % H];
    }
    float xv[2], y[4];  // inputs of the thread's two entries, targets of the lane's outputs (waves 0 .. 3)
    bool live_x[2], mine;
    auto stage = [&](int64_t tile) {
        if (tid < T) {
            const int64_t row = tile * T + tid;
            src[tid] = row >= p.n ? -1 : p.total > 0 ? sample_row(p.key, row, p.total) : row;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int64_t g = src[32 * k + tid / IN];
            live_x[k] = g >= 0;
            xv[k] = p.X[max(g, (int64_t)0) * IN + tid % IN];
        }
        const int64_t g = src[16 * (w & 3) + r];
        mine = w < 4 && g >= 0;
        if (w < 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = p.Y[max(g, (int64_t)0) * OUT + min(4 * q + j, OUT - 1)];
        }
    };
    const int64_t ntiles = (p.n + T - 1) / T;
    stage(blockIdx.x);
    __builtin_amdgcn_sched_barrier(0);
    // weight fragments of this wave (rows 16 w .. of W, and of W^T)
    const bf16x8 w1 = q < 2 ? frag8(p.W[0] + (16 * w + r) * IN + 8 * q) : zero8;
    const bf16x8 t4 = q < 2 ? frag8(p.WT[3] + (16 * w + r) * OUTP + 8 * q) : zero8;
    bf16x8 w2[4], w3[4], w4[4], t2[4], t3[4];
    auto fragments = [&](bf16x8 (&f)[4], const uint16_t* W, int row) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) f[ks] = frag8(W + row * H + 32 * ks + 8 * q);
    };
    fragments(w2, p.W[1], 16 * w + r);
    fragments(w3, p.W[2], 16 * w + r);
    fragments(w4, p.W[3], r);
    fragments(t3, p.WT[2], 16 * w + r);
    fragments(t2, p.WT[1], 16 * w + r);
    __builtin_amdgcn_sched_barrier(0);
    auto bias_of = [&](int l) { return *reinterpret_cast<const f32x4*>(&bias[l * H + (l < 3 ? f0 : 4 * q)]); };
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};

    // Z = W A + b of 16 features x 16 samples; relu to both layouts; the mask Z > 0, bit 4 cb + j
    auto activate = [&](const f32x4& acc, const f32x4& b, int cb, uint16_t* os, uint16_t* ot) {
        uint32_t mask = 0;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float z = acc[j] + b[j];
            mask |= (z > 0.f ? 1u : 0u) << (4 * cb + j);
            v[j] = fmaxf(z, 0.f);
        }
        put4(v, os + (16 * cb + r) * kLs + f0, ot + f0 * kLt + 16 * cb + r);
        return mask;
    };
    auto forward = [&](const bf16x8 (&wk)[4], f32x4 b, const uint16_t* in, uint16_t* os, uint16_t* ot) {
        uint32_t mask = 0;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            f32x4 acc = zero4;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk[ks], frag8(in + (16 * cb + r) * kLs + 32 * ks + 8 * q),
                                                              acc, 0, 0, 0);
            mask |= activate(acc, b, cb, os, ot);
        }
        return mask;
    };
    // dZ_in = (W^T dZ) masked, to both layouts (os may be null)
    auto masked = [&](const f32x4& acc, uint32_t mask, int cb, uint16_t* os, uint16_t* ot) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (mask >> (4 * cb + j)) & 1u ? acc[j] : 0.f;
        put4(v, os ? os + (16 * cb + r) * kLs + f0 : nullptr, ot + f0 * kLt + 16 * cb + r);
    };
    auto backward = [&](const bf16x8 (&tk)[4], uint32_t mask, const uint16_t* in, uint16_t* os, uint16_t* ot) {
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            f32x4 acc = zero4;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tk[ks], frag8(in + (16 * cb + r) * kLs + 32 * ks + 8 * q),
                                                              acc, 0, 0, 0);
            masked(acc, mask, cb, os, ot);
        }
    };

    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int live = (int)min((int64_t)T, p.n - tile * T);
        uint16_t* out = p.tiles + tile * TileAt::size;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int s = 32 * k + tid / IN, c = tid % IN;
            const uint16_t v = live_x[k] ? bf16_bits((xv[k] - xmu) / xsd) : (uint16_t)0;
            xs[s * kLx + c] = v;
            xt[c * kLt + s] = v;
        }
        __syncthreads();
        // ---- forward
        uint32_t m1 = 0;
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const bf16x8 x = q < 2 ? frag8(xs + (16 * cb + r) * kLx + 8 * q) : zero8;
            m1 |= activate(__builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, x, zero4, 0, 0, 0), bias_of(0), cb, as[0], ft[0]);
        }
        store_block(xt, IN, live, out + TileAt::x, tid);
        __syncthreads();
        const uint32_t m2 = forward(w2, bias_of(1), as[0], as[1], ft[1]);
        store_block(ft[0], H, live, out + TileAt::a(0), tid);
        __syncthreads();
        const uint32_t m3 = forward(w3, bias_of(2), as[1], as[0], ft[0]);
        store_block(ft[1], H, live, out + TileAt::a(1), tid);
        __syncthreads();
        // ---- output layer, loss and its gradient: waves 0 .. 3, 16 samples each
        if (w < 4) {
            const int s = 16 * w + r;
            f32x4 acc = zero4;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w4[ks], frag8(as[0] + s * kLs + 32 * ks + 8 * q), acc, 0, 0,
                                                              0);
            const f32x4 b4 = bias_of(3);
            float v[4], se[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = se[j] = 0.f;
                if (4 * q + j < OUT && mine) {
                    const float d = acc[j] + b4[j] - (y[j] - ymu[j]) / ysd[j];
                    se[j] = d * d;
                    v[j] = 2.f * d / (float)(p.n * OUT);
                }
            }
            put4(v, ds4 + s * kLx + 4 * q, dt4 + 4 * q * kLt + s);
            // the wave's 16 x 16 squares by halves: rows 8, 4, 2, 1 apart, then columns
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                se[j] += __shfl_xor(se[j], 8);
                se[j] += __shfl_xor(se[j], 4);
                se[j] += __shfl_xor(se[j], 2);
                se[j] += __shfl_xor(se[j], 1);
                se[j] += __shfl_xor(se[j], 32);
                se[j] += __shfl_xor(se[j], 16);
            }
            if (lane == 0 && 16 * w < live) p.loss[tile * 4 + w] = (se[0] + se[2]) + (se[1] + se[3]);
        }
        store_block(ft[0], H, live, out + TileAt::a(2), tid);
        __syncthreads();
        // ---- backward
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
            const bf16x8 d = q < 2 ? frag8(ds4 + (16 * cb + r) * kLx + 8 * q) : zero8;
            masked(__builtin_amdgcn_mfma_f32_16x16x32_bf16(t4, d, zero4, 0, 0, 0), m3, cb, as[1], ft[1]);
        }
        store_block(dt4, OUTP, live, out + TileAt::d4, tid);
        if (p.bias && w >= 4) tile_bias_out(dt4, p.bias + tile * kBiases + 3 * H, tid - 256);
        __syncthreads();
        backward(t3, m2, as[1], as[0], ft[0]);
        store_block(ft[1], H, live, out + TileAt::d(2), tid);
        if (p.bias && w < 4) tile_bias(ft[1], p.bias + tile * kBiases + 2 * H, tid);
        __syncthreads();
        backward(t2, m1, as[0], nullptr, ft[1]);
        store_block(ft[0], H, live, out + TileAt::d(1), tid);
        if (p.bias && w >= 4) tile_bias(ft[0], p.bias + tile * kBiases + H, tid - 256);
        __syncthreads();
        store_block(ft[1], H, live, out + TileAt::d(0), tid);
        if (p.bias && w < 4) tile_bias(ft[1], p.bias + tile * kBiases, tid);
        if (tile + gridDim.x < ntiles) stage(tile + gridDim.x);
    }
}

// Rows of one slab of a batch's weight gradients: up to 64 slabs of at least 512 rows, so that a batch
// of 32,768 has enough of them for the chip; a multiple of the MFMA's k.
inline int64_t wgrad_split(int64_t n) {
    const int64_t slabs = std::min<int64_t>(kMaxSlabs, std::max<int64_t>(1, n / 512));
    return ((n + slabs - 1) / slabs + 31) / 32 * 32;
}
// Rows of one block of its bias gradients.
inline int64_t bias_rows(int64_t n) { return std::max<int64_t>(64, (n + kMaxBiasBlocks - 1) / kMaxBiasBlocks); }

struct GradArgs {
    int64_t n;
    const uint16_t* tiles;
    int64_t ksplit;  // wgrad_split(n)
    int nslab;
    float* slab;  // [nslab][kWeights]
    int64_t R;    // bias_rows(n)
    int nblock;   // row blocks whose bias gradients are formed here (0: the tiles' own)
    float* bias;  // [nblock][kBiases]
};

// STEPS k-steps of a (16 MB x 16 NB) block of dW, all their loads in flight; dp and ap point at the lane's
// first values of dZ and A in the first tile's block.
template <int STEPS, int MB, int NB>
__device__ __forceinline__ void grad_steps(const uint16_t* __restrict__ dp, const uint16_t* __restrict__ ap, int64_t k,
                                           f32x4 (&acc)[MB][NB]) {
    bf16x8 df[STEPS][MB], af[STEPS][NB];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
        const int64_t ks = k + 32 * u, at = (ks >> 6) * TileAt::size + (ks & 63);
#pragma unroll
        for (int m = 0; m < MB; ++m) df[u][m] = frag8(dp + at + m * 16 * kTrainCols);
#pragma unroll
        for (int c = 0; c < NB; ++c) af[u][c] = frag8(ap + at + c * 16 * kTrainCols);
    }
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int c = 0; c < NB; ++c)
                acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(df[u][m], af[u][c], acc[m][c], 0, 0, 0);
}

// (16 MB x 16 NB) of dW = dZ^T A over the samples [k0, k1), from row m0 of dZ and row n0 of A in the
// tiles' blocks at d and a.  The last step's samples past the batch are zeros.
template <int MB, int NB>
__device__ __forceinline__ void grad_block(const uint16_t* __restrict__ tiles, int d, int m0, int a, int n0, int64_t k0,
                                           int64_t k1, float* __restrict__ out, int ld) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    f32x4 acc[MB][NB] = {};
    const uint16_t *dp = tiles + d + (m0 + r) * kTrainCols + 8 * q, *ap = tiles + a + (n0 + r) * kTrainCols + 8 * q;
    int64_t k = k0;
    for (; k + 7 * 32 < k1; k += 8 * 32) grad_steps<8>(dp, ap, k, acc);
    for (; k + 32 < k1; k += 2 * 32) grad_steps<2>(dp, ap, k, acc);
    if (k < k1) grad_steps<1>(dp, ap, k, acc);
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) out[(m0 + 16 * m + 4 * q + j) * ld + n0 + 16 * c + r] = acc[m][c][j];
}

// One wave per workgroup and job: 40 blocks of the weights for each slab, then 6 + 4 groups of 64
// bias sums for each row block.  A slab's workgroups are eight apart, so that they run on one XCD,
// whose L2 then reads the slab's tiles once.  A batch of 8,192 takes 8.1 us; 10.2 with four waves per
// workgroup, whose 160 workgroups leave CUs idle.
constexpr int kSlabJobs = 40, kBiasJobs = 10;
inline int64_t slab_grid(int nslab) { return (int64_t)(nslab + 7) / 8 * 8 * kSlabJobs; }
__global__ void __launch_bounds__(64) k_mlp_wgrad(GradArgs p) {
    constexpr int H = MlpDims::H, IN = MlpDims::IN;
    const int lane = threadIdx.x, first_bias = (p.nslab + 7) / 8 * 8 * kSlabJobs;
    if ((int)blockIdx.x < first_bias) {
        const int y = blockIdx.x >> 3, z = (blockIdx.x & 7) + 8 * (y / kSlabJobs), b = y % kSlabJobs;
        if (z >= p.nslab) return;
        const int64_t k0 = z * p.ksplit, k1 = min(p.n, k0 + p.ksplit);
        float* out = p.slab + (size_t)z * kWeights;
        if (b < 32) {
            const int l = 1 + (b >> 4), m0 = 32 * ((b >> 2) & 3), n0 = 32 * (b & 3);
            grad_block<2, 2>(p.tiles, TileAt::d(l), m0, TileAt::a(l - 1), n0, k0, k1, out + kOffW[l], H);
        } else if (b < 36) {
            grad_block<2, 1>(p.tiles, TileAt::d(0), 32 * (b - 32), TileAt::x, 0, k0, k1, out + kOffW[0], IN);
        } else {
            grad_block<1, 2>(p.tiles, TileAt::d4, 0, TileAt::a(2), 32 * (b - 36), k0, k1, out + kOffW[3], H);
        }
        return;
    }
    const int job = (int)blockIdx.x - first_bias;
    const int block = job / kBiasJobs, b = job % kBiasJobs;
    const int64_t r0 = block * p.R, r1 = min(p.n, r0 + p.R);
    auto f32 = [](uint16_t v) { return __uint_as_float((uint32_t)v << 16); };
    if (b < 6) {  // a hidden layer's column: the sums of its even and of its odd rows
        const int l = b >> 1, c = 64 * (b & 1) + lane;
        const uint16_t* col = p.tiles + TileAt::d(l) + c * kTrainCols;
        typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
        float sum[2] = {0.f, 0.f};
        for (int64_t g0 = r0 >> 3; 8 * g0 < r1; g0 += 8) {
            u16x8 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t g = min(g0 + u, (r1 - 1) >> 3);
                v[u] = *reinterpret_cast<const u16x8*>(col + (g >> 3) * TileAt::size + 8 * (g & 7));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int64_t row = 8 * (g0 + u) + j;
                    if (row >= r0 && row < r1) sum[j & 1] += f32(v[u][j]);
                }
        }
        p.bias[(size_t)block * kBiases + l * H + c] = sum[0] + sum[1];
    } else {  // an output column: sixteen sums of every sixteenth row, added in order
        const int c = 4 * (b - 6) + (lane >> 4);
        const uint16_t* col = p.tiles + TileAt::d4 + c * kTrainCols;
        float s = 0.f, t = 0.f;
        for (int64_t row0 = r0 + (lane & 15); row0 < r1; row0 += 64) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t row = min(row0 + 16 * u, r1 - 1);
                v[u] = f32(col[(row >> 6) * TileAt::size + (row & 63)]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (row0 + 16 * u < r1) s += v[u];
        }
        for (int k = 0; k < 16; ++k) t += __shfl(s, (lane & 48) + k);
        if ((lane & 15) == 0) p.bias[(size_t)block * kBiases + 3 * H + c] = t;
    }
}

struct UpdateArgs {
    const float* slab;
    int nslab;
    const float* bias;
    int nblock;
    const float* loss;
    int64_t nloss;
    double loss_scale;
    double* loss_acc;  // += loss_scale * (sum of loss[])
    float *p[8], *m[8], *v[8], *g[8];  // W1 b1 W2 b2 W3 b3 W4 b4
    uint16_t *pb[4], *pbT[4];          // BF16 weights and their transposes
    float lr, c1, c2;
};

// entry i of parameter tensor seg: an Adam step with its gradient, or the gradient itself
struct AdamState {
    float p, m, v;
};
__device__ __forceinline__ AdamState load_state(const UpdateArgs& a, int seg, int i) {
    return AdamState{a.p[seg][i], a.m[seg][i], a.v[seg][i]};
}
template <bool ADAM>
__device__ __forceinline__ void update_param(const UpdateArgs& a, int seg, int i, const AdamState& st, float gt) {
    if constexpr (ADAM) {
        if (seg == 6 ? i >= MlpDims::OUT * MlpDims::H : seg == 7 && i >= MlpDims::OUT) return;  // padding rows stay
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        const float mt = b1 * st.m + (1.f - b1) * gt;
        const float vt = b2 * st.v + (1.f - b2) * gt * gt;
        a.m[seg][i] = mt;
        a.v[seg][i] = vt;
        const float pt = st.p - a.lr * (mt / a.c1) / (sqrtf(vt / a.c2) + eps);
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

// Blocks: 256 weights each, one per thread; then 32 biases each, eight threads per bias; the last
// one adds the batch's loss.  No block spans two layers.
constexpr int kWeightBlocks = kWeights / 256, kBiasBlocks = (kBiases + 31) / 32;
template <bool ADAM>
__global__ void __launch_bounds__(256) k_mlp_update(UpdateArgs a) {
    __shared__ double red[256];
    const int tid = threadIdx.x, blk = blockIdx.x;
    if (blk < kWeightBlocks) {
        const int t0 = blk * 256, l = t0 < kOffW[1] ? 0 : t0 < kOffW[2] ? 1 : t0 < kOffW[3] ? 2 : 3;
        const int t = t0 + tid, i = t - kOffW[l];
        const AdamState st = load_state(a, 2 * l, i);
        float acc = 0.f;
        if (a.nslab == 1) {
            acc = a.slab[t];
        } else {
            for (int z = 0; z < a.nslab; z += 16) {  // sixteen loads in flight, added in slab order
                float v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = a.slab[(size_t)min(z + u, a.nslab - 1) * kWeights + t];
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    if (z + u < a.nslab) acc += v[u];
            }
        }
        update_param<ADAM>(a, 2 * l, i, st, acc);
    } else if (blk < kWeightBlocks + kBiasBlocks) {
        // The row blocks' sums by halves of 256: thread g of a bias adds those 8 apart from g on,
        // 128, 64 .. 8 apart, then the eight threads 4, 2 and 1 apart.
        const int b0 = 32 * (blk - kWeightBlocks), l = b0 / MlpDims::H, g = tid & 7;
        const int cc = b0 + (tid >> 3), c = min(cc, kBiases - 1), i = c - l * MlpDims::H;
        const AdamState st = load_state(a, 2 * l + 1, i);
        float v[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = a.bias[(size_t)min(g + 8 * k, a.nblock - 1) * kBiases + c];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = g + 8 * k < a.nblock ? 0.f + v[k] : 0.f;
        if (a.nblock > 256) {
            float h[32];
#pragma unroll
            for (int k = 0; k < 32; ++k) h[k] = a.bias[(size_t)min(256 + g + 8 * k, a.nblock - 1) * kBiases + c];
#pragma unroll
            for (int k = 0; k < 32; ++k)
                if (256 + g + 8 * k < a.nblock) v[k] += h[k];
        }
#pragma unroll
        for (int o = 16; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < o; ++k) v[k] += v[k + o];
        float s = v[0];
        s += __shfl_xor(s, 4);
        s += __shfl_xor(s, 2);
        s += __shfl_xor(s, 1);
        if (g == 0 && cc < kBiases) update_param<ADAM>(a, 2 * l + 1, i, st, s);
    } else {
        double e = 0;
        for (int64_t k = tid; k < a.nloss; k += 256) e += a.loss[k];
        red[tid] = e;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o) red[tid] += red[tid + o];
            __syncthreads();
        }
        if (tid == 0) *a.loss_acc += red[0] * a.loss_scale;
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
    const int64_t ntiles = (n + kTrainCols - 1) / kTrainCols;
    const int blocks = (int)std::min<int64_t>(ntiles, max_blocks);
    GradArgs ga{};
    ga.n = n;
    ga.ksplit = wgrad_split(n);
    ga.nslab = (int)((n + ga.ksplit - 1) / ga.ksplit);
    ga.R = bias_rows(n);
    const int nblock = (int)((n + ga.R - 1) / ga.R);
    // A row block of one tile is summed where the tile is in LDS (n <= 32768); longer ones, which cross
    // tiles, from memory.
    const bool by_tile = ga.R == kTrainCols;
    ga.nblock = by_tile ? 0 : nblock;
    const size_t nloss = (size_t)(n + 15) / 16;
    if (tiles.n < (size_t)ntiles * TileAt::size) tiles.alloc((size_t)ntiles * TileAt::size);
    if (slab.n < (size_t)ga.nslab * kWeights) slab.alloc((size_t)ga.nslab * kWeights);
    if (bias_part.n < (size_t)nblock * kBiases) bias_part.alloc((size_t)nblock * kBiases);
    if (loss_part.n < nloss) loss_part.alloc(nloss);
    TrainArgs a{};
    a.n = n;
    a.total = total;
    a.key = key;
    a.X = X;
    a.Y = Y;
    a.norm = norm.p;
    UpdateArgs u{};
    for (int l = 0; l < 4; ++l) {
        a.W[l] = u.pb[l] = Wb[l].p;
        a.WT[l] = u.pbT[l] = WbT[l].p;
        a.b[l] = bvec[l].p;
        const int kw = 2 * l, kb = 2 * l + 1;
        u.p[kw] = W[l].p, u.m[kw] = mW[l].p, u.v[kw] = vW[l].p, u.g[kw] = gW[l].p;
        u.p[kb] = bvec[l].p, u.m[kb] = mb[l].p, u.v[kb] = vb[l].p, u.g[kb] = gb[l].p;
    }
    a.tiles = tiles.p;
    a.loss = loss_part.p;
    a.bias = by_tile ? bias_part.p : nullptr;
    ga.tiles = tiles.p;
    u.slab = ga.slab = slab.p;
    u.bias = ga.bias = bias_part.p;
    u.nslab = ga.nslab;
    u.nblock = nblock;
    u.loss = loss_part.p;
    u.nloss = (int64_t)nloss;
    u.loss_scale = 1.0 / (double)(n * MlpDims::OUT);
    u.loss_acc = loss_dev.p;
    const int64_t wgrid = slab_grid(ga.nslab) + (int64_t)ga.nblock * kBiasJobs;
    hipLaunchKernelGGL(k_mlp_train, dim3(blocks), dim3(kTrainThreads), 0, stream, a);
    hipLaunchKernelGGL(k_mlp_wgrad, dim3((unsigned)wgrid), dim3(64), 0, stream, ga);
    const dim3 ug(kWeightBlocks + kBiasBlocks + 1);
    if (adam) {
        ++t_adam;
        u.lr = lr;
        u.c1 = 1.f - std::pow(0.9f, (float)t_adam);
        u.c2 = 1.f - std::pow(0.999f, (float)t_adam);
        hipLaunchKernelGGL(k_mlp_update<true>, ug, dim3(256), 0, stream, u);
    } else {
        hipLaunchKernelGGL(k_mlp_update<false>, ug, dim3(256), 0, stream, u);
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
    batch_pass(X.p, Y.p, n, 0, 0, false, 0.f);
    std::vector<float> part((n + 15) / 16);
    PB_HIP(hipMemcpyAsync(part.data(), loss_part.p, part.size() * 4, hipMemcpyDeviceToHost, stream));
    PB_HIP(hipStreamSynchronize(stream));
    double loss = 0;
    for (float v : part) loss += v;
    if (grads_host) get_params(grads_host, true);
    return loss / (double)(n * MlpDims::OUT);
}

}  // namespace pb
