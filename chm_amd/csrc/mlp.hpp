// Per-face network of the learned warm start (mlp.hip).
#pragma once

#include "kernels.hpp"

namespace pb {

struct MlpDims {
    static constexpr int IN = 16;   // features of a face and its three neighbours
    static constexpr int H = 128;   // hidden width (three hidden layers)
    static constexpr int OUT = 11;  // 10 layer concentrations + deposition flux
    static constexpr int OUTP = 16; // output padded to one MFMA tile
    static int din(int l);
    static int dout(int l);
};

class Mlp {
  public:
    Mlp(int device, uint64_t seed);
    ~Mlp();
    // X: [n x IN] f32, Y: [n x OUT] f32 device arrays (raw units; normalised inside)
    double train(const float* X, const float* Y, int64_t n, int epochs, int batch, float lr, uint64_t seed);
    // inference: the fused one-launch kernel, or layer by layer through a GEMM (a check of the
    // fused one: the two agree bit for bit)
    void predict(const float* X, float* Y, int64_t n, hipStream_t s) {
        if (n > 0) predict_fused(X, Y, n, s);
    }
    void predict_fused(const float* X, float* Y, int64_t n, hipStream_t s);
    void predict_layers(const float* X, float* Y, int64_t n, hipStream_t s);
    double gradients(const float* Xh, const float* Yh, int64_t n, float* grads_host);  // MSE gradients, host arrays
    static int64_t param_count();
    void get_params(float* host, bool grads);
    void set_params(const float* host);
    void set_normalization(const float* host);  // x_mean[IN], x_std[IN], y_mean[OUT], y_std[OUT]

    int device = 0;
    hipStream_t stream = nullptr;
    int max_blocks = 256;  // workgroups of the fused kernels (one per CU)

  private:
    void ensure(int64_t n);
    void forward_prepared(int64_t n, hipStream_t s);
    // gradients of one batch (total > 0: rows sampled from total by key), then an Adam step or
    // the gradients into gW / gb; adds the batch's mean squared error to loss_dev
    void batch_pass(const float* X, const float* Y, int64_t n, int64_t total, uint64_t key, bool adam, float lr);
    const float* xmu() const;
    const float* xsd() const;
    const float* ymu() const;
    const float* ysd() const;

    DevBuf<float> W[4], bvec[4], gW[4], gb[4], mW[4], vW[4], mb[4], vb[4];
    DevBuf<uint16_t> Wb[4], WbT[4];  // BF16 weights [dout x din], and transposed
    DevBuf<float> norm;
    int64_t cap = 0;
    DevBuf<uint16_t> Xb, Ab[3];  // workspace of the layer-by-layer forward
    DevBuf<float> Yp;
    DevBuf<uint16_t> tiles;    // a batch's activations and gradients by 64-sample tile
    DevBuf<float> slab;        // its weight gradients, one slab per row range
    DevBuf<float> bias_part;   // its bias gradients, one row per row block
    DevBuf<float> loss_part;   // summed squared error per 16 rows
    DevBuf<double> loss_dev;   // the epoch's summed batch losses
    int64_t t_adam = 0;
};

}  // namespace pb
