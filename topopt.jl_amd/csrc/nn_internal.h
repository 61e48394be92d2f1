// Internal declarations of the learned warm-start network kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tohip {

// One stride-1 zero-padded 3D convolution over NDHWC BF16 tensors.
struct ConvDesc {
    int B;             // batch
    int D, H, W;       // input spatial size
    int OD, OH, OW;    // output spatial size (D + 2 pd - kd + 1, ...)
    int Cin, Cin32;    // input channels (multiple of 8); Cin rounded up to 32
    int Cout;          // output channels
    int kd, kh, kw;    // kernel size
    int pd, ph, pw;    // zero padding
    int out_cstride;   // channels of the output tensor (writes into a concat view)
    int out_coff;      // channel offset of the view
    int out_cvalid;    // FP32 output: channels stored
    int act;           // 0 identity, 1 SiLU, 2 times silu'(Z) (Z read, not written)
};

hipError_t launch_conv_fwd(const ConvDesc& c, const uint16_t* X, const uint16_t* W,
                           const float* bias, uint16_t* Y, uint16_t* Z, float* Yf,
                           hipStream_t s);
// dW [Cout][taps][Cin], db [Cout]; part: conv_bwd_w_floats(c) floats of scratch,
// 16-byte aligned like X and dY.  Cubic kernels up to 3, Cout a divisor of 256.
size_t conv_bwd_w_floats(const ConvDesc& c);
hipError_t launch_conv_bwd_w(const ConvDesc& c, const uint16_t* X, const uint16_t* dY,
                             float* part, float* dW, float* db, hipStream_t s);
// Layers whose FP32 weights go to BF16, in one launch.
struct ConvWeights {
    static constexpr int kMax = 16;
    struct Layer {
        int Cout, T, Cin, Cin32, Cout32;
        const float* w;
        uint16_t *wf, *wt;
    } layer[kMax];
    int count;
};
hipError_t launch_weights_to_bf16(const ConvWeights& t, hipStream_t s);
// Samples of the data set into a batch (16-byte words and floats a sample).
struct NNBatch {
    static constexpr int kMax = 64;
    int idx[kMax];
    int count;
};
hipError_t launch_nn_gather(const NNBatch& t, int64_t nf, const void* src_f, void* dst_f, int64_t nu,
                            const float* src_u, float* dst_u, hipStream_t s);
hipError_t launch_silu_bwd(int64_t n, const uint16_t* dA, const uint16_t* Z, uint16_t* dZ,
                           hipStream_t s);
hipError_t launch_avgpool_fwd(int B, int D, int H, int W, int C, const uint16_t* in, int in_cs,
                              int in_co, uint16_t* out, hipStream_t s);
hipError_t launch_skip_bwd(int B, int D, int H, int W, int C, const uint16_t* dpool,
                           const uint16_t* dskip, int cs, int co, const uint16_t* Z, uint16_t* dZ,
                           hipStream_t s);
hipError_t launch_upsample_fwd(int B, int D, int H, int W, int C, const uint16_t* in,
                               uint16_t* out, int out_cs, int out_co, hipStream_t s);
hipError_t launch_upsample_bwd(int B, int D, int H, int W, int C, const uint16_t* dout,
                               int out_cs, int out_co, const uint16_t* Z, uint16_t* dZ,
                               hipStream_t s);

}  // namespace tohip
