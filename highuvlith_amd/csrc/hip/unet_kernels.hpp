// Launchers of the U-Net kernels (unet_kernels.hip): BF16 storage, FP32
// accumulation on the matrix cores (v_mfma_f32_32x32x16_bf16).  Activations
// are NHWC; conv weights [Cout][3][3][Cin].  All pointers are device
// pointers; every launcher is asynchronous on `s`.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace huvk {

typedef uint16_t bf16_t;  // raw BF16 bits

// A convolution's input: C channels of X (N, H, W), after Cu channels of the
// half-resolution U (N, H/2, W/2) read by nearest 2x upsampling when Cu > 0 (the
// decoder's concatenation, which is not written out where conv3x3_by_rows).  C, Cu
// multiples of 8.
struct ConvIn {
  const bf16_t* X = nullptr;
  int C = 0;
  const bf16_t* U = nullptr;
  int Cu = 0;
  __device__ __forceinline__ const bf16_t* at(int n, int y, int x, int H, int W, int c) const {
    if (c < Cu) return U + (((size_t)n * (H / 2) + y / 2) * (W / 2) + x / 2) * Cu + c;
    return X + (((size_t)n * H + y) * W + x) * C + (c - Cu);
  }
};
// A convolution's output: Y, with Cout - Cu channels.  mask (optional, Y's shape): Y
// zeroed where mask <= 0.  pool (optional): the 2 x 2 maximum of Y, (N, H/2, W/2, Cout).
// Cu > 0 (neither mask nor pool; only where conv3x3_by_rows): the first Cu channels go
// to dU (N, H/2, W/2, Cu) instead, summed over 2 x 2 and zero where U, of that shape, is
// not positive: the gradient of the upsampled half of a concatenation.  head (only where
// conv3x3_by_rows, Cout <= 64): head_b[0] + sum over the channels of Y head_w, FP32 per
// pixel; Y may then be null.
struct ConvOut {
  bf16_t* Y = nullptr;
  const bf16_t* mask = nullptr;
  bf16_t* pool = nullptr;
  bf16_t* dU = nullptr;
  const bf16_t* U = nullptr;
  int Cu = 0;
  float* head = nullptr;
  const float *head_w = nullptr, *head_b = nullptr;
};
// out = act(conv3x3(in) + bias), pad 1, stride 1, Cout channels (a multiple of 8).
// relu: 0/1.  bias may be NULL.  Cu > 0 only where conv3x3_by_rows.
hipError_t launch_conv3x3_fwd(const ConvIn& in, int N, int H, int W, const bf16_t* Wt,
                              const float* bias, int Cout, int relu, const ConvOut& out,
                              hipStream_t s);
bool conv3x3_by_rows(const ConvIn& in, int N, int H, int W, int Cout);
// Wr[ci][t][co] = W[co][8 - t][ci] (the kernel of the data gradient).
hipError_t launch_conv_weight_rot(const bf16_t* Wt, int Cout, int Cin, bf16_t* Wr, hipStream_t s);
// XT[n][c][y][x] = X[n][y][x][c] (H W a multiple of 64, C of 8; likewise below).
hipError_t launch_nhwc_to_nchw(const bf16_t* X, int N, int H, int W, int C, bf16_t* XT,
                               hipStream_t s);
// Split-K weight gradient partials: part[split][co][t][ci] (FP32), W % 16 == 0,
// Cin % 8 == 0; rows (n, y) are split into `splits` contiguous ranges.
hipError_t launch_conv3x3_wgrad(const bf16_t* dYT, const bf16_t* XT, int N, int H, int W,
                                int Cin, int Cout, int splits, float* part, hipStream_t s);
// Weight and bias gradient partials straight from the NHWC tensors dY (ReLU
// already applied) and `in`: part[split] = [co][t][ci] then [co]; W % 64 == 0, Cout
// a multiple of 8, Cu of 32; the rows of the 64-pixel column strips are split into
// `splits` contiguous ranges (wgrad_nhwc_splits: as many as fill the card).
int wgrad_nhwc_splits(int N, int H, int W, int Cin, int Cout);
hipError_t launch_conv3x3_wgrad_nhwc(const bf16_t* dY, const ConvIn& in, int N, int H, int W,
                                     int Cout, int splits, float* part, hipStream_t s);
// out[i] = sum_s part[s][i] (fixed order), i < count.
hipError_t launch_sum_splits(const float* part, int splits, int64_t count, float* out,
                             hipStream_t s);
// db[c] = sum over n, pixels of dYT[n][c][.]  (NCHW): `splits` chunk
// partials in part (splits x C floats), then summed in a fixed order.
hipError_t launch_channel_sum(const bf16_t* dYT, int N, int HW, int C, float* part, int splits,
                              float* db, hipStream_t s);
// 2 x 2 max pooling (H, W even).
hipError_t launch_maxpool_fwd(const bf16_t* X, int N, int H, int W, int C, bf16_t* Y,
                              hipStream_t s);
// Gradient of an encoder output X (N, H, W, C): dP of its pooled map to the first
// maximum of each window, plus channels Cu .. of dcat, zero where X <= 0.
hipError_t launch_skip_pool_bwd(const bf16_t* X, const bf16_t* dP, const bf16_t* dcat, int Cu,
                                int N, int H, int W, int C, bf16_t* dX, hipStream_t s);
// cat[n][y][x] = [nearest-2x(U)[n][y][x][0..Cu), S[n][y][x][0..Cs)] at (H, W);
// U is (H/2, W/2).  Backward of the first part: dU = sum of the 4 children of
// dcat, zero where U <= 0.
hipError_t launch_upcat_fwd(const bf16_t* U, int Cu, const bf16_t* S, int Cs, int N, int H,
                            int W, bf16_t* cat, hipStream_t s);
hipError_t launch_upcat_bwd_u(const bf16_t* dcat, int Cu, int Cs, int N, int H, int W,
                              const bf16_t* U, bf16_t* dU, hipStream_t s);
// out[p] = sum_c Y[p][c] w[c] + b (FP32); C in {16, 32, 64}.
hipError_t launch_head_fwd(const bf16_t* Y, int64_t P, int C, const float* w, const float* b,
                           float* out, hipStream_t s);
// dY[p][c] = dout[p] w[c] where Y > 0, else 0; partial sums for dw (C per block)
// and db.
hipError_t launch_head_bwd(const bf16_t* Y, const float* dout, int64_t P, int C, const float* w,
                           bf16_t* dY, float* part, int nblk, hipStream_t s);
// loss partials (FP64) and dout = 2 (out - target) / P.
hipError_t launch_mse(const float* out, const float* target, int64_t P, float* dout,
                      double* part, int nblk, hipStream_t s);
// X8[n][y][x][0..8) = (in[n][y][x], 0, ..., 0) as BF16.
hipError_t launch_pack_input(const float* in, int64_t P, bf16_t* X8, hipStream_t s);
// Adam on the FP32 master parameters; BF16 copies refreshed for conv weights.
hipError_t launch_adam(float* p, const float* g, float* m, float* v, int64_t count, float lr,
                       float b1, float b2, float eps, float c1, float c2, hipStream_t s);
hipError_t launch_to_bf16(const float* x, int64_t count, bf16_t* y, hipStream_t s);

}  // namespace huvk
