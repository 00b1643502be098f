// HIP kernels of the U-Net warm start (gfx950): BF16 activations and
// weights, FP32 accumulation on the matrix cores.
//
// 3x3 convolutions are implicit GEMMs on v_mfma_f32_32x32x16_bf16
// (D[32 x 32] += A[32 x 16] B[16 x 32]; lane l supplies A row l % 32 and
// B column l % 32 for k in 8 (l / 32) .. 8 (l / 32) + 7, and holds
// D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32] in accumulator r):
//   forward:  rows = output pixels, columns = output channels, k = (tap, ci);
//             NHWC activations and [co][tap][ci] weights give each lane's
//             8 consecutive k as one 16-byte load.
//   data gradient: the forward kernel on the ReLU-masked output gradient
//             with the rotated, transposed weights.
//   weight gradient: rows = output channels, columns = input channels of
//             one tap, k = pixels (16 consecutive x of one row), read
//             from LDS copies of the NHWC tensors by transposing reads (rows a
//             multiple of 64 wide) or from NCHW copies (narrower rows); the +-1
//             column shift of a tap is a 2-byte funnel shift of aligned
//             words.  Split-K partials are summed in a fixed order.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "unet_kernels.hpp"

namespace huvk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)0x7fc0;  // NaN
  u += 0x7fffu + ((u >> 16) & 1u);                              // round to nearest even
  return (bf16_t)(u >> 16);
}

// Two values rounded to nearest even, the first in the low half (one instruction).
__device__ __forceinline__ uint32_t f2bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

__device__ __forceinline__ bf16x8 ld8(const bf16_t* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}
__device__ __forceinline__ bf16x8 zero8() { return __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0)); }

// Eight BF16 values as one 16-byte word.
union B8 {
  uint4 u;
  bf16_t h[8];
};

// Four as one 8-byte word.
union B4 {
  uint2 u;
  bf16_t h[4];
};

// The maximum of four, channel by channel, keeping the winner's bits.
__device__ __forceinline__ B8 max4(const B8& v0, const B8& v1, const B8& v2, const B8& v3) {
  B8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    bf16_t m = v0.h[e];
    if (bf2f(v1.h[e]) > bf2f(m)) m = v1.h[e];
    if (bf2f(v2.h[e]) > bf2f(m)) m = v2.h[e];
    if (bf2f(v3.h[e]) > bf2f(m)) m = v3.h[e];
    o.h[e] = m;
  }
  return o;
}

// The sum of four, channel by channel, zero where u (a ReLU's output) is not positive.
__device__ __forceinline__ B8 sum4_masked(const B8& a0, const B8& a1, const B8& a2, const B8& a3,
                                          const B8& u) {
  B8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bf16_t sum = f2bf((bf2f(a0.h[e]) + bf2f(a1.h[e])) + (bf2f(a2.h[e]) + bf2f(a3.h[e])));
    o.h[e] = bf2f(u.h[e]) <= 0.f ? (bf16_t)0 : sum;
  }
  return o;
}

// ---------------------------------------------------------------------------
// Forward 3x3 convolution.  Work-group = 4 waves along pixels; each wave
// computes BM x BN blocks of 32 pixels x 32 output channels.  The operands
// of step s + 1 are loaded before the products of step s are issued.  The products are
// weights x pixels: a lane has four consecutive channels of its pixel at a time, so the
// output and the ReLU mask (which two-byte accesses made a third of a masked layer's
// epilogue) go in 8-byte words.  One source: a choice between two at every load cost all
// layers a tenth of their time, and the concatenation a third of its own, where writing
// it once takes 5 us.  Bound by the latency of its loads, each operand read anew for
// every tap: a gradient of 2 fields of 96 x 32, base 64, takes 766 us (with pixels x
// weights 821, and the choice of sources 854), of 8 of 96 x 96, base 32, 603 (651).
// ---------------------------------------------------------------------------
template <int BM, int BN>
__global__ __launch_bounds__(256) void k_conv3x3_fwd(const bf16_t* __restrict__ X, int N, int H,
                                                     int W, int Cin,
                                                     const bf16_t* __restrict__ Wt,
                                                     const float* __restrict__ bias, int Cout,
                                                     int relu, const bf16_t* __restrict__ mask,
                                                     bf16_t* __restrict__ Y) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, li = lane & 31;
  const int64_t NP = (int64_t)N * H * W;
  const int64_t pbase = ((int64_t)blockIdx.x * 4 + wave) * (32 * BM);
  const int cobase = blockIdx.y * 32 * BN;
  if (pbase >= NP) return;  // whole wave; no barriers in this kernel
  const int CB = Cin / 8, KB = 9 * CB, steps = (KB + 1) / 2;
  const int HW = H * W;
  int pn[BM], py[BM], px[BM];
  bool pv[BM];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm) {
    const int64_t p = pbase + 32 * bm + li;
    pv[bm] = p < NP;
    const int64_t pp = pv[bm] ? p : 0;
    pn[bm] = (int)(pp / HW);
    const int rem = (int)(pp - (int64_t)pn[bm] * HW);
    py[bm] = rem / W;
    px[bm] = rem - py[bm] * W;
  }
  int co[BN];
#pragma unroll
  for (int bn = 0; bn < BN; ++bn) co[bn] = cobase + 32 * bn + li;

  auto load = [&](int s, bf16x8* a, bf16x8* b) {
    const int kb = 2 * s + half;
    const bool kv = kb < KB;
    const int tap = kv ? kb / CB : 0, cb = kv ? kb - (kb / CB) * CB : 0;
    const int dy = tap / 3 - 1, dx = tap - (tap / 3) * 3 - 1;
#pragma unroll
    for (int bm = 0; bm < BM; ++bm) {
      const int yy = py[bm] + dy, xx = px[bm] + dx;
      const bool v = kv && pv[bm] && yy >= 0 && yy < H && xx >= 0 && xx < W;
      a[bm] = v ? ld8(X + (((int64_t)pn[bm] * H + yy) * W + xx) * Cin + cb * 8) : zero8();
    }
#pragma unroll
    for (int bn = 0; bn < BN; ++bn) {
      const bool v = kv && co[bn] < Cout;
      b[bn] = v ? ld8(Wt + ((int64_t)co[bn] * 9 + tap) * Cin + cb * 8) : zero8();
    }
  };

  f32x16 acc[BM][BN];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm)
#pragma unroll
    for (int bn = 0; bn < BN; ++bn)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bm][bn][r] = 0.f;
  bf16x8 a[BM], b[BN], an[BM], bnx[BN];
  load(0, a, b);
  for (int s = 0; s < steps; ++s) {
    if (s + 1 < steps) load(s + 1, an, bnx);
#pragma unroll
    for (int bm = 0; bm < BM; ++bm)
#pragma unroll
      for (int bn = 0; bn < BN; ++bn)
        acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[bn], a[bm], acc[bm][bn], 0, 0, 0);
#pragma unroll
    for (int bm = 0; bm < BM; ++bm) a[bm] = an[bm];
#pragma unroll
    for (int bn = 0; bn < BN; ++bn) b[bn] = bnx[bn];
  }
  // a lane's pixel of block bm, four channels of block bn at a time
#pragma unroll
  for (int bn = 0; bn < BN; ++bn)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = cobase + 32 * bn + 8 * q + 4 * half;
      if (c >= Cout) continue;
      float bv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[e] = bias ? bias[c + e] : 0.f;
#pragma unroll
      for (int bm = 0; bm < BM; ++bm) {
        const int64_t p = pbase + 32 * bm + li;
        if (p >= NP) continue;
        B4 v, m;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float f = acc[bm][bn][4 * q + e] + bv[e];
          if (relu) f = fmaxf(f, 0.f);
          v.h[e] = f2bf(f);
        }
        if (mask) {
          m.u = *reinterpret_cast<const uint2*>(mask + p * Cout + c);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (bf2f(m.h[e]) <= 0.f) v.h[e] = 0;
        }
        *reinterpret_cast<uint2*>(Y + p * Cout + c) = v.u;
      }
    }
}

// ---------------------------------------------------------------------------
// Forward 3x3 convolution of the first layer's 8 input channels, input and weights staged
// in LDS.  Work-group = 4 waves over an output tile of TH = 2 BM rows x 64 columns of one
// image; wave w takes columns x0 + 32 (w % 2) .. + 31 of the BM rows from y0 + BM (w / 2),
// and BN blocks of 32 output channels, so one weight fragment feeds BM products.  The
// (TH + 2) x (64 + 2) x 8 halo and the 9 x 8 weights of the 32 BN output channels are
// loaded once (zero outside the image and beyond Cout) and read by all four waves from
// LDS; A = 32 pixels x 16 k per MFMA step, two taps of 8 channels.  The output leaves
// through LDS in 16-byte runs of channels.  Bound by the writes: 32 fields of 512^2, 32
// channels, 184 us.  Needs W % 64 == 0 and H % TH == 0.
// ---------------------------------------------------------------------------
template <int BM, int BN>
__global__ __launch_bounds__(256) void k_conv3x3_fwd_lds(const bf16_t* __restrict__ X, int H, int W,
                                                         const bf16_t* __restrict__ Wt,
                                                         const float* __restrict__ bias, int Cout,
                                                         int relu, bf16_t* __restrict__ Y) {
  constexpr int CC = 8, KB = 9, STEPS = (KB + 1) / 2;  // channels, taps, products
  constexpr int TH = 2 * BM, TW = 64, HR = TH + 2, HC = TW + 2;
  constexpr int PS = CC + 8;  // pixel stride in the tile (bf16), spreads the LDS banks
  constexpr int WS = KB * CC + 8;  // output-channel stride of the staged weights (bf16)
  constexpr int OS = 32 * BN + 8;  // pixel stride of the staged output (bf16)
  constexpr int IN_LDS = HR * HC * PS, OUT_LDS = TH * TW * OS;
  __shared__ __attribute__((aligned(16))) bf16_t tile[IN_LDS > OUT_LDS ? IN_LDS : OUT_LDS];
  __shared__ __attribute__((aligned(16))) bf16_t wts[32 * BN * WS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, li = lane & 31;
  const int tilesX = W / TW, tilesY = H / TH;
  const int x0 = (int)blockIdx.x % tilesX * TW, y0 = (int)blockIdx.x / tilesX % tilesY * TH;
  const int n = (int)blockIdx.x / (tilesX * tilesY);
  const int cobase = blockIdx.y * 32 * BN;
  const int px = 32 * (wave & 1) + li;  // this lane's A row (pixel column) in the tile
  const int py0 = BM * (wave >> 1);     // first output row of the wave in the tile
  constexpr int HALO = HR * HC, HIT = (HALO + 255) / 256;
  constexpr int WGT = 32 * BN * KB, WIT = (WGT + 255) / 256;
  f32x16 acc[BM][BN];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm)
#pragma unroll
    for (int bn = 0; bn < BN; ++bn)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bm][bn][r] = 0.f;
  // Every load is issued before the first LDS store, so their latencies overlap: buffer
  // loads with 32-bit offsets into the image, where a pixel outside it, and an output
  // channel beyond Cout, gets an offset past the end, which reads zero.
  uint4 hv[HIT], wv[WIT];
  const int image = H * W * CC;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(X + (size_t)n * image), (short)0, image * (int)sizeof(bf16_t), 0x00020000);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16_t*>(Wt), (short)0, Cout * KB * CC * (int)sizeof(bf16_t), 0x00020000);
#pragma unroll
  for (int k = 0; k < HIT; ++k) {
    const int i = threadIdx.x + 256 * k;
    const int yy = y0 - 1 + i / HC, xx = x0 - 1 + i % HC;
    const bool v = i < HALO && yy >= 0 && yy < H && xx >= 0 && xx < W;
    const int off = (yy * W + xx) * CC * (int)sizeof(bf16_t);
    hv[k] = __builtin_bit_cast(uint4,
                               __builtin_amdgcn_raw_buffer_load_b128(xr, v ? off : -1, 0, 0));
  }
#pragma unroll
  for (int k = 0; k < WIT; ++k) {
    const int i = threadIdx.x + 256 * k;
    const int tap = i % KB, col = i / KB, c = cobase + col;
    const bool v = i < WGT && c < Cout;
    const int off = (c * KB + tap) * CC * (int)sizeof(bf16_t);
    wv[k] = __builtin_bit_cast(uint4,
                               __builtin_amdgcn_raw_buffer_load_b128(wr, v ? off : -1, 0, 0));
  }
#pragma unroll
  for (int k = 0; k < HIT; ++k) {
    const int i = threadIdx.x + 256 * k;
    if (i < HALO) *reinterpret_cast<uint4*>(tile + i * PS) = hv[k];
  }
#pragma unroll
  for (int k = 0; k < WIT; ++k) {
    const int i = threadIdx.x + 256 * k;
    if (i < WGT) *reinterpret_cast<uint4*>(wts + (i / KB) * WS + CC * (i % KB)) = wv[k];
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < STEPS; ++s) {
    const int kb = 2 * s + half;
    const bool kv = kb < KB;
    const int tap = kv ? kb : 0;
    const int dy = tap / 3, dx = tap % 3;
    bf16x8 bw[BN];
#pragma unroll
    for (int bn = 0; bn < BN; ++bn) {
      const bf16x8 w = ld8(wts + (32 * bn + li) * WS + CC * tap);
      bw[bn] = kv ? w : zero8();
    }
#pragma unroll
    for (int bm = 0; bm < BM; ++bm) {
      const bf16x8 a0 = ld8(tile + ((py0 + bm + dy) * HC + px + dx) * PS);
      const bf16x8 a = kv ? a0 : zero8();
#pragma unroll
      for (int bn = 0; bn < BN; ++bn)
        acc[bm][bn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, bw[bn], acc[bm][bn], 0, 0, 0);
    }
  }
  __syncthreads();  // the tile has been read by every wave
#pragma unroll
  for (int bn = 0; bn < BN; ++bn) {
    const int co = cobase + 32 * bn + li;
    const float bv = bias && co < Cout ? bias[co] : 0.f;
#pragma unroll
    for (int bm = 0; bm < BM; ++bm)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r / 4) + 4 * half + (r % 4);
        float v = acc[bm][bn][r] + bv;
        if (relu) v = fmaxf(v, 0.f);
        tile[((py0 + bm) * TW + 32 * (wave & 1) + i) * OS + 32 * bn + li] = f2bf(v);
      }
  }
  __syncthreads();
  constexpr int G8 = 4 * BN;  // 8-channel groups of the block
  for (int i = threadIdx.x; i < TH * TW * G8; i += 256) {
    const int g = i % G8, q = i / G8, c = cobase + 8 * g;
    if (c >= Cout) continue;
    const size_t at = (((size_t)n * H + y0 + q / TW) * W + x0 + q % TW) * Cout + c;
    *reinterpret_cast<uint4*>(Y + at) = *reinterpret_cast<const uint4*>(tile + q * OS + 8 * g);
  }
}

// ---------------------------------------------------------------------------
// Forward 3x3 convolution with channels in chunks of CC = 16 or 32, staged in LDS.
// Work-group = 4 waves over a tile of TH rows x 64 columns of one image and 32 COW
// output channels: wave w takes one block of 32 output channels, 32 columns and BM
// rows.  A chunk's weights of the block (9 taps x CC channels) stay in the wave's
// registers; each input row of the tile is read from LDS once per column shift and
// feeds the output rows above, at and below it, so a chunk costs (BM + 2) + 3 operand
// reads of 16 bytes per 3 BM products.  The sums run over (chunk, tap, channel) for
// every output, whatever BM.
//
// The products are weights x pixels: a lane ends up with four consecutive channels
// of one pixel at a time, which leave through LDS in 16-byte runs, where the ReLU
// mask of the layer below (mask: dX zeroed where that layer's output is not positive)
// and the 2 x 2 maximum (pool) cost no pass of their own; the decoder's input is
// read from its two sources (the half-resolution map and the skip), so the
// concatenation is never written.
//
// What bounds it: at 64 and more output channels the matrix cores, 1030 TFLOP/s over
// the layers of a forward pass (a large library product: 1190); at 32 the copies of
// halo and weights, 0.7 of the card's copy rate.  Blocks of 2 rows x 32 columns x 64
// channels per wave, with both operands read anew for every tap and copied through
// registers, took 2557 and 1262 us of a forward pass of 32 fields of 512^2 (4 levels,
// base 32), now 1874 and 1246: 3790 -> 3110 us altogether, and 4245 -> 3670 for the
// loss gradient of 8 of them.  Needs W % 64 == 0 and H % TH == 0.
// ---------------------------------------------------------------------------
template <int BM, int COW, int CC>
__global__ __launch_bounds__(256, 2) void k_conv3x3_rows(ConvIn in, int N, int H, int W,
                                                         const bf16_t* __restrict__ Wt,
                                                         const float* __restrict__ bias, int Cout,
                                                         int relu, ConvOut out) {
  constexpr int TH = 2 * BM / COW, TW = 64, HR = TH + 2, HC = TW + 2;
  constexpr int CB = CC / 8, S = CC / 16;  // 16-byte pieces of a pixel; products per tap
  constexpr int OS = 32 * COW + 8;         // pixel stride of the staged output
  constexpr int IN_RUNS = (HR * HC * CB + 63) / 64;  // 64 pieces a wave copies at once
  constexpr int W_RUNS = 32 * COW * 9 * CB / 64;
  constexpr int IN_LDS = IN_RUNS * 512, W_LDS = W_RUNS * 512, OUT_LDS = TH * TW * OS;
  __shared__ __attribute__((aligned(16)))
  bf16_t lds[IN_LDS + W_LDS > OUT_LDS ? IN_LDS + W_LDS : OUT_LDS];
  const int Cin = in.Cu + in.C;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wv = __builtin_amdgcn_readfirstlane(wave);
  const int half = lane >> 5, li = lane & 31;
  const int cw = wave % COW, col = wave / COW % 2, rg = wave / (2 * COW);
  const int tilesX = W / TW, tilesY = H / TH;
  const int tiles = N * tilesY * tilesX, cogroups = (Cout + 32 * COW - 1) / (32 * COW);
  // The channel groups of a tile, and tiles with a common edge, run on one XCD
  // (work-groups are dealt to the 8 XCDs in turn) where the tiles can be dealt out.
  int t = blockIdx.x / cogroups, cg = blockIdx.x % cogroups;
  if (tiles % 8 == 0) {
    const int j = blockIdx.x / 8;
    cg = j % cogroups;
    t = (int)blockIdx.x % 8 * (tiles / 8) + j / cogroups;
  }
  const int x0 = t % tilesX * TW, y0 = t / tilesX % tilesY * TH, n = t / (tilesX * tilesY);
  const int cobase = cg * 32 * COW;
  // The 16-byte pieces of a pixel (or of one tap of an output channel) are permuted by
  // its column (channel), so that the reads of consecutive lanes do not meet in a bank.
  auto swz = [](int c) { return CB == 4 ? (c >> 1) & 3 : (c >> 2) & 1; };
  int abase[3][S], wbase[S];  // this lane's operand pieces at the wave's first row, and tap 0
#pragma unroll
  for (int q = 0; q < S; ++q) {
#pragma unroll
    for (int dx = 0; dx < 3; ++dx) {
      const int c = 32 * col + li + dx;
      abase[dx][q] = (rg * BM * HC + c) * CC + 8 * ((2 * q + half) ^ swz(c));
    }
    wbase[q] = IN_LDS + (32 * cw + li) * CC + 8 * ((2 * q + half) ^ swz(li));
  }
  f32x16 acc[BM];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[bm][r] = 0.f;
  for (int c0 = 0; c0 < Cin; c0 += CC) {
    // The chunk goes from memory to LDS without registers, 64 pieces per wave and copy,
    // by buffer loads with 32-bit offsets into the image (or its half-resolution part):
    // a pixel outside it, and an output channel beyond Cout, gets an offset past the
    // end, which reads zero.
    const bool up = c0 < in.Cu;
    const int sh = up ? 1 : 0, cs = up ? in.Cu : in.C, ws = W >> sh;
    const int image = (H >> sh) * ws * cs;
    const bf16_t* src = (up ? in.U : in.X) + (size_t)n * image;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(src), (short)0, image * (int)sizeof(bf16_t), 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(Wt), (short)0, Cout * 9 * Cin * (int)sizeof(bf16_t), 0x00020000);
    const int soff = (up ? c0 : c0 - in.Cu) * (int)sizeof(bf16_t);
    __syncthreads();  // the previous chunk has been consumed
#pragma unroll 1
    for (int k = wv; k < W_RUNS; k += 4) {
      const int i = 64 * k + lane, c = i / CB % (32 * COW), tap = i / (CB * 32 * COW);
      const int cb = i % CB ^ swz(c);
      const int off = (((cobase + c) * 9 + tap) * Cin + c0 + 8 * cb) * (int)sizeof(bf16_t);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(lds + IN_LDS + 512 * k), 16,
                                               cobase + c < Cout ? off : -1, 0, 0, 0);
    }
#pragma unroll 1
    for (int k = wv; k < IN_RUNS; k += 4) {
      const int i = 64 * k + lane, pix = i / CB, row = pix / HC, c = pix - row * HC;
      const int cb = i % CB ^ swz(c);
      const int yy = y0 - 1 + row, xx = x0 - 1 + c;
      const bool v = row < HR && yy >= 0 && yy < H && xx >= 0 && xx < W;
      const int off = (((yy >> sh) * ws + (xx >> sh)) * cs + 8 * cb) * (int)sizeof(bf16_t);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(lds + 512 * k), 16,
                                               v ? off + soff : -1, 0, 0, 0);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's copies have landed (vmcnt 0)
    __syncthreads();
    bf16x8 wf[9 * S];
#pragma unroll
    for (int k = 0; k < 9 * S; ++k) wf[k] = ld8(lds + wbase[k % S] + k / S * (32 * COW * CC));
    // units of one input row and column shift, the next one's operands being read
    // during this one's products (and no earlier: registers)
    bf16x8 a[S], an[S];
#pragma unroll
    for (int q = 0; q < S; ++q) a[q] = ld8(lds + abase[0][q]);
#pragma unroll
    for (int u = 0; u < 3 * (BM + 2); ++u) {
      const int rho = u / 3, dx = u % 3, rn = (u + 1) / 3, dn = (u + 1) % 3;
      if (rn < BM + 2) {
#pragma unroll
        for (int q = 0; q < S; ++q) an[q] = ld8(lds + abase[dn][q] + rn * (HC * CC));
      }
#pragma unroll
      for (int q = 0; q < S; ++q)
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) {
          const int bm = rho - dy;
          if (bm >= 0 && bm < BM)
            acc[bm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[(dy * 3 + dx) * S + q], a[q],
                                                              acc[bm], 0, 0, 0);
        }
#pragma unroll
      for (int q = 0; q < S; ++q) a[q] = an[q];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();  // the tile has been read by every wave
  int hb = half;
  asm volatile("" : "+v"(hb));  // the biases are not loaded before the products
  float bv[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int co = cobase + 32 * cw + 8 * (r / 4) + 4 * hb + (r % 4);
    bv[r] = bias && co < Cout ? bias[co] : 0.f;
  }
#pragma unroll
  for (int bm = 0; bm < BM; ++bm) {
    bf16_t* o = lds + ((rg * BM + bm) * TW + 32 * col + li) * OS + 32 * cw + 4 * half;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[bm][4 * q + e] + bv[4 * q + e];
        if (relu) v[e] = fmaxf(v[e], 0.f);
      }
      *reinterpret_cast<uint2*>(o + 8 * q) = make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
    }
  }
  __syncthreads();
  constexpr int G8 = 4 * COW;  // 8-channel groups of the block
  if (out.head) {
    // the 1 x 1 head on this block's channels, which are all there are
    for (int i = tid; i < TH * TW; i += 256) {
      float h = out.head_b[0];
      for (int c = 0; c < Cout; c += 8) {
        B8 v;
        v.u = *reinterpret_cast<const uint4*>(lds + i * OS + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) h += bf2f(v.h[e]) * out.head_w[c + e];
      }
      out.head[((size_t)n * H + y0 + i / TW) * W + x0 + i % TW] = h;
    }
    if (!out.Y) return;
  }
  const int Cu = out.Cu, Cy = Cout - Cu;
  for (int i = tid; i < TH * TW * G8; i += 256) {
    const int g = i % G8, q = i / G8, c = cobase + 8 * g;
    if (c >= Cout || c < Cu) continue;
    const size_t at = (((size_t)n * H + y0 + q / TW) * W + x0 + q % TW) * Cy + c - Cu;
    B8 v;
    v.u = *reinterpret_cast<const uint4*>(lds + q * OS + 8 * g);
    if (out.mask) {
      B8 m;
      m.u = *reinterpret_cast<const uint4*>(out.mask + at);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (bf2f(m.h[e]) <= 0.f) v.h[e] = 0;
    }
    *reinterpret_cast<uint4*>(out.Y + at) = v.u;
  }
  if (!out.pool && cobase >= Cu) return;
  for (int i = tid; i < TH * TW / 4 * G8; i += 256) {
    const int g = i % G8, q = i / G8, c = cobase + 8 * g;
    if (c >= Cout || (!out.pool && c >= Cu)) continue;
    const int yo = q / (TW / 2), xo = q % (TW / 2);
    const bf16_t* b = lds + (2 * yo * TW + 2 * xo) * OS + 8 * g;
    B8 v0, v1, v2, v3;
    v0.u = *reinterpret_cast<const uint4*>(b);
    v1.u = *reinterpret_cast<const uint4*>(b + OS);
    v2.u = *reinterpret_cast<const uint4*>(b + TW * OS);
    v3.u = *reinterpret_cast<const uint4*>(b + (TW + 1) * OS);
    const size_t p = ((size_t)n * (H / 2) + y0 / 2 + yo) * (W / 2) + x0 / 2 + xo;
    if (out.pool) {
      *reinterpret_cast<uint4*>(out.pool + p * Cout + c) = max4(v0, v1, v2, v3).u;
    } else {
      B8 u;
      u.u = *reinterpret_cast<const uint4*>(out.U + p * Cu + c);
      *reinterpret_cast<uint4*>(out.dU + p * Cu + c) = sum4_masked(v0, v1, v2, v3, u).u;
    }
  }
}

// Wr[ci][t][co] = W[co][8 - t][ci].
__global__ void k_conv_weight_rot(const bf16_t* __restrict__ Wt, int Cout, int Cin,
                                  bf16_t* __restrict__ Wr) {
  const int64_t total = (int64_t)Cout * 9 * Cin;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int ci = (int)(i % Cin);
    const int t = (int)((i / Cin) % 9);
    const int co = (int)(i / (9 * (int64_t)Cin));
    Wr[((int64_t)ci * 9 + (8 - t)) * Cout + co] = Wt[i];
  }
}

// ---------------------------------------------------------------------------
// NHWC -> NCHW through a 64-pixel x 32-channel LDS tile (HW % 64 == 0, C % 8
// == 0): each thread reads one 16-byte run of 8 channels of a pixel and
// writes one 16-byte run of 8 pixels of a channel.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_transpose_t(const bf16_t* __restrict__ X, int N, int HW,
                                                     int C, bf16_t* __restrict__ out) {
  constexpr int TP = 64, TC = 32, LP = TP + 8;  // padded pixel stride (16-byte aligned rows)
  __shared__ __align__(16) bf16_t tile[TC][LP];
  const int64_t p0 = (int64_t)blockIdx.x * TP;  // flat pixel over N * HW
  const int c0 = blockIdx.y * TC;
  {
    const int px = threadIdx.x >> 2, ch = 8 * (threadIdx.x & 3);
    if (c0 + ch < C) {
      B8 v;
      v.u = *reinterpret_cast<const uint4*>(X + (p0 + px) * C + c0 + ch);
#pragma unroll
      for (int k = 0; k < 8; ++k) tile[ch + k][px] = v.h[k];
    }
  }
  __syncthreads();
  const int n = (int)(p0 / HW);
  const int hw0 = (int)(p0 - (int64_t)n * HW);
  const int c = threadIdx.x >> 3, pc = 8 * (threadIdx.x & 7);
  if (c0 + c < C)
    *reinterpret_cast<uint4*>(out + ((int64_t)n * C + c0 + c) * HW + hw0 + pc) =
        *reinterpret_cast<const uint4*>(&tile[c][pc]);
}

// ---------------------------------------------------------------------------
// Weight gradient (split K over rows).  Grid x = co-block groups (BM blocks
// of 32) * ci blocks * 3 kernel rows kh, grid y = splits.  Each wave loads a
// 16-pixel segment of dY (per co block) and of the input row y + kh - 1 once
// and feeds all three column taps kw from it (the -1 / +1 shifts are 2-byte
// funnel shifts), i.e. 3 BM products per BM + 1 operand loads.  The 4 waves
// take interleaved rows of the split and are reduced through LDS in a fixed
// order, one output tile at a time.
// ---------------------------------------------------------------------------
template <int BM>
__global__ __launch_bounds__(256) void k_conv3x3_wgrad(const bf16_t* __restrict__ dYT,
                                                       const bf16_t* __restrict__ XT, int N,
                                                       int H, int W, int Cin, int Cout,
                                                       int rows_per_split,
                                                       float* __restrict__ part) {
  __shared__ float red[4][32][33];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5, li = lane & 31;
  const int ciblocks = (Cin + 31) / 32;
  const int tile = blockIdx.x;
  const int kh = tile % 3, rest = tile / 3;
  const int cib = rest % ciblocks, cog = rest / ciblocks;
  const int dy = kh - 1;
  const int split = blockIdx.y;
  const int rows = N * H;
  const int r0 = split * rows_per_split;
  const int r1 = min(rows, r0 + rows_per_split);
  int coA[BM];
  bool av[BM];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm) {
    coA[bm] = (cog * BM + bm) * 32 + li;
    av[bm] = coA[bm] < Cout;
  }
  const int ciB = cib * 32 + li;
  const bool bv = ciB < Cin;
  f32x16 acc[BM][3];
#pragma unroll
  for (int bm = 0; bm < BM; ++bm)
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[bm][k][r] = 0.f;
  for (int row = r0 + wave; row < r1; row += 4) {
    const int n = row / H, y = row - n * H;
    const int yy = y + dy;
    const bool rv = bv && yy >= 0 && yy < H;
    const bf16_t* arow[BM];
#pragma unroll
    for (int bm = 0; bm < BM; ++bm)
      arow[bm] = dYT + (((int64_t)n * Cout + (av[bm] ? coA[bm] : 0)) * H + y) * W;
    const bf16_t* brow = XT + (((int64_t)n * Cin + (bv ? ciB : 0)) * H + (rv ? yy : 0)) * W;
    // One 16-pixel segment: the dY rows (A), the input row (B) and its two
    // neighbouring words for the -1 / +1 column shifts.
    struct Seg {
      bf16x8 a[BM];
      uint4 w;
      uint32_t prev, next;
    };
    auto load = [&](int x0, Seg& g) {
      const int xs = x0 + 8 * half;
#pragma unroll
      for (int bm = 0; bm < BM; ++bm) g.a[bm] = av[bm] ? ld8(arow[bm] + xs) : zero8();
      g.w = make_uint4(0, 0, 0, 0);
      g.prev = 0u;
      g.next = 0u;
      if (rv) {
        g.w = *reinterpret_cast<const uint4*>(brow + xs);
        if (xs > 0) g.prev = *reinterpret_cast<const uint32_t*>(brow + xs - 2);
        if (xs + 8 < W) g.next = *reinterpret_cast<const uint32_t*>(brow + xs + 8);
      }
    };
    auto mma = [&](const Seg& g) {
      const uint4 w = g.w;
      // kw = 0: input column x - 1; kw = 1: x; kw = 2: x + 1
      const bf16x8 b0 = __builtin_bit_cast(
          bf16x8, make_uint4(__builtin_amdgcn_alignbit(w.x, g.prev, 16),
                             __builtin_amdgcn_alignbit(w.y, w.x, 16),
                             __builtin_amdgcn_alignbit(w.z, w.y, 16),
                             __builtin_amdgcn_alignbit(w.w, w.z, 16)));
      const bf16x8 b1 = __builtin_bit_cast(bf16x8, w);
      const bf16x8 b2 = __builtin_bit_cast(
          bf16x8, make_uint4(__builtin_amdgcn_alignbit(w.y, w.x, 16),
                             __builtin_amdgcn_alignbit(w.z, w.y, 16),
                             __builtin_amdgcn_alignbit(w.w, w.z, 16),
                             __builtin_amdgcn_alignbit(g.next, w.w, 16)));
#pragma unroll
      for (int bm = 0; bm < BM; ++bm) {
        acc[bm][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g.a[bm], b0, acc[bm][0], 0, 0, 0);
        acc[bm][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g.a[bm], b1, acc[bm][1], 0, 0, 0);
        acc[bm][2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g.a[bm], b2, acc[bm][2], 0, 0, 0);
      }
    };
    // Segments in groups of U, every load of a group issued before its
    // products, so the loads' latencies overlap.
    constexpr int U = 4;
    int x0 = 0;
    for (; x0 + 16 * U <= W; x0 += 16 * U) {
      Seg g[U];
#pragma unroll
      for (int u = 0; u < U; ++u) load(x0 + 16 * u, g[u]);
#pragma unroll
      for (int u = 0; u < U; ++u) mma(g[u]);
    }
    for (; x0 < W; x0 += 16) {
      Seg g;
      load(x0, g);
      mma(g);
    }
  }
#pragma unroll
  for (int bm = 0; bm < BM; ++bm)
#pragma unroll
    for (int kw = 0; kw < 3; ++kw) {
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave][8 * (r / 4) + 4 * half + (r % 4)][li] = acc[bm][kw][r];
      __syncthreads();
      for (int e = threadIdx.x; e < 32 * 32; e += 256) {
        const int i = e / 32, j = e % 32;
        const float v = ((red[0][i][j] + red[1][i][j]) + red[2][i][j]) + red[3][i][j];
        const int co = (cog * BM + bm) * 32 + i, ci = cib * 32 + j;
        if (co < Cout && ci < Cin)
          part[(((int64_t)split * Cout + co) * 9 + kh * 3 + kw) * Cin + ci] = v;
      }
      __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Weight and bias gradients read straight from the NHWC tensors.  Work-group = 4
// waves on COB x CIB blocks of 32 output x 32 input channels and a contiguous range
// of units (split K), a unit being one row of one 64-pixel column strip, strip by
// strip.  Each stage takes R = 4 / (COB CIB) rows y .. y + R - 1 of a strip: wave
// (kr, channel block pair) takes row y + kr and all nine taps of its pair, 36
// products per stage.  dY's rows and the input rows y + 1 .. y + R (columns x0 - 1 ..
// x0 + 64) are copied to LDS as they stand, pixel by pixel, in planes of 32
// channels; the input rows y - 1 and y are there from the stage before (a ring of
// 2 R + 2 rows, dY in two halves, so one barrier per stage).  The next stage's loads
// are in flight during the products.
//
// A and B need consecutive pixels of one channel in a lane, which is what the
// transposing LDS read gives: 16 lanes read a 4 pixel x 16 channel block as 8-byte
// pieces and each gets four pixels of one channel.  A plane's 64-byte pixel stride
// puts the four pixels and two channel halves that 32 lanes read on different banks.
// A tap's column shift is a funnel shift of the aligned pixels and the next two.
//
// What bounds it: the matrix cores at 700 - 830 TFLOP/s, with 0.6 of the LDS cycles a
// product has.  The loss gradient of 8 fields of 512^2 (4 levels, base 32) spent 1788
// us here with one 32 x 32 block per three waves, channel-major staging by 2-byte
// stores and two barriers per row, now 908.  Eight waves and half the splits on 64 x
// 64 channels: 38 us less in the split sums, 45 more here; storing the next stage
// between a stage's products: 3% slower.
//
// part[split]: [co][tap][ci], then [co] biases (the order of the parameters).  Needs
// W % 64 == 0, Cin % 8 == 0, Cout % 8 == 0, Cu % 32 == 0.
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(3))) bf16_t lds_bf16;
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// Four consecutive pixels of one channel: lane i of 16 passes the address of the
// 4-channel piece i % 4 of pixel i / 4, and gets channel i.
__device__ __forceinline__ uint2 lds_tr4(const lds_bf16* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p));
}

template <int COB, int CIB>
__global__ __launch_bounds__(256, 2) void k_conv3x3_wgrad_nhwc(
    const bf16_t* __restrict__ dY, ConvIn in, int N, int H, int W, int Cout, int splits,
    int units_per_split, float* __restrict__ part) {
  constexpr int R = 4 / (COB * CIB);            // rows of a stage
  constexpr int SEG = 64, PX = SEG + 4;         // input pixels of a row: x0 - 1 .. (66 used)
  constexpr int YP = SEG * 32, XP = PX * 32;    // a plane's 32-channel rows
  constexpr int XR = 2 * R + 2;                 // the ring of input rows
  constexpr int kY = 2 * R * COB * YP, kX = XR * CIB * XP;
  constexpr int kRed = R > 1 ? 4 * 48 * 64 * 2 : 0;  // the waves' sums of one ky, in bf16 units
  constexpr int kLds = kY + kX > kRed ? kY + kX : kRed;
  __shared__ __attribute__((aligned(16))) bf16_t lds[kLds];
  const int Cin = in.Cu + in.C;
  const size_t stride = (size_t)Cout * 9 * Cin + Cout;  // a split's weights, then biases
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5, li = lane & 31;
  const int pair = wave % (COB * CIB), kr = wave / (COB * CIB);
  const int wco = pair % COB, wci = pair / COB;
  const int cogroups = (Cout + 32 * COB - 1) / (32 * COB);
  const int tiles = cogroups * ((Cin + 32 * CIB - 1) / (32 * CIB));
  // The tiles of one split read the same rows: they run on one XCD (work-groups are
  // dealt to the 8 XCDs in turn) where the number of splits allows it.
  int tile, split;
  if (splits % 8 == 0) {
    const int j = blockIdx.x / 8;
    tile = j % tiles;
    split = j / tiles * 8 + (int)blockIdx.x % 8;
  } else {
    tile = blockIdx.x % tiles;
    split = blockIdx.x / tiles;
  }
  const int co0 = tile % cogroups * 32 * COB, ci0 = tile / cogroups * 32 * CIB;
  const int strips = W / SEG;
  const int64_t u0 = (int64_t)split * units_per_split;
  const int64_t u1 = min((int64_t)N * strips * H, u0 + units_per_split);
  const bool bias = ci0 == 0 && wci == 0;
  const int tpx = tid >> 2, tc = 8 * (tid & 3);  // the pixel and channels this thread copies

  f32x16 acc[3][3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  float bsum = 0.f;

  // Row yy of the input planes (64 pixels from x0 - 1): one 16-byte piece per thread
  // and plane; a buffer of exactly the row's bytes makes pixels outside it read zero.
  auto load_x = [&](int n, int yy, int x0, int b) -> uint4 {
    const int c = ci0 + 32 * b;
    const bool up = c < in.Cu;
    const int sh = up ? 1 : 0, cs = up ? in.Cu : in.C, ws = W >> sh;
    const bool v = yy >= 0 && yy < H && c < Cin;
    const bf16_t* row =
        (up ? in.U : in.X) + ((size_t)n * (H >> sh) + (v ? yy >> sh : 0)) * ws * cs;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(row), (short)0, v ? ws * cs * (int)sizeof(bf16_t) : 0, 0x00020000);
    const int x = x0 - 1 + tpx, cc = (up ? c : c - in.Cu) + tc;
    const int off = ((x >> sh) * cs + cc) * (int)sizeof(bf16_t);
    return __builtin_bit_cast(
        uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, x >= 0 && cc < cs ? off : -1, 0, 0));
  };
  // Pixels 64 and 65 of `rows` rows from yy0: threads 0 .. 8 CIB rows - 1.
  auto load_tail = [&](int n, int yy0, int rows, int x0) -> uint4 {
    const int b = tid / 8 % CIB, r = tid / (8 * CIB), c = ci0 + 32 * b + tc;
    const int yy = yy0 + r, x = x0 + 63 + (tid >> 2) % 2;
    if (r < rows && yy >= 0 && yy < H && x < W && c < Cin)
      return *reinterpret_cast<const uint4*>(in.at(n, yy, x, H, W, c));
    return make_uint4(0, 0, 0, 0);
  };
  auto store_tail = [&](int yy0, int rows, const uint4& v) {
    const int b = tid / 8 % CIB, r = tid / (8 * CIB);
    if (r < rows)
      *reinterpret_cast<uint4*>(lds + kY + ((yy0 + r + XR) % XR * CIB + b) * XP +
                                (SEG + (tid >> 2) % 2) * 32 + tc) = v;
  };
  auto store_x = [&](int yy, int b, const uint4& v) {
    *reinterpret_cast<uint4*>(lds + kY + ((yy + XR) % XR * CIB + b) * XP + 8 * tid) = v;
  };
  auto load_y = [&](int n, int yy, int yend, int x0, int b) -> uint4 {
    const int c = co0 + 32 * b;
    const bool v = yy < yend && c < Cout;
    const bf16_t* row = dY + ((size_t)n * H + (v ? yy : 0)) * W * Cout;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(row), (short)0, v ? W * Cout * (int)sizeof(bf16_t) : 0, 0x00020000);
    const int off = ((x0 + tpx) * Cout + c + tc) * (int)sizeof(bf16_t);
    return __builtin_bit_cast(
        uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, c + tc < Cout ? off : -1, 0, 0));
  };

  const int trl = (8 * half + ((lane & 15) >> 2)) * 32 + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
  int buf = 0;
  for (int64_t u = u0; u < u1;) {
    const int strip = (int)(u / H), ya = (int)(u - (int64_t)strip * H);
    const int yb = (int)min((int64_t)H, ya + (u1 - u));
    const int n = strip / strips, x0 = strip % strips * SEG;
    u += yb - ya;
    uint4 vy[R * COB], vx[R * CIB], vt;
    uint4 px[2 * CIB], pt;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int b = 0; b < CIB; ++b) px[r * CIB + b] = load_x(n, ya - 1 + r, x0, b);
    pt = load_tail(n, ya - 1, 2, x0);
    auto fetch = [&](int y) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int b = 0; b < COB; ++b) vy[r * COB + b] = load_y(n, y + r, yb, x0, b);
#pragma unroll
        for (int b = 0; b < CIB; ++b) vx[r * CIB + b] = load_x(n, y + 1 + r, x0, b);
      }
      vt = load_tail(n, y + 1, R, x0);
    };
    fetch(ya);
    __syncthreads();  // the strip before has been read
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int b = 0; b < CIB; ++b) store_x(ya - 1 + r, b, px[r * CIB + b]);
    store_tail(ya - 1, 2, pt);
    for (int y = ya; y < yb; y += R) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int b = 0; b < COB; ++b)
          *reinterpret_cast<uint4*>(lds + ((buf * R + r) * COB + b) * YP + 8 * tid) =
              vy[r * COB + b];
#pragma unroll
        for (int b = 0; b < CIB; ++b) store_x(y + 1 + r, b, vx[r * CIB + b]);
      }
      store_tail(y + 1, R, vt);
      if (y + R < yb) fetch(y + R);
      __syncthreads();
      const lds_bf16* ya_ = (const lds_bf16*)lds + ((buf * R + kr) * COB + wco) * YP + trl;
      const lds_bf16* xa[3];
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
        xa[ky] = (const lds_bf16*)lds + kY + ((y + kr + ky - 1 + XR) % XR * CIB + wci) * XP + trl;
#pragma unroll
      for (int ks = 0; ks < SEG / 16; ++ks) {
        const uint2 a0 = lds_tr4(ya_ + 512 * ks), a1 = lds_tr4(ya_ + 512 * ks + 128);
        B8 ab;
        ab.u = make_uint4(a0.x, a0.y, a1.x, a1.y);
        const bf16x8 a = __builtin_bit_cast(bf16x8, ab.u);
        if (bias) {
#pragma unroll
          for (int e = 0; e < 8; ++e) bsum += bf2f(ab.h[e]);
        }
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) {
          const uint2 p = lds_tr4(xa[ky] + 512 * ks), q = lds_tr4(xa[ky] + 512 * ks + 128);
          const uint32_t nx = lds_tr4(xa[ky] + 512 * ks + 256).x;
          const bf16x8 b0 = __builtin_bit_cast(bf16x8, make_uint4(p.x, p.y, q.x, q.y));
          const bf16x8 b1 = __builtin_bit_cast(
              bf16x8, make_uint4(__builtin_amdgcn_alignbit(p.y, p.x, 16),
                                 __builtin_amdgcn_alignbit(q.x, p.y, 16),
                                 __builtin_amdgcn_alignbit(q.y, q.x, 16),
                                 __builtin_amdgcn_alignbit(nx, q.y, 16)));
          const bf16x8 b2 = __builtin_bit_cast(bf16x8, make_uint4(p.y, q.x, q.y, nx));
          acc[ky][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b0, acc[ky][0], 0, 0, 0);
          acc[ky][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b1, acc[ky][1], 0, 0, 0);
          acc[ky][2] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b2, acc[ky][2], 0, 0, 0);
        }
      }
      buf ^= 1;
    }
  }
  // Lane (li, half) holds rows 8 (r / 4) + 4 half + r % 4 (output channels) of column
  // li (input channel) of its pair's nine taps; the R rows' sums are added in row order.
  float* red = reinterpret_cast<float*>(lds);
  const int ci = ci0 + 32 * wci + li;
  float* out = part + (size_t)split * stride;
  bsum += __shfl_xor(bsum, 32);  // the two pixel halves of channel li
#pragma unroll
  for (int ky = 0; ky < 3; ++ky) {
    if constexpr (R > 1) {
      __syncthreads();
#pragma unroll
      for (int kx = 0; kx < 3; ++kx)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[(wave * 48 + 16 * kx + r) * 64 + lane] = acc[ky][kx][r];
      __syncthreads();
      // wave (kr, pair) finishes every R-th value of its pair
#pragma unroll
      for (int k = 0; k < 48 / R; ++k) {
        const int e = k * R + kr, kx = e / 16, r = e % 16;
        float s = red[(pair * 48 + e) * 64 + lane];
#pragma unroll
        for (int q = 1; q < R; ++q) s += red[((q * COB * CIB + pair) * 48 + e) * 64 + lane];
        const int co = co0 + 32 * wco + 8 * (r / 4) + 4 * half + (r % 4);
        if (co < Cout && ci < Cin) out[((size_t)co * 9 + 3 * ky + kx) * Cin + ci] = s;
      }
    } else {
#pragma unroll
      for (int kx = 0; kx < 3; ++kx)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int co = co0 + 32 * wco + 8 * (r / 4) + 4 * half + (r % 4);
          if (co < Cout && ci < Cin)
            out[((size_t)co * 9 + 3 * ky + kx) * Cin + ci] = acc[ky][kx][r];
        }
    }
  }
  if constexpr (R > 1) {
    __syncthreads();
    red[wave * 64 + lane] = bsum;
    __syncthreads();
    bsum = red[pair * 64 + lane];
#pragma unroll
    for (int q = 1; q < R; ++q) bsum += red[(q * COB * CIB + pair) * 64 + lane];
  }
  const int co = co0 + 32 * wco + li;
  if (bias && kr == 0 && half == 0 && co < Cout) out[(size_t)Cout * 9 * Cin + co] = bsum;
}

// out[i] = sum over k of part[k][i]: 32 columns of V outputs per work-group, the
// splits dealt round-robin over 32 groups of 32 lanes (each summed in increasing k,
// eight loads in flight), then the 32 group sums added in group order, so the result
// does not depend on scheduling.  V = 4 where the rows are 16-byte aligned: it is bound
// by the reads, 266 -> 168 us in a gradient with 0.7 GB of partials against V = 1.
template <int V>
__global__ __launch_bounds__(1024) void k_sum_splits(const float* __restrict__ part, int splits,
                                                     int64_t count, float* __restrict__ out) {
  typedef float fv __attribute__((ext_vector_type(V)));
  constexpr int U = 8;
  __shared__ float sh[32][32 * V + 1];
  const int j = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int64_t i = ((int64_t)blockIdx.x * 32 + j) * V;
  fv s = (fv)0.f;
  if (i < count)
    for (int k0 = g; k0 < splits; k0 += 32 * U) {
      fv v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = min(k0 + 32 * u, splits - 1);
        v[u] = *reinterpret_cast<const fv*>(part + (int64_t)k * count + i);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) s += k0 + 32 * u < splits ? v[u] : (fv)0.f;
    }
#pragma unroll
  for (int e = 0; e < V; ++e) sh[g][V * j + e] = s[e];
  __syncthreads();
  const int c = threadIdx.x;
  const int64_t o = (int64_t)blockIdx.x * 32 * V + c;
  if (c < 32 * V && o < count) {
    float t = 0.f;
#pragma unroll
    for (int q = 0; q < 32; ++q) t += sh[q][c];
    out[o] = t;
  }
}

// part[s][c] = sum of dYT[n][c][hw] over the s-th of `splits` contiguous
// chunks of the flat (n, hw) range (fixed order within a chunk).
__global__ __launch_bounds__(256) void k_channel_partial(const bf16_t* __restrict__ dYT, int N,
                                                         int HW, int C, int64_t chunk,
                                                         float* __restrict__ part) {
  __shared__ float sh[256];
  const int c = blockIdx.x, sp = blockIdx.y;
  const int64_t total = (int64_t)N * HW;
  const int64_t i0 = (int64_t)sp * chunk, i1 = min(total, i0 + chunk);
  float s = 0.f;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) {
    const int64_t n = i / HW, hw = i - n * HW;
    s += bf2f(dYT[(n * C + c) * HW + hw]);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[(int64_t)sp * C + c] = sh[0];
}

// ---------------------------------------------------------------------------
// Pooling, upsampling + concatenation, head, loss, optimiser.
// ---------------------------------------------------------------------------
// Element-wise kernels on NHWC tensors with channel counts that are multiples
// of 8: one thread per (pixel, 8-channel group), 16-byte loads and stores.
__device__ __forceinline__ B8 ld_b8(const bf16_t* p) {
  B8 r;
  r.u = *reinterpret_cast<const uint4*>(p);
  return r;
}
__device__ __forceinline__ void st_b8(bf16_t* p, const B8& v) {
  *reinterpret_cast<uint4*>(p) = v.u;
}

__global__ void k_maxpool_fwd(const bf16_t* __restrict__ X, int N, int H, int W, int C,
                              bf16_t* __restrict__ Y) {
  const int Ho = H / 2, Wo = W / 2, G = C / 8;
  const int total = N * Ho * Wo * G;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int g = i % G, q = i / G;
    const int xo = q % Wo, t = q / Wo, yo = t % Ho, n = t / Ho;
    const bf16_t* b = X + (((size_t)n * H + 2 * yo) * W + 2 * xo) * C + 8 * g;
    const B8 v0 = ld_b8(b), v1 = ld_b8(b + C), v2 = ld_b8(b + (size_t)W * C),
             v3 = ld_b8(b + (size_t)W * C + C);
    const B8 o = max4(v0, v1, v2, v3);
    st_b8(Y + (size_t)q * C + 8 * g, o);
  }
}

// The gradient of an encoder level's output X (N, H, W, C): dP (of the pooled
// map) routed to the first maximum of each 2 x 2 window, added to the skip's part
// of dcat (channels Cu .. Cu + C - 1 of Cu + C), zero where X is not positive (the
// ReLU that made X): one pass over the four tensors.
__global__ void k_skip_pool_bwd(const bf16_t* __restrict__ X, const bf16_t* __restrict__ dP,
                                const bf16_t* __restrict__ dcat, int Cu, int N, int H, int W,
                                int C, bf16_t* __restrict__ dX) {
  const int Ho = H / 2, Wo = W / 2, G = C / 8, Ct = Cu + C;
  const int total = N * Ho * Wo * G;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int g = i % G, q = i / G;
    const int xo = q % Wo, t = q / Wo, yo = t % Ho, n = t / Ho;
    const size_t p = ((size_t)n * H + 2 * yo) * W + 2 * xo;
    const size_t o[4] = {p, p + 1, p + W, p + W + 1};
    B8 v[4], d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = ld_b8(X + o[k] * C + 8 * g);
      d[k] = ld_b8(dcat + o[k] * Ct + Cu + 8 * g);
    }
    const B8 dy = ld_b8(dP + (size_t)q * C + 8 * g);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int arg = 0;
      float m = bf2f(v[0].h[e]);
#pragma unroll
      for (int k = 1; k < 4; ++k) {
        const float x = bf2f(v[k].h[e]);
        if (x > m) { m = x; arg = k; }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bf16_t r = k == arg ? dy.h[e] : (bf16_t)0;
        const bf16_t sum = f2bf(bf2f(d[k].h[e]) + bf2f(r));
        d[k].h[e] = bf2f(v[k].h[e]) <= 0.f ? (bf16_t)0 : sum;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) st_b8(dX + o[k] * C + 8 * g, d[k]);
  }
}

// cat = [nearest 2x upsample of U (Cu channels), S (Cs channels)]
__global__ void k_upcat_fwd(const bf16_t* __restrict__ U, int Cu, const bf16_t* __restrict__ S,
                            int Cs, int N, int H, int W, bf16_t* __restrict__ cat) {
  const int Ct = Cu + Cs, G = Ct / 8, Gu = Cu / 8;
  const int total = N * H * W * G;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int g = i % G, p = i / G;
    B8 v;
    if (g < Gu) {
      const int x = p % W, t = p / W, y = t % H, n = t / H;
      v = ld_b8(U + (((size_t)n * (H / 2) + y / 2) * (W / 2) + x / 2) * Cu + 8 * g);
    } else {
      v = ld_b8(S + (size_t)p * Cs + 8 * (g - Gu));
    }
    st_b8(cat + (size_t)p * Ct + 8 * g, v);
  }
}

// dU = sum of dcat's first Cu channels over each 2 x 2 block, zero where U (a
// ReLU's output) is not positive
__global__ void k_upcat_bwd_u(const bf16_t* __restrict__ dcat, int Cu, int Cs, int N, int H,
                              int W, const bf16_t* __restrict__ U, bf16_t* __restrict__ dU) {
  const int Ct = Cu + Cs, Hh = H / 2, Wh = W / 2, G = Cu / 8;
  const int total = N * Hh * Wh * G;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int g = i % G, q = i / G;
    const int x = q % Wh, t = q / Wh, y = t % Hh, n = t / Hh;
    const size_t b = (((size_t)n * H + 2 * y) * W + 2 * x) * Ct + 8 * g;
    const B8 a0 = ld_b8(dcat + b), a1 = ld_b8(dcat + b + Ct), a2 = ld_b8(dcat + b + (size_t)W * Ct),
             a3 = ld_b8(dcat + b + (size_t)W * Ct + Ct);
    const B8 u = ld_b8(U + (size_t)q * Cu + 8 * g);
    const B8 o = sum4_masked(a0, a1, a2, a3, u);
    st_b8(dU + (size_t)q * Cu + 8 * g, o);
  }
}

template <int C>
__global__ void k_head_fwd(const bf16_t* __restrict__ Y, int64_t P, const float* __restrict__ w,
                           const float* __restrict__ b, float* __restrict__ out) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < P;
       p += (int64_t)gridDim.x * blockDim.x) {
    float s = b[0];
#pragma unroll
    for (int c = 0; c < C; ++c) s += bf2f(Y[p * C + c]) * w[c];
    out[p] = s;
  }
}

// Block-partial dw (C values) and db (1 value) per block, fixed order.
constexpr int kHeadThreads = 256;
template <int C>
__global__ __launch_bounds__(kHeadThreads) void k_head_bwd(
    const bf16_t* __restrict__ Y, const float* __restrict__ dout, int64_t P,
    const float* __restrict__ w, bf16_t* __restrict__ dY, float* __restrict__ part) {
  __shared__ float sh[kHeadThreads];
  float acc[C + 1], wr[C];
#pragma unroll
  for (int c = 0; c <= C; ++c) acc[c] = 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c) wr[c] = w[c];
  for (int64_t p = blockIdx.x * (int64_t)kHeadThreads + threadIdx.x; p < P;
       p += (int64_t)gridDim.x * kHeadThreads) {
    const float g = dout[p];
#pragma unroll
    for (int c8 = 0; c8 < C; c8 += 8) {
      const B8 y = ld_b8(Y + p * C + c8);
      B8 d;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = bf2f(y.h[e]);
        d.h[e] = v <= 0.f ? (bf16_t)0 : f2bf(g * wr[c8 + e]);  // the ReLU that made Y
        acc[c8 + e] += g * v;
      }
      st_b8(dY + p * C + c8, d);
    }
    acc[C] += g;
  }
#pragma unroll
  for (int c = 0; c <= C; ++c) {
    sh[threadIdx.x] = acc[c];
    __syncthreads();
    for (int s = kHeadThreads / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) part[(int64_t)blockIdx.x * (C + 1) + c] = sh[0];
    __syncthreads();
  }
}

constexpr int kMseThreads = 256;
__global__ __launch_bounds__(kMseThreads) void k_mse(const float* __restrict__ out,
                                                     const float* __restrict__ target, int64_t P,
                                                     float* __restrict__ dout,
                                                     double* __restrict__ part) {
  __shared__ double sh[kMseThreads];
  double s = 0.0;
  const float sc = 2.0f / (float)P;
  for (int64_t p = blockIdx.x * (int64_t)kMseThreads + threadIdx.x; p < P;
       p += (int64_t)gridDim.x * kMseThreads) {
    const float d = out[p] - target[p];
    s += (double)d * d;
    dout[p] = sc * d;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = kMseThreads / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

__global__ void k_pack_input(const float* __restrict__ in, int64_t P, bf16_t* __restrict__ X8) {
  for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < P;
       p += (int64_t)gridDim.x * blockDim.x) {
    uint4 v = make_uint4((uint32_t)f2bf(in[p]), 0u, 0u, 0u);
    *reinterpret_cast<uint4*>(X8 + p * 8) = v;
  }
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

__global__ void k_to_bf16(const float* __restrict__ x, int64_t n, bf16_t* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

// ===========================================================================
// Launchers
// ===========================================================================
static dim3 grid1d(int64_t n, int threads = 256) {
  int64_t b = (n + threads - 1) / threads;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return dim3((unsigned)b);
}

// A chunk of input channels comes from one source.
static int conv_chunk(const ConvIn& in) {
  const int Cin = in.Cu + in.C;
  return Cin == 8 ? 8 : Cin % 32 != 0 || in.Cu % 32 != 0 ? 16 : 32;
}

bool conv3x3_by_rows(const ConvIn& in, int N, int H, int W, int Cout) {
  const int chunk = conv_chunk(in);
  return chunk > 8 && W % 64 == 0 && H % 8 == 0 && (in.Cu + in.C) % chunk == 0 &&
         in.Cu % chunk == 0 &&
         (int64_t)H * W * std::max(in.C, in.Cu) < (1ll << 30) &&  // 32-bit byte offsets
         (int64_t)N * (H / 4) * (W / 64) * ((Cout + 31) / 32) < (1ll << 31);
}

hipError_t launch_conv3x3_fwd(const ConvIn& in, int N, int H, int W, const bf16_t* Wt,
                              const float* bias, int Cout, int relu, const ConvOut& out,
                              hipStream_t s) {
  const int Cin = in.Cu + in.C;
  const bf16_t* mask = out.mask;
  bf16_t *Y = out.Y, *pool = out.pool;
  const bool rows = conv3x3_by_rows(in, N, H, W, Cout);
  if (in.C % 8 != 0 || in.Cu % 8 != 0 || Cout % 8 != 0 || Cout < 8 || N < 1 || H < 1 || W < 1 ||
      (pool && (H % 2 != 0 || W % 2 != 0)) || (in.Cu > 0 && !rows) ||
      (out.head && (!rows || Cout > 64 || !out.head_w || !out.head_b)) || (!Y && !out.head) ||
      (out.Cu > 0 && (!rows || pool || mask || out.Cu % 8 != 0 || out.Cu > Cout)))
    return hipErrorInvalidValue;
  const int64_t NP = (int64_t)N * H * W;
  const int chunk = conv_chunk(in);
  if (rows) {
    const int cow = Cout <= 32 ? 1 : 2, groups = (Cout + 32 * cow - 1) / (32 * cow);
    auto blocks = [&](int th) { return (int64_t)N * (H / th) * (W / 64) * groups; };
    // Tiles of 8 rows where two work-groups per CU come of it, else of 4 (more reads per
    // product): with the limit at 256, 3790 -> 3810 us for the gradient of 8 of 512^2.
    const int th = blocks(8) >= 512 ? 8 : 4;
#define HUV_CONV_ROWS(BM_, COW_, CC_)                                                          \
  hipLaunchKernelGGL((k_conv3x3_rows<BM_, COW_, CC_>), dim3((unsigned)blocks(th)), dim3(256), \
                     0, s, in, N, H, W, Wt, bias, Cout, relu, out)
      if (cow == 1) {
        if (chunk == 16) { if (th == 8) HUV_CONV_ROWS(4, 1, 16); else HUV_CONV_ROWS(2, 1, 16); }
        else { if (th == 8) HUV_CONV_ROWS(4, 1, 32); else HUV_CONV_ROWS(2, 1, 32); }
      } else {
        if (chunk == 16) { if (th == 8) HUV_CONV_ROWS(8, 2, 16); else HUV_CONV_ROWS(4, 2, 16); }
        else { if (th == 8) HUV_CONV_ROWS(8, 2, 32); else HUV_CONV_ROWS(4, 2, 32); }
      }
#undef HUV_CONV_ROWS
    return hipGetLastError();
  }
  // the first layer's form: neither mask nor pool
  if (chunk == 8 && !mask && !pool && W % 64 == 0 && H % 4 == 0 &&
      (int64_t)N * (H / 4) * (W / 64) < (1ll << 31) && (int64_t)H * W * in.C < (1ll << 30)) {
    // tiles of 4 rows x 64 columns: BM = 2 pixel blocks per wave
    dim3 grid((unsigned)((int64_t)N * (H / 4) * (W / 64)),
              (unsigned)((Cout + (Cout <= 32 ? 31 : 63)) / (Cout <= 32 ? 32 : 64)));
#define HUV_CONV_LDS(BN_)                                                                     \
  hipLaunchKernelGGL((k_conv3x3_fwd_lds<2, BN_>), grid, dim3(256), 0, s, in.X, H, W, Wt, bias, \
                     Cout, relu, Y)
    if (Cout <= 32) HUV_CONV_LDS(1);
    else HUV_CONV_LDS(2);
#undef HUV_CONV_LDS
    return hipGetLastError();
  }
  constexpr int BM = 2;
  if (Cout <= 32) {
    dim3 grid((unsigned)((NP + 4 * 32 * BM - 1) / (4 * 32 * BM)), (unsigned)((Cout + 31) / 32));
    hipLaunchKernelGGL((k_conv3x3_fwd<BM, 1>), grid, dim3(256), 0, s, in.X, N, H, W, Cin, Wt, bias,
                       Cout, relu, mask, Y);
  } else {
    dim3 grid((unsigned)((NP + 4 * 32 * BM - 1) / (4 * 32 * BM)), (unsigned)((Cout + 63) / 64));
    hipLaunchKernelGGL((k_conv3x3_fwd<BM, 2>), grid, dim3(256), 0, s, in.X, N, H, W, Cin, Wt, bias,
                       Cout, relu, mask, Y);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !pool) return e;
  return launch_maxpool_fwd(Y, N, H, W, Cout, pool, s);
}

hipError_t launch_conv_weight_rot(const bf16_t* Wt, int Cout, int Cin, bf16_t* Wr,
                                  hipStream_t s) {
  hipLaunchKernelGGL(k_conv_weight_rot, grid1d((int64_t)Cout * 9 * Cin), dim3(256), 0, s, Wt,
                     Cout, Cin, Wr);
  return hipGetLastError();
}

hipError_t launch_nhwc_to_nchw(const bf16_t* X, int N, int H, int W, int C, bf16_t* XT,
                               hipStream_t s) {
  if ((H * W) % 64 != 0 || C % 8 != 0) return hipErrorInvalidValue;
  dim3 grid((unsigned)((int64_t)N * H * W / 64), (unsigned)((C + 31) / 32));
  hipLaunchKernelGGL(k_transpose_t, grid, dim3(256), 0, s, X, N, H * W, C, XT);
  return hipGetLastError();
}

hipError_t launch_conv3x3_wgrad(const bf16_t* dYT, const bf16_t* XT, int N, int H, int W,
                                int Cin, int Cout, int splits, float* part, hipStream_t s) {
  if (W % 16 != 0 || Cin % 8 != 0 || splits < 1) return hipErrorInvalidValue;
  const int rows = N * H;
  const int rps = (rows + splits - 1) / splits;
  const int coblocks = (Cout + 31) / 32, ciblocks = (Cin + 31) / 32;
  if (coblocks >= 2) {
    const int tiles = ((coblocks + 1) / 2) * ciblocks * 3;
    hipLaunchKernelGGL(k_conv3x3_wgrad<2>, dim3(tiles, splits), dim3(256), 0, s, dYT, XT, N, H,
                       W, Cin, Cout, rps, part);
  } else {
    const int tiles = coblocks * ciblocks * 3;
    hipLaunchKernelGGL(k_conv3x3_wgrad<1>, dim3(tiles, splits), dim3(256), 0, s, dYT, XT, N, H,
                       W, Cin, Cout, rps, part);
  }
  return hipGetLastError();
}

// 32-channel blocks of a work-group of the NHWC weight gradient: two of each kind
// where there are two.
static void wgrad_blocks(int Cin, int Cout, int* cob, int* cib) {
  *cob = Cout > 32 ? 2 : 1;
  *cib = (Cin + 31) / 32 % 2 == 0 ? 2 : 1;
}

int wgrad_nhwc_splits(int N, int H, int W, int Cin, int Cout) {
  int cob, cib;
  wgrad_blocks(Cin, Cout, &cob, &cib);
  const int tiles =
      ((Cout + 32 * cob - 1) / (32 * cob)) * ((Cin + 32 * cib - 1) / (32 * cib));
  const int64_t units = (int64_t)N * H * (W / 64);
  int64_t s = std::max(1, 512 / tiles);  // two work-groups per CU
  if (s >= 8) s -= s % 8;
  return (int)std::min(s, units);
}

hipError_t launch_conv3x3_wgrad_nhwc(const bf16_t* dY, const ConvIn& in, int N, int H, int W,
                                     int Cout, int splits, float* part, hipStream_t s) {
  const int64_t units = (int64_t)N * H * (W / 64);
  if (W % 64 != 0 || in.C % 8 != 0 || in.Cu % 32 != 0 || Cout % 8 != 0 || splits < 1 ||
      splits > units || (int64_t)W * std::max(std::max(in.C, in.Cu), Cout) >= (1ll << 30) ||
      (units + splits - 1) / splits >= (1ll << 31))
    return hipErrorInvalidValue;
  int cob, cib;
  wgrad_blocks(in.Cu + in.C, Cout, &cob, &cib);
  const int tiles = ((Cout + 32 * cob - 1) / (32 * cob)) *
                    ((in.Cu + in.C + 32 * cib - 1) / (32 * cib));
  const int ups = (int)((units + splits - 1) / splits);
#define HUV_WGRAD(A_, B_)                                                                       \
  hipLaunchKernelGGL((k_conv3x3_wgrad_nhwc<A_, B_>), dim3((unsigned)(tiles * splits)), dim3(256), \
                     0, s, dY, in, N, H, W, Cout, splits, ups, part)
  if (cob == 1 && cib == 1) HUV_WGRAD(1, 1);
  else if (cob == 1) HUV_WGRAD(1, 2);
  else if (cib == 1) HUV_WGRAD(2, 1);
  else HUV_WGRAD(2, 2);
#undef HUV_WGRAD
  return hipGetLastError();
}

hipError_t launch_sum_splits(const float* part, int splits, int64_t count, float* out,
                             hipStream_t s) {
  if (count <= 0 || splits < 1 || (count + 31) / 32 >= (1ll << 31)) return hipErrorInvalidValue;
  if (count % 4 == 0 && ((uintptr_t)part | (uintptr_t)out) % 16 == 0)
    hipLaunchKernelGGL(k_sum_splits<4>, dim3((unsigned)((count + 127) / 128)), dim3(1024), 0, s,
                       part, splits, count, out);
  else
    hipLaunchKernelGGL(k_sum_splits<1>, dim3((unsigned)((count + 31) / 32)), dim3(1024), 0, s,
                       part, splits, count, out);
  return hipGetLastError();
}

hipError_t launch_channel_sum(const bf16_t* dYT, int N, int HW, int C, float* part, int splits,
                              float* db, hipStream_t s) {
  const int64_t total = (int64_t)N * HW;
  const int64_t chunk = (total + splits - 1) / splits;
  hipLaunchKernelGGL(k_channel_partial, dim3(C, splits), dim3(256), 0, s, dYT, N, HW, C, chunk,
                     part);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_sum_splits(part, splits, C, db, s);
}

hipError_t launch_maxpool_fwd(const bf16_t* X, int N, int H, int W, int C, bf16_t* Y,
                              hipStream_t s) {
  if (C % 8 != 0 || (int64_t)N * H * W * C / 8 >= (1ll << 30)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_maxpool_fwd, grid1d((int64_t)N * (H / 2) * (W / 2) * C / 8), dim3(256), 0,
                     s, X, N, H, W, C, Y);
  return hipGetLastError();
}

hipError_t launch_skip_pool_bwd(const bf16_t* X, const bf16_t* dP, const bf16_t* dcat, int Cu,
                                int N, int H, int W, int C, bf16_t* dX, hipStream_t s) {
  if (C % 8 != 0 || Cu % 8 != 0 || (int64_t)N * H * W * (Cu + C) / 8 >= (1ll << 30))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_skip_pool_bwd, grid1d((int64_t)N * (H / 2) * (W / 2) * C / 8), dim3(256), 0,
                     s, X, dP, dcat, Cu, N, H, W, C, dX);
  return hipGetLastError();
}

hipError_t launch_upcat_fwd(const bf16_t* U, int Cu, const bf16_t* S, int Cs, int N, int H,
                            int W, bf16_t* cat, hipStream_t s) {
  if (Cu % 8 != 0 || Cs % 8 != 0 || (int64_t)N * H * W * (Cu + Cs) / 8 >= (1ll << 30))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_upcat_fwd, grid1d((int64_t)N * H * W * (Cu + Cs) / 8), dim3(256), 0, s, U, Cu,
                     S, Cs, N, H, W, cat);
  return hipGetLastError();
}

hipError_t launch_upcat_bwd_u(const bf16_t* dcat, int Cu, int Cs, int N, int H, int W,
                              const bf16_t* U, bf16_t* dU, hipStream_t s) {
  if (Cu % 8 != 0 || Cs % 8 != 0 || (int64_t)N * H * W * (Cu + Cs) / 8 >= (1ll << 30))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_upcat_bwd_u, grid1d((int64_t)N * (H / 2) * (W / 2) * Cu / 8), dim3(256), 0,
                     s, dcat, Cu, Cs, N, H, W, U, dU);
  return hipGetLastError();
}

hipError_t launch_head_fwd(const bf16_t* Y, int64_t P, int C, const float* w, const float* b,
                           float* out, hipStream_t s) {
  switch (C) {
    case 16: hipLaunchKernelGGL(k_head_fwd<16>, grid1d(P), dim3(256), 0, s, Y, P, w, b, out); break;
    case 32: hipLaunchKernelGGL(k_head_fwd<32>, grid1d(P), dim3(256), 0, s, Y, P, w, b, out); break;
    case 64: hipLaunchKernelGGL(k_head_fwd<64>, grid1d(P), dim3(256), 0, s, Y, P, w, b, out); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_head_bwd(const bf16_t* Y, const float* dout, int64_t P, int C, const float* w,
                           bf16_t* dY, float* part, int nblk, hipStream_t s) {
  switch (C) {
    case 16: hipLaunchKernelGGL(k_head_bwd<16>, dim3(nblk), dim3(kHeadThreads), 0, s, Y, dout, P, w, dY, part); break;
    case 32: hipLaunchKernelGGL(k_head_bwd<32>, dim3(nblk), dim3(kHeadThreads), 0, s, Y, dout, P, w, dY, part); break;
    case 64: hipLaunchKernelGGL(k_head_bwd<64>, dim3(nblk), dim3(kHeadThreads), 0, s, Y, dout, P, w, dY, part); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_mse(const float* out, const float* target, int64_t P, float* dout,
                      double* part, int nblk, hipStream_t s) {
  hipLaunchKernelGGL(k_mse, dim3(nblk), dim3(kMseThreads), 0, s, out, target, P, dout, part);
  return hipGetLastError();
}

hipError_t launch_pack_input(const float* in, int64_t P, bf16_t* X8, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_input, grid1d(P), dim3(256), 0, s, in, P, X8);
  return hipGetLastError();
}

hipError_t launch_adam(float* p, const float* g, float* m, float* v, int64_t count, float lr,
                       float b1, float b2, float eps, float c1, float c2, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, grid1d(count), dim3(256), 0, s, p, g, m, v, count, lr, b1, b2, eps,
                     c1, c2);
  return hipGetLastError();
}

hipError_t launch_to_bf16(const float* x, int64_t count, bf16_t* y, hipStream_t s) {
  hipLaunchKernelGGL(k_to_bf16, grid1d(count), dim3(256), 0, s, x, count, y);
  return hipGetLastError();
}

}  // namespace huvk
