// Exact mask spectrum of masks given as rectangles and simple polygons,
// evaluated on the device (polygons: see k_poly_band below).
//
// The spectrum convention is the one of mask.rs:31-45 (crates/highuvlith-core):
// for the field [-L/2, L/2)^2, L = N p, and the signed order m,
//   S[m] = N^2 c(m) e^{-i pi (mx + my)(N - 1)/N},
//   c(m) = (1/L^2) \iint t(x, y) e^{-2 pi i (mx x + my y)/L} dx dy,
// which equals FFT_N(raster) in the fine-pixel limit.  A rectangle cell
// [x0, x1) x [y0, y1) of weight w contributes w X(mx) Y(my) with
//   X(m) = N (wx/L) sinc(pi m wx/L) e^{-i pi m ((x0 + x1)/L + (N - 1)/N)}
// (mask.rs:1426-1477, axis_coefficients for a finite interval), and the
// background b adds b N^2 at m = 0 (mask.rs:633).  Axis tables are computed
// once per cell in FP64; the band box sums w X Y over the cells of a clip in
// cell order (FP64 accumulation, one FP32 rounding at the store).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mask_kernels.hpp"

namespace huvk {

// N (w/L) sinc(pi m w/L) e^{-i pi m ((a + b)/L + (N - 1)/N)}
__device__ __forceinline__ double2 axis_coeff(double a, double b, int m, int n, double L) {
  const double w = b - a;
  const double u = (double)m * w / L;
  const double sinc = m == 0 ? 1.0 : sinpi(u) / (M_PI * u);
  const double amp = (double)n * (w / L) * sinc;
  // phase / (-pi), reduced to [-1, 1] before the sine and cosine
  double t = (double)m * ((a + b) / L + (double)(n - 1) / (double)n);
  t -= 2.0 * rint(0.5 * t);
  double sv, cv;
  sincospi(-t, &sv, &cv);
  return make_double2(amp * cv, amp * sv);
}

__global__ __launch_bounds__(256) void k_rect_tables(const double* __restrict__ cells,
                                                     int64_t ncells, int n, double L, int B,
                                                     double2* __restrict__ X,
                                                     double2* __restrict__ Y) {
  const int nk = 2 * B + 1;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= ncells * nk) return;
  const int64_t c = idx / nk;
  const int m = (int)(idx - c * nk) - B;
  const double* p = cells + 6 * c;
  const double2 xa = axis_coeff(p[0], p[1], m, n, L);
  const double2 ya = axis_coeff(p[2], p[3], m, n, L);
  const double wr = p[4], wi = p[5];
  X[idx] = make_double2(wr * xa.x - wi * xa.y, wr * xa.y + wi * xa.x);
  Y[idx] = ya;
}

// A lane takes a tile of kRectT consecutive rows (ky + BB) x kRectT consecutive
// columns (kx + BB), row tiles fastest: per cell it loads kRectT row and
// kRectT column coefficients for kRectT^2 products.  The SL waves of a
// work-group share its 64 tiles and take every SL-th cell each, the next cell's
// coefficients requested before the current one's products; their sums are
// added in a fixed tree.  Work-groups [clip * gpc, (clip + 1) * gpc) cover one
// clip's box.  A chain of loads over the cells bounds a small batch (one clip,
// 100 cells, B = 13: 50 us with one wave a tile group and no request ahead,
// 7.5 us so), so it takes eight waves; a full chip takes two (96 clips of 43
// cells, B = 47: 25.6 us).
constexpr int kRectT = 4;
constexpr int kPolySlices = 8;

template <int SL>
__global__ __launch_bounds__(64 * SL) void k_rect_band(const double2* __restrict__ X,
                                                       const double2* __restrict__ Y,
                                                       const int64_t* __restrict__ coff,
                                                       const double* __restrict__ bg, int n, int B,
                                                       int BB, int gpc, float2* __restrict__ Mq,
                                                       float2* __restrict__ Mp) {
  __shared__ double red[SL / 2][2 * kRectT * kRectT][64];
  const int W = 2 * BB + 1, nk = 2 * B + 1;
  const int G = (W + kRectT - 1) / kRectT;
  const int clip = blockIdx.x / gpc;
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int t = (blockIdx.x - clip * gpc) * 64 + lane;
  const bool tile = t < G * G;
  const int gc = tile ? t / G : 0, gr = tile ? t - gc * G : 0;
  int xi[kRectT], yi[kRectT];
  bool xl[kRectT], yl[kRectT];
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    const int kx = kRectT * gc + j - BB, ky = kRectT * gr + j - BB;
    xl[j] = kx >= -B && kx <= B && kRectT * gc + j < W;
    yl[j] = ky >= -B && ky <= B && kRectT * gr + j < W;
    // clamped: dead rows and columns compute and are discarded
    xi[j] = min(max(kx + B, 0), nk - 1);
    yi[j] = min(max(ky + B, 0), nk - 1);
  }
  double re[kRectT][kRectT], im[kRectT][kRectT];
#pragma unroll
  for (int i = 0; i < kRectT; ++i)
#pragma unroll
    for (int j = 0; j < kRectT; ++j) re[i][j] = im[i][j] = 0.0;
  const int64_t c0 = coff[clip] + slice, c1 = coff[clip + 1];
  if (c0 < c1) {
    double2 x[kRectT], y[kRectT];
    auto load = [&](int64_t c, double2* a, double2* b) {
#pragma unroll
      for (int j = 0; j < kRectT; ++j) {
        a[j] = X[c * nk + xi[j]];
        b[j] = Y[c * nk + yi[j]];
      }
    };
    load(c0, x, y);
    for (int64_t c = c0; c < c1; c += SL) {
      double2 xn[kRectT], yn[kRectT];
      load(c + SL < c1 ? c + SL : c, xn, yn);
#pragma unroll
      for (int i = 0; i < kRectT; ++i)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          re[i][j] = fma(x[j].x, y[i].x, re[i][j]);
          re[i][j] = fma(-x[j].y, y[i].y, re[i][j]);
          im[i][j] = fma(x[j].x, y[i].y, im[i][j]);
          im[i][j] = fma(x[j].y, y[i].x, im[i][j]);
        }
#pragma unroll
      for (int j = 0; j < kRectT; ++j) {
        x[j] = xn[j];
        y[j] = yn[j];
      }
    }
  }
#pragma unroll
  for (int h = SL / 2; h >= 1; h /= 2) {
    if (slice >= h && slice < 2 * h) {
#pragma unroll
      for (int i = 0; i < kRectT; ++i)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          red[slice - h][2 * (i * kRectT + j)][lane] = re[i][j];
          red[slice - h][2 * (i * kRectT + j) + 1][lane] = im[i][j];
        }
    }
    __syncthreads();
    if (slice < h) {
#pragma unroll
      for (int i = 0; i < kRectT; ++i)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          re[i][j] += red[slice][2 * (i * kRectT + j)][lane];
          im[i][j] += red[slice][2 * (i * kRectT + j) + 1][lane];
        }
    }
    __syncthreads();
  }
  if (slice != 0 || !tile) return;
  const double nn = (double)n * (double)n;
  float2* mq = Mq + (size_t)clip * W * W;
  float2* mp = Mp ? Mp + (size_t)clip * (W + 1) * W : nullptr;
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    const int col = kRectT * gc + j;
    if (col >= W) break;
#pragma unroll
    for (int i = 0; i < kRectT; ++i) {
      const int row = kRectT * gr + i;
      if (row >= W) break;
      const bool live = xl[j] && yl[i];
      double vr = live ? re[i][j] : 0.0, vi = live ? im[i][j] : 0.0;
      if (col == BB && row == BB) {  // kx = ky = 0: the background
        vr += bg[2 * clip] * nn;
        vi += bg[2 * clip + 1] * nn;
      }
      const float2 v = make_float2((float)vr, (float)vi);
      mq[(size_t)col * W + row] = v;
      if (mp) {
        // column-paired copy: (col, row) at [(col + 1) / 2][row][(col + 1) % 2], column -1 zero
        mp[((size_t)((col + 1) >> 1) * W + row) * 2 + ((col + 1) & 1)] = v;
        if (col == 0) mp[(size_t)row * 2] = make_float2(0.f, 0.f);
      }
    }
  }
}

// One edge's term of a tile's bins: x the edge's column table, yv its row entries.
__device__ __forceinline__ void poly_edge(const double4* x, const int* xi, const double4* yv,
                                          double dx, double dy, double dk, int mx0, int my0,
                                          double (&ar)[kRectT][kRectT],
                                          double (&ai)[kRectT][kRectT]) {
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    const double4 xv = x[xi[j]];  // one column at a time (register budget)
    const double kx = dk * (mx0 + j);
#pragma unroll
    for (int i = 0; i < kRectT; ++i) {
      const double ky = dk * (my0 + i);
      const double kn = kx * dy - ky * dx;
      const double u = 0.5 * (kx * dx + ky * dy);
      const double su = xv.w * yv[i].z + xv.z * yv[i].w;
      double r = __builtin_amdgcn_rcp(u);
      r = fma(r, fma(-u, r, 1.0), r);
      r = fma(r, fma(-u, r, 1.0), r);
      const double sc = fabs(u) < 1e-4 ? 1.0 - u * u * (1.0 / 6.0) : su * r;
      const double a = kn * sc;
      const double hr = xv.x * yv[i].x - xv.y * yv[i].y;
      const double hi = xv.x * yv[i].y + xv.y * yv[i].x;
      ar[i][j] = fma(a, hr, ar[i][j]);
      ai[i][j] = fma(a, hi, ai[i][j]);
    }
  }
}

// The bin of orders (mx, my) from its edge sum (re, im): i / |k|^2 of it, or the area at
// the origin, in the box's scale and phase.
__device__ __forceinline__ double2 poly_bin(int mx, int my, double re, double im,
                                            const double* pdc, double dk, double scale, double nf) {
  double fr, fi;
  if (mx == 0 && my == 0) {
    fr = pdc[0];
    fi = pdc[1];
  } else {
    const double kx = dk * mx, ky = dk * my;
    const double inv = 1.0 / (kx * kx + ky * ky);
    fr = -im * inv;
    fi = re * inv;
  }
  double tt = (double)(mx + my) * (nf - 1.0) / nf;
  tt -= 2.0 * rint(0.5 * tt);
  double sv, cv;
  sincospi(-tt, &sv, &cv);
  return make_double2(scale * (fr * cv - fi * sv), scale * (fr * sv + fi * cv));
}

// Adds v to what the rectangle pass stored at (col, row).
__device__ __forceinline__ void poly_add(float2* mq, float2* mp, int W, int col, int row,
                                         double vr, double vi) {
  float2* q = mq + (size_t)col * W + row;
  const float2 old = *q;
  const float2 v = make_float2((float)((double)old.x + vr), (float)((double)old.y + vi));
  *q = v;
  if (mp) mp[((size_t)((col + 1) >> 1) * W + row) * 2 + ((col + 1) & 1)] = v;
}

// Simple polygons (mask.rs:1286-1352): for k = 2 pi m / L != 0
//   \iint_P e^{-ik.r} = (i/|k|^2) sum_e s (kx dy - ky dx) sinc(k.d/2) e^{-ik.r_mid}
// with s the polygon's orientation sign, and the area at k = 0.  edges:
// (dx, dy, cx, cy, re, im) with (re, im) = s (value - background); pdc per
// clip = sum of (value - background) area.  The box bins |kx|, |ky| <= B get
//   (N^2/L^2) e^{-i pi (mx + my)(N - 1)/N} x integral
// added to what the rectangle pass stored (plain and column-paired).
// The form for bands above 63: wpc work-groups per clip (of up to 512 threads), one
// thread per tile of kRectT rows x kRectT columns.  The clip's edges
// are taken in chunks; for each chunk the work-group first tabulates, per edge
// and order m in [-B, B], w e^{-i kx cx} with (cos, sin)(kx dx / 2) and
// e^{-i ky cy} with (cos, sin)(ky dy / 2) in LDS, then every tile reads its
// kRectT columns and rows from there: sin(k.d/2) is the sine of the sum of
// the two half-angles, sinc switches to its Taylor series below |u| = 1e-4
// (where that sum loses relative accuracy), and 1/u is the hardware
// reciprocal refined by two Newton steps.
__global__ __launch_bounds__(512) void k_poly_band(const double* __restrict__ edges,
                                                   const int64_t* __restrict__ eoff,
                                                   const double* __restrict__ pdc, int n,
                                                   double L, int B, int BB, int chunk, int wpc,
                                                   float2* __restrict__ Mq,
                                                   float2* __restrict__ Mp) {
  extern __shared__ double4 tab[];  // [axis][edge in chunk][m + B]
  const int W = 2 * BB + 1, nk = 2 * B + 1;
  const int G = (W + kRectT - 1) / kRectT;
  const int clip = blockIdx.x / wpc;
  const int t = (blockIdx.x - clip * wpc) * blockDim.x + threadIdx.x;  // tile index
  const int64_t e0 = eoff[clip], e1 = eoff[clip + 1];
  if (e0 == e1) return;  // uniform over the work-group
  const bool active = t < G * G;
  const int gc = active ? t / G : 0, gr = active ? t - (t / G) * G : 0;
  const int mx0 = kRectT * gc - BB, my0 = kRectT * gr - BB;
  const double dk = 2.0 * M_PI / L;
  int xi[kRectT], yi[kRectT];
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    xi[j] = min(max(mx0 + j + B, 0), nk - 1);
    yi[j] = min(max(my0 + j + B, 0), nk - 1);
  }
  double ar[kRectT][kRectT], ai[kRectT][kRectT];
#pragma unroll
  for (int i = 0; i < kRectT; ++i)
#pragma unroll
    for (int j = 0; j < kRectT; ++j) ar[i][j] = ai[i][j] = 0.0;
  for (int64_t cb = e0; cb < e1; cb += chunk) {
    const int ne = (int)min((int64_t)chunk, e1 - cb);
    __syncthreads();  // the previous chunk's tables are consumed
    for (int q = threadIdx.x; q < 2 * ne * nk; q += blockDim.x) {
      const int axis = q / (ne * nk), r = q - axis * ne * nk;
      const int el = r / nk, mi = r - el * nk;
      const double* p = edges + 6 * (cb + el);
      const double k = dk * (mi - B);
      double sv, cv, sh, ch;
      sincos(k * (axis == 0 ? p[2] : p[3]), &sv, &cv);
      sincos(0.5 * k * (axis == 0 ? p[0] : p[1]), &sh, &ch);
      // e^{-i k c}, times the edge weight on the x axis
      double pr = cv, pi = -sv;
      if (axis == 0) {
        const double wr = p[4], wi = p[5];
        const double tr = wr * pr - wi * pi;
        pi = wr * pi + wi * pr;
        pr = tr;
      }
      tab[(axis * chunk + el) * nk + mi] = make_double4(pr, pi, ch, sh);
    }
    __syncthreads();
    if (active) {
      for (int el = 0; el < ne; ++el) {
        const double dx = edges[6 * (cb + el)], dy = edges[6 * (cb + el) + 1];
        double4 yv[kRectT];
#pragma unroll
        for (int i = 0; i < kRectT; ++i) yv[i] = tab[(chunk + el) * nk + yi[i]];
        // poly_edge's sum written out: as a call it is scheduled 3 to 5 % slower here (24
        // clips, band 64: 331 against 317 us; the sliced form below does not mind)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          const double4 xv = tab[el * nk + xi[j]];  // one column at a time (register budget)
          const double kx = dk * (mx0 + j);
#pragma unroll
          for (int i = 0; i < kRectT; ++i) {
            const double ky = dk * (my0 + i);
            const double kn = kx * dy - ky * dx;
            const double u = 0.5 * (kx * dx + ky * dy);
            const double su = xv.w * yv[i].z + xv.z * yv[i].w;
            double r = __builtin_amdgcn_rcp(u);
            r = fma(r, fma(-u, r, 1.0), r);
            r = fma(r, fma(-u, r, 1.0), r);
            const double sc = fabs(u) < 1e-4 ? 1.0 - u * u * (1.0 / 6.0) : su * r;
            const double a = kn * sc;
            const double hr = xv.x * yv[i].x - xv.y * yv[i].y;
            const double hi = xv.x * yv[i].y + xv.y * yv[i].x;
            ar[i][j] = fma(a, hr, ar[i][j]);
            ai[i][j] = fma(a, hi, ai[i][j]);
          }
        }
      }
    }
  }
  if (!active) return;
  const double nf = (double)n, scale = nf * nf / (L * L);
  float2* mq = Mq + (size_t)clip * W * W;
  float2* mp = Mp ? Mp + (size_t)clip * (W + 1) * W : nullptr;
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    const int col = kRectT * gc + j, mx = mx0 + j;
    if (col >= W) break;
#pragma unroll
    for (int i = 0; i < kRectT; ++i) {
      const int row = kRectT * gr + i, my = my0 + i;
      if (row >= W) break;
      if (mx < -B || mx > B || my < -B || my > B) continue;
      const double2 v = poly_bin(mx, my, ar[i][j], ai[i][j], pdc + 2 * clip, dk, scale, nf);
      poly_add(mq, mp, W, col, row, v.x, v.y);
    }
  }
}

// The same for bands up to 63.  Work-group = 64 tiles x 8 waves, each wave taking every
// eighth edge (one of a chunk of eight), so that few clips fill the chip: wpc
// work-groups per clip.  The tables of a chunk are products of two short ones, orders
// 16 a and b < 16 (m = 16 a + b), so an edge and axis take at most 24 pairs of sincos
// instead of 2 B + 1.  HERM, where no edge has an imaginary weight: only the columns
// kx <= 0 are summed, each bin's conjugate going to its mirror image.
// What bounds it: the FP64 products and one work-group's registers per CU.  96 clips of
// real polygons, B = 47: 430 us with one thread per tile, every bin and long tables
// (192 work-groups of five waves), 413 with half the bins and half the work-groups, 238
// so; at 128 registers, for two work-groups per CU, it spills (416).
template <bool HERM>
__global__ __launch_bounds__(512) void k_poly_band_sliced(
    const double* __restrict__ edges, const int64_t* __restrict__ eoff,
    const double* __restrict__ pdc, int n, double L, int B, int BB, int wpc,
    float2* __restrict__ Mq, float2* __restrict__ Mp) {
  constexpr int E = kPolySlices;
  extern __shared__ double4 tab[];  // [axis][edge in chunk][m + B], then the short tables
  const int W = 2 * BB + 1, nk = 2 * B + 1;
  const int G = (W + kRectT - 1) / kRectT;
  const int clip = blockIdx.x / wpc;
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int t = (blockIdx.x - clip * wpc) * 64 + lane;  // tile index
  const int64_t e0 = eoff[clip], e1 = eoff[clip + 1];
  if (e0 == e1) return;  // uniform over the work-group
  const bool active = t < (HERM ? BB / kRectT + 1 : G) * G;
  const int gc = active ? t / G : 0, gr = active ? t - (t / G) * G : 0;
  const int mx0 = kRectT * gc - BB, my0 = kRectT * gr - BB;
  const double dk = 2.0 * M_PI / L;
  const int A = (B + 15) / 16, NS = 2 * A + 1 + 16;  // orders 16 (-A .. A), then 0 .. 15
  double4* const sht = tab + 2 * E * nk;             // [axis][edge][NS]
  int xi[kRectT], yi[kRectT];
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    xi[j] = min(max(mx0 + j + B, 0), nk - 1);
    yi[j] = min(max(my0 + j + B, 0), nk - 1);
  }
  double ar[kRectT][kRectT], ai[kRectT][kRectT];
#pragma unroll
  for (int i = 0; i < kRectT; ++i)
#pragma unroll
    for (int j = 0; j < kRectT; ++j) ar[i][j] = ai[i][j] = 0.0;
  for (int64_t cb = e0; cb < e1; cb += E) {
    const int ne = (int)min((int64_t)E, e1 - cb);
    for (int q = threadIdx.x; q < 2 * ne * NS; q += 512) {
      const int axis = q / (ne * NS), r = q - axis * ne * NS;
      const int el = r / NS, i = r - el * NS;
      const double* p = edges + 6 * (cb + el);
      const double k = dk * (i <= 2 * A ? 16 * (i - A) : i - 2 * A - 1);
      double sv, cv, sh, ch;
      sincos(k * (axis == 0 ? p[2] : p[3]), &sv, &cv);
      sincos(0.5 * k * (axis == 0 ? p[0] : p[1]), &sh, &ch);
      double pr = cv, pi = -sv;  // e^{-i k c}, times the edge weight on the x axis, once
      if (axis == 0 && i <= 2 * A) {
        const double wr = p[4], wi = p[5];
        const double tr = wr * pr - wi * pi;
        pi = wr * pi + wi * pr;
        pr = tr;
      }
      sht[(axis * E + el) * NS + i] = make_double4(pr, pi, ch, sh);
    }
    __syncthreads();  // the short tables; and the previous chunk has been consumed
    for (int q = threadIdx.x; q < 2 * ne * nk; q += 512) {
      const int axis = q / (ne * nk), r = q - axis * ne * nk;
      const int el = r / nk, mi = r - el * nk, m = mi - B + 16 * A;
      const double4* s = sht + (axis * E + el) * NS;
      const double4 u = s[m >> 4], v = s[2 * A + 1 + (m & 15)];
      tab[(axis * E + el) * nk + mi] =
          make_double4(u.x * v.x - u.y * v.y, u.x * v.y + u.y * v.x, u.z * v.z - u.w * v.w,
                       u.w * v.z + u.z * v.w);
    }
    __syncthreads();
    if (active && slice < ne) {
      const double dx = edges[6 * (cb + slice)], dy = edges[6 * (cb + slice) + 1];
      double4 yv[kRectT];
#pragma unroll
      for (int i = 0; i < kRectT; ++i) yv[i] = tab[(E + slice) * nk + yi[i]];
      poly_edge(tab + slice * nk, xi, yv, dx, dy, dk, mx0, my0, ar, ai);
    }
  }
  // the waves' sums, by halves
  double* const red = reinterpret_cast<double*>(tab);
#pragma unroll
  for (int h = E / 2; h >= 1; h /= 2) {
    __syncthreads();
    if (slice >= h && slice < 2 * h) {
#pragma unroll
      for (int i = 0; i < kRectT; ++i)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          double* r = red + ((slice - h) * 2 * kRectT * kRectT + 2 * (i * kRectT + j)) * 64 + lane;
          r[0] = ar[i][j];
          r[64] = ai[i][j];
        }
    }
    __syncthreads();
    if (slice < h) {
#pragma unroll
      for (int i = 0; i < kRectT; ++i)
#pragma unroll
        for (int j = 0; j < kRectT; ++j) {
          const double* r = red + (slice * 2 * kRectT * kRectT + 2 * (i * kRectT + j)) * 64 + lane;
          ar[i][j] += r[0];
          ai[i][j] += r[64];
        }
    }
  }
  if (!active || slice != 0) return;
  const double nf = (double)n, scale = nf * nf / (L * L);
  float2* mq = Mq + (size_t)clip * W * W;
  float2* mp = Mp ? Mp + (size_t)clip * (W + 1) * W : nullptr;
#pragma unroll
  for (int j = 0; j < kRectT; ++j) {
    const int col = kRectT * gc + j, mx = mx0 + j;
    if (col >= W || (HERM && mx > 0)) break;
#pragma unroll
    for (int i = 0; i < kRectT; ++i) {
      const int row = kRectT * gr + i, my = my0 + i;
      if (row >= W) break;
      if (mx < -B || mx > B || my < -B || my > B) continue;
      const double2 v = poly_bin(mx, my, ar[i][j], ai[i][j], pdc + 2 * clip, dk, scale, nf);
      poly_add(mq, mp, W, col, row, v.x, v.y);
      if (HERM && mx < 0) poly_add(mq, mp, W, 2 * BB - col, 2 * BB - row, v.x, -v.y);
    }
  }
}

hipError_t launch_poly_band(const double* edges, const int64_t* eoff, const double* pdc,
                            bool real, int nclips, int n, double L, int B, int BB, float2* Mq,
                            float2* Mp, hipStream_t s) {
  if (nclips <= 0) return hipSuccess;
  if (B < 0 || BB < B || B > kPolyMaxBand || BB > 1024) return hipErrorInvalidValue;
  const int W = 2 * BB + 1, nk = 2 * B + 1;
  const int G = (W + kRectT - 1) / kRectT;
  // Eight edges' tables take up to 78 KiB of LDS at 63, the widest band of an image; a
  // wider one would leave most waves without an edge.
  if (B <= 63) {
    const int tiles = (real ? BB / kRectT + 1 : G) * G, wpc = (tiles + 63) / 64;
    if ((int64_t)wpc * nclips >= (1ll << 31)) return hipErrorInvalidValue;
    const int ns = 2 * ((B + 15) / 16) + 17;
    const size_t lds = std::max((size_t)2 * kPolySlices * (nk + ns) * sizeof(double4),
                                (size_t)kPolySlices * kRectT * kRectT * 64 * sizeof(double));
    auto kern = real ? k_poly_band_sliced<true> : k_poly_band_sliced<false>;
    // sized for B = 63, once each
    constexpr int most = 2 * kPolySlices * (127 + 25) * (int)sizeof(double4);
    static const hipError_t attr[2] = {
        hipFuncSetAttribute((const void*)k_poly_band_sliced<false>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, most),
        hipFuncSetAttribute((const void*)k_poly_band_sliced<true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, most)};
    if (attr[real] != hipSuccess) return attr[real];
    hipLaunchKernelGGL(kern, dim3((unsigned)(wpc * nclips)), dim3(512), lds, s, edges, eoff, pdc, n,
                       L, B, BB, wpc, Mq, Mp);
    return hipGetLastError();
  }
  const int wpc = (G * G + 511) / 512;
  const int threads = ((((G * G + wpc - 1) / wpc) + 63) / 64) * 64;
  if ((int64_t)wpc * nclips >= (1ll << 31)) return hipErrorInvalidValue;
  // edges per chunk: two tables of nk 32-byte entries per edge within 48 KiB of LDS
  const int chunk = std::max(1, (48 * 1024) / (2 * nk * (int)sizeof(double4)));
  const size_t lds = (size_t)2 * chunk * nk * sizeof(double4);
  hipLaunchKernelGGL(k_poly_band, dim3((unsigned)(wpc * nclips)), dim3(threads), lds, s, edges,
                     eoff, pdc, n, L, B, BB, chunk, wpc, Mq, Mp);
  return hipGetLastError();
}

hipError_t launch_rect_tables(const double* cells, int64_t ncells, int n, double L, int B,
                              double2* X, double2* Y, hipStream_t s) {
  if (ncells <= 0) return hipSuccess;
  const int64_t total = ncells * (2 * B + 1);
  const int64_t blocks = (total + 255) / 256;
  if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_rect_tables, dim3((unsigned)blocks), dim3(256), 0, s, cells, ncells, n, L,
                     B, X, Y);
  return hipGetLastError();
}

hipError_t launch_rect_band(const double2* X, const double2* Y, const int64_t* coff,
                            int64_t ncells, const double* bg, int nclips, int n, int B, int BB,
                            float2* Mq, float2* Mp, hipStream_t s) {
  if (nclips <= 0) return hipSuccess;
  if (B < 0 || BB < B || BB > 1024) return hipErrorInvalidValue;
  const int W = 2 * BB + 1;
  const int G = (W + kRectT - 1) / kRectT;
  const int gpc = (G * G + 63) / 64;
  if ((int64_t)gpc * nclips >= (1ll << 31)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(gpc * nclips));
  // Eight waves where there is at most one work-group per CU and each wave has a cell or
  // two, else two.  Band 47, us with two and eight waves: 24 clips (216 work-groups) of 8
  // cells 8.1 and 8.8, of 16 10.0 and 9.4, of 43 16.0 and 12.3; 56 clips (504) of 43 18.3
  // and 19.6, of none 6.8 and 10.3.
  if (gpc * nclips <= 256 && ncells >= 12 * (int64_t)nclips)
    hipLaunchKernelGGL(k_rect_band<8>, grid, dim3(512), 0, s, X, Y, coff, bg, n, B, BB, gpc, Mq,
                       Mp);
  else
    hipLaunchKernelGGL(k_rect_band<2>, grid, dim3(128), 0, s, X, Y, coff, bg, n, B, BB, gpc, Mq,
                       Mp);
  return hipGetLastError();
}

}  // namespace huvk
