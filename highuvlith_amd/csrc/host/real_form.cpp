// The real fields of a SOCS kernel set, for masks with a real transmittance.
//
// The spectrum of a real mask is Hermitian, M(-f) = conj M(f).  A Hermitian
// function H then gives a real field (the product H M is Hermitian), and every
// kernel splits into two of them, K = H + i A with H = (K(f) + conj K(-f)) / 2
// and A = (K(f) - conj K(-f)) / (2 i), so
//   I = sum_k lambda_k |E_k|^2 = sum_k lambda_k (h_k^2 + a_k^2)
// is a real quadratic form on the 2K real fields.  Its eigenvectors are real
// fields v_j with I = sum_j v_j^2 exactly; where the optics make the 2K fields
// dependent (an in-focus pupil with a point-symmetric source: every kernel is
// real up to a phase) only about K of them are non-zero, and two real fields
// travel as one complex field v_j + i v_{j+1} (|.|^2 = v_j^2 + v_{j+1}^2).
// The decomposition is computed from the kernels themselves (no assumption on
// the optics), in FP64.
#include <algorithm>
#include <cmath>

#include "engine.hpp"

namespace huv {

namespace {

// Two doubles of a row, at the 8-byte alignment of any element.
typedef double v2 __attribute__((vector_size(16), aligned(8), may_alias));

// Hermitian functions on the (2B+1)^2 box as real vectors of the same length:
// the Gram products sum over both f and -f, so the half box carries sqrt(2).
// Rows of such vectors lie at an even stride, zero behind the last element.
size_t row_stride(size_t n) { return (n + 1) / 2 * 2; }

// out[i][j] = a_i . b_j (ra x rb), of rows of length n at stride row_stride(n);
// symmetric: a == b and only j >= i - 3 is computed.  Tiles of 4 x 2 products over
// stretches of the rows that stay in cache: 256 rows of 109^2 take 0.06 s, row pair
// by row pair 0.14.
void dots(const double* a, int ra, const double* b, int rb, size_t n, bool symmetric,
          std::vector<double>& out) {
  const size_t st = row_stride(n), kStretch = 512;
  out.assign((size_t)ra * rb, 0.0);
  for (size_t x0 = 0; x0 < st; x0 += kStretch) {
    const size_t x1 = std::min(st, x0 + kStretch);
    for (int i = 0; i < ra; i += 4)
      for (int j = symmetric ? i : 0; j < rb; j += 2) {
        const double *p[4], *q[2];  // rows past the last are read as it, not stored
        for (int u = 0; u < 4; ++u) p[u] = a + (size_t)std::min(i + u, ra - 1) * st;
        for (int u = 0; u < 2; ++u) q[u] = b + (size_t)std::min(j + u, rb - 1) * st;
        v2 s[4][2] = {};
        for (size_t x = x0; x < x1; x += 2) {
          const v2 q0 = *(const v2*)(q[0] + x), q1 = *(const v2*)(q[1] + x);
          for (int u = 0; u < 4; ++u) {
            const v2 w = *(const v2*)(p[u] + x);
            s[u][0] += w * q0;
            s[u][1] += w * q1;
          }
        }
        for (int u = 0; u < 4 && i + u < ra; ++u)
          for (int t = 0; t < 2 && j + t < rb; ++t)
            out[(size_t)(i + u) * rb + j + t] += s[u][t][0] + s[u][t][1];
      }
  }
}

// o_j += sum_i u[j][i] f_i (ro x rf) for rows as above; 4 rows x 4 columns at a time.
void combine(const double* u, const double* f, int rf, size_t n, int ro, double* o) {
  const size_t st = row_stride(n), kStretch = 128;
  for (size_t x0 = 0; x0 < st; x0 += kStretch) {
    const size_t x1 = std::min(st, x0 + kStretch);
    for (int j = 0; j < ro; j += 4) {
      const double* c[4];
      for (int t = 0; t < 4; ++t) c[t] = u + (size_t)std::min(j + t, ro - 1) * rf;
      size_t x = x0;
      for (; x + 4 <= x1; x += 4) {
        v2 s[4][2] = {};
        for (int i = 0; i < rf; ++i) {
          const double* fi = f + (size_t)i * st + x;
          const v2 f0 = *(const v2*)fi, f1 = *(const v2*)(fi + 2);
          for (int t = 0; t < 4; ++t) {
            const v2 k = {c[t][i], c[t][i]};
            s[t][0] += k * f0;
            s[t][1] += k * f1;
          }
        }
        for (int t = 0; t < 4 && j + t < ro; ++t) {
          *(v2*)(o + (size_t)(j + t) * st + x) += s[t][0];
          *(v2*)(o + (size_t)(j + t) * st + x + 2) += s[t][1];
        }
      }
      for (; x < x1; ++x)
        for (int t = 0; t < 4 && j + t < ro; ++t) {
          double s = 0.0;
          for (int i = 0; i < rf; ++i) s += c[t][i] * f[(size_t)i * st + x];
          o[(size_t)(j + t) * st + x] += s;
        }
    }
  }
}

// Both limits are parts of the largest intensity that one unit order gives (peak),
// the clear field where the optics pass the zero order: a form of norm q moves no
// image of a mask by more than q times the mean of its squared transmittance.
// (The trace would be no such scale: it grows with the band's area, to 153 .. 2469
// clear fields for the annular source at 2 nm, 512^2 .. 2048^2.)
// The dropped eigenvalues' sum: what one FP32 rounding of the clear field is.
constexpr double kDrop = 1.0 / (double)(1 << 25);
// How far two planes' forms may differ (Frobenius norm) to count as one: half of
// that.  Opposite focus planes of a point-symmetric source are 1e-12 apart.
constexpr double kSame = 1.0 / (double)(1 << 26);

// The real and imaginary parts h_k, a_k of every kernel as rows, scaled by the root
// of its eigenvalue (2K x row_stride((2B + 1)^2)); false for input without a form.
bool kernel_rows(int n, int B, int K, int64_t S, const int64_t* support, const double* eig,
                 const double* values, std::vector<double>& v) {
  if (K < 1 || K > kRealFieldsMaxKernels) return false;
  double emax = 0.0;
  for (int k = 0; k < K; ++k) {
    if (!std::isfinite(eig[k]) || eig[k] < 0.0) return false;
    emax = std::max(emax, eig[k]);
  }
  for (int64_t t = 0; t < 2 * K * S; ++t)
    if (!std::isfinite(values[t])) return false;
  if (!(emax > 0.0)) return false;
  const int W = 2 * B + 1;
  const size_t N = (size_t)W * W, half = (N - 1) / 2;  // box index of -f: N - 1 - index
  const size_t st = row_stride(N);
  const double r2 = std::sqrt(2.0);
  v.assign((size_t)2 * K * st, 0.0);
  std::vector<cd> box(N);
  for (int k = 0; k < K; ++k) {
    std::fill(box.begin(), box.end(), cd(0, 0));
    const double s = std::sqrt(eig[k]);
    for (int64_t t = 0; t < S; ++t) {
      const int64_t i = support[t] / n, j = support[t] % n;
      const int64_t ky = i < n / 2 ? i : i - n, kx = j < n / 2 ? j : j - n;
      box[(size_t)(kx + B) * W + (ky + B)] =
          s * cd(values[2 * (k * S + t)], values[2 * (k * S + t) + 1]);
    }
    double* h = v.data() + (size_t)(2 * k) * st;
    double* a = h + st;
    for (size_t i = 0; i < half; ++i) {
      const cd p = box[i], q = std::conj(box[N - 1 - i]);
      const cd hh = 0.5 * (p + q), aa = cd(0.0, -0.5) * (p - q);
      h[2 * i] = r2 * hh.real();
      h[2 * i + 1] = r2 * hh.imag();
      a[2 * i] = r2 * aa.real();
      a[2 * i + 1] = r2 * aa.imag();
    }
    h[N - 1] = box[half].real();
    a[N - 1] = box[half].imag();
  }
  return true;
}

}  // namespace

bool real_form(int n, int B, int K, int64_t S, const int64_t* support, const double* eig,
               const double* values, bool fewer_only, RealFields& out) {
  out = RealFields();
  std::vector<double> v, g;
  if (!kernel_rows(n, B, K, S, support, eig, values, v)) return false;
  const int F = 2 * K;
  const size_t N = (size_t)(2 * B + 1) * (2 * B + 1), st = row_stride(N);
  dots(v.data(), F, v.data(), F, N, true, g);
  for (int i = 0; i < F; ++i)
    for (int j = i; j < F; ++j) g[(size_t)j * F + i] = g[(size_t)i * F + j];
  std::vector<double> mu, U;
  if (!symmetric_eigen_desc(g, F, 0, mu, U)) return false;
  double trace = 0.0, peak = 0.0;
  for (double m : mu) trace += std::max(m, 0.0);
  std::vector<double> power((N + 1) / 2, 0.0);  // sum of |v(f)|^2 over the half box
  for (int i = 0; i < F; ++i) {
    const double* p = v.data() + (size_t)i * st;
    for (size_t x = 0; x + 1 < N; x += 2)
      power[x / 2] += 0.5 * (p[x] * p[x] + p[x + 1] * p[x + 1]);
    power[N / 2] += p[N - 1] * p[N - 1];
  }
  for (double p : power) peak = std::max(peak, p);
  if (!(peak > 0.0) || !std::isfinite(trace)) return false;
  int R = F;
  double tail = 0.0;
  while (R > 1 && tail + std::max(mu[R - 1], 0.0) <= kDrop * peak) tail += std::max(mu[--R], 0.0);
  const bool fields = !fewer_only || (R + 1) / 2 < K;
  if (fields && !symmetric_eigen_desc(g, F, R, mu, U)) return false;
  out.B = B;
  out.R = R;
  out.trace = trace;
  out.peak = peak;
  out.mu.assign(mu.begin(), mu.begin() + R);
  if (fields) {
    out.v.assign((size_t)R * st, 0.0);
    combine(U.data(), v.data(), F, N, R, out.v.data());
  }
  return true;
}

cd real_field_value(const RealFields& f, int j, int kx, int ky) {
  const int W = 2 * f.B + 1;
  const size_t N = (size_t)W * W, half = (N - 1) / 2;
  const size_t i = (size_t)(kx + f.B) * W + (ky + f.B);
  const double* v = f.v.data() + (size_t)j * row_stride(N);
  const double s = std::sqrt(0.5);
  if (i == half) return cd(v[N - 1], 0.0);
  if (i < half) return s * cd(v[2 * i], v[2 * i + 1]);
  return s * cd(v[2 * (N - 1 - i)], -v[2 * (N - 1 - i) + 1]);
}

bool same_eigenvalues(const RealFields& a, const RealFields& b) {
  if (a.R < 1 || a.R != b.R || a.B != b.B) return false;
  for (int j = 0; j < a.R; ++j)
    if (!(std::fabs(a.mu[j] - b.mu[j]) <= kSame * a.peak)) return false;
  return true;
}

// I = sum v_j^2 is the same form for both sets when b's fields lie in a's span
// with orthonormal coordinates; both defects are formed without cancellation.
bool same_real_form(const RealFields& a, const RealFields& b) {
  if (!same_eigenvalues(a, b) || a.v.empty() || b.v.empty()) return false;
  const int R = a.R;
  const size_t N = (size_t)(2 * a.B + 1) * (2 * a.B + 1), st = row_stride(N);
  std::vector<double> c, cc;  // c[i][l] = a_i . b_l; b_l = sum_i c[i][l] a_i / mu_i
  dots(a.v.data(), R, b.v.data(), R, N, false, c);
  // || M^(1/2) (C C^T - 1) M^(1/2) ||_F^2, C = M^-1 c
  std::vector<double> rows((size_t)R * row_stride(R), 0.0);
  for (int i = 0; i < R; ++i)
    std::copy(c.begin() + (size_t)i * R, c.begin() + (size_t)(i + 1) * R,
              rows.begin() + (size_t)i * row_stride(R));
  dots(rows.data(), R, rows.data(), R, R, false, cc);
  double in = 0.0;
  for (int i = 0; i < R; ++i)
    for (int k = 0; k < R; ++k) {
      const double w = std::sqrt(a.mu[i] * a.mu[k]);
      const double d = cc[(size_t)i * R + k] / w - (i == k ? a.mu[i] : 0.0);
      in += d * d;
    }
  // squared norm of what leaves the span
  std::vector<double> left(b.v), coef((size_t)R * R);
  for (int l = 0; l < R; ++l)
    for (int i = 0; i < R; ++i) coef[(size_t)l * R + i] = -c[(size_t)i * R + l] / a.mu[i];
  combine(coef.data(), a.v.data(), R, N, R, left.data());
  double res = 0.0;
  for (size_t x = 0; x < (size_t)R * st; ++x) res += left[x] * left[x];
  return std::sqrt(in) + 2.0 * std::sqrt(res * a.trace) <= kSame * a.peak;
}

}  // namespace huv
