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

// Hermitian functions on the (2B+1)^2 box as real vectors of the same length:
// the Gram products sum over both f and -f, so the half box carries sqrt(2).
double dotr(const double* a, const double* b, size_t n) {
  double s[8] = {};
  size_t i = 0;
  for (; i + 8 <= n; i += 8)
    for (int u = 0; u < 8; ++u) s[u] += a[i + u] * b[i + u];
  for (; i < n; ++i) s[0] += a[i] * b[i];
  return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
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

}  // namespace

bool real_fields(int n, int B, int K, int64_t S, const int64_t* support, const double* eig,
                 const double* values, RealFields& out) {
  out = RealFields();
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
  const int F = 2 * K;
  const double r2 = std::sqrt(2.0);
  std::vector<double> v((size_t)F * N, 0.0);
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
    double* h = v.data() + (size_t)(2 * k) * N;
    double* a = h + N;
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
  std::vector<cd> gram((size_t)F * F);
  for (int i = 0; i < F; ++i)
    for (int j = i; j < F; ++j)
      gram[(size_t)j * F + i] = gram[(size_t)i * F + j] =
          dotr(v.data() + (size_t)i * N, v.data() + (size_t)j * N, N);
  std::vector<double> mu;
  std::vector<cd> U;
  if (!hermitian_eigen_desc(gram, F, F, mu, U)) return false;
  double trace = 0.0;
  for (double m : mu) trace += std::max(m, 0.0);
  std::vector<double> power(half + 1, 0.0);  // sum of |v(f)|^2 over the half box
  for (int i = 0; i < F; ++i) {
    const double* p = v.data() + (size_t)i * N;
    for (size_t x = 0; x < half; ++x)
      power[x] += 0.5 * (p[2 * x] * p[2 * x] + p[2 * x + 1] * p[2 * x + 1]);
    power[half] += p[N - 1] * p[N - 1];
  }
  double peak = 0.0;
  for (double p : power) peak = std::max(peak, p);
  if (!(peak > 0.0) || !std::isfinite(trace)) return false;
  int R = F;
  double tail = 0.0;
  while (R > 1 && tail + std::max(mu[R - 1], 0.0) <= kDrop * peak) tail += std::max(mu[--R], 0.0);
  for (int j = 0; j < R; ++j) {
    double im = 0.0;
    for (int i = 0; i < F; ++i) im = std::max(im, std::fabs(U[(size_t)j * F + i].imag()));
    if (im > 1e-10) return false;  // a real symmetric matrix has real eigenvectors
  }
  out.B = B;
  out.R = R;
  out.trace = trace;
  out.peak = peak;
  out.mu.assign(mu.begin(), mu.begin() + R);
  out.v.assign((size_t)R * N, 0.0);
  for (int j = 0; j < R; ++j) {
    double* o = out.v.data() + (size_t)j * N;
    for (int i = 0; i < F; ++i) {
      const double u = U[(size_t)j * F + i].real();
      const double* f = v.data() + (size_t)i * N;
      for (size_t x = 0; x < N; ++x) o[x] += u * f[x];
    }
  }
  return true;
}

cd real_field_value(const RealFields& f, int j, int kx, int ky) {
  const int W = 2 * f.B + 1;
  const size_t N = (size_t)W * W, half = (N - 1) / 2;
  const size_t i = (size_t)(kx + f.B) * W + (ky + f.B);
  const double* v = f.v.data() + (size_t)j * N;
  const double s = std::sqrt(0.5);
  if (i == half) return cd(v[N - 1], 0.0);
  if (i < half) return s * cd(v[2 * i], v[2 * i + 1]);
  return s * cd(v[2 * (N - 1 - i)], -v[2 * (N - 1 - i) + 1]);
}

// I = sum v_j^2 is the same form for both sets when b's fields lie in a's span
// with orthonormal coordinates; both defects are formed without cancellation.
bool same_real_form(const RealFields& a, const RealFields& b) {
  if (a.R < 1 || a.R != b.R || a.B != b.B) return false;
  for (int j = 0; j < a.R; ++j)
    if (std::fabs(a.mu[j] - b.mu[j]) > kSame * a.peak) return false;
  const int R = a.R;
  const size_t N = (size_t)(2 * a.B + 1) * (2 * a.B + 1);
  std::vector<double> c((size_t)R * R);  // c[i][l]: b_l = sum_i c[i][l] a_i / mu_i
  for (int i = 0; i < R; ++i)
    for (int l = 0; l < R; ++l)
      c[(size_t)i * R + l] = dotr(a.v.data() + (size_t)i * N, b.v.data() + (size_t)l * N, N);
  double in = 0.0;  // || M^(1/2) (C C^T - 1) M^(1/2) ||_F^2, C = M^-1 c
  for (int i = 0; i < R; ++i)
    for (int k = 0; k < R; ++k) {
      const double cc = dotr(c.data() + (size_t)i * R, c.data() + (size_t)k * R, R);
      const double w = std::sqrt(a.mu[i] * a.mu[k]);
      const double d = cc / w - (i == k ? a.mu[i] : 0.0);
      in += d * d;
    }
  double res = 0.0;  // squared norm of what leaves the span
  std::vector<double> r(N);
  for (int l = 0; l < R; ++l) {
    std::copy(b.v.begin() + (size_t)l * N, b.v.begin() + (size_t)(l + 1) * N, r.begin());
    for (int i = 0; i < R; ++i) {
      const double x = c[(size_t)i * R + l] / a.mu[i];
      const double* f = a.v.data() + (size_t)i * N;
      for (size_t k = 0; k < N; ++k) r[k] -= x * f[k];
    }
    res += dotr(r.data(), r.data(), N);
  }
  return std::sqrt(in) + 2.0 * std::sqrt(res * a.trace) <= kSame * a.peak;
}

}  // namespace huv
