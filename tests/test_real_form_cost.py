"""What a first call spends on a kernel set's real form: the eigenvalues alone where
nothing is gained, at a fraction of the fields' cost, and they say the same.  The
blocked sums agree with plain ones at row counts off their tiles.
"""
import os
import subprocess

import highuvlith_amd as H

HOST = os.path.join(os.path.dirname(os.path.abspath(H.__file__)), "csrc", "host")

FORMS = r"""
#include <chrono>
#include <cmath>
#include <cstdio>
#include <random>
#include "engine.hpp"
using namespace huv;
struct Set { int n, B, K; std::vector<int64_t> sup; std::vector<double> eig, val; };
static Set make(int K, int B, int seed) {
  Set s{512, B, K, {}, std::vector<double>(K), {}};
  for (int y = -B; y <= B; ++y)
    for (int x = -B; x <= B; ++x)
      if (x * x + y * y <= B * B) s.sup.push_back((int64_t)((y + s.n) % s.n) * s.n + (x + s.n) % s.n);
  std::mt19937_64 g(seed);
  std::normal_distribution<double> nd;
  for (int k = 0; k < K; ++k) s.eig[k] = std::pow(0.9, k);
  s.val.resize(2 * K * s.sup.size());
  for (double& v : s.val) v = nd(g) / std::sqrt(2.0 * s.sup.size());
  return s;
}
static bool form(const Set& s, bool fields, RealFields& rf) {
  return real_form(s.n, s.B, s.K, (int64_t)s.sup.size(), s.sup.data(), s.eig.data(),
                   s.val.data(), !fields, rf);
}
static double seconds(const Set& s, bool fields) {
  RealFields rf;
  double best = 1e9;
  for (int r = 0; r < 3; ++r) {
    const auto t = std::chrono::steady_clock::now();
    if (!form(s, fields, rf)) return 1e9;
    best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t).count());
  }
  return best;
}
int main() {
  for (int K : {1, 2, 3, 5, 7, 33})
    for (int B : {1, 2, 9, 20}) {
      const Set s = make(K, B, K + B);
      RealFields a, b;
      if (!form(s, false, a) || !form(s, true, b)) return 1;
      if (a.R != b.R || a.B != b.B || a.mu != b.mu || a.peak != b.peak ||
          !a.v.empty() != ((a.R + 1) / 2 < K))
        return 2;
      // each field's squared norm is its eigenvalue, and the fields are orthogonal
      const int W = 2 * B + 1;
      for (int i = 0; i < b.R; ++i)
        for (int j = 0; j <= i; ++j) {
          double d = 0.0;
          for (int x = -B; x <= B; ++x)
            for (int y = -B; y <= B; ++y)
              d += (std::conj(real_field_value(b, i, x, y)) * real_field_value(b, j, x, y)).real();
          if (std::fabs(d - (i == j ? b.mu[i] : 0.0)) > 1e-12 * b.mu[0]) return 3;
        }
      // the sum of the squared fields is the sum of the squared kernels, order by order
      double got = 0.0, want = 0.0;
      for (int j = 0; j < b.R; ++j) got += std::norm(real_field_value(b, j, 0, 0));
      for (int k = 0; k < K; ++k)
        for (size_t t = 0; t < s.sup.size(); ++t)
          if (s.sup[t] == 0)
            want += s.eig[k] * std::norm(cd(s.val[2 * (k * s.sup.size() + t)],
                                            s.val[2 * (k * s.sup.size() + t) + 1]));
      if (std::fabs(got - want) > 1e-6 * b.peak || W < 3) return 4;
      if (!same_eigenvalues(a, b) || !same_real_form(b, b)) return 5;
    }
  const Set big = make(128, 27, 1);
  const double less = seconds(big, false), all = seconds(big, true);
  std::printf("128 kernels, band 27: eigenvalues %.3f s, fields %.3f s\n", less, all);
  return less <= 0.6 * all ? 0 : 6;
}
"""


def test_eigenvalues_alone(tmp_path):
    src, exe = tmp_path / "forms.cpp", tmp_path / "forms"
    src.write_text(FORMS)
    subprocess.run(["g++", "-O3", "-std=c++17", "-I", HOST, str(src),
                    os.path.join(HOST, "real_form.cpp"), os.path.join(HOST, "linalg.cpp"),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
