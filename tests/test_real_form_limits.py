"""The real form of a kernel set against the set itself, as operators: the limits on
what it drops and on what counts as one image for two planes are parts of the clear
field (2^-25 and 2^-26), whatever the trace of the form, which grows with the area of
the band.

|I - I'| <= ||Q - Q'|| ||M||^2, Q the quadratic form on Hermitian spectra, and ||M||^2
the mean of a mask's squared transmittance, at most 1 here.
"""
import os
import subprocess

import numpy as np
import pytest

import highuvlith_amd as H
from highuvlith_amd import engine as E
from highuvlith_amd import workloads as W

HOST = os.path.join(os.path.dirname(os.path.abspath(H.__file__)), "csrc", "host")


def _rows(boxes):
    """Real rows with the Gram products of the Hermitian parts h and a of each box."""
    flip = boxes[:, ::-1, ::-1].conj()
    parts = np.concatenate([(boxes + flip) / 2, (boxes - flip) / 2j]).reshape(2 * len(boxes), -1)
    return np.concatenate([parts.real, parts.imag], 1)


def _set_rows(ks, band):
    n, w = ks.n, 2 * band + 1
    ky, kx = (np.where(t < n // 2, t, t - n) for t in (ks.support // n, ks.support % n))
    box = np.zeros((ks.num_kernels, w, w), complex)
    box[:, kx + band, ky + band] = ks.values * np.sqrt(
        ks.eigenvalues / ks.normalization_divisor)[:, None]
    return _rows(box)


def _norm(a, b):
    """Spectral norm of a^T a - b^T b."""
    q = np.linalg.qr(np.concatenate([a, b]).T)[0]
    a, b = a @ q, b @ q
    return np.abs(np.linalg.eigvalsh(a.T @ a - b.T @ b)).max()


@pytest.mark.parametrize("setup,z", [(W.arf_lines_256_setup(), 0.0),
                                     (W.arf_annular_2nm_setup(512), 0.0),
                                     (W.arf_annular_2nm_setup(1024), 0.0),
                                     (W.euv_dipole_1024_setup(), 0.01)])
def test_dropped_fields_are_below_a_rounding_of_the_clear_field(setup, z):
    src, opt, grid, k = setup
    ks = H.AerialImageEngine(src, opt, grid, max_kernels=k).kernel_set(z)
    v = E.real_fields(ks)
    assert len(v)
    want = _set_rows(ks, (v.shape[1] - 1) // 2)
    got = v.reshape(len(v), -1)
    got = np.concatenate([got.real, got.imag], 1)
    assert _norm(want, got) <= 2.0 ** -25 * (1 + 1e-6)


FORMS = r"""
#include <cstdio>
#include <random>
#include "engine.hpp"
using namespace huv;
// K orthogonal kernels, one order each (two with their mirror images), eigenvalue 1 but
// for the last, which is 1 + eps: the trace is K, the peak 1.
static RealFields form(int B, bool mirrored, double eps) {
  const int n = 64, W = 2 * B + 1;
  std::vector<int64_t> sup;
  for (int y = -B; y <= B; ++y)
    for (int x = -B; x <= B; ++x) sup.push_back((int64_t)((y + n) % n) * n + (x + n) % n);
  const int K = W * W / 2;
  std::vector<double> eig(K, 1.0), val((size_t)2 * K * sup.size(), 0.0);
  eig[K - 1] += eps;
  for (int k = 0; k < K; ++k) {
    const int t = mirrored ? W * W - 1 - k : k;
    val[2 * ((size_t)k * sup.size() + t)] = 1.0;
  }
  RealFields rf;
  real_fields(n, B, K, (int64_t)sup.size(), sup.data(), eig.data(), val.data(), rf);
  return rf;
}
int main() {
  const RealFields a = form(7, false, 0.0);
  const double one = 1.0 / (1 << 26);
  if (a.R != 2 * 112) return 1;
  if (!same_real_form(a, a)) return 2;
  if (!same_real_form(a, form(7, true, 0.0))) return 3;   // f and -f: the same images
  if (!same_real_form(a, form(7, true, 0.01 * one))) return 4;
  for (double eps : {4 * one, 40 * one, -4 * one, -40 * one})
    for (bool mirrored : {false, true})
      if (same_real_form(a, form(7, mirrored, eps))) return 5;
  if (same_real_form(a, form(6, false, 0.0))) return 6;
  return 0;
}
"""


def test_forms_that_differ_do_not_count_as_one(tmp_path):
    src, exe = tmp_path / "forms.cpp", tmp_path / "forms"
    src.write_text(FORMS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", HOST, str(src),
                    os.path.join(HOST, "real_form.cpp"), os.path.join(HOST, "linalg.cpp"),
                    "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
