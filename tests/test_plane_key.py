"""What a context keeps per plane list (kernel stacks, pointer tables, recorded
launches) goes when one of the list's own kernel sets dies, and only then: the ids
count up from 1 and so equal the layout flags and coarse sizes of a key's form.

CPU: the keys and their removal, as the library compiles them.  GPU: a process whose
first kernel set is destroyed goes on replaying and serving the lists of the others.
"""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

KEYS = r"""
#include <cstdio>
#include <map>
#include "plane_key.hpp"
using huvi::PlaneKey;
int main() {
  std::map<PlaneKey, int> m;
  const unsigned long long sizes[] = {32, 64, 128, 192, 256};
  int n = 0;
  for (unsigned long long m32 : sizes)
    for (unsigned long long paired : {0, 1})
      for (unsigned long long real : {0, 1}) {
        m[PlaneKey{{7}, {m32, paired, real}}] = n++;
        m[PlaneKey{{7, 9}, {m32, paired, real}}] = n++;
      }
  if ((int)m.size() != n) return 1;  // lists and forms are told apart
  if (m.count(PlaneKey{{7, 9, 64}, {0, 1}})) return 2;
  for (unsigned long long id : {0, 1, 32, 64, 128, 192, 256})
    huvi::forget_entries(m, id, [](int) {});
  if ((int)m.size() != n) return 3;  // none of these is a set of a list
  int dropped = 0;
  huvi::forget_entries(m, 9, [&](int v) { dropped += v % 2; });
  if (dropped != n / 2 || (int)m.size() != n / 2) return 4;
  huvi::forget_entries(m, 7, [&](int v) { dropped += v % 2 == 0; });
  return dropped == n && m.empty() ? 0 : 5;
}
"""


def test_flags_are_not_taken_for_ids(tmp_path):
    src, exe = tmp_path / "keys.cpp", tmp_path / "keys"
    src.write_text(KEYS)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "highuvlith_amd/csrc/host"),
                    str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


REPLAYS = r"""
import ctypes as C, sys
import numpy as np, torch
import highuvlith_amd as H
from highuvlith_amd import _lib

def engine(grid, k, ctx):
    return H.AerialImageEngine(H.Source.arf(H.IlluminationShape.Annular(0.7, 0.9)),
                               H.ProjectionOptics.immersion_193i(), grid, max_kernels=k,
                               context=ctx)

ctx = H.DeviceContext(0)
small = H.GridConfig(256, 1.0)   # band below 8: coarse grid 32, one lane per row
first = engine(small, 5, ctx)
first.device_kernel_set(0.0)     # the process's first kernel set
cases = []
for grid in (small, H.GridConfig(256, 4.0)):
    eng = engine(grid, 6, ctx)
    rng = np.random.default_rng(3)
    masks = torch.from_numpy((rng.random((2, 256, 256)) > 0.5).astype(np.float32)).cuda()
    out = torch.empty((2, 2, 256, 256), device="cuda")
    zs = (0.0, 30.0)
    want = eng.compute_batch(masks, zs)
    eng.compute_batch(masks, zs, out=out, graph=True)
    cases.append((eng, masks, out, zs, want))
assert cases[0][0].device_kernel_set(0.0).band <= 7
first.device_kernel_set(0.0).__del__()
junk = [torch.full((1 << 18,), 1e30, device="cuda") for _ in range(8)]  # over what was freed
for rep in range(3):
    for eng, masks, out, zs, want in cases:
        out.fill_(-1.0)
        eng.compute_batch(masks, zs, out=out, graph=True)
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
        got = torch.full_like(out, -1.0)
        planes = [eng.device_kernel_set(z) for z in zs]
        arr = (C.c_void_p * 2)(*[p.handle.value for p in planes])
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        st = ctx.lib.huv_socs_images_noalloc(ctx.handle, 2, 256, C.c_void_p(masks.data_ptr()), 2,
                                             arr, C.c_void_p(got.data_ptr()), 0)
        assert st == _lib.HUV_OK, ctx.lib.huv_last_error()
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep
print("replays served", len(junk))
"""


@pytest.mark.gpu
def test_lists_outlive_the_process_first_set():
    r = subprocess.run([sys.executable, "-c", REPLAYS], cwd=ROOT, capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "replays served 8" in r.stdout
