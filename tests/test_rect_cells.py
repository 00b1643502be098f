"""Cells of rectangle lists (resolve_rect_cells): the picture is the painter's one, and
no list is cut into more cells than one grid over all its edges gives, with equal
neighbours along x and equal neighbouring rows joined.
"""
import os
import subprocess

import pytest

import highuvlith_amd as H

HOST = os.path.join(os.path.dirname(os.path.abspath(H.__file__)), "csrc", "host")

HEAD = r"""
#include <chrono>
#include <cmath>
#include <cstdio>
#include <functional>
#include <random>
#include <set>
#include "engine.hpp"
using namespace huv;
typedef std::vector<RectFeature> List;
static const int N = 1024;
static const double PX = 1.0, HALF = 512.0;
static std::mt19937_64 gen(11);
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(gen); }

// Cells of one grid over all edges, and the value at (x, y).
static long one_grid(const List& l, cd bg) {
  std::set<double> xs, ys;
  for (auto& r : l) {
    for (double s : {-0.5, 0.5}) {
      xs.insert(std::min(HALF, std::max(-HALF, r.x + s * r.w)));
      ys.insert(std::min(HALF, std::max(-HALF, r.y + s * r.h)));
    }
  }
  auto near = [](const std::set<double>& s) {
    std::vector<double> o;
    for (double v : s) if (o.empty() || v - o.back() > 1e-12 * 2 * HALF) o.push_back(v);
    return o;
  };
  const std::vector<double> x = near(xs), y = near(ys);
  auto at = [](const std::vector<double>& e, double v) {
    return std::lower_bound(e.begin(), e.end(), std::min(HALF, std::max(-HALF, v)) - 1e-9) - e.begin();
  };
  const long nx = (long)x.size() - 1, ny = (long)y.size() - 1;
  if (nx < 1 || ny < 1) return 0;
  std::vector<std::vector<cd>> c(ny, std::vector<cd>(nx, bg));
  for (auto& r : l)
    for (long i = at(y, r.y - r.h / 2); i < std::min<long>(ny, at(y, r.y + r.h / 2)); ++i)
      for (long j = at(x, r.x - r.w / 2); j < std::min<long>(nx, at(x, r.x + r.w / 2)); ++j)
        c[i][j] = r.value;
  long cells = 0;
  for (long i = 0; i < ny; ++i) {
    if (i && c[i] == c[i - 1]) continue;
    for (long j = 0; j < nx; ++j) cells += c[i][j] != bg && (j == 0 || c[i][j] != c[i][j - 1]);
  }
  return cells;
}

static List tiles(int nx, int ny, double sx, double sy, double fill, double shift, cd v) {
  List l;
  for (int i = 0; i < ny; ++i)
    for (int j = 0; j < nx; ++j)
      l.push_back({sx * (j - 0.5 * nx + 0.5) + shift * (i % 2), sy * (i - 0.5 * ny + 0.5), sx * fill,
                   sy * fill, v});
  return l;
}

static List scatter(int n, double most, int values) {
  List l;
  for (int i = 0; i < n; ++i)
    l.push_back({std::round(uni(-520, 520)), std::round(uni(-520, 520)), std::round(uni(1, most)),
                 std::round(uni(1, most)), cd(1.0 + i % values, 0.25 * (i % 3))});
  return l;
}

// 0, or what is wrong with the cells of l
static int check(const List& l, cd bg) {
  std::vector<RectCell> cells;
  if (!resolve_rect_cells(l, bg, N, PX, 1 << 20, cells)) return 1;
  if ((long)cells.size() > one_grid(l, bg)) {
    std::printf("%zu rectangles: %zu cells, one grid %ld\n", l.size(), cells.size(), one_grid(l, bg));
    return 2;
  }
  for (int t = 0; t < 400; ++t) {
    double x = uni(-HALF, HALF), y = uni(-HALF, HALF);
    if (t % 2 && !l.empty()) {  // near a rectangle
      const RectFeature& r = l[(size_t)uni(0, l.size()) % l.size()];
      x = r.x + uni(-0.6, 0.6) * r.w;
      y = r.y + uni(-0.6, 0.6) * r.h;
    }
    if (std::fabs(x) >= HALF || std::fabs(y) >= HALF) continue;
    cd want = bg, got = bg;
    for (auto& r : l)
      if (std::fabs(x - r.x) < r.w / 2 && std::fabs(y - r.y) < r.h / 2) want = r.value;
    int in = 0;
    for (auto& c : cells)
      if (x > c.x0 && x < c.x1 && y > c.y0 && y < c.y1) {
        got = bg + c.w;
        ++in;
      }
    if (in > 1 || std::abs(got - want) > 1e-12) return 3;
  }
  return 0;
}
"""

BODIES = {
    # layouts with common edges take one grid's time: far less than groups would
    "common": r"""
int main() {
  for (cd bg : {cd(0, 0), cd(1, 0)})
    for (const List& l : {tiles(32, 32, 16, 16, 1, 0, 1.0), tiles(20, 40, 40, 20, 1, 20, 1.0),
                          tiles(12, 11, 40, 30, 1, 0, 1.0), tiles(9, 1, 20, 800, 0.5, 0, 1.0),
                          tiles(2, 1, 20, 40, 1, 0, 1.0), tiles(50, 45, 16, 16, 0.5, 0, 1.0),
                          tiles(13, 10, 40, 40, 1.2, 0, 0.5)})
      if (int e = check(l, bg)) return e;
  const List tiling = tiles(32, 32, 16, 16, 1, 0, 1.0);
  List apart = tiles(32, 32, 16, 16, 0.5, 0, 1.0);  // as many, none alike
  for (auto& r : apart) {
    r.x += uni(0, 4);
    r.y += uni(0, 4);
    r.w += uni(0, 3);
  }
  std::vector<RectCell> cells;
  double cost[2] = {1e9, 1e9};
  for (int k = 0; k < 30; ++k)
    for (int c = 0; c < 2; ++c) {
      const auto t0 = std::chrono::steady_clock::now();
      resolve_rect_cells(c ? apart : tiling, cd(0, 0), N, PX, 1 << 30, cells);
      cost[c] = std::min(cost[c], std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
    }
  std::printf("%.3f ms, apart %.3f ms\n", 1e3 * cost[0], 1e3 * cost[1]);
  return cost[0] <= 2.0 * cost[1] ? 0 : 7;
}
""",
    # a call's limit counts one grid's cells, whatever the clip is cut into; the bound
    # that spares the count holds, and lets 512 clips of 200 scattered contacts pass
    "apart": r"""
// A plan that compares all pairs and gives each rectangle a list of its own.
static size_t all_pairs(const List& l) {
  struct Box { double x0, x1, y0, y1; };
  std::vector<Box> b;
  for (auto& r : l) b.push_back({r.x - r.w / 2, r.x + r.w / 2, r.y - r.h / 2, r.y + r.h / 2});
  std::vector<int> root(b.size());
  for (size_t i = 0; i < b.size(); ++i) {
    root[i] = (int)i;
    for (size_t j = 0; j < i; ++j)
      if (b[i].x0 < b[j].x1 && b[j].x0 < b[i].x1 && b[i].y0 < b[j].y1 && b[j].y0 < b[i].y1)
        root[i] = root[j];
  }
  std::vector<std::vector<int>> members(b.size());
  for (size_t i = 0; i < b.size(); ++i) members[root[i]].push_back((int)i);
  std::vector<RectCell> cells;
  for (auto& m : members)
    for (int i : m) cells.push_back({b[i].x0, b[i].x1, b[i].y0, b[i].y1, l[i].value});
  return cells.size();
}
static List apart(int n) {  // an array with no common edges
  List l = tiles(8, (n + 7) / 8, 128, 60, 0.4, 0, 1.0);
  l.resize(n);
  for (auto& r : l) {
    r.x += uni(-6, 6);
    r.y += uni(-6, 6);
    r.w += uni(0, 30);
  }
  return l;
}
int main() {
  // the first rectangles of a list are like its others, or are not
  for (int n : {2, 3, 4, 5, 6, 9, 10, 16, 17, 43, 128, 129})
    for (int k = 1; k <= n; k += std::max(1, n / 6)) {
      const List a = apart(n);
      List t = tiles(8, (n + 7) / 8, 60, 50, 1, 0, 1.0);
      t.resize(n);
      List at(a.begin(), a.begin() + k), ta(t.begin(), t.begin() + k);
      at.insert(at.end(), t.begin() + k, t.end());
      ta.insert(ta.end(), a.begin() + k, a.end());
      for (const List& l : {a, t, at, ta})
        if (int e = check(l, cd(0, 0))) return e;
    }
  std::vector<List> clips;
  for (int i = 0; i < 24; ++i) clips.push_back(apart(64));
  double cost[2] = {1e9, 1e9};
  size_t cells = 0, other = 0;
  std::vector<RectCell> out;
  for (int k = 0; k < 200; ++k)
    for (int c = 0; c < 2; ++c) {
      cells = c ? cells : 0;
      other = c ? 0 : other;
      const auto t0 = std::chrono::steady_clock::now();
      for (auto& l : clips) {
        if (c) {
          other += all_pairs(l);
        } else {
          resolve_rect_cells(l, cd(0, 0), N, PX, 1 << 30, out);
          cells += out.size();
        }
      }
      cost[c] = std::min(cost[c], std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
    }
  std::printf("%.1f us, all pairs %.1f us, %zu %zu cells\n", 1e6 * cost[0], 1e6 * cost[1], cells, other);
  return cost[0] <= 1.1 * cost[1] ? 0 : 8;
}
""",
    "limit": r"""
int main() {
  std::vector<RectCell> with, without;
  for (int values : {1, 5, 100})
    for (int n : {0, 1, 2, 9, 60, 200})
      for (double most : {20.0, 300.0}) {
        const List l = scatter(n, most, values);
        int64_t grid = -1;
        if (!resolve_rect_cells(l, cd(0, 0), N, PX, 1 << 20, with, &grid)) return 1;
        if (grid != one_grid(l, cd(0, 0))) return 2;
        if (rect_grid_cells_bound(l, N, PX) < grid) return 3;
        resolve_rect_cells(l, cd(0, 0), N, PX, 1 << 20, without);
        if (with.size() != without.size()) return 4;
      }
  for (const List& l : {tiles(32, 32, 16, 16, 1, 0, 1.0), tiles(20, 40, 40, 20, 1, 20, 1.0),
                        tiles(50, 45, 16, 16, 0.5, 0, 1.0)}) {
    int64_t grid = -1;
    if (!resolve_rect_cells(l, cd(0, 0), N, PX, 1 << 20, with, &grid)) return 5;
    if (grid != one_grid(l, cd(0, 0)) || rect_grid_cells_bound(l, N, PX) < grid) return 6;
  }
  int64_t calls = 0;
  for (int c = 0; c < 512; ++c) {
    List l;
    for (int i = 0; i < 200; ++i)
      l.push_back({-480 + 64.0 * (i % 15) + uni(0, 8), -480 + 64.0 * (i / 15) + uni(0, 8), uni(12, 24),
                   uni(12, 24), 1.0});
    calls += rect_grid_cells_bound(l, N, PX);
  }
  return calls <= 1 << 26 ? 0 : 7;
}
""",
    # an aligned array of 2025 rectangles takes less than one look at every pair does
    "array": r"""
static volatile long sink;
int main() {
  for (double shift : {0.0, 3.0})
    for (bool turned : {false, true}) {
      List l = tiles(45, 45, 16, 20, 0.5, shift, 1.0);
      if (turned)
        for (auto& r : l) {
          std::swap(r.x, r.y);
          std::swap(r.w, r.h);
        }
      if (int e = check(l, cd(0, 0))) return e;
      std::vector<RectCell> cells;
      double cost[2] = {1e9, 1e9};
      for (int k = 0; k < 20; ++k) {
        const auto t0 = std::chrono::steady_clock::now();
        resolve_rect_cells(l, cd(0, 0), N, PX, 1 << 20, cells);
        const auto t1 = std::chrono::steady_clock::now();
        long n = 0;
        for (size_t i = 0; i < l.size(); ++i)
          for (size_t j = 0; j < i; ++j)
            n += l[i].x - l[i].w / 2 < l[j].x + l[j].w / 2 && l[j].x - l[j].w / 2 < l[i].x + l[i].w / 2 &&
                 l[i].y - l[i].h / 2 < l[j].y + l[j].h / 2 && l[j].y - l[j].h / 2 < l[i].y + l[i].h / 2;
        sink = n;
        const auto t2 = std::chrono::steady_clock::now();
        cost[0] = std::min(cost[0], std::chrono::duration<double>(t1 - t0).count());
        cost[1] = std::min(cost[1], std::chrono::duration<double>(t2 - t1).count());
      }
      std::printf("%.3f ms, every pair %.3f ms\n", 1e3 * cost[0], 1e3 * cost[1]);
      if (cost[0] > cost[1]) return 7;
    }
  return 0;
}
""",
    # equal neighbours are joined however many values the clip has
    "values": r"""
int main() {
  for (int values : {3, 15, 16, 17, 63, 64, 65, 66, 150}) {
    List l;
    for (int i = 0; i < 300; ++i)  // a strip of pairs of equal slabs, then one over them
      l.push_back({-500.0 + 3 * i, 100, 3, 50, cd(1.0 + i / 2 % values, 0)});
    for (int i = 0; i < 60; ++i) l.push_back({-300.0 + 8 * i, 90, 8, 9, cd(1.0 + values - i / 4 % 3, 0)});
    l.push_back({0, 0, 30, 30, cd(-0.0, 0.0)});
    l.push_back({0, 40, 30, 30, cd(0.0, -0.0)});
    for (cd bg : {cd(0, 0), cd(5, 0)})
      if (int e = check(l, bg)) return e;
    for (int r = 0; r < 4; ++r)
      if (int e = check(scatter(120, 200, values), cd(0, 0))) return e;
  }
  return 0;
}
""",
    # shapes made of slabs, tilings, steps and bricks: joined across touching edges
    "touching": r"""
int main() {
  for (cd bg : {cd(0, 0), cd(0.3, -0.1)}) {
    std::vector<RectCell> cells;
    if (!resolve_rect_cells(tiles(32, 32, 16, 16, 1, 0, 1.0), bg, N, PX, 1 << 20, cells)) return 9;
    if (cells.size() != 1) return 8;
    List steps, ls;
    for (int i = 0; i < 60; ++i) steps.push_back({-300.0 + 10 * i, 4.0 * i, 10, 20, 1.0});
    for (int i = 0; i < 5; ++i)
      for (int j = 0; j < 5; ++j) {
        ls.push_back({-440.0 + 180 * j, -440.0 + 180 * i, 20, 80, 1.0});
        ls.push_back({-405.0 + 180 * j, -470.0 + 180 * i, 50, 20, 1.0});
      }
    for (const List& l : {tiles(32, 32, 16, 16, 1, 0, 1.0), tiles(20, 40, 40, 20, 1, 20, 1.0),
                          tiles(9, 9, 30, 30, 1, 3.7, 0.5), tiles(7, 7, 40, 40, 0.5, 0, 1.0),
                          steps, ls, List{}, scatter(1, 90, 1)})
      if (int e = check(l, bg)) return e;
    for (int n : {2, 3, 8, 30, 90})
      for (double most : {40.0, 200.0})
        for (int r = 0; r < 6; ++r)
          if (int e = check(scatter(n, most, 1 + r), bg)) return e;
  }
  return 0;
}
""",
}


@pytest.mark.parametrize("case", sorted(BODIES))
def test_cells(tmp_path, case):
    src, exe = tmp_path / "cells.cpp", tmp_path / "cells"
    src.write_text(HEAD + BODIES[case])
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", HOST, str(src)]
                   + [os.path.join(HOST, f) for f in ("kernels_build.cpp", "linalg.cpp",
                                                      "optics_source.cpp")]
                   + ["-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_a_call_of_many_rectangles(gpu_ctx):
    """520 clips of 190 contacts: above the limit by their number, far below by their
    cells.  Tolerance as for the groups: one rounding to FP32 of FP64 sums."""
    import numpy as np
    from test_gpu_rect_groups import _reference
    rng = np.random.default_rng(1)
    n, px, band = 256, 2.0, 7
    site = np.arange(190)
    lists = [[(*map(float, p), 1.0) for p in np.stack(
        [-240 + 34 * (site % 14) + rng.uniform(0, 8, 190), -240 + 34 * (site // 14)
         + rng.uniform(0, 8, 190), rng.uniform(8, 30, 190), rng.uniform(8, 30, 190)], 1)]
             for _ in range(520)]
    got = H.engine.band_spectrum_rects_device(gpu_ctx, lists, H.GridConfig(n, px), band).cpu().numpy()
    for c in range(0, 520, 40):
        assert np.abs(got[c] - _reference(lists[c], 0.0, n, px, band)).max() <= 1.2e-7 * n * n, c
