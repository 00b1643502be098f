"""Band spectra of rectangle lists resolved group by group (overlapping
rectangles on their own edges) and summed by two or eight waves per tile group,
against the painter's rule on one edge grid in FP64.

Tolerance: the device sums FP64 products and rounds once to FP32, so a bin is
off by at most 2^-24 of its size plus FP64 noise; 1.2e-7 n^2 |value| covers it.
"""
import numpy as np
import pytest

import highuvlith_amd as H

pytestmark = pytest.mark.gpu


def _reference(rects, bg, n, px, band):
    L = n * px
    clip = lambda t: min(max(t, -L / 2), L / 2)  # noqa: E731
    b = [(clip(x - w / 2), clip(x + w / 2), clip(y - h / 2), clip(y + h / 2), v)
         for x, y, w, h, v in rects if w > 0 and h > 0]
    k = np.arange(-band, band + 1)
    out = np.zeros((len(k), len(k)), complex)
    out[band, band] = bg * n * n
    if not b:
        return out
    ex = np.unique([e for r in b for e in r[:2]])
    ey = np.unique([e for r in b for e in r[2:4]])
    cell = np.full((len(ex) - 1, len(ey) - 1), bg, complex)
    for x0, x1, y0, y1, v in b:
        cell[np.searchsorted(ex, x0):np.searchsorted(ex, x1),
             np.searchsorted(ey, y0):np.searchsorted(ey, y1)] = v

    def axis(e):
        lo, hi = e[:-1, None], e[1:, None]
        return n * (hi - lo) / L * np.sinc(k * (hi - lo) / L) * np.exp(
            -1j * np.pi * k * ((lo + hi) / L + (n - 1) / n))

    return out + axis(ex).T @ (cell - bg) @ axis(ey)


def _clip(rng, L, count, spread, values):
    return [(*rng.uniform(-0.5 * L, 0.5 * L, 2), *rng.uniform(0.01, spread, 2) * L,
             complex(rng.choice(values))) for _ in range(count)]


@pytest.mark.parametrize("band,clips", [(6, 1), (13, 5), (40, 2), (40, 12), (1, 600)])
def test_groups_match_one_grid(gpu_ctx, band, clips):
    rng = np.random.default_rng(band + clips)
    n, px = 256, 1.7
    L = n * px
    lists = []
    for c in range(clips):
        count = (0, 1, 2, 7, 8, 9, 40)[c % 7] if clips > 1 else 23
        lists.append(_clip(rng, L, count, (0.05, 0.3)[c % 2], (1.0, 0.5, -0.245 + 0.1j, 0.0)))
    lists[0] += [(0.0, 0.0, 20.0, 20.0, 1.0), (20.0, 0.0, 20.0, 20.0, 0.5),  # shared edge
                 (0.0, 0.0, 8.0, 8.0, 0.0),                                   # back to background
                 (40.0, 50.0, 10.0, 10.0, 1.0), (40.0, 50.0, 10.0, 10.0, 0.25)]
    got = H.engine.band_spectrum_rects_device(gpu_ctx, lists, H.GridConfig(n, px), band)
    got = got.cpu().numpy()
    for c in range(0, clips, max(1, clips // 12)):
        ref = _reference(lists[c], 0.0, n, px, band)
        assert np.abs(got[c] - ref).max() <= 1.2e-7 * n * n, c


def test_many_values_and_many_rectangles(gpu_ctx):
    rng = np.random.default_rng(4)
    n, px, band = 256, 1.0, 9
    many = [(*rng.uniform(-120, 120, 2), *rng.uniform(1, 40, 2), float(v))
            for v in np.linspace(0.01, 1.0, 90)]
    grid = [(x, y, 1.5, 1.5, 1.0) for x in np.arange(-126, 126, 5.0)
            for y in np.arange(-126, 126, 5.0)]  # 2601 rectangles: one group
    got = H.engine.band_spectrum_rects_device(gpu_ctx, [many, grid], H.GridConfig(n, px), band,
                                              backgrounds=[0.3, 0.0]).cpu().numpy()
    for c, (r, bg) in enumerate(((many, 0.3), (grid, 0.0))):
        assert np.abs(got[c] - _reference(r, bg, n, px, band)).max() <= 1.2e-7 * n * n


def test_calls_in_a_row_keep_their_own_geometry(gpu_ctx):
    """Calls issued without waiting (two staging slots in turn) see their own lists."""
    import torch
    rng = np.random.default_rng(8)
    n, px, band = 256, 2.0, 11
    lists = [[_clip(rng, n * px, 30 + 60 * (i % 3), 0.1, (1.0,))] for i in range(7)]
    outs = [H.engine.band_spectrum_rects_device(gpu_ctx, ls, H.GridConfig(n, px), band)
            for ls in lists]
    torch.cuda.synchronize()
    for ls, o in zip(lists, outs):
        ref = _reference(ls[0], 0.0, n, px, band)
        assert np.abs(o[0].cpu().numpy() - ref).max() <= 1.2e-7 * n * n
