"""Polygons of real value, whose half box and mirror image are computed, against the
oracle's edge sum in FP64, at bands around the tiles and around the widest one that is
shared by eight waves.

Tolerance: the device sums in FP64 and rounds once to FP32 onto a rounded rectangle
pass, at most two roundings of bins up to n^2 (1.2e-7 n^2).
"""
import numpy as np
import pytest

import oracle
import highuvlith_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [0, 1, 3, 4, 5, 7, 8, 47, 62, 63, 64])
def test_real_polygons(gpu_ctx, band):
    rng = np.random.default_rng(band)
    n, px = 256, 1.5
    clips, polys = [], []
    for c in range(4):
        own = []
        for j in range((0, 1, 5, 9)[c]):  # 9 polygons: more edges than one chunk of eight
            # corners around a centre, less than a half turn apart: no edges cross
            t = 2 * np.pi * (np.arange(3 + j) + rng.uniform(0, 0.4, 3 + j)) / (3 + j)
            own.append(([(-150 + 35 * j + r * np.cos(a), 40 + r * np.sin(a))
                         for a, r in zip(t, rng.uniform(6, 17, 3 + j))], (1.0, -0.245, 0.5)[j % 3]))
        polys.append(own)
        clips.append([(-60.0, -100.0, 50.0, 30.0, 1.0)] if c % 2 else [])
    got = H.engine.band_spectrum_features_device(gpu_ctx, clips, polys, H.GridConfig(n, px),
                                                 band).cpu().numpy()
    k = np.arange(-band, band + 1) % n
    for c in range(4):
        ref = oracle.mask_spectrum(n, px, [("rect", *r[:4]) for r in clips[c]], dark_field=True)
        for verts, value in polys[c]:
            ref = oracle.polygon_spectrum(n, px, verts, value, spectrum=ref)
        assert np.abs(got[c] - ref[np.ix_(k, k)].T).max() <= 1.2e-7 * n * n, c
