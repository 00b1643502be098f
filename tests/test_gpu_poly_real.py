"""Polygons of real value fill half of the band box and its mirror image; the same
polygons with an imaginary part of 1e-30 take the general pass over every bin.  Both
sum in FP64 and round once to FP32, onto the same rectangle pass: at most two roundings
apart, 1.2e-7 n^2.
"""
import numpy as np
import pytest

import highuvlith_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("band", [0, 3, 4, 5, 6, 47, 70])
def test_half_box_equals_whole_box(gpu_ctx, band):
    rng = np.random.default_rng(band)
    n, px = 256, 1.5
    t = np.sort(rng.uniform(0, 2 * np.pi, (4, 9)), axis=1)
    polys = [[(-90 + 60 * j + r * np.cos(a), 40 + r * np.sin(a)) for a, r in zip(t[j], rng.uniform(8, 28, 9))]
             for j in range(4)]
    rects = [[(-60.0, -100.0, 50.0, 30.0, 1.0)], [(30.0, -90.0, 20.0, 44.0, 0.4 + 0.2j)], []]
    def run(eps):
        clips = [[(polys[0], 1.0 + eps), (polys[1], 0.5 + eps)], [(polys[2], -0.3 + eps)],
                 [(p, 1.0 + eps) for p in polys]]
        return H.engine.band_spectrum_features_device(gpu_ctx, rects, clips, H.GridConfig(n, px),
                                                      band).cpu().numpy()
    assert np.abs(run(0.0) - run(1e-30j)).max() <= 1.2e-7 * n * n
