"""The autotuner times only what it can choose: the factor of the band transforms has no
effect on an image and is recorded as its default, whatever the timing noise."""
import pytest

import highuvlith_amd as H

pytestmark = pytest.mark.gpu


def test_the_band_factor_is_not_timed():
    import torch
    src = H.Source.arf(H.IlluminationShape.Annular(0.7, 0.9))
    for n, n1 in ((256, 16), (512, 16), (1024, 32)):
        eng = H.AerialImageEngine(src, H.ProjectionOptics.immersion_193i(), H.GridConfig(n, 2.0),
                                  max_kernels=4)
        ctx, ks = eng.context(), eng.device_kernel_set(0.0)
        ctx.set_autotune(True)
        masks = torch.rand((2, n, n), device="cuda")
        for planes in (1, 2, 3, 4):  # a shape class each
            eng.compute_batch(masks, (0.0,) * planes)
            t = ctx.tuning(n, ks.band, planes, ks.host.num_kernels)
            assert t[1] == n1, (n, planes, t)
