"""Kernel sets with negative eigenvalues (a caller's own; no optics give them) are summed
with the negative kernels first and subtracted, whichever share of the kernels a
work-group takes: one clip splits the sum over many work-groups, a batch does not.

Reference: the oracle's FP64 sum; gate 1e-5 of the clear field.
"""
import numpy as np
import pytest

import oracle
import highuvlith_amd as H
from highuvlith_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("negative", [(0,), (8,), (1, 3, 4), (2, 3, 4, 5, 6, 7, 8), tuple(range(9))])
def test_negative_eigenvalues(negative):
    import torch
    n = 256
    eng = H.AerialImageEngine(H.Source.arf(H.IlluminationShape.Annular(0.7, 0.9)),
                              H.ProjectionOptics.immersion_193i(), H.GridConfig(n, 4.0),
                              max_kernels=9)
    ks = eng.kernel_set(0.0)
    assert ks.num_kernels == 9
    ks.eigenvalues = ks.eigenvalues.copy()
    ks.eigenvalues[list(negative)] *= -1.0
    assert len(E.real_fields(ks)) == 0
    ctx = eng.context()
    dev = ctx.upload(ks, eng.flare_fraction())
    rng = np.random.default_rng(len(negative))
    masks = torch.from_numpy((rng.random((96, n, n)) > 0.5).astype(np.float32)).cuda()
    refs = [oracle.socs_image(ks, oracle.fft2(masks[c].cpu().numpy().astype(np.complex128)),
                              eng.flare_fraction(), threads=8) for c in (0, 95)]
    for clips in (1, 5, 96):
        m = masks[96 - clips:].contiguous()
        out = torch.empty((clips, 1, n, n), device="cuda")
        E.socs_images_device(ctx, m, [dev], out)
        assert np.abs(out[-1, 0].cpu().numpy() - refs[1]).max() <= 1e-5, clips
        both = torch.empty((clips, 2, n, n), device="cuda")  # beside a set of the usual kind
        E.socs_images_complex_device(ctx, m.to(torch.complex64), [dev, eng.device_kernel_set(40.0)],
                                     both)
        assert np.abs(both[-1, 0].cpu().numpy() - refs[1]).max() <= 1e-5, clips
    assert np.abs(out[0, 0].cpu().numpy() - refs[0]).max() <= 1e-5
