"""The U-Net on fields narrower than a tile at every level, where the decoder's input is
written out for the general convolution, against the FP64 oracle with BF16 emulation.
Tolerances as for wider fields.
"""
import numpy as np
import pytest

from oracle import unet_ref as U
import highuvlith_amd as H
from highuvlith_amd import unet as UN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,base,n,h,w", [(2, 64, 2, 96, 32), (3, 16, 3, 64, 64), (2, 32, 1, 32, 96)])
def test_output_and_gradient(gpu_ctx, levels, base, n, h, w):
    import torch
    rng = np.random.default_rng(w)
    net = UN.UNet(gpu_ctx, levels=levels, base=base, seed=1)
    p = net.get_params()
    p += 0.02 * rng.standard_normal(p.shape).astype(np.float32)
    net.set_params(p)
    lay = U.Layout(levels, base)
    x = (rng.random((n, h // 8, w // 8)) > 0.5).astype(np.float32).repeat(8, 1).repeat(8, 2)
    t = (x - 0.5 + 0.1 * rng.standard_normal(x.shape)).astype(np.float32)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref, _ = U.forward(p.astype(np.float64), lay, x.astype(np.float64), bf=True)
    assert np.abs(out - ref).max() / np.abs(ref).max() <= 1e-2
    loss, g = net.loss_and_grad(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(),
                                want_grad=True)
    lref, gref = U.loss_grad(p.astype(np.float64), lay, x.astype(np.float64),
                             t.astype(np.float64), bf=True)
    assert abs(loss - lref) <= 2e-3 * lref
    for name in ("enc1", "enc2", "dec1", "dec2"):
        for l, s in enumerate(getattr(lay, name)):
            for off, shape in s[:2]:
                cnt = int(np.prod(shape))
                a, b = g[off:off + cnt], gref[off:off + cnt]
                assert np.linalg.norm(a - b) <= 3e-2 * np.linalg.norm(b), (name, l, shape)
