"""The U-Net on fields that are not square, single and odd batches, every base
width and level count that changes a convolution's route (tiles staged in LDS or
not, the concatenation read from two tensors, 8-, 16- and 32-channel chunks,
row blocks that end inside an image), against the FP64 oracle with BF16
emulation.  Tolerances as for the square fields: BF16 storage (2^-9 per value)
through up to 14 layers.
"""
import numpy as np
import pytest

from oracle import unet_ref as U
import highuvlith_amd as H
from highuvlith_amd import unet as UN

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return H.DeviceContext(0)


@pytest.mark.parametrize("levels,base,n,h,w", [(3, 16, 1, 64, 192), (2, 64, 3, 32, 64),
                                               (3, 32, 1, 192, 64), (2, 16, 5, 96, 128),
                                               (4, 16, 1, 128, 256)])
def test_output_and_gradient(ctx, levels, base, n, h, w):
    import torch
    rng = np.random.default_rng(levels * base + h)
    net = UN.UNet(ctx, levels=levels, base=base, seed=1)
    p = net.get_params()
    p += 0.02 * rng.standard_normal(p.shape).astype(np.float32)  # biases away from zero
    net.set_params(p)
    lay = U.Layout(levels, base)
    x = (rng.random((n, h // 8, w // 8)) > 0.5).astype(np.float32).repeat(8, 1).repeat(8, 2)
    t = (x - 0.5 + 0.1 * rng.standard_normal(x.shape)).astype(np.float32)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref, _ = U.forward(p.astype(np.float64), lay, x.astype(np.float64), bf=True)
    err = np.abs(out - ref).max() / np.abs(ref).max()
    print("forward", err)
    assert err <= 1e-2
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
                rel = np.linalg.norm(a - b) / np.linalg.norm(b)
                assert rel <= 3e-2, (name, l, shape, rel)
    # the same inputs again: the same bits
    loss2, g2 = net.loss_and_grad(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda(),
                                  want_grad=True)
    assert loss2 == loss and np.array_equal(g, g2)


@pytest.mark.parametrize("levels,base", [(3, 64), (3, 32), (2, 16)])
def test_batch_equals_its_fields(ctx, levels, base):
    """A batch is convolved in taller tiles than a single field: the same bits."""
    import torch
    net = UN.UNet(ctx, levels=levels, base=base, seed=2)
    x = torch.rand((16, 256, 256), generator=torch.Generator().manual_seed(base)).cuda()
    out = net.forward(x).cpu().numpy()
    for k in (0, 7, 15):
        one = net.forward(x[k:k + 1].contiguous()).cpu().numpy()
        assert np.array_equal(one[0], out[k])
