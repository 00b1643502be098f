"""Calls captured into a caller's graph with only the other mask kind's kernel stacks
built: real masks after eager complex calls and complex masks after eager real calls,
which one stack served before real masks had their own.

Tolerance against eager calls: real masks captured on the general stacks and eager on
the real ones are each within 2.5e-6 of the FP64 image, so within 5e-6 of each other;
complex masks have one form, bit for bit.
"""
import numpy as np
import pytest

import highuvlith_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", ["complex", "real"])
def test_captured_after_the_other_kind(first):
    import torch
    eng = H.AerialImageEngine(H.Source.arf(H.IlluminationShape.Annular(0.7, 0.9)),
                              H.ProjectionOptics.immersion_193i(), H.GridConfig(256, 4.0),
                              max_kernels=9, context=H.DeviceContext(0))
    zs = (0.0, 40.0)
    rng = np.random.default_rng(2)
    masks = torch.from_numpy((rng.random((8, 256, 256)) > 0.5).astype(np.float32)).cuda()
    cmasks = (masks * torch.exp(0.4j * masks)).to(torch.complex64).contiguous()
    calls = {"real": (eng.compute_batch, masks), "complex": (eng.compute_batch_complex, cmasks)}
    eager, data = calls[first]
    eager(data, zs)              # the workspace of 8 clips holds the captured call's 3
    call, data = calls["real" if first == "complex" else "complex"]
    data = data[:3].contiguous()
    out = torch.full((3, 2, 256, 256), -1.0, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(data, zs, out=out)
    want = call(data, zs).clone()
    for rep in range(3):
        out.fill_(-1.0)
        graph.replay()
        torch.randn(1 << 18, device="cuda").sum().item()
        assert (out - want).abs().max().item() <= (5e-6 if first == "complex" else 0.0), rep
