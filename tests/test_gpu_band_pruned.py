"""Band spectra of rasters at the edges of the pruned transforms: every size, bands of
one bin, at the limits of the two and four outer bins (31 | 32, 63) and one beyond
(64, the general four-step path), against NumPy in 64 bits.  Tolerance: FP32
transforms of up to 2^22 zero-mean points err by a few 2^-24 per stage and
dimension, 2e-6 of the largest bin.  Complex rasters: a constant phase leaves the
image as it is, so the complex path must give the real path's image; each is within
2.5e-6 of the FP64 image, so they differ by less than 5e-6.
"""
import numpy as np
import pytest

import highuvlith_amd as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [256, 512, 1024, 2048])
@pytest.mark.parametrize("band", [1, 15, 31, 32, 63, 64])
def test_band_spectrum(gpu_ctx, n, band):
    import torch
    rng = np.random.default_rng(n + band)
    masks = rng.standard_normal((3, n, n)).astype(np.float32)
    got = H.engine.band_spectrum_device(gpu_ctx, torch.from_numpy(masks).cuda(), band).cpu().numpy()
    ks = np.arange(-band, band + 1) % n
    for c in range(3):
        ref = np.fft.fft2(masks[c].astype(np.float64))[np.ix_(ks, ks)].T
        err = np.abs(got[c] - ref).max() / np.abs(ref).max()
        assert err < 2e-6, err


@pytest.mark.parametrize("n,px", [(256, 4.0), (512, 2.0), (512, 4.0), (1024, 4.0), (2048, 2.0)])
def test_complex_rasters_equal_real_ones(n, px):
    import torch
    eng = H.AerialImageEngine(H.Source.arf(H.IlluminationShape.Annular(0.7, 0.9)),
                              H.ProjectionOptics.immersion_193i(), H.GridConfig(n, px),
                              max_kernels=8)
    rng = np.random.default_rng(n)
    m = (rng.random((2, n // 16, n // 16)) > 0.5).repeat(16, 1).repeat(16, 2).astype(np.float32)
    real = eng.compute_batch(torch.from_numpy(m).cuda(), (0.0, 40.0)).cpu().numpy()
    z = torch.from_numpy(m * np.exp(0.7j).astype(np.complex64)).cuda()
    cplx = eng.compute_batch_complex(z, (0.0, 40.0)).cpu().numpy()
    err = np.abs(real - cplx).max()
    print(n, px, err)
    assert err < 5e-6
