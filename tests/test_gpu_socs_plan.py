"""What the device images per clip: planes share an image only where their real forms
are one, and no plane takes more steps than it has kernels."""
import pytest

import highuvlith_amd as H
from highuvlith_amd import engine as E

pytestmark = pytest.mark.gpu


def _engine(source, optics, px, k):
    return H.AerialImageEngine(source, optics, H.GridConfig(256, px), max_kernels=k)


def test_plans():
    dipole = _engine(H.Source(13.5, H.IlluminationShape.SectorPoles(0.7, 0.9, 35.0, 0.0, 2)),
                     H.EuvProjectionOptics.nxe_033(), 1.0, 12)
    pole = _engine(H.Source.arf(H.IlluminationShape.SectorPoles(0.5, 0.8, 60.0, 20.0, 1)),
                   H.ProjectionOptics.immersion_193i(), 2.0, 7)
    assert dipole.kernel_set(30.0).num_kernels == 12 and pole.kernel_set(-25.0).num_kernels == 7
    for eng, zs, images, steps in (
            (dipole, (0.0,), 1, 6),                  # 12 real fields
            (dipole, (30.0,), 1, 12),                # 24: its own kernels
            (dipole, (-30.0, 0.0, 30.0), 2, 18),     # opposite defocus, one image
            (dipole, (30.0, 30.0), 1, 12),           # listed twice
            (dipole, (30.0, 30.05), 2, 24),          # close is not the same
            (pole, (-25.0, 25.0), 2, 14)):           # no point symmetry
        planes = [eng.device_kernel_set(z) for z in zs]
        assert E.socs_plan(planes) == (images, steps), zs
        assert E.socs_plan(planes, real_masks=False) == (
            len(zs), sum(p.host.num_kernels for p in planes))
        for p in planes:
            fields = len(E.real_fields(p.host))
            own = min(p.host.num_kernels, (fields + 1) // 2)
            assert E.socs_plan([p]) == (1, own)
    near = [dipole.device_kernel_set(z) for z in (0.0, 0.02)]
    assert E.socs_plan(near)[0] == 2
    with pytest.raises(H.HuvError):
        E.socs_plan([pole.device_kernel_set(0.0), dipole.device_kernel_set(0.0)])
