"""The rho-sweep's automatic shape: every size that has a shape keeps one, and it covers the line."""
import pytest

from ionization_amd import engine
from ionization_amd.exceptions import DeviceError


def test_every_rho_size_has_a_shape():
    for n in range(2, 2049):
        _, _, cr, mr, lanes = engine.choose_cyl_layout(64, n)
        assert cr * mr >= n and (cr * lanes) % 64 == 0 and cr <= engine.CYL_RHO_SHAPES[(mr, lanes)], n
    with pytest.raises(DeviceError):
        engine.choose_cyl_layout(64, 2049)


@pytest.mark.parametrize("points, shape", [(2, (4, 4)), (320, (4, 4)), (321, (8, 4)), (400, (4, 4)), (512, (8, 4)),
                                           (1000, (8, 4)), (1025, (16, 4))])
def test_rho_shape_rule(points, shape):
    assert engine.choose_cyl_layout(64, points)[3:] == shape
