"""Up to 32 rho points the rho-sweep's automatic shape pads to 32 rows, not to 64: a batch of such meshes is bound by its rows."""

import pytest

from ionization_amd import engine


@pytest.mark.parametrize("z_points, rho_points, shape, rows", [
    (300, 2, (4, 8), 32), (300, 30, (4, 8), 32), (65, 32, (4, 8), 32), (300, 33, (4, 4), 64), (300, 64, (4, 4), 64),
])
def test_small_rho_shapes(z_points, rho_points, shape, rows):
    _, _, cr, mr, lanes = engine.choose_cyl_layout(z_points, rho_points)
    assert (mr, lanes) == shape and cr * mr == rows
