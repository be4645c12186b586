"""
Downloads on both sides of the size up to which g comes with the stored data and the host reorders it: the state that was
uploaded, bit for bit.
"""

import numpy as np
import pytest

from ionization_amd import engine
from tests.cases import line_case, sh_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("r_points, l_bound, rows", [(60, 36, 2), (128, 36, 2), (129, 16, 4), (60, 37, 2), (700, 1, 16), (700, 2, 16)])
def test_sh_downloads(device_ctx, r_points, l_bound, rows):
    c = sh_case(r_points=r_points, l_bound=l_bound, rows=rows, t_half_as=2.0, n_basis_l=1)["compiled"]
    g = np.random.default_rng(5).standard_normal((l_bound, r_points)) * (1 - 2j)
    slot = device_ctx.add_sh(c)
    device_ctx.upload_state(engine.KIND_SH, slot, g, 0)
    assert np.array_equal(device_ctx.download_sh(slot).g, g)
    assert device_ctx.download_sh(slot, with_g=False).g is None
    device_ctx.remove(engine.KIND_SH, slot)


@pytest.mark.parametrize("z_points, rows", [(3, 2), (1000, 16), (1024, 8), (1025, 6)])
def test_line_downloads(device_ctx, z_points, rows):
    c = line_case(z_points=z_points, rows=rows, n_steps=4)["compiled"]
    g = np.random.default_rng(6).standard_normal(z_points) * (1 + 1j)
    slot = device_ctx.add_line(c)
    device_ctx.upload_state(engine.KIND_LINE, slot, g, 0)
    assert np.array_equal(device_ctx.download_line(slot)[0], g)
    device_ctx.remove(engine.KIND_LINE, slot)
