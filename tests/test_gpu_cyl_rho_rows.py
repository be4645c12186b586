"""
Where the last row of a cylindrical line can sit, on the device: followed by a padding row of the same
thread, of the next one, or by none at all. In the rho-sweep its coupling to the next row is zero; in the
z-sweep, whose couplings are all alike, the padding rows' pivots are made zero. The sizes put it at each of
these, in both sweeps; the mask's ramp crosses every one of them.
"""
import numpy as np
import pytest

from tests.cases import cyl_case
from tests.conftest import rel_l2
from tests.test_gpu_cyl import OBS_ATOL, WF_RTOL, _run_device

pytestmark = pytest.mark.gpu


def _check(case, g_dev, norms_dev, ips_dev):
    g, norms, ips = case["oracle"].run(case["g0"], case["times"], case["store_every"], basis=case["basis"])
    assert len(norms_dev) == len(norms)
    assert rel_l2(g_dev, g) <= WF_RTOL
    assert np.max(np.abs(norms_dev - norms)) <= OBS_ATOL
    assert np.max(np.abs(ips_dev - ips)) <= OBS_ATOL


@pytest.mark.parametrize("rho_shape, rho_points", [
    ((8, 4), 128),  # no padding row
    ((8, 4), 127), ((8, 4), 121), ((8, 4), 120), ((8, 4), 9), ((8, 4), 2),
    ((4, 4), 64), ((4, 4), 61), ((4, 4), 5),
    ((8, 8), 64), ((16, 4), 256), ((16, 4), 241),
])
def test_last_rho_row(device_ctx, rho_shape, rho_points):
    case = cyl_case(z_points=96, rho_points=rho_points, rho_shape=rho_shape, t_half_as=6.0, store_every=3)
    c = case["compiled"]
    print(f"Cyl last rho row, shape={rho_shape} points={rho_points} Cr={c.Cr}", flush=True)
    _check(case, *_run_device(device_ctx, c))


@pytest.mark.parametrize("z_rows, z_points", [(4, 256), (4, 253), (8, 512), (8, 505), (2, 128)])
def test_last_z_row(device_ctx, z_rows, z_points):
    case = cyl_case(z_points=z_points, rho_points=40, z_rows=z_rows, t_half_as=6.0, store_every=3)
    c = case["compiled"]
    print(f"Cyl last z row, rows={z_rows} points={z_points} Pz={c.Pz}", flush=True)
    _check(case, *_run_device(device_ctx, c))
