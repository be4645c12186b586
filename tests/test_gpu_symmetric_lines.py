"""
The Crank-Nicolson solvers against the oracle for every rows-per-thread instance, on the radial lines of the length
gauge (SH) and on a Line: with the last row at each place it can have in its thread (first, last but one, last), and with no
padding row at all.
"""
import pytest

from tests.cases import line_case, sh_case
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

# Every pivot has a real part of at least 1, so a step's solve is backward stable: some 4 eps (2.2e-16) times the
# entries of tau H (up to about 1e2). 12 steps and two solvers: 12 * 2 * 4 * 1e2 * eps = 2e-12, rounded up.
RTOL = 1e-11
ROWS = [2, 4, 6, 8, 10, 12, 14, 16]


def _points(rows, last):
    return 64 * rows if last is None else 37 * rows + last % rows + 1


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("last", [0, -2, -1, None])
def test_sh_length_lines(device_ctx, rows, last):
    n = _points(rows, last)
    case = sh_case(r_points=n, l_bound=4, rows=rows, r_bound_bohr=0.2 * n, t_half_as=6.0, store_every=-1, n_basis_l=1)
    comp = case["compiled"]
    print(f"SH symmetric lines: rows={rows} points={n} P={comp.P}", flush=True)
    assert comp.m == rows
    slot = device_ctx.add_sh(comp)
    device_ctx.run(comp.n_steps + 1)
    out = device_ctx.download_sh(slot)
    device_ctx.remove(0, slot)
    g = case["oracle"].run(case["g0"], case["times"], case["dt"], -1, basis=case["basis"])[0]
    assert rel_l2(out.g, g) <= RTOL


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("last", [0, -2, -1, None])
def test_line_adi(device_ctx, rows, last):
    n = _points(rows, last)
    case = line_case(z_bound_bohr=0.1 * n, z_points=n, rows=rows, n_steps=12, store_every=-1)
    comp = case["compiled"]
    print(f"Line symmetric: rows={rows} points={n} P={comp.P}", flush=True)
    assert comp.m == rows
    slot = device_ctx.add_line(comp)
    device_ctx.line_run(comp.n_steps)
    out = device_ctx.download_line(slot)
    device_ctx.remove(1, slot)
    g = case["oracle"].run(case["g0"], case["times"], case["store_every"], basis=case["basis"])[0]
    assert rel_l2(out[0], g) <= RTOL
