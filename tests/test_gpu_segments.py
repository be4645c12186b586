"""
The L-phase gives a wave as many l-rows as the batch can afford (4 rows in a small batch, up to 64 in a large one).
A simulation's wavefunction, norms, largest-l norms, norms by l and inner products must be the same bits either way:
the same simulation alone (4-row segments) and beside fillers that push the batch to the longest segments.
"""

import numpy as np
import pytest

from ionization_amd import engine
from ionization_amd import units as u
from ionization_amd.engine import DeviceContext
from tests.cases import sh_case

pytestmark = pytest.mark.gpu


def _filler(r_points=4000, l_bound=300):
    r_bound = 400 * u.bohr_radius
    g0 = np.zeros((l_bound, r_points), dtype=np.complex128)
    g0[0] = 1.0
    return engine.compile_sh(
        r_bound=r_bound, r_points=r_points, l_bound=l_bound, potential=lambda r: -1e-18 * np.ones_like(r),
        field=lambda t: 1e9 * np.ones_like(t), mask=None, times=np.linspace(0, 40 * u.asec, 41), time_step=u.asec,
        g0=g0, store_every=-1)


@pytest.mark.parametrize("gauge", ["length", "velocity"])
@pytest.mark.parametrize("l_bound, store_every", [(1, 1), (9, 1), (17, 3), (64, 1), (73, 1), (130, 7)])
def test_results_do_not_depend_on_the_segment_length(l_bound, store_every, gauge):
    if gauge == "velocity" and l_bound < 2:
        pytest.skip("the velocity gauge needs two l")
    case = sh_case(r_points=131, l_bound=l_bound, t_half_as=12.0, store_every=store_every, norm_by_l=True, gauge=gauge)
    comp = case["compiled"]
    print(f"segments: l_bound={l_bound} every={store_every} {gauge}", flush=True)

    def run(fillers):
        with DeviceContext(pool_bytes=(comp.footprint_bytes + sum(f.footprint_bytes for f in fillers)) * 2 + (64 << 20)) as ctx:
            slot = ctx.add_sh(comp)
            for f in fillers:
                ctx.add_sh(f)
            ctx.run(comp.n_steps + 1)
            return ctx.download_sh(slot)

    fill = _filler()
    # columns of 64 positions times 64-row segments: enough for more than 4096 waves of 64 rows
    n = 1 + 4096 // ((fill.npad // 64) * (fill.l_bound // 64))
    alone, batch = run([]), run([fill] * n)
    for name in ("g", "norms", "lnorms", "ips", "norm_by_l"):
        assert np.array_equal(getattr(alone, name), getattr(batch, name)), name
    # and the norms add up: by l to the total, each sum in its own order
    assert np.allclose(alone.norm_by_l.sum(axis=1), alone.norms, rtol=1e-13, atol=0)
    assert np.allclose(alone.norm_by_l[:, -1], alone.lnorms, rtol=1e-13, atol=1e-300)
