"""
What a simulation takes of the pool is what admission counts for it: its footprint and the allocations' rounding. Meshes
whose norm partials, stored norms by l or second field table are a visible part of it.
"""

import numpy as np
import pytest

from ionization_amd import engine, serve
from ionization_amd import units as u
from tests.cases import cyl_case, line_case

pytestmark = pytest.mark.gpu


def _sh(r_points, l_bound, steps, **kwargs):
    return engine.compile_sh(r_bound=0.1 * r_points * u.bohr_radius, r_points=r_points, l_bound=l_bound,
                             potential=lambda r: np.zeros_like(r), field=lambda t: np.zeros_like(t), mask=None,
                             times=np.linspace(0, steps * u.asec, steps + 1), time_step=u.asec,
                             g0=np.zeros((l_bound, r_points)), **kwargs)


@pytest.mark.parametrize("name, make", [
    ("sh 1000 x 4096", lambda: _sh(1000, 4096, 4)),
    ("sh 1000 x 4095, norm by l", lambda: _sh(1000, 4095, 4, norm_by_l=True)),
    ("sh 100 x 300, norm by l of 1000 steps", lambda: _sh(100, 300, 1000, norm_by_l=True)),
    ("sh adi 60 x 3, 20000 steps", lambda: _sh(60, 3, 20000, store_every=-1, method="adi")),
    ("sh velocity 3000 x 50", lambda: _sh(3000, 50, 4, gauge="velocity")),
    ("sh 5000 x 1, 40 states", lambda: _sh(5000, 1, 4, basis=[(np.ones(5000), 0)] * 40)),
    ("line", lambda: line_case(z_points=8192, n_steps=50)["compiled"]),
    ("cyl", lambda: cyl_case(z_points=90, rho_points=70, t_half_as=10.0)["compiled"]),
])
def test_a_simulation_takes_what_admission_reserves(name, make):
    c = make()
    with engine.DeviceContext(pool_bytes=int(1.2 * c.footprint_bytes) + (4 << 20)) as ctx:
        before = ctx.pool_usage()[0]
        {engine.CompiledSH: ctx.add_sh, engine.CompiledLine: ctx.add_line, engine.CompiledCyl: ctx.add_cyl}[type(c)](c)
        used = ctx.pool_usage()[0] - before
    print(f"footprint: {name}: {used} B used, {c.footprint_bytes} counted", flush=True)
    assert 0.9 * used < c.footprint_bytes and used <= c.footprint_bytes + serve._ALLOC_SLACK
