"""
A batch that mixes layouts must not pay for sharing launches: one deep mesh beside many shallow ones, whose workgroups
would all take the deep one's threads, LDS and registers. A step of the whole batch may take no longer than a step of the
deep mesh followed by a step of the shallow ones, with 20 % for the clock. And many ADI meshes of one layout, which
have nothing to share, may take no longer than by the launches of their layout (25 % for the clock).
"""

import numpy as np
import pytest

from ionization_amd import engine
from ionization_amd import units as u

pytestmark = pytest.mark.gpu

STEPS = 80


def _mesh(r_points, l_bound, gauge, method):
    g0 = np.zeros((l_bound, r_points), dtype=np.complex128)
    g0[0] = 1.0
    return engine.compile_sh(
        r_bound=0.2 * r_points * u.bohr_radius, r_points=r_points, l_bound=l_bound,
        potential=lambda r: -1e-18 * np.ones_like(r), field=lambda t: 1e9 * np.ones_like(t), mask=None,
        times=np.linspace(0, STEPS * u.asec, STEPS + 1), time_step=u.asec, g0=g0, store_every=-1, gauge=gauge,
        method=method)


def _us_per_step(comps, each_layout=False):
    with engine.DeviceContext(pool_bytes=int(1.1 * sum(c.footprint_bytes for c in comps)) + (64 << 20)) as ctx:
        for c in comps:
            ctx.add_sh(c)
        ctx.profile(each_layout)  # a profiled pass launches each layout by itself
        ctx.run(16, use_graph=not each_layout)
        return 1e3 * min(ctx.run(8, use_graph=not each_layout) for _ in range(6)) / 8


@pytest.mark.parametrize("gauge, method", [("length", "sio"), ("velocity", "sio"), ("length", "adi")])
def test_a_deep_mesh_does_not_slow_many_shallow_ones(gauge, method):
    deep, shallow = _mesh(4000, 50, gauge, method), _mesh(250, 50, gauge, method)
    alone = _us_per_step([deep]) + _us_per_step([shallow] * 300)
    batch = _us_per_step([deep] + [shallow] * 300)
    print(f"{method} {gauge}: {batch:.1f} us, one after the other {alone:.1f} us", flush=True)
    assert batch < 1.2 * alone


def test_adi_meshes_of_one_layout():
    meshes = [_mesh(250, 100, "length", "adi")] * 448
    batch, each = _us_per_step(meshes), _us_per_step(meshes, each_layout=True)
    print(f"448 ADI meshes of one layout: {batch:.1f} us, by their layout's launches {each:.1f} us", flush=True)
    assert batch < 1.25 * each
