"""States as uploads take them: the mesh's own shape, flat, or of fewer points (the rest is zero, as in position order)."""

import numpy as np
import pytest

from ionization_amd import engine


@pytest.mark.parametrize("shape, P, m", [((3, 131), 64, 4), ((389,), 64, 8)])
@pytest.mark.parametrize("points", ["all", "fewer"])
def test_line_states(shape, P, m, points):
    n = shape[-1] if points == "all" else shape[-1] - 30
    g = np.random.default_rng(1).standard_normal(shape[:-1] + (n,)) * (1 + 2j)
    got = engine.mesh_state(g, shape)
    assert got.shape == shape and got.dtype == np.complex128 and got.flags.c_contiguous
    assert np.array_equal(engine.to_positions(got, P, m), engine.to_positions(g, P, m))


@pytest.mark.parametrize("have", [(75, 33), (70, 33), (75, 20), (11, 4)])
def test_cylinder_states(have):
    shape, Pz, Mz, nrpad = (75, 33), 64, 2, 64
    g = np.random.default_rng(2).standard_normal(have)  # real states too
    got = engine.mesh_state(g, shape)
    assert got.shape == shape and got.dtype == np.complex128
    assert np.array_equal(engine.to_cyl_positions(got, Pz, Mz, nrpad), engine.to_cyl_positions(g, Pz, Mz, nrpad))


def test_flat_and_strided_states():
    g = np.random.default_rng(3).standard_normal((6, 8)) + 0j
    assert np.array_equal(engine.mesh_state(g.reshape(-1), (6, 8)), g)
    assert np.array_equal(engine.mesh_state(np.asfortranarray(g), (6, 8)), g)
    assert np.array_equal(engine.mesh_state(np.repeat(g, 2, axis=1)[:, ::2], (6, 8)), g)


@pytest.mark.parametrize("have", [(7, 8), (6, 9), (49,), (2, 3, 9)])
def test_states_of_more_points_are_refused(have):
    with pytest.raises(ValueError):
        engine.mesh_state(np.zeros(have), (6, 8))
