"""
Tridiagonal lines that split into uncoupled runs (rows t - 1 and t with sub[t] = sup[t - 1] = 0): solved by several waves,
each run must equal its solution alone, bit for bit, and the whole must match the oracle's sequential sweep. One zero
coupling alone does not split a line. A run that overflows takes its NaN through the whole line, as one sweep does.
"""

import numpy as np
import pytest

from oracle import mesh_cpu
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu


def _line(rng, n, cuts=(), half=()):
    z = lambda: rng.standard_normal(n) + 1j * rng.standard_normal(n)
    sub, sup, d, diag = z(), z(), z(), z() + 4.0
    for t in cuts:
        sub[t] = sup[t - 1] = 0.0
    for i, t in enumerate(half):
        (sub if i % 2 else sup)[t - (0 if i % 2 else 1)] = 0.0
    return sub, diag, sup, d


@pytest.mark.parametrize("n, cuts, half", [
    (1, (), ()), (64, (), (10, 30)), (65, (64,), ()), (128, (64,), (1, 100)), (129, (1, 2, 3, 128), ()),
    (1000, (250, 500, 750), (251, 499)), (1003, (63, 65, 130, 640, 1002), (64,)), (5000, (), (64, 128, 2500)),
    (300, tuple(range(1, 300)), ()),
])
def test_runs_equal_their_solutions_alone(device_ctx, n, cuts, half):
    rng = np.random.default_rng(n)
    sub, diag, sup, d = _line(rng, n, cuts, half)
    x = device_ctx.tdma(sub, diag, sup, d)
    edges = [0, *cuts, n]
    for b, e in zip(edges[:-1], edges[1:]):
        assert np.array_equal(x[b:e], device_ctx.tdma(sub[b:e], diag[b:e], sup[b:e], d[b:e])), (b, e)
    ref = mesh_cpu.thomas(sub, diag, sup, d) if n > 1 else d / diag  # the oracle takes two rows or more
    # both sweeps carry rounding errors of a few n eps times the conditioning of these rows (|diag| > 4 on average)
    assert rel_l2(x, ref) < 1e-11


def test_ragged_systems_with_runs(device_ctx):
    rng = np.random.default_rng(3)
    lengths = np.array([700, 1, 64, 65, 2, 333], dtype=np.int64)
    offsets = np.concatenate([[0], np.cumsum(lengths + 3)[:-1]])
    total = int(offsets[-1] + lengths[-1])
    sub, diag, sup, d = _line(rng, total)
    for t in (100, 164, 300, 699, offsets[5] + 64):
        sub[t] = sup[t - 1] = 0.0
    x = device_ctx.tdma_batched(sub, diag, sup, d, offsets, lengths)
    for o, n in zip(offsets, lengths):
        s = slice(int(o), int(o + n))
        assert np.array_equal(x[s], device_ctx.tdma(sub[s], diag[s], sup[s], d[s]))


def test_a_run_that_is_not_finite_spoils_the_line_as_in_one_sweep(device_ctx):
    rng = np.random.default_rng(5)
    sub, diag, sup, d = _line(rng, 400, cuts=(150, 300))
    d[200] = np.inf
    x = device_ctx.tdma(sub, diag, sup, d)
    with np.errstate(all="ignore"):
        ref = mesh_cpu.thomas(sub, diag, sup, d)
    assert np.array_equal(np.isfinite(x), np.isfinite(ref))
    assert not np.isfinite(x).any()
