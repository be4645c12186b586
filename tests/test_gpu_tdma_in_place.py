"""
tdse_tdma_batched_noalloc with the right-hand side as the output (x is d): the same bits as with an output of its own, also
where a line splits into uncoupled runs and where one of these is not finite, which takes a second sweep of the line.
"""

import numpy as np
import pytest

from ionization_amd import _lib
from tests.test_gpu_tdma_many import _systems
from tests.test_zz_no_alloc import DeviceArrays, ctx, hip  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name, lengths, cuts, overflow", [
    ("one line, runs", [1000], (64, 250, 500, 640), None),
    ("one line, overflow in the elimination", [1000], (64, 250, 500, 640), "forward"),
    ("one line, overflow in the back substitution", [1000], (64, 250, 500, 640), "backward"),
    ("ragged lines, overflow in the back substitution", [700, 1, 64, 65, 333], (100, 164, 300, 699), "backward"),
    ("many lines by threads", [20] * 10000, (10,), "backward"),
])
def test_output_over_the_right_hand_side(ctx, hip, name, lengths, cuts, overflow):  # noqa: F811
    rng = np.random.default_rng(12)
    (sub, diag, sup, d), offsets, lengths = _systems(rng, lengths)
    for t in cuts:
        sub[t] = sup[t - 1] = 0.0
    t = cuts[0] + 3
    if overflow == "forward":  # one sweep carries it on to the line's end, and back
        d[t] = np.inf
    if overflow == "backward":  # x_t = d'_t - 1e200 x_{t+1}, x_{t+1} about 1e200: the rows before it, not the later runs
        sub[t] = sub[t + 1] = 0.0
        diag[t] = diag[t + 1] = 1.0
        sup[t], d[t + 1] = 1e200, 1e200
    print(f"tridiagonal lines in place: {name}", flush=True)
    dev = DeviceArrays(hip, [np.ascontiguousarray(a) for a in (sub, diag, sup, d, np.zeros_like(d))])

    def solve(out):
        _lib.check(_lib.load().tdse_tdma_batched_noalloc(
            ctx, *dev.ptrs[:4], dev.ptrs[out], offsets.ctypes.data_as(_lib.c_int64_p),
            lengths.ctypes.data_as(_lib.c_int64_p), len(lengths), len(d)), ctx)
        return dev.download(out, d)

    apart, over = solve(4), solve(3)
    dev.free()
    if overflow:
        assert not np.isfinite(apart[:t + 1]).any()
        assert np.isfinite(apart[cuts[1] if len(cuts) > 1 else 20:]).all() == (overflow == "backward")
    else:
        assert np.isfinite(apart).all()
    assert np.array_equal(apart, over, equal_nan=True)
