"""A download of a small state is one call of the library, its copy reordered by the host; a larger one is reordered on the device."""

import ctypes
from types import SimpleNamespace

import numpy as np
import pytest

from ionization_amd import engine


class _Library:
    """Stands in for the native library: records the copies it is asked for, and hands out a ramp as position-order g."""

    def __init__(self, size):
        self.size, self.calls = size, []

    def tdse_sim_state(self, ctx, kind, slot, step, n, nd):
        for p, v in ((step, 4), (n, 4), (nd, 5)):
            ctypes.cast(p, ctypes.POINTER(ctypes.c_int32))[0] = v
        return 0

    def tdse_download(self, ctx, kind, slot, g, *data):
        self.calls.append("data and g" if g else "data")
        for i in range(2 * self.size if g else 0):
            g[i] = i
        return 0

    def tdse_download_g(self, ctx, kind, slot, g):
        self.calls.append("g")
        return 0


def _context(c, kind):
    ctx = engine.DeviceContext.__new__(engine.DeviceContext)
    ctx._ctx, ctx._sh, ctx._line, ctx._cyl = None, {0: c}, {0: c}, {}
    ctx._lib = _Library(getattr(c, "l_bound", 1) * c.npad)
    return ctx


@pytest.mark.parametrize("points, P, m, calls", [(100, 64, 2, ["data and g"]), (1000, 64, 16, ["data and g"]),
                                                 (1025, 64, 18, ["data", "g"]), (8192, 512, 16, ["data", "g"])])
def test_line(points, P, m, calls):
    c = SimpleNamespace(z_points=points, P=P, m=m, npad=P * m, basis=[])
    ctx = _context(c, engine.KIND_LINE)
    g, norms, ips = ctx.download_line(0)
    assert ctx._lib.calls == calls and g.shape == (points,) and norms.shape == (5,)
    if len(calls) == 1:
        j = np.arange(points)
        p = (j % m) * P + j // m
        assert np.array_equal(g, 2.0 * p + 1j * (2 * p + 1))


@pytest.mark.parametrize("L, calls", [(1, ["data and g"]), (36, ["data and g"]), (37, ["data", "g"])])
@pytest.mark.parametrize("with_g", [True, False])
def test_sh(L, calls, with_g):
    c = SimpleNamespace(r_points=100, l_bound=L, P=64, m=2, npad=128, basis_l=[], norm_by_l=False)
    ctx = _context(c, engine.KIND_SH)
    r = ctx.download_sh(0, with_g=with_g)
    assert ctx._lib.calls == (calls if with_g else ["data"])
    assert r.g.shape == (L, 100) if with_g else r.g is None
