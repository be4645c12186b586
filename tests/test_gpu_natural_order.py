"""
Wavefunctions cross between natural order and device positions on the device. They must equal the host's own
reordering (to_positions, to_cyl_positions) of the raw copy, keep the padding positions zero, survive a round trip bit
for bit, and do so when the pool has no room for a staging copy (row by row, or through a block outside the pool).
"""

import ctypes

import numpy as np
import pytest

from ionization_amd import _lib, engine
from ionization_amd.engine import DeviceContext
from tests.cases import cyl_case, line_case, sh_case

pytestmark = pytest.mark.gpu


def _sims():
    yield "sh", sh_case(r_points=131, l_bound=5, t_half_as=3.0)["compiled"]
    yield "sh one row", sh_case(r_points=640, l_bound=1, rows=10, t_half_as=3.0, n_basis_l=1)["compiled"]
    yield "line", line_case(z_points=389, rows=6, n_steps=5)["compiled"]
    yield "cyl odd rho", cyl_case(z_points=75, rho_points=33, t_half_as=3.0)["compiled"]


def _raw(ctx, kind, slot, shape):
    g = np.empty(shape, dtype=np.complex128)
    _lib.check(ctx._lib.tdse_download(ctx._ctx, kind, slot, _lib.dptr(g), None, None, None), ctx._ctx)
    return g


@pytest.mark.parametrize("spare", ["room", "some rows", "full"])
def test_natural_order_round_trip(spare):
    rng = np.random.default_rng(1)
    for name, c in _sims():
        print(f"natural order: {name}, pool {spare}", flush=True)
        kind = {engine.CompiledSH: 0, engine.CompiledLine: 1, engine.CompiledCyl: 2}[type(c)]
        shape = {0: lambda: (c.l_bound, c.r_points), 1: lambda: (c.z_points,),
                 2: lambda: (c.z_points, c.rho_points)}[kind]()
        with DeviceContext(pool_bytes=c.footprint_bytes + (1 << 20)) as ctx:
            slot = {0: ctx.add_sh, 1: ctx.add_line, 2: ctx.add_cyl}[kind](c)
            if spare != "room":
                # fill the pool with idle lines until the staging copy does not fit
                small = line_case(z_points=3, rows=2, n_steps=2)["compiled"]
                try:
                    while True:
                        last = ctx.add_line(small)
                except Exception:
                    pass
                if spare == "some rows":
                    ctx.remove(engine.KIND_LINE, last)
            g = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
            ctx.upload_state(kind, slot, g, 0)
            if kind == 2:
                raw = _raw(ctx, kind, slot, (c.nrpad, c.npz))
                assert np.array_equal(raw, engine.to_cyl_positions(g, c.Pz, c.Mz, c.nrpad)), name
                back = ctx.download_cyl(slot)[0]
            else:
                raw = _raw(ctx, kind, slot, shape[:-1] + (c.npad,))
                assert np.array_equal(raw, engine.to_positions(g, c.P, c.m)), name
                back = ctx.download_sh(slot).g if kind == 0 else ctx.download_line(slot)[0]
            assert back.shape == shape and np.array_equal(back, g), name


def test_bad_slots_are_refused(device_ctx):
    g = np.zeros(4, dtype=np.complex128)
    for kind, slot in ((0, 9999), (1, -1), (2, 9999), (3, 0)):
        assert device_ctx._lib.tdse_download_g(device_ctx._ctx, kind, slot, _lib.dptr(g)) != 0
        assert device_ctx._lib.tdse_upload_g(device_ctx._ctx, kind, slot, _lib.dptr(g), 0) != 0
    assert device_ctx._lib.tdse_download_g(device_ctx._ctx, 0, 0, ctypes.cast(None, _lib.c_double_p)) != 0
