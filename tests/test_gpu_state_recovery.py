"""
A slot whose state stopped being finite is as good as new after a fresh upload. The solves carry a NaN into the padding
rows that share a line with it, so an upload has to write zeros there too (both buffers of an SH mesh);
run again, the simulation must give the bits of one that never held a NaN. Sizes with a thread whose last
rows are padding, with threads that are all padding, and (where the layout allows it) with no padding at all.
"""

import numpy as np
import pytest

from ionization_amd import _lib, engine
from tests.cases import cyl_case, line_case, sh_case

pytestmark = pytest.mark.gpu

CASES = {
    "sh 131 x 10, 4 rows": lambda: sh_case(r_points=131, l_bound=10, t_half_as=12.0, store_every=5, rows=4),
    "sh 120 x 9, 2 rows": lambda: sh_case(r_points=120, l_bound=9, t_half_as=12.0, store_every=5, rows=2),
    "sh velocity 649 x 6, 12 rows": lambda: sh_case(r_points=649, l_bound=6, t_half_as=12.0, store_every=5, rows=12,
                                                    gauge="velocity"),
    "sh adi 131 x 10, 6 rows": lambda: sh_case(r_points=131, l_bound=10, t_half_as=12.0, store_every=5, rows=6,
                                               method="adi"),
    "line 389, 6 rows": lambda: line_case(z_points=389, rows=6, n_steps=24, store_every=5),
    "line 128, 2 rows": lambda: line_case(z_points=128, rows=2, n_steps=24, store_every=5),
    "line velocity 301": lambda: line_case(z_points=301, n_steps=24, store_every=5, method="sio", gauge="velocity"),
    "cyl 75 x 33": lambda: cyl_case(z_points=75, rho_points=33, t_half_as=10.0, store_every=5),
    "cyl 128 x 30, no z padding": lambda: cyl_case(z_points=128, rho_points=30, z_rows=2, t_half_as=10.0, store_every=5),
    "cyl 70 x 64, no rho padding": lambda: cyl_case(z_points=70, rho_points=64, rho_shape=(4, 4), t_half_as=10.0,
                                                   store_every=5),
}


def _kind(c):
    return {engine.CompiledSH: engine.KIND_SH, engine.CompiledLine: engine.KIND_LINE, engine.CompiledCyl: engine.KIND_CYL}[type(c)]


def _run(ctx, c, slot):
    kind = _kind(c)
    ctx.run(c.n_steps + (kind == engine.KIND_SH))
    if kind == engine.KIND_SH:
        r = ctx.download_sh(slot)
        return r.g, r.norms, r.lnorms, r.ips
    return ctx.download_line(slot) if kind == engine.KIND_LINE else ctx.download_cyl(slot)


@pytest.mark.parametrize("raw", [False, True])
@pytest.mark.parametrize("at", ["first row", "last row"])
@pytest.mark.parametrize("name", list(CASES))
def test_fresh_upload_after_a_nan(name, at, raw):
    case = CASES[name]()
    c, kind = case["compiled"], _kind(case["compiled"])
    print(f"state recovery: {name}, NaN in the {at}, {'position' if raw else 'natural'} order", flush=True)
    bad = np.array(case["g0"], dtype=np.complex128)
    bad.reshape(-1)[0 if at == "first row" else -1] = np.nan
    with engine.DeviceContext(pool_bytes=2 * c.footprint_bytes + (16 << 20)) as ctx:
        slot = {engine.KIND_SH: ctx.add_sh, engine.KIND_LINE: ctx.add_line, engine.KIND_CYL: ctx.add_cyl}[kind](c)
        clean = _run(ctx, c, slot)
        assert all(np.isfinite(x).all() for x in clean)
        ctx.upload_state(kind, slot, bad, 0)
        assert not np.isfinite(_run(ctx, c, slot)[0]).all()
        if raw:
            _lib.check(ctx._lib.tdse_upload_state(ctx._ctx, kind, slot, _lib.dptr(np.ascontiguousarray(c.g0)), 0), ctx._ctx)
        else:
            ctx.upload_state(kind, slot, case["g0"], 0)
        again = _run(ctx, c, slot)
        for a, b in zip(clean, again):
            assert np.array_equal(a, b)
