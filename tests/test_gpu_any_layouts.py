"""
SH batches of several layouts share one launch per sweep while they are small; larger ones, and the profiled pass, launch
each layout by itself. Both routes must give the same bits: observables of every step and the wavefunctions, for
every rows-per-thread instance in the length gauge, the velocity gauge and ADI.
"""

import numpy as np
import pytest

from ionization_amd.engine import DeviceContext
from tests.cases import sh_case

pytestmark = pytest.mark.gpu

# (radial points, rows per thread, l): one, two and four waves per line; odd, even, single and paired l rows
SHAPES = [(100, 2, 5), (250, 4, 8), (310, 6, 2), (512, 8, 7), (900, 8, 4), (640, 10, 9), (1500, 12, 4), (890, 14, 6),
          (1024, 16, 3), (3000, 16, 5)]


@pytest.mark.parametrize("kind", ["length", "velocity", "adi", "mixed"])
def test_one_launch_for_all_layouts_gives_the_layout_launches_bits(kind):
    comps = []
    for i, (n, m, L) in enumerate(SHAPES):
        method = {"mixed": ["length", "velocity", "adi"][i % 3]}.get(kind, kind)
        comps.append(sh_case(r_points=n, l_bound=L, rows=m, t_half_as=6.0, store_every=2, n_basis_l=2,
                             r_bound_bohr=0.2 * n, gauge="velocity" if method == "velocity" else "length",
                             method="adi" if method == "adi" else "sio")["compiled"])
    print(f"any layouts: {kind}", flush=True)

    def run(each_layout):
        with DeviceContext(pool_bytes=256 << 20) as ctx:
            slots = [ctx.add_sh(c) for c in comps]
            ctx.profile(each_layout)
            for k in (5, 8):
                ctx.run(k, use_graph=not each_layout)
            ctx.profile(False)
            return [ctx.download_sh(s) for s in slots]

    for c, a, b in zip(comps, run(False), run(True)):
        for name in ("g", "norms", "lnorms", "ips"):
            assert np.array_equal(getattr(a, name), getattr(b, name)), (c.r_points, c.m, c.gauge, c.method, name)
