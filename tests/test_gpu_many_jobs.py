"""
A batch with more than 1024 observation jobs gives them, and with them the counting of the steps, a launch of their own
instead of letting them ride in the next one: beside the solves on a side stream where each layout has a launch, on
the main stream otherwise. Every simulation must give the bits that it gives alone.
"""

import numpy as np
import pytest

from ionization_amd.engine import DeviceContext
from tests.cases import sh_case

pytestmark = pytest.mark.gpu

STATES = 24  # of each simulation; with the norm and the count 26 jobs


def _case(r_points, l_bound, gauge="length", method="sio", rows=None):
    c = sh_case(r_points=r_points, l_bound=l_bound, t_half_as=4.0, store_every=3, n_basis_l=2, gauge=gauge, method=method,
                rows=rows, r_bound_bohr=0.2 * r_points)["compiled"]
    n = len(c.basis_l)  # the eigenstates over and over
    pick = [i % n for i in range(STATES)]
    c.basis, c.basis_l = np.ascontiguousarray(c.basis[pick]), np.ascontiguousarray(c.basis_l[pick])
    return c


def _results(comps):
    with DeviceContext(pool_bytes=int(1.2 * sum(c.footprint_bytes for c in comps)) + (32 << 20)) as ctx:
        slots = [ctx.add_sh(c) for c in comps]
        for k in (4, 3, 2):
            ctx.run(k)
        return [ctx.download_sh(s) for s in slots]


@pytest.mark.parametrize("name, kinds", [
    ("one layout", [dict(r_points=70, l_bound=5)]),
    ("several layouts in one launch", [dict(r_points=70, l_bound=5), dict(r_points=200, l_bound=4, rows=4)]),
    ("a launch for each layout", [dict(r_points=70, l_bound=5), dict(r_points=4200, l_bound=2)]),
    ("velocity gauge", [dict(r_points=70, l_bound=5, gauge="velocity"), dict(r_points=200, l_bound=4, gauge="velocity")]),
    ("adi", [dict(r_points=70, l_bound=5, method="adi"), dict(r_points=200, l_bound=4, method="adi")]),
    ("adi beside the split operator", [dict(r_points=70, l_bound=5, method="adi"), dict(r_points=200, l_bound=4)]),
])
def test_more_jobs_than_ride(name, kinds):
    own = [_case(**k) for k in kinds]
    count = -(-1024 // (STATES + 2)) + 1
    comps = [own[0]] * count + own[1:]
    print(f"many jobs: {name}, {len(comps) * (STATES + 2)} jobs", flush=True)
    assert len(comps) * (STATES + 1) > 1024  # also where the ADI simulations' counts are not among them
    alone = [_results([c])[0] for c in own]
    for i, got in enumerate(_results(comps)):
        want = alone[0 if i < count else i - count + 1]
        for field in ("g", "norms", "lnorms", "ips"):
            assert np.array_equal(getattr(got, field), getattr(want, field)), (i, field)
