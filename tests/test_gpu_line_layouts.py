"""
LineMesh batches of mixed layouts: up to one line per CU they share one launch (a workgroup of the longest line's
threads, whose extra waves leave), larger batches get a launch for each layout on several streams. Each line must be
the same bits as alone, in its own layout's launch.
"""

import numpy as np
import pytest

from ionization_amd.engine import DeviceContext
from tests.cases import line_case

pytestmark = pytest.mark.gpu

# (points, rows per thread): every rows instance, one and several waves, ragged ends
SHAPES = [(3, 2), (130, 2), (250, 4), (389, 6), (513, 8), (1000, 8), (641, 10), (1535, 12), (900, 14), (2049, 16)]


@pytest.mark.parametrize("copies", [1, 30])  # 10 lines: one launch; 300 lines: a launch for each layout
@pytest.mark.parametrize("method, gauge", [("adi", "length"), ("sio", "length"), ("sio", "velocity")])
def test_line_layouts_together_equal_alone(method, gauge, copies):
    print(f"line layouts {method} {gauge} x{copies}", flush=True)
    comps = [line_case(z_points=n, rows=m, n_steps=12, store_every=5, method=method, gauge=gauge)["compiled"]
             for n, m in SHAPES]

    def run(cs):
        with DeviceContext(pool_bytes=64 << 20 if len(cs) < 50 else 512 << 20) as ctx:
            slots = [ctx.add_line(c) for c in cs]
            ctx.line_run(5)
            ctx.line_run(7)
            return [ctx.download_line(s) for s in slots]

    together = run(comps * copies)
    for i, c in enumerate(comps):
        alone = run([c])[0]
        for k in range(copies):
            got = together[k * len(comps) + i]
            for a, b in zip(alone, got):
                assert np.array_equal(a, b), (SHAPES[i], k)
