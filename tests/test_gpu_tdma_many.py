"""
Batches of many tridiagonal lines: they are solved by one thread or by one or more waves a line, whichever is faster
for their number and lengths, with the same bits. Batches on both sides of that rule, at its edges, with a span of more
than 64 rows per wave, and with a line that is not finite; and a batch of lines that do not split has to use the whole chip.
"""

import time

import numpy as np
import pytest

from ionization_amd import _lib
from tests.test_zz_no_alloc import DeviceArrays, ctx, hip  # noqa: F401

pytestmark = pytest.mark.gpu


def _systems(rng, lengths, gap=0):
    lengths = np.asarray(lengths, dtype=np.int64)
    offsets = np.concatenate([[0], np.cumsum(lengths + gap)[:-1]]).astype(np.int64)
    total = int(offsets[-1] + lengths[-1])
    z = lambda: rng.standard_normal(total) + 1j * rng.standard_normal(total)
    return [z(), z() + 4.0, z(), z()], offsets, lengths


@pytest.mark.parametrize("name, lengths", [
    ("1024 x 4", [4] * 1024), ("1024 x 5", [5] * 1024), ("8192 x 93", [93] * 8192), ("8192 x 94", [94] * 8192),
    ("65535 x 16", [16] * 65535), ("65536 x 15", [15] * 65536),
    ("65536 x 16", [16] * 65536), ("300001 x 3", [3] * 300001),
    ("ragged by threads", [1 + (7 * i) % 40 for i in range(20000)]),
    ("ragged by waves", [1 + (7 * i) % 400 for i in range(1500)]),
])
def test_lines_of_a_large_batch_equal_themselves_alone(device_ctx, name, lengths):
    rng = np.random.default_rng(len(lengths))
    (sub, diag, sup, d), offsets, lengths = _systems(rng, lengths, gap=1)
    print(f"tridiagonal lines: {name}", flush=True)
    x = device_ctx.tdma_batched(sub, diag, sup, d, offsets, lengths)
    for i in [0, 1, 63, 64, len(lengths) // 2, len(lengths) - 2, len(lengths) - 1]:
        s = slice(int(offsets[i]), int(offsets[i] + lengths[i]))
        assert np.array_equal(x[s], device_ctx.tdma(sub[s], diag[s], sup[s], d[s])), i
    # every line's residual: rounding of about ten operations per row on terms of up to ten times the largest |x|,
    # times the growth that pivots of at least 0.1 allow in an elimination without pivoting
    first = np.zeros(len(x), dtype=bool)
    first[offsets] = True
    last = np.zeros(len(x), dtype=bool)
    last[offsets + lengths - 1] = True
    inside = np.zeros(len(x), dtype=bool)
    for k in range(int(lengths.max())):
        inside[(offsets + k)[lengths > k]] = True
    r = diag * x - d
    r[1:] += np.where(first[1:], 0, sub[1:] * x[:-1])
    r[:-1] += np.where(last[:-1], 0, sup[:-1] * x[1:])
    size = np.maximum(1.0, np.abs(x)).max()
    assert np.abs(r[inside]).max() < 1e-11 * size


def test_waves_of_more_than_64_rows(device_ctx):
    """4095 short lines leave a long one 256 waves: 79 rows for each, so a wave looks for a restart in two blocks."""
    rng = np.random.default_rng(8)
    (sub, diag, sup, d), offsets, lengths = _systems(rng, [3] * 4000 + [20000] + [2] * 95)
    o = int(offsets[4000])
    cuts = [1, 78, 79, 80, 157, 158, 316, 1000, 1070, 9999, 19999]
    for t in cuts:
        sub[o + t] = sup[o + t - 1] = 0.0
    x = device_ctx.tdma_batched(sub, diag, sup, d, offsets, lengths)
    for b, e in zip([0, *cuts], [*cuts, 20000]):
        s = slice(o + b, o + e)
        assert np.array_equal(x[s], device_ctx.tdma(sub[s], diag[s], sup[s], d[s])), (b, e)
    for i in (0, 3999, 4001, 4095):
        s = slice(int(offsets[i]), int(offsets[i] + lengths[i]))
        assert np.array_equal(x[s], device_ctx.tdma(sub[s], diag[s], sup[s], d[s])), i


def test_a_line_that_is_not_finite_spoils_itself_only(device_ctx):
    rng = np.random.default_rng(9)
    (sub, diag, sup, d), offsets, lengths = _systems(rng, [20] * 10000)
    sub[offsets[7] + 10] = sup[offsets[7] + 9] = 0.0
    d[offsets[7] + 15] = np.inf
    x = device_ctx.tdma_batched(sub, diag, sup, d, offsets, lengths).reshape(10000, 20)
    assert not np.isfinite(x[7]).any()
    assert np.isfinite(np.delete(x, 7, axis=0)).all()


def test_lines_that_do_not_split_use_the_whole_chip(ctx, hip):  # noqa: F811
    """2048 lines of 1000 rows are two waves for each SIMD: they may take little longer than 256 such lines. With a
    line's 16 waves side by side in the grid their work fell on one XCD, and took more than six times as long."""
    rng = np.random.default_rng(10)
    best = {}
    for n in (256, 2048):
        arrays, offsets, lengths = _systems(rng, [1000] * n)
        dev = DeviceArrays(hip, [np.ascontiguousarray(a) for a in arrays] + [np.zeros(1000 * n, dtype=complex)])
        times = []
        for _ in range(6):
            t = time.perf_counter()
            _lib.check(_lib.load().tdse_tdma_batched_noalloc(
                ctx, *dev.ptrs, offsets.ctypes.data_as(_lib.c_int64_p), lengths.ctypes.data_as(_lib.c_int64_p), n,
                1000 * n), ctx)
            times.append(time.perf_counter() - t)
        dev.free()
        best[n] = min(times)
    print(f"256 lines {best[256] * 1e6:.0f} us, 2048 lines {best[2048] * 1e6:.0f} us")
    assert best[2048] < 3 * best[256]
