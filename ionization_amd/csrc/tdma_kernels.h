// Op-level Thomas solve: the device counterpart of cy.tdma (ionization/cy.pyx:9-50).
#pragma once

#include "common.h"

// Line i occupies [off[i], off[i] + len[i]) of the packed arrays. a[t] multiplies x[t-1], c[t] multiplies
// x[t+1] (a[first] and c[last] are ignored). cp holds the primed super-diagonal; x holds the primed
// right-hand side during the forward sweep and the solution after the back substitution. Recurrence of
// cy.pyx:31-48 with one reciprocal of the pivot instead of two divisions.
//
// The recurrence is a serial chain, about 12 dependent FP64 operations and a reciprocal per row; what
// bounded one thread per line was the wait for each row's loads on top of it (530 ns per row). One wave
// works on a run of rows: the lanes load 64 rows of the four arrays at once, one row a lane and the next
// 64 ahead of need, and put them in LDS; every lane then walks the chain, lane t keeping row t's results
// for one coalesced store.
//
// A line splits where rows t - 1 and t are uncoupled (a[t] = c[t-1] = 0): the recurrence then restarts by
// itself, so the runs on either side are solved by different waves with the same products. The
// reference's own calls are of this kind, an operator of a two-dimensional mesh flattened to one line
// (mesh_operators.py:75-89). Wave w of a line takes the rows from the first such restart in its `span` rows
// to the first one past them; without any restart the line's first wave takes it whole.
//
// An overflowing or singular run would, in one sweep over the whole line, carry its NaN through the
// zero couplings (0 * NaN) into the other runs. A wave of a split line that meets a value that is not
// finite sets *redo, and a second launch (redo_pass) then solves every line as one run.
//
// 100 lines of 250 rows flattened to one call (25 000 unknowns), whole call on host arrays: 13.4 ms ->
// 0.20 ms; the same length without a restart: 5.3 ms.
//
// A wave's instruction costs the same for one row as for 64 lines' rows, so lines that fill the chip by
// themselves are faster with one thread each (k_tdma_threads; tdma_by_threads has the line between the two).
constexpr int kTdmaTile = TDSE_WAVE;

__device__ __forceinline__ bool tdma_zero(double2 v) { return v.x == 0.0 && v.y == 0.0; }
__device__ __forceinline__ bool tdma_finite(double2 v) {
    return fabs(v.x) <= 1.7976931348623157e308 && fabs(v.y) <= 1.7976931348623157e308;
}

// First row in [t, end) where the line restarts, or end. All lanes of the wave take part.
__device__ __forceinline__ int64_t tdma_restart(const double2* __restrict__ a, const double2* __restrict__ c,
                                                int64_t t, int64_t end, int lane) {
    for (; t < end; t += TDSE_WAVE) {
        const int64_t i = t + lane;
        const bool cut = i < end && (i == 0 || (tdma_zero(a[i]) && tdma_zero(c[i - 1])));
        const unsigned long long m = __ballot(cut);
        if (m) return t + __ffsll(m) - 1;
    }
    return end;
}

__global__ void __launch_bounds__(TDSE_WAVE) k_tdma_lines(
    const double2* __restrict__ a, const double2* __restrict__ b, const double2* __restrict__ c,
    const double2* __restrict__ d, double2* __restrict__ x, double2* __restrict__ cp,
    const int64_t* __restrict__ off, const int64_t* __restrict__ len, int64_t n_lines, int64_t span,
    int64_t waves_per_line, int redo_pass, int* __restrict__ redo) {
    // the lines' first waves first, then their second ones: with a line's waves side by side, 8 or 16 of them put all the
    // first waves, which have the whole line to do where it does not split, on one XCD
    const int64_t line = blockIdx.x % (unsigned)n_lines, w = blockIdx.x / (unsigned)n_lines;
    if (w >= waves_per_line || (redo_pass && *redo == 0)) return;
    const int64_t o = off[line], n = len[line];
    if (w * span >= n) return;
    a += o, b += o, c += o, d += o, x += o, cp += o;
    const int lane = threadIdx.x;
    int64_t begin = 0, end = n;
    if (waves_per_line > 1) {
        const int64_t stop = min(n, (w + 1) * span);
        begin = tdma_restart(a, c, w * span, stop, lane);
        if (begin == stop) return;
        end = tdma_restart(a, c, stop, n, lane);
    }
    __shared__ double2 tile[4][kTdmaTile];
    const double2 zero = cmk(0.0, 0.0);
    bool fine = true;
    // forward: primed super-diagonal and right-hand side
    auto fetch = [&](int64_t t0, double2& fa, double2& fb, double2& fc, double2& fd) {
        const int64_t i = t0 + lane;
        const bool in = i < end;
        fa = (in && i > begin) ? a[i] : zero;  // no coupling into the run
        fb = in ? b[i] : cmk(1.0, 0.0);
        fc = (in && i + 1 < n) ? c[i] : zero;
        fd = in ? d[i] : zero;
    };
    double2 fa, fb, fc, fd;
    fetch(begin, fa, fb, fc, fd);
    double2 cprev = zero, dprev = zero;
    for (int64_t t0 = begin; t0 < end; t0 += kTdmaTile) {
        __syncthreads();
        tile[0][lane] = fa;
        tile[1][lane] = fb;
        tile[2][lane] = fc;
        tile[3][lane] = fd;
        __syncthreads();
        if (t0 + kTdmaTile < end) fetch(t0 + kTdmaTile, fa, fb, fc, fd);
        const int rows = (int)min((int64_t)kTdmaTile, end - t0);
        double2 my_c = zero, my_d = zero;
#pragma unroll 4
        for (int t = 0; t < rows; ++t) {
            const double2 at = tile[0][t];
            const double2 r = crecip(csub(tile[1][t], cmul(at, cprev)));
            dprev = cmul(csub(tile[3][t], cmul(at, dprev)), r);
            cprev = cmul(tile[2][t], r);
            if (t == lane) {
                my_c = cprev;
                my_d = dprev;
            }
        }
        if (lane < rows) {
            cp[t0 + lane] = my_c;
            x[t0 + lane] = my_d;
            fine = fine && tdma_finite(my_c) && tdma_finite(my_d);
        }
    }
    // back substitution, tiles from the run's end
    auto fetch_back = [&](int64_t t1, double2& fc, double2& fd) {  // rows t1 - 64 .. t1 - 1
        const int64_t i = t1 - kTdmaTile + lane;
        const bool in = i >= begin;
        fc = (in && i + 1 < end) ? cp[i] : zero;
        fd = in ? x[i] : zero;
    };
    __threadfence_block();
    fetch_back(end, fc, fd);
    double2 xn = zero;
    for (int64_t t1 = end; t1 > begin; t1 -= kTdmaTile) {
        __syncthreads();
        tile[0][lane] = fc;
        tile[1][lane] = fd;
        __syncthreads();
        if (t1 - kTdmaTile > begin) fetch_back(t1 - kTdmaTile, fc, fd);
        const int low = (int)max((int64_t)0, begin - (t1 - kTdmaTile));
        double2 my_x = zero;
#pragma unroll 4
        for (int t = kTdmaTile - 1; t >= low; --t) {
            xn = csub(tile[1][t], cmul(tile[0][t], xn));
            if (t == lane) my_x = xn;
        }
        if (lane >= low) {
            x[t1 - kTdmaTile + lane] = my_x;
            fine = fine && tdma_finite(my_x);
        }
    }
    if (waves_per_line > 1 && !fine) *redo = 1;  // the same value from every wave
}

// One thread per line, the same recurrence and bits.
__global__ void __launch_bounds__(TDSE_WAVE) k_tdma_threads(
    const double2* __restrict__ a, const double2* __restrict__ b, const double2* __restrict__ c,
    const double2* __restrict__ d, double2* __restrict__ x, double2* __restrict__ cp,
    const int64_t* __restrict__ off, const int64_t* __restrict__ len, int64_t n_lines) {
    const int64_t line = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (line >= n_lines) return;
    const int64_t o = off[line], n = len[line];
    double2 cprev = cmk(0.0, 0.0), dprev = cmk(0.0, 0.0);
    for (int64_t t = 0; t < n; ++t) {
        const double2 at = t > 0 ? a[o + t] : cmk(0.0, 0.0);
        const double2 ct = t + 1 < n ? c[o + t] : cmk(0.0, 0.0);
        const double2 r = crecip(csub(b[o + t], cmul(at, cprev)));
        dprev = cmul(csub(d[o + t], cmul(at, dprev)), r);
        cprev = cmul(ct, r);
        x[o + t] = dprev;
        cp[o + t] = cprev;
    }
    double2 xn = dprev;
    for (int64_t t = n - 2; t >= 0; --t) {
        xn = csub(x[o + t], cmul(cp[o + t], xn));
        x[o + t] = xn;
    }
}

// Whether lines are solved by one thread each: when a wave for every line would take longer to issue (about 1.1 ns
// for its workgroup and 0.092 ns for each row, over the whole chip) than the longest line takes as one thread's
// chain (850 ns a row). Past 64 K lines the threads' rows no longer stay in the L2s (each keeps a 128 B line
// of five arrays in use), and waves are faster again from 16 rows on. Device us, threads / waves:
//   lines x rows    1024 x 4    4096 x 8    4096 x 16    8192 x 32   8192 x 250   32768 x 32   65536 x 8   65536 x 32
//                  4.6 / 5.5   8.2 / 9.2  14.4 / 12.6    28 / 32     236 / 230     96 / 102     50 / 79    226 / 201
//   lines x rows   1024 x 100  4096 x 100  16384 x 100  16384 x 1000  65536 x 1   262144 x 4  262144 x 64
//                   67 / 26     84 / 57     100 / 168   1075 / 1550    3.5 / 77    61 / 289   2177 / 1460
// A launch holds fewer than 2^32 threads: past 2^25 lines it is always threads.
inline bool tdma_by_threads(int64_t n_lines, int64_t rows, int64_t longest) {
    if (n_lines >= int64_t(1) << 25) return true;
    if (n_lines >= int64_t(1) << 16 && rows >= 16 * n_lines) return false;
    return 850.0 * (double)longest <= 1.1 * (double)n_lines + 0.092 * (double)rows;
}
