// Crank-Nicolson line solve by the partition method, complex128, one chunk per thread.
//
// Solves   (1 + w H) y = (1 - w H) x   for one line, where H is tridiagonal and
// w = i tau (tau = dt / 2 hbar; complex tau gives imaginary-time relaxation).
// This is the pair DotOperator(1 - i tau H) then TDMAOperator(1 + i tau H)
// of evolution_methods.py:56-77 / 99-110; the reference solves the implicit
// half with the sequential Thomas recurrence of cy.pyx:31-48, which here is
// replaced by an algebraically equivalent parallel elimination:
//
//  * The line is cut into P chunks of m rows; the calling thread owns chunk k
//    (rows j = k m + i, i < m) in registers.
//  * Rows 0..m-2 of the chunk are eliminated downward in terms of the left
//    unknown L_k = y_{k m - 1}:  y_i = delta_i - alpha_i L_k - gamma_i y_{i+1}.
//  * A running backward pass expresses row 0 through (L_k, Y_k),
//    Y_k = y_{k m + m - 1}; the chunk's last row then gives one equation in
//    (Y_{k-1}, Y_k, Y_{k+1}).
//  * The P-unknown reduced system (every equation normalised to a unit
//    diagonal) is solved in LDS (reduced_cr).
//  * Each thread back-substitutes its rows.
//
// M is the exact number of rows per chunk (a compile-time constant, 2 <= M).
// Requirements: all P threads of the line call this together
// (block-wide barriers), lds holds 3 P double2 for this line and kRedScratch more. Rows beyond the
// physical line are padding rows with H = 0 and x = 0 (they stay 0).
#pragma once

#include <type_traits>

#include "common.h"

template <bool IMAG>
__device__ __forceinline__ double2 wmul(double2 w, double2 v) {
    if constexpr (IMAG) return cimul(w.y, v);
    else return cmul(w, v);
}

// coef(i, hm, h, hp): H_{j,j-1}, H_{j,j}, H_{j,j+1} of the thread's row i.
// xl / xr: x_{km-1} and x_{km+m} (zero at the line ends).
// The reduced system  a_k Y_{k-1} + Y_k + c_k Y_{k+1} = d_k,  k < P  (one equation
// per thread, unit diagonal, a_0 = c_{P-1} = 0): returns Y_k and Y_{k-1}.
//
// Cyclic reduction with compacted threads down to what one wave holds. At stride s the
// surviving equations kk = 2 s (t + 1) - 1 are updated by threads t = 0, 1, ... (so
// whole waves drop out as the system shrinks), eliminating kk - s and kk + s. Once
// the survivors of the block's lines fit 64 lanes, the first wave finishes them without
// block barriers; the eliminated equations s (2 t + 1) - 1 then follow from their solved
// neighbours. The wave's own part takes one of two forms:
//  * pcr: parallel cyclic reduction, log2 levels in which every lane updates its own
//    equation, where cyclic reduction takes as many levels up and again down at the same
//    issue cost (a wave's instruction costs the same with one lane active);
//  * otherwise cyclic reduction, the same products as the block-wide levels form. SH
//    simulations mix rows of very different size, and what a pulse leaves in the largest l is
//    the rounding of amplitudes that cancel: there the bits of a solve show in a stored value
//    (the norm in the largest l), which any change in rounding would move.
// Against cyclic reduction behind block barriers throughout, us per step: one 8192-point
// line (P = 512) 12.2 -> 10.5, 250 x 100 cylinder 20.2 -> 18.4 (pcr).
//
// LANES > 1: LANES independent lines share the block, thread k LANES + ln on equation
// k of line ln, which sits at LDS index k * LANES + ln (each array of 3 holds P * LANES
// entries); all lines have the same P and step through the levels together. The
// wave's own part takes kRedScratch more entries after them, contiguous so that
// neighbouring lanes do not conflict.
constexpr int kRedScratch = 3 * TDSE_WAVE;

template <int LANES = 1>
__device__ __forceinline__ void reduced_cr(double2 A, double2 C, double2 D, const int k, const int P,
                                           double2* __restrict__ lds, double2& Yk, double2& Ykm1,
                                           const int ln = 0, const bool pcr = true) {
    double2* pa = lds + ln;
    double2* pc = lds + P * LANES + ln;
    double2* pd = lds + 2 * P * LANES + ln;
    // a0 Y_- + Y + c0 Y_+ = d0 without its neighbours (am, cm, dm) and (apl, cpl, dpl)
    auto eliminate = [](double2& a0, double2& c0, double2& d0, double2 am, double2 cm, double2 dm, double2 apl,
                        double2 cpl, double2 dpl) {
        const double2 bn = csub(csub(cmk(1.0, 0.0), cmul(a0, cm)), cmul(c0, apl));
        const double2 an2 = cneg(cmul(a0, am));
        const double2 cn2 = cneg(cmul(c0, cpl));
        const double2 dn2 = csub(csub(d0, cmul(a0, dm)), cmul(c0, dpl));
        const double2 ib = crecip(bn);
        a0 = cmul(an2, ib);
        c0 = cmul(cn2, ib);
        d0 = cmul(dn2, ib);
    };
    __syncthreads();
    pa[k * LANES] = A;
    pc[k * LANES] = C;
    pd[k * LANES] = D;
    int s = 1, left = P;  // equations s (t + 1) - 1, t < left, survive
    for (; left * LANES > TDSE_WAVE; s <<= 1, left = P / s) {
        __syncthreads();
        const int kk = 2 * s * (k + 1) - 1;
        if (kk < P) {
            const int e = kk * LANES, em = (kk - s) * LANES, ep = (kk + s) * LANES;
            double2 a0 = pa[e], c0 = pc[e], d0 = pd[e];
            double2 apl = cmk(0.0, 0.0), cpl = cmk(0.0, 0.0), dpl = cmk(0.0, 0.0);
            if (kk + s < P) {
                apl = pa[ep];
                cpl = pc[ep];
                dpl = pd[ep];
            }
            eliminate(a0, c0, d0, pa[em], pc[em], pd[em], apl, cpl, dpl);
            pa[e] = a0;
            pc[e] = c0;
            pd[e] = d0;
        }
    }
    __syncthreads();
    const int t = k * LANES + ln;
    if (t < TDSE_WAVE) {
        double2* __restrict__ w = lds + 3 * P * LANES + t;
        const double2 zero = cmk(0.0, 0.0);
        const bool on = k < left;
        const int e = (s * (k + 1) - 1) * LANES;
        double2 a0 = zero, c0 = zero, d0 = zero;
        if (on) {
            a0 = pa[e];
            c0 = pc[e];
            d0 = pd[e];
        }
        // one wave: its LDS operations complete in order, only the compiler has to keep it
        auto ordered = []() {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        auto publish = [&]() {
            w[0] = a0;
            w[TDSE_WAVE] = c0;
            w[2 * TDSE_WAVE] = d0;
        };
        // this equation without the ones q before and after it
        auto update = [&](int q) {
            double2 am = zero, cm = zero, dm = zero, apl = zero, cpl = zero, dpl = zero;
            if (k >= q) {
                am = w[-q * LANES];
                cm = w[TDSE_WAVE - q * LANES];
                dm = w[2 * TDSE_WAVE - q * LANES];
            }
            if (k + q < left) {
                apl = w[q * LANES];
                cpl = w[TDSE_WAVE + q * LANES];
                dpl = w[2 * TDSE_WAVE + q * LANES];
            }
            __builtin_amdgcn_wave_barrier();
            eliminate(a0, c0, d0, am, cm, dm, apl, cpl, dpl);
        };
        if (pcr) {
            for (int q = 1; q < left; q <<= 1) {
                publish();
                ordered();
                update(q);
            }
        } else {
            publish();
            int q = 1;
            for (; q < left; q <<= 1) {
                ordered();
                if (on && ((k + 1) & (2 * q - 1)) == 0) {
                    update(q);
                    publish();
                }
            }
            for (q >>= 1; q >= 1; q >>= 1) {
                ordered();
                if (on && ((k + 1) & (2 * q - 1)) == q) {
                    const double2 ym = (k >= q) ? w[2 * TDSE_WAVE - q * LANES] : zero;
                    const double2 yp = (k + q < left) ? w[2 * TDSE_WAVE + q * LANES] : zero;
                    d0 = csub(csub(d0, cmul(a0, ym)), cmul(c0, yp));
                    w[2 * TDSE_WAVE] = d0;
                }
            }
        }
        if (on) pd[e] = d0;  // no neighbours left: its d is its solution
    }
    for (s >>= 1; s >= 1; s >>= 1) {
        __syncthreads();
        const int kk = s * (2 * k + 1) - 1;
        if (kk < P) {
            const double2 ym = (kk - s >= 0) ? pd[(kk - s) * LANES] : cmk(0.0, 0.0);
            const double2 yp = (kk + s < P) ? pd[(kk + s) * LANES] : cmk(0.0, 0.0);
            pd[kk * LANES] = csub(csub(pd[kk * LANES], cmul(pa[kk * LANES], ym)), cmul(pc[kk * LANES], yp));
        }
    }
    __syncthreads();
    Yk = pd[k * LANES];
    Ykm1 = (k > 0) ? pd[(k - 1) * LANES] : cmk(0.0, 0.0);
}

// Off-diagonal coefficients w*hm, w*hp: complex in general; for IMAG (w = i s)
// they are i times a real number and are kept as that real number.
template <bool IMAG>
struct OffDiag {
    double2 v;
    __device__ __forceinline__ static OffDiag make(double2 w, double h) {
        OffDiag o;
        o.v = cmk(w.x * h, w.y * h);
        return o;
    }
    __device__ __forceinline__ double2 mul(double2 a) const { return cmul(v, a); }
};
template <>
struct OffDiag<true> {
    double s;  // the coefficient is i * s
    __device__ __forceinline__ static OffDiag make(double2 w, double h) {
        OffDiag o;
        o.s = w.y * h;
        return o;
    }
    __device__ __forceinline__ double2 mul(double2 a) const { return cimul(s, a); }
};

// RHS_IS_X: the right-hand side is x itself (implicit solve only, no explicit
// half); xl / xr are then unused.
template <int M, bool IMAG, class Coef, bool RHS_IS_X = false>
__device__ __forceinline__ void cn_partition(double2 (&x)[M], const int k, const int P,
                                             const double2 xl, const double2 xr, const double2 w,
                                             Coef coef, double2* __restrict__ lds, const bool sync_first) {
    using Off = OffDiag<IMAG>;
    double2 al[M - 1], ga[M - 1], de[M - 1];
    double2 alm = cmk(0.0, 0.0), gam = cmk(0.0, 0.0), dem = cmk(0.0, 0.0);  // row m-2
    double2 dlast = cmk(0.0, 0.0), diaglast = cmk(1.0, 0.0);
    Off sublast = Off::make(w, 0.0), suplast = Off::make(w, 0.0);
#pragma unroll
    for (int i = 0; i < M; ++i) {
        {
            double hm, h, hp;
            coef(i, hm, h, hp);
            double2 d = x[i];
            if constexpr (!RHS_IS_X) {
                const double2 xm = (i == 0) ? xl : x[i > 0 ? i - 1 : 0];
                const double2 xp = (i + 1 < M) ? x[i + 1 < M ? i + 1 : i] : xr;
                // explicit half: d = x - w (hm x_{j-1} + h x_j + hp x_{j+1})
                const double2 hx =
                    cmk(fma(hm, xm.x, fma(h, x[i].x, hp * xp.x)), fma(hm, xm.y, fma(h, x[i].y, hp * xp.y)));
                d = csub(x[i], wmul<IMAG>(w, hx));
            }
            // implicit half coefficients: sub = w hm, diag = 1 + w h, sup = w hp
            const Off sub = Off::make(w, hm);
            const Off sup = Off::make(w, hp);
            const double2 diag = cadd(cmk(1.0, 0.0), wmul<IMAG>(w, cmk(h, 0.0)));
            if (i < M - 1) {
                const double2 den = (i == 0) ? diag : csub(diag, sub.mul(ga[i > 0 ? i - 1 : 0]));
                const double2 r = crecip(den);
                const double2 rsub = sub.mul(r);
                if (i == 0) {
                    al[0] = rsub;
                    de[0] = cmul(r, d);
                } else {
                    al[i] = cneg(cmul(rsub, al[i - 1]));
                    de[i] = csub(cmul(r, d), cmul(rsub, de[i - 1]));
                }
                ga[i] = sup.mul(r);
                alm = al[i];
                gam = ga[i];
                dem = de[i];
            } else {
                dlast = d;
                diaglast = diag;
                sublast = sub;
                suplast = sup;
            }
        }
    }
    // running backward pass: row 0 in terms of (L_k, Y_k), starting from row m-2
    double2 ap0 = alm, gp0 = gam, dp0 = dem;
#pragma unroll
    for (int i = M - 3; i >= 0; --i) {
        ap0 = csub(al[i], cmul(ga[i], ap0));
        gp0 = cneg(cmul(ga[i], gp0));
        dp0 = csub(de[i], cmul(ga[i], dp0));
    }
    if (sync_first) __syncthreads();
    lds[k] = ap0;
    lds[P + k] = gp0;
    lds[2 * P + k] = dp0;
    __syncthreads();
    double2 na = cmk(0.0, 0.0), ng = cmk(0.0, 0.0), nd = cmk(0.0, 0.0);
    if (k + 1 < P) {
        na = lds[k + 1];
        ng = lds[P + k + 1];
        nd = lds[2 * P + k + 1];
    }
    // reduced equation of the chunk's last row: A Y_{k-1} + B Y_k + C Y_{k+1} = D
    double2 A = cneg(sublast.mul(alm));
    const double2 B = csub(csub(diaglast, sublast.mul(gam)), suplast.mul(na));
    double2 C = cneg(suplast.mul(ng));
    double2 D = csub(csub(dlast, sublast.mul(dem)), suplast.mul(nd));
    {
        const double2 ib = crecip(B);
        A = cmul(A, ib);
        C = cmul(C, ib);
        D = cmul(D, ib);
    }
    double2 Lk, Yk;
    reduced_cr(A, C, D, k, P, lds, Yk, Lk);
    D = Yk;
    double2 y = D;
#pragma unroll
    for (int i = M - 1; i >= 0; --i) {
        if (i < M - 1) y = csub(csub(de[i], cmul(al[i], Lk)), cmul(ga[i], y));
        x[i] = y;
    }
}

// Implicit solve (1 + i H) z = x for real H with a smaller register footprint
// than cn_partition: per row only gamma and delta are kept (4 doubles).
//
//  pass 1 (forward): pivots r_i, gamma_i = r_i sup_i, delta_i = r_i (x_i - sub_i delta_{i-1})
//          and the running alpha_i = -r_i sub_i alpha_{i-1}; the row-0 coefficients
//          through (L_k, Y_k) that the previous chunk needs are accumulated forward,
//          alpha'_0 = sum_i pi_i alpha_i, delta'_0 = sum_i pi_i delta_i,
//          gamma'_0 = pi_{m-2} gamma_{m-2}, with pi_i = prod_{k<i} (-gamma_k);
//  reduced system (one equation per chunk, unit diagonal) by cyclic reduction;
//  pass 2 (forward): the left-boundary term mu_i = alpha_i L_k = -r_i sub_i mu_{i-1},
//          pivots recomputed from the stored gamma, delta_i <- delta_i - mu_i;
//  pass 3 (backward): z_{m-1} = Y_k, z_i = delta_i - gamma_i z_{i+1}.
// coef(i, hm, h, hp) as for cn_partition; sub = i hm, diag = 1 + i h, sup = i hp.
// coef2 is called in pass 2 and must re-read the coefficients (not reuse
// pass-1 values held in registers across the reduced solve).
// EXPLICIT: the right-hand side is the explicit half (1 - i H~) x, formed
// row by row in pass 1 from x and the chunk neighbours xl = x_{km-1},
// xr = x_{km+m} (chunk_neighbours); otherwise it is x itself.
// LANES / ln: several interleaved lines per block, as for reduced_cr (in its in-wave reduction form).
//
// ALPHA_LDS (fewer instructions and registers; used where the two-line kernel
// would otherwise spill):
//  * pass 1 forms the pivots from the chunk's leading principal minors (no
//    division in the recurrence) and stores alpha_i, i < m - 2, in LDS after
//    the reduced system's entries, at 3 P LANES + kRedScratch + (i P + k) LANES + ln
//    (M - 2 more P LANES double2; alpha_{m-2} stays in its register);
//  * the row-0 coefficients through (L_k, Y_k) come from a backward sweep over
//    the stored alpha_i instead of the running forward sums;
//  * pass 2 disappears: pass 3 reads alpha_i back and forms
//    z_i = delta_i - alpha_i L_k - gamma_i z_{i+1} (coef2 is not called).
// Every thread reads back only what it wrote, so no barrier is needed.
template <int M, class Coef, class Coef2, bool EXPLICIT = false, int LANES = 1, bool ALPHA_LDS = false>
__device__ __forceinline__ void cn_implicit_lowreg(double2 (&x)[M], const int k, const int P, Coef coef,
                                                   Coef2 coef2, double2* __restrict__ lds,
                                                   const double2 xl = make_double2(0.0, 0.0),
                                                   const double2 xr = make_double2(0.0, 0.0), const int ln = 0) {
    double2* __restrict__ alds = lds + (3 * P + k) * LANES + kRedScratch + ln;  // alpha_i at alds[i P LANES]
    double2 ga[M - 1], de[M - 1];
    double2 al = cmk(0.0, 0.0), pi = cmk(1.0, 0.0), sa = cmk(0.0, 0.0), sd = cmk(0.0, 0.0);
    double2 gprev = cmk(0.0, 0.0), dprev = cmk(0.0, 0.0);
    double2 dlast = cmk(0.0, 0.0), diaglast = cmk(1.0, 0.0);
    double sublast = 0.0, suplast = 0.0;
    double2 Dm1 = cmk(1.0, 0.0), Dm2 = cmk(0.0, 0.0);  // ALPHA_LDS: D_{i-1}, D_{i-2}
    double hpp = 0.0;                                  // ALPHA_LDS: hp_{i-1}
#pragma unroll
    for (int i = 0; i < M; ++i) {
        double hm, h, hp;
        coef(i, hm, h, hp);
        double2 rhs = x[i];
        if constexpr (EXPLICIT) {
            // (1 - i H~) x on row i: x_i - i (hm x_{i-1} + h x_i + hp x_{i+1})
            const double2 xm = (i == 0) ? xl : x[i > 0 ? i - 1 : 0];
            const double2 xp = (i + 1 < M) ? x[i + 1 < M ? i + 1 : i] : xr;
            const double2 hx =
                cmk(fma(hm, xm.x, fma(h, x[i].x, hp * xp.x)), fma(hm, xm.y, fma(h, x[i].y, hp * xp.y)));
            rhs = cmk(x[i].x + hx.y, x[i].y - hx.x);
        }
        if (i < M - 1) {
            double2 r;
            if constexpr (ALPHA_LDS) {
                // The pivots den_i = (1 + i h) - (i hm) gamma_{i-1} are ratios D_i / D_{i-1} of the
                // chunk's leading principal minors, D_i = (1 + i h_i) D_{i-1} + hm_i hp_{i-1} D_{i-2}
                // (D_{-1} = 1, D_{-2} = 0): the recurrence carries no division, and
                // r_i = D_{i-1} / D_i is formed off it. |D_i| >= |D_{i-1}|: every pivot has
                // real part >= 1 (the Hermitian part of 1 + i H, H real symmetric, is the
                // identity, and Schur complements keep that bound), so nothing underflows.
                const double c = hm * hpp;
                const double2 Di = cmk(fma(c, Dm2.x, fma(-h, Dm1.y, Dm1.x)), fma(c, Dm2.y, fma(h, Dm1.x, Dm1.y)));
                const double inv = tdse_rcp(fma(Di.x, Di.x, Di.y * Di.y));
                r = cmk(fma(Dm1.x, Di.x, Dm1.y * Di.y) * inv, fma(Dm1.y, Di.x, -Dm1.x * Di.y) * inv);
                Dm2 = Dm1;
                Dm1 = Di;
                hpp = hp;
            } else {
                // den = (1 + i h) - (i hm) gamma_{i-1}
                const double2 den = (i == 0) ? cmk(1.0, h) : cmk(fma(hm, gprev.y, 1.0), fma(-hm, gprev.x, h));
                r = crecip(den);
            }
            const double2 rsub = cimul(hm, r);
            al = (i == 0) ? rsub : cneg(cmul(rsub, al));
            if constexpr (ALPHA_LDS) {
                if (i < M - 2) alds[(size_t)i * P * LANES] = al;
            }
            const double2 d = (i == 0) ? cmul(r, rhs) : csub(cmul(r, rhs), cmul(rsub, dprev));
            const double2 g = cimul(hp, r);
            if constexpr (!ALPHA_LDS) {
                sa = cadd(sa, cmul(pi, al));
                sd = cadd(sd, cmul(pi, d));
                if (i < M - 2) pi = cneg(cmul(pi, g));
            }
            ga[i] = g;
            de[i] = d;
            gprev = g;
            dprev = d;
        } else {
            dlast = rhs;
            diaglast = cmk(1.0, h);
            sublast = hm;
            suplast = hp;
        }
    }
    double2 gp0;
    if constexpr (ALPHA_LDS) {
        // row 0 through (L_k, Y_k) by a backward sweep from row m-2 over the stored alpha_i
        double2 ap0 = al, dp0 = dprev;
        gp0 = gprev;
#pragma unroll
        for (int i = M - 3; i >= 0; --i) {
            int off = i * P * LANES;
            asm("" : "+v"(off));  // an opaque offset: read back from LDS, not forwarded from the store
            const double2 a = alds[off];
            ap0 = csub(a, cmul(ga[i], ap0));
            gp0 = cneg(cmul(ga[i], gp0));
            dp0 = csub(de[i], cmul(ga[i], dp0));
        }
        sa = ap0;
        sd = dp0;
    } else {
        gp0 = cmul(pi, gprev);  // pi_{m-2} gamma_{m-2}
    }
    __syncthreads();
    lds[k * LANES + ln] = sa;
    lds[(P + k) * LANES + ln] = gp0;
    lds[(2 * P + k) * LANES + ln] = sd;
    __syncthreads();
    double2 na = cmk(0.0, 0.0), ng = cmk(0.0, 0.0), nd = cmk(0.0, 0.0);
    if (k + 1 < P) {
        na = lds[(k + 1) * LANES + ln];
        ng = lds[(P + k + 1) * LANES + ln];
        nd = lds[(2 * P + k + 1) * LANES + ln];
    }
    // reduced equation of the chunk's last row: A Y_{k-1} + B Y_k + C Y_{k+1} = D
    double2 A = cneg(cimul(sublast, al));
    const double2 B = csub(csub(diaglast, cimul(sublast, gprev)), cimul(suplast, na));
    double2 C = cneg(cimul(suplast, ng));
    double2 D = csub(csub(dlast, cimul(sublast, dprev)), cimul(suplast, nd));
    {
        const double2 ib = crecip(B);
        A = cmul(A, ib);
        C = cmul(C, ib);
        D = cmul(D, ib);
    }
    double2 Lk, Yk;
    reduced_cr<LANES>(A, C, D, k, P, lds, Yk, Lk, ln, false);
    if constexpr (ALPHA_LDS) {
        // passes 2 and 3 in one: z_i = delta_i - alpha_i L_k - gamma_i z_{i+1}
        double2 z = Yk;
        x[M - 1] = z;
#pragma unroll
        for (int i = M - 2; i >= 0; --i) {
            const double2 a = (i == M - 2) ? al : alds[(size_t)i * P * LANES];
            z = csub(csub(de[i], cmul(a, Lk)), cmul(ga[i], z));
            x[i] = z;
        }
        return;
    }
    // pass 2: subtract alpha_i L_k
    double2 mu = cmk(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < M - 1; ++i) {
        double hm, h;
        coef2(i, hm, h);
        const double2 den = (i == 0) ? cmk(1.0, h) : cmk(fma(hm, ga[i - 1 > 0 ? i - 1 : 0].y, 1.0),
                                                          fma(-hm, ga[i - 1 > 0 ? i - 1 : 0].x, h));
        const double2 rsub = cimul(hm, crecip(den));
        mu = (i == 0) ? cmul(rsub, Lk) : cneg(cmul(rsub, mu));
        de[i] = csub(de[i], mu);
    }
    // pass 3: back substitution
    double2 z = Yk;
    x[M - 1] = z;
#pragma unroll
    for (int i = M - 2; i >= 0; --i) {
        z = csub(de[i], cmul(ga[i], z));
        x[i] = z;
    }
}

// Implicit solve (1 + i H) z = x for real symmetric H: Line and the cylinder (the SH meshes keep
// cn_implicit_lowreg). Symmetry leaves one real coupling o_i = H_{i,i+1} per row, and per row the solver keeps the
// reciprocal pivot r_i and the eliminated right-hand side u_i (4 doubles):
//
//  pass 1 (forward): r_i = 1 / (1 + i h_i + o_{i-1}^2 r_{i-1}), u_i = r_i (x_i - i o_{i-1} u_{i-1}); the response
//          q_i = r_i p_i, p_{i+1} = -i o_i q_i (p_0 = 1) to a unit right-hand side in row 0, which by symmetry is also
//          row 0's dependence on the other rows: z_0 = sum p_i u_i - i o_left L_k sum p_i q_i + p_{m-1} Y_k;
//  reduced system (one equation per chunk, unit diagonal), reduced_cr;
//  pass 2 (forward): the left neighbour's term, w_0 = -i o_left L_k: u_i <- u_i + r_i w_i, w_{i+1} = -i o_i r_i w_i;
//  pass 3 (backward): z_{m-1} = Y_k, z_i = u_i - r_i (i o_i z_{i+1}).
// Every real factor (i o) stays apart from the complex ones, pass 2 needs neither the pivots' reciprocals nor the
// diagonal again, and sums are fused (cmla): about 62 FP64 operations per row where the general form
// takes 92. Per step, general -> this: an 8192-point line 10.5 -> 8.9 us, 24 velocity-gauge lines 15.6 -> 11.7,
// a 250 x 100 cylinder 16.2 -> 16.0, four of 2000 x 1000
// 137 -> 133. The SH lines would gain too (256 simulations 1.55 -> 1.48 ms per step), but keep their bits (reduced_cr).
//
// coef(i, h, o): row i's diagonal h_i and its coupling o_i to row i + 1, rows in order; off(i): o_i again in
// passes 2 and 3 (in order forwards, then backwards; to be read again, not held across the reduced solve);
// o_left: the coupling of row 0 to the previous chunk's last row. Couplings past the line's last row are 0, or,
// with live(i) (row i is no padding), anything: a padding row's r_i is made 0, and with it all that could pass through
// the row, its own z_i included. One selection per row instead of one for each use of o_i and for h_i (an 8192-point
// line 8.9 -> 8.1 us per step, 24 lines 11.7 -> 10.7). Padding rows hold zeros.
// EXPLICIT, xl, xr, LANES, ln: as for cn_implicit_lowreg. lds: 3 P LANES + kRedScratch double2.
struct AllLive {};

template <int M, bool EXPLICIT, int LANES, class Coef, class Off, class Live = AllLive>
__device__ __forceinline__ void cn_symmetric(double2 (&x)[M], const int k, const int P, const double o_left, Coef coef,
                                             Off off, double2* __restrict__ lds, const double2 xl, const double2 xr,
                                             const int ln = 0, Live live = Live{}) {
    constexpr bool kSelect = !std::is_same_v<Live, AllLive>;
    auto pivot = [&](int i, const double2 den) {
        if constexpr (kSelect) {
            const double inv = live(i) ? tdse_rcp(cabs2(den)) : 0.0;
            return cmk(den.x * inv, -den.y * inv);
        } else {
            return crecip(den);
        }
    };
    double2 r[M - 1], u[M - 1];
    double2 p = cmk(1.0, 0.0), q = p, sa = p, sd = p, flast = p;
    double ob = o_left, hlast = 0.0, olast = 0.0;  // ob: o_{i-1}
#pragma unroll
    for (int i = 0; i < M; ++i) {
        double h, o;
        coef(i, h, o);
        if constexpr (kSelect) {
            if (i == M - 1) ob = live(i) ? ob : 0.0;  // the last row has no r_i
        }
        double2 f = x[i];
        if constexpr (EXPLICIT) {
            // (1 - i H) x on row i: x_i - i (o_{i-1} x_{i-1} + h x_i + o_i x_{i+1})
            const double2 xm = (i == 0) ? xl : x[i > 0 ? i - 1 : 0];
            const double2 xp = (i + 1 < M) ? x[i + 1 < M ? i + 1 : i] : xr;
            f = cmk(fma(ob, xm.y, fma(h, f.y, fma(o, xp.y, f.x))), fma(-ob, xm.x, fma(-h, f.x, fma(-o, xp.x, f.y))));
        }
        if (i < M - 1) {
            if (i == 0) {
                r[0] = pivot(0, cmk(1.0, h));
                q = r[0];
                u[0] = cmul(q, f);
                sa = q;
                sd = u[0];
            } else {
                const double2 rb = r[i > 0 ? i - 1 : 0], ub = u[i > 0 ? i - 1 : 0];
                const double c = ob * ob;
                const double2 ri = pivot(i, cmk(fma(c, rb.x, 1.0), fma(c, rb.y, h)));
                const double2 ui = cmul(ri, cmk(fma(ob, ub.y, f.x), fma(-ob, ub.x, f.y)));
                q = cmul(ri, p);
                sa = cmla(sa, p, q);
                sd = cmla(sd, p, ui);
                r[i < M - 1 ? i : 0] = ri;
                u[i < M - 1 ? i : 0] = ui;
            }
            p = cmk(o * q.y, -o * q.x);
            ob = o;
        } else {
            flast = f;
            hlast = h;
            olast = o;
        }
    }
    __syncthreads();
    lds[k * LANES + ln] = cimul(o_left, sa);
    lds[(P + k) * LANES + ln] = p;
    lds[(2 * P + k) * LANES + ln] = sd;
    __syncthreads();
    double2 na = cmk(0.0, 0.0), np = cmk(0.0, 0.0), nd = cmk(0.0, 0.0);
    if (k + 1 < P) {
        na = lds[(k + 1) * LANES + ln];
        np = lds[(P + k + 1) * LANES + ln];
        nd = lds[(2 * P + k + 1) * LANES + ln];
    }
    // reduced equation of the chunk's last row: A Y_{k-1} + B Y_k + C Y_{k+1} = D, with
    // z_{m-2} = u_{m-2} - i o_left q L_k - i ob r_{m-2} Y_k and the next chunk's z_0 = nd - na Y_k + np Y_{k+1}
    const double c = ob * ob;
    const double2 B = cmk(fma(c, r[M - 2].x, fma(olast, na.y, 1.0)), fma(c, r[M - 2].y, fma(-olast, na.x, hlast)));
    const double2 iB = crecip(B);
    const double2 A = cmul(cscale(ob * o_left, q), iB), C = cmul(cimul(olast, np), iB);
    const double2 D = cmul(cmk(fma(olast, nd.y, fma(ob, u[M - 2].y, flast.x)),
                               fma(-olast, nd.x, fma(-ob, u[M - 2].x, flast.y))), iB);
    double2 Lk, z;
    reduced_cr<LANES>(A, C, D, k, P, lds, z, Lk, ln);
    double2 w = cmk(o_left * Lk.y, -o_left * Lk.x);
#pragma unroll
    for (int i = 0; i < M - 1; ++i) {
        const double2 t = cmul(r[i], w);
        u[i] = cadd(u[i], t);
        if (i < M - 2) {
            const double o = off(i);
            w = cmk(o * t.y, -o * t.x);
        }
    }
    x[M - 1] = z;
#pragma unroll
    for (int i = M - 2; i >= 0; --i) {
        const double o = off(i);
        z = cmla(u[i], r[i], cmk(o * z.y, -o * z.x));
        x[i] = z;
    }
}

// Exchange the first / last rows of every chunk through LDS so each thread
// knows x_{km-1} and x_{km+m}. lds: 2 P double2.
template <int M, int LANES = 1>
__device__ __forceinline__ void chunk_neighbours(const double2 (&x)[M], const int k, const int P,
                                                 double2* __restrict__ lds, double2& xl, double2& xr,
                                                 const bool sync_first, const int ln = 0) {
    if (sync_first) __syncthreads();
    lds[k * LANES + ln] = x[0];
    lds[(P + k) * LANES + ln] = x[M - 1];
    __syncthreads();
    xl = (k > 0) ? lds[(P + k - 1) * LANES + ln] : cmk(0.0, 0.0);
    xr = (k + 1 < P) ? lds[(k + 1) * LANES + ln] : cmk(0.0, 0.0);
}
