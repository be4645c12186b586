// CylindricalSliceMesh, length gauge, alternating-direction implicit step on gfx950.
//
// One reference step n (evolution_methods.py:52-77 with the total Hamiltonian
// of mesh_operators.py:282-298, then the mask of meshes.py:256-257) is
//     g <- M . I_rho . E_z . I_z . E_rho . g
// with E_d = 1 - i tau_n H_d (DotOperator) and I_d = (1 + i tau_n H_d)^-1
// (TDMAOperator) along direction d. H_z and H_rho each carry the kinetic term
// of their direction (mesh_operators.py:561-600) plus half of the Coulomb
// potential and half of the length-gauge interaction -z q E(t_{n+1})
// (mesh_operators.py:244-298, 602-628); tau_n = (t_{n+1} - t_n) / (2 hbar).
//
// Two HBM sweeps per step (64 B per mesh point):
//   z-sweep   E_z I_z = 2 (1 + i tau H_z)^-1 - 1 along every z-line (the two
//             halves share one matrix, so they collapse to the Cayley form);
//   rho-sweep E_rho(n+1) . [observe] . M . I_rho(n) along every rho-line: the
//             implicit half of step n, the mask, the observables of the exact
//             g after n+1 steps, and the explicit half of step n+1.
// A simulation held at an exact state (phase 1: its last rho-sweep skipped the
// explicit half, at the end of the run or when the host asked for exact states)
// gets that half from the pre-sweep at the start of its next step.
//
// Layout of one simulation in HBM: g[rho][p], rho in [0, nrpad), p in [0, npz),
// npz = Pz * Mz. The z index of position p is jz = (p % Pz) * Mz + p / Pz, as
// for the SphericalHarmonicMesh radial layout, so the z-sweep thread k holds
// rows jz = k Mz .. k Mz + Mz - 1 of one rho-line at unit stride across the
// wave. The rho-sweep puts LANES consecutive positions (LANES z-lines) side by
// side in every wave: a wave reads 64 / LANES runs of LANES * 16 B. Padding
// (jz >= nz, rho >= nr) is zero in g and gets zero coefficients.
#pragma once

#include "common.h"
#include "line_solver.h"
#include "sh_kernels.h"

struct CylSim {
    double2* g;             // [nrpad][npz]
    const double* zt;       // [npz] z of every position (0 for padding)
    const double* roff;     // [nrpad] off-diagonal rp c(j + 1) of rho between j = c Mr + i and j + 1, at i Cr + c; 0 past
                            // the line
    const double* fs;       // [N] E(t_{n+1})
    const double* ts;       // [N] tau_n = (t_{n+1} - t_n) / (2 hbar)
    double* part;           // [n_groups][1 + 2 n_basis] observation partials of the rho-sweep blocks
    double* out_norm;       // [n_data]
    double2* out_ip;        // [n_data][n_basis]
    const double2* basis;   // [n_basis][nrpad][npz] test states in device layout
    double zp, rp;          // kinetic prefactors -hbar^2 / (2 mu dz^2), -hbar^2 / (2 mu drho^2)
    double kc;              // Coulomb numerator k Q q: V = kc / r
    double q;               // test charge
    double delta;           // inner-product weight dz drho
    double m_inner, m_outer, m_inv_s;  // RadialCosineMask (inner, outer, 1 / smoothness)
    double z0, dz, rho0, drho;         // grids: z_j = z0 + j dz, rho_j = rho0 + j drho
    int has_mask;
    int m_roots;  // smoothness = 2^m_roots: the root is m_roots square roots; -1 otherwise
    int nz, nr, Pz, Mz, npz, Cr, Mr, nrpad, lanes, n_groups;
    int N, store_every, n_basis;
    int step;   // steps already advanced; read by the z-sweep and the host, written by the rho-sweep
    int rstep;  // the step under way: written by the z-sweep, read by the rho-sweep
    int obs;    // time index whose observation partials are in `part`, or -1
    int active;
    int phase;  // 1: g is the reference g after `step` steps; 0: the explicit rho half of step `step` is applied
    int hold;   // 1: end every step at an exact state (phase 1)
    int flags;  // health flags (norm_health), device-updated at data times
};

// 1 / sqrt(x): the hardware estimate y refined by the series
// x^(-1/2) = y (1 - e)^(-1/2) = y (1 + e/2 + 3 e^2 / 8 + ...), e = 1 - x y^2,
// to third order (5 operations instead of 8 for two Newton steps; the
// truncation error ~e^3 is far below the final rounding).
__device__ __forceinline__ double cyl_rsqrt(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y), y, 1.0);
    return fma(y, e * fma(e, 0.375, 0.5), y);
}

// Half the Coulomb potential plus half the interaction at (z, rho):
// internal_hamiltonian adds V / 2, total_hamiltonian adds (-z q E) / 2.
__device__ __forceinline__ double cyl_half_potential(const CylSim& S, double z, double rho, double E) {
    return 0.5 * (S.kc * cyl_rsqrt(z * z + rho * rho)) + 0.5 * (-z * S.q * E);
}

// Device order of a cylindrical g (and of its basis states): rho rows in pairs
// (2 q, 2 q + 1) interleaved position by position, element (r, p) at
// ((r / 2) npz + p) 2 + r % 2 (nrpad is even). The z-sweep's threads then read
// whole lines in pairs and the rho-sweep's four positions whole 128 B lines.
__device__ __forceinline__ size_t cyl_at(int r, int p, int npz) {
    return ((size_t)(r >> 1) * npz + p) * 2 + (r & 1);
}

// RadialCosineMask.__call__ (potentials/masks.py:76-89) at r.
__device__ __forceinline__ double cyl_mask_r(const CylSim& S, double r) {
    if (r < S.m_inner) return 1.0;
    if (r >= S.m_outer) return 0.0;
    double sn, cs;
    tdse_sincos(0.5 * 3.141592653589793 * (r - S.m_inner) / fabs(S.m_outer - S.m_inner), &sn, &cs);
    // |cos|^(1/s): for the usual s = 2^k (default 8) k square roots, a few
    // times cheaper than pow (1.49 -> 1.45 ms per cylinder step)
    if (S.m_roots >= 0) {
        double c = fabs(cs);
        for (int i = 0; i < S.m_roots; ++i) c = sqrt(c);
        return c;
    }
    return pow(fabs(cs), S.m_inv_s);
}

// Job table entry (sim, b): b == -1 reduces the rho-sweep partials of a data time to the norm, b >= 0
// to the inner product with test state b. One wave per job, sums in a fixed order. The partials of a
// step are reduced by job waves in the leading workgroups of the next step's z-sweep launch (CylJobs), or
// after the run's last step by a launch of their own. Job -3 rides with both sweeps and counts: the
// z-sweep reads S.step, its job copies it to S.rstep; the rho-sweep reads S.rstep, its job sets S.step
// for the next z-sweep. The two launches per step that this replaces took 8 us of the 23 us step of one
// 250 x 100 mesh.
struct CylJobs {
    CylSim* sims;  // as ShObs
    const int2* jobs;
    int n_jobs;
    int blocks;  // leading workgroups of the launch that take jobs, blockDim.x / 64 each
};

__device__ __forceinline__ void cyl_observe_job(CylSim& S, const int b, const int n, const int lane) {
    const int slot = sh_data_slot(n, S.N, S.store_every);
    const int stride = 1 + 2 * S.n_basis;
    const int off = b < 0 ? 0 : 1 + 2 * b;
    const double* __restrict__ part = S.part;
    const int n_groups = S.n_groups;
    double re = 0.0, im = 0.0;
#pragma unroll 4
    for (int g = lane; g < n_groups; g += TDSE_WAVE) {
        re += ld1(part, (size_t)g * stride + off);
        if (b >= 0) im += ld1(part, (size_t)g * stride + off + 1);
    }
    re = wave_sum_last(re);
    im = wave_sum_last(im);
    if (lane != TDSE_WAVE - 1) return;
    if (b < 0) {
        const double nrm = re * S.delta;
        const int health = norm_health(S.out_norm, slot, nrm);
        S.out_norm[slot] = nrm;
        if (health) S.flags |= health;
    } else {
        S.out_ip[(size_t)slot * S.n_basis + b] = cmk(re * S.delta, im * S.delta);
    }
}

// Time index observed by the step that ends at n + 1 (MAIN) or by the pre-sweep (n = 0), or -1.
__device__ __forceinline__ int cyl_observed(const CylSim& S, int n) {
    return sh_is_data_step(n, S.N, S.store_every) ? n : -1;
}

// AFTER_RHO false: with the z-sweep, or after the last step. A simulation's pending partials are those of
// the g it now holds: reduced once per data time (again with the same result if it stays at that step).
template <bool AFTER_RHO>
__device__ __forceinline__ void cyl_job_block(const CylJobs& jobs) {
    const int job = blockIdx.x * (blockDim.x / TDSE_WAVE) + threadIdx.x / TDSE_WAVE;
    if (job >= jobs.n_jobs) return;
    const int2 jb = jobs.jobs[job];
    CylSim& S = jobs.sims[jb.x];
    const int lane = threadIdx.x % TDSE_WAVE;
    if (!S.active) return;
    if (AFTER_RHO) {
        const int n = S.rstep;
        if (jb.y != -3 || lane != 0 || n >= S.N) return;
        S.obs = cyl_observed(S, n + 1);
        S.phase = (n + 1 < S.N && !S.hold) ? 0 : 1;  // whether g is exact
        S.step = n + 1;
    } else {
        const int n = S.step;
        if (jb.y == -3) {
            if (lane == 0) S.rstep = n;
        } else if (S.obs == n) {
            cyl_observe_job(S, jb.y, n, lane);
        }
    }
}

__global__ void __launch_bounds__(256) k_cyl_observe(CylJobs jobs) { cyl_job_block<false>(jobs); }

// ------------------------------------------------------------------ z-sweep
//
// One workgroup of 2 Pz threads per (simulation, pair of rho-lines 2 q, 2 q + 1);
// Mz rows per thread. Thread t works on line ln = t & 1 and chunk k = t >> 1:
// the two lines of a pair are interleaved in memory (cyl_at), so neighbouring
// threads read neighbouring 16 B and a wave reads 1 KiB contiguous.
// (1 + i tau H_z) y = (1 - i tau H_z) x with H_z tridiagonal: diagonal
// -2 zp + V/2 - z q E / 2, off-diagonals zp inside the line
// (mesh_operators.py:561-575); the launch uses the explicit form. A pair may end in a
// padding line (r = nr for odd nr): it holds zeros and stays zero.
template <int M, int MAXT, int WPE, int FORM>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(WPE, 8)))
k_cyl_z(CylSim* __restrict__ sims, const int2* __restrict__ pairs, int n_pairs, CylJobs jobs) {
    extern __shared__ double2 lds[];  // 3 * Pz * 2 + kRedScratch
    if ((int)blockIdx.x < jobs.blocks) {
        cyl_job_block<false>(jobs);
        return;
    }
    const int job = blockIdx.x - jobs.blocks;
    if (job >= n_pairs) return;
    const int2 lt = pairs[job];
    CylSim& S = sims[lt.x];
    const int n = S.step;
    if (!S.active || n >= S.N) return;  // uniform across the block
    const int P = S.Pz, nz = S.nz;
    const int ln = threadIdx.x & 1, k = threadIdx.x >> 1;
    const double tau = ld1(S.ts, n);
    const double E = ld1(S.fs, n);
    const double rho = fma((double)(2 * lt.y + ln), S.drho, S.rho0);
    const double tzp = tau * S.zp;
    const double tdiag = tau * (S.zp * -2.0);
    double2* __restrict__ gl = S.g + cyl_at(2 * lt.y + ln, k, S.npz);
    const double z0 = S.z0, dz = S.dz;

    double2 x[M];
#pragma unroll
    for (int i = 0; i < M; ++i) x[i] = ld2(gl, (size_t)i * P * 2);
    // coefficients from the grid, no table reads
    auto off = [&](int) { return tzp; };
    auto coef = [&](int i, double& h, double& o) {
        const double z = fma((double)(k * M + i), dz, z0);
        h = fma(tau, cyl_half_potential(S, z, rho, E), tdiag);
        o = tzp;
    };
    const int rows = nz - k * M;  // of this chunk that are no padding
    auto live = [&](int i) { return i < rows; };
    auto solve = [&](auto expl, const double2 xl, const double2 xr) {
        cn_symmetric<M, decltype(expl)::value, 2>(x, k, P, k > 0 ? tzp : 0.0, coef, off, lds, xl, xr, ln, live);
    };
    cn_line_finish<M, FORM, 2>(x, gl, k, P, lds, solve, ln, 2 * P, true);
}

// ---------------------------------------------------------------- rho-sweep
//
// One workgroup of LANES * Cr threads per (simulation, group of LANES
// consecutive positions): thread t works on line ln = t % LANES (position
// p = LANES * group + ln) and chunk c = t / LANES (rho rows c Mr .. c Mr + Mr - 1).
// H_rho: diagonal -2 rp + V/2 - z q E / 2, off-diagonals rp c(j + 1), c(m) = m / sqrt(m^2 - 1/4)
// (mesh_operators.py:578-600).
//
// What bounds it: FP64 issue at 4 waves per SIMD (128 VGPRs). The couplings come from the simulation's table,
// staged in LDS once per workgroup: formed from m each time, they were a reciprocal square root three times per row
// and kept registers busy over the solve. With half the potential in LDS too, the
// explicit half gained nothing (139.6 us against 140.1 per step of four 2000 x 1000 simulations), so it is formed
// again. A wave whose points all lie inside the mask's ramp skips it. Padding rows hold zeros, so nothing selects on
// them. Per step, before and after (with cn_symmetric): one 250 x 100 simulation 18.4 -> 16.0 us, four of 2000 x 1000
// 151 -> 133, 32 of them 1070 -> 942.
//
// MAIN (every step n < N):  implicit half of step n, mask, observables of the
//     exact g after n + 1 steps at data times, explicit half of step n + 1
//     unless n + 1 == N or the simulation holds exact states.
// PRE (phase 1 only): observables of g at step 0, explicit half of step n.
enum { CYL_PRE = 0, CYL_MAIN = 1 };

// LDS of the rho-sweep: the solver's rows, the couplings, reduction scratch.
constexpr size_t cyl_rho_lds_bytes(int M, int LANES, int P) {
    return ((size_t)3 * P * LANES + kRedScratch) * sizeof(double2) +
           ((size_t)M * P + 16) * sizeof(double);
}

template <int LANES>
__device__ __forceinline__ double cyl_block_sum(double v, double* red, int t, int nthreads) {
    v = wave_sum(v);
    __syncthreads();
    if ((t & (TDSE_WAVE - 1)) == 0) red[t / TDSE_WAVE] = v;
    __syncthreads();
    double s = 0.0;
    const int nw = (nthreads + TDSE_WAVE - 1) / TDSE_WAVE;
    for (int w = 0; w < nw; ++w) s += red[w];  // fixed order
    return s;
}

template <int M, int LANES, int MODE, int MAXT, int WPE>
__global__ void __launch_bounds__(MAXT) __attribute__((amdgpu_waves_per_eu(WPE, 8))) k_cyl_rho(CylSim* __restrict__ sims, const int2* __restrict__ groups,
                                                  int n_groups, CylJobs jobs) {
    extern __shared__ double2 lds[];  // cyl_rho_lds_bytes(M, LANES, Cr)
    if ((int)blockIdx.x < jobs.blocks) {
        if (MODE == CYL_MAIN) cyl_job_block<true>(jobs);
        return;
    }
    // neighbouring position groups share 128 B lines: keep them on one XCD
    const int2 gt = groups[xcd_remap(blockIdx.x - jobs.blocks, n_groups)];
    CylSim& S = sims[gt.x];
    const int n = (MODE == CYL_PRE) ? S.step : S.rstep;
    if (!S.active || n >= S.N) return;
    if (MODE == CYL_PRE && S.phase != 1) return;
    const int t = threadIdx.x;
    const int ln = t % LANES, c = t / LANES;
    const int P = S.Cr, npz = S.npz;
    const int p = gt.y * LANES + ln;
    double z = ld1(S.zt, p);
    // rows c M .. c M + M - 1 (M even): row c M + i at gl[cyl_at(i, 0, npz)]; with the two
    // rows of a pair adjacent, LANES = 4 neighbouring positions read whole 128 B lines
    double2* __restrict__ gl = S.g + cyl_at(c * M, p, npz);
    double* const off = reinterpret_cast<double*>(lds + 3 * P * LANES + kRedScratch);  // [M][P]
    double* const red = off + M * P;

    double2 x[M];
#pragma unroll
    for (int i = 0; i < M; ++i) x[i] = ld2(gl, cyl_at(i, 0, npz));
    for (int i = t; i < M * P; i += P * LANES) off[i] = ld1(S.roff, i);
    __syncthreads();

    const double hk = 0.5 * S.kc, drho = S.drho, rp = S.rp;
    double rho_c = fma((double)(c * M), drho, S.rho0);  // of row c M
    auto radius2 = [&](int i) {
        const double rho = fma((double)i, drho, rho_c);
        return fma(rho, rho, z * z);
    };
    const double left = c > 0 ? off[(M - 1) * P + c - 1] : 0.0;  // off_{c M - 1}

    if constexpr (MODE == CYL_MAIN) {
        const double tau = ld1(S.ts, n), w = 0.5 * (-z * S.q * ld1(S.fs, n)), kin = tau * (rp * -2.0);
        auto off_at = [&](int i) {
            int c2 = c;
            asm volatile("" : "+v"(c2));  // the table is read again, its rows are not kept over the solve
            return tau * off[i * P + c2];
        };
        auto coef = [&](int i, double& h, double& o) {
            h = fma(tau, fma(hk, cyl_rsqrt(radius2(i)), w), kin);
            o = tau * off[i * P + c];
        };
        cn_symmetric<M, false, LANES>(x, c, P, tau * left, coef, off_at, lds, cmk(0.0, 0.0), cmk(0.0, 0.0), ln);
        asm volatile("" : "+v"(rho_c), "+v"(z), "+v"(gl));  // radii and addresses are formed again, not kept over the solve
        if (S.has_mask) {
            // rows lie at growing radius: inside the inner radius (most points) the mask is 1, from the outer on 0
            const double in2 = S.m_inner * S.m_inner, out2 = S.m_outer * S.m_outer;
            if (!__all(radius2(M - 1) < in2)) {
#pragma unroll
                for (int i = 0; i < M; ++i) {
                    const double r2 = radius2(i);
                    double mk = r2 < in2 ? 1.0 : 0.0;
                    if (r2 >= in2 && r2 < out2) mk = cyl_mask_r(S, sqrt(r2));
                    x[i] = cscale(mk, x[i]);
                }
            }
        }
    }

    // observables of the exact g after n + 1 (MAIN) or 0 (PRE) steps
    const int obs = (MODE == CYL_MAIN) ? n + 1 : 0;
    if (MODE == CYL_PRE && n == 0 && gt.y == 0 && t == 0) jobs.sims[gt.x].obs = cyl_observed(S, 0);
    const bool observe = (MODE == CYL_MAIN || n == 0) && sh_is_data_step(obs, S.N, S.store_every);
    if (observe) {
        const int nb = S.n_basis;
        double* part = S.part + (size_t)gt.y * (1 + 2 * nb);
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < M; ++i) acc += cabs2(x[i]);
        const double tot = cyl_block_sum<LANES>(acc, red, t, blockDim.x);
        if (t == 0) part[0] = tot;
        for (int b = 0; b < nb; ++b) {
            const double2* phi = S.basis + (size_t)b * S.nrpad * npz + cyl_at(c * M, p, npz);
            double re = 0.0, im = 0.0;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                const double2 f = ld2(phi, cyl_at(i, 0, npz));  // conj(f) x
                re += fma(f.x, x[i].x, f.y * x[i].y);
                im += fma(f.x, x[i].y, -f.y * x[i].x);
            }
            const double sre = cyl_block_sum<LANES>(re, red, t, blockDim.x);
            const double sim = cyl_block_sum<LANES>(im, red, t, blockDim.x);
            if (t == 0) {
                part[1 + 2 * b] = sre;
                part[2 + 2 * b] = sim;
            }
        }
    }

    // explicit half of the next step (MAIN) or of step n (PRE)
    const int ne = (MODE == CYL_MAIN) ? n + 1 : n;
    const bool expl = (MODE == CYL_PRE) || (ne < S.N && !S.hold);
    if (expl) {
        const double tau = ld1(S.ts, ne), w = 0.5 * (-z * S.q * ld1(S.fs, ne)), kin = tau * (rp * -2.0);
        double2 xl, xr;
        chunk_neighbours<M, LANES>(x, c, P, lds, xl, xr, true, ln);
        double2 prev = xl;
        int c1 = c;
        asm volatile("" : "+v"(c1));  // as above
        double carry = c1 > 0 ? off[(M - 1) * P + c1 - 1] : 0.0;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const double v = fma(hk, cyl_rsqrt(radius2(i)), w);
            const double o = off[i * P + c1];
            const double h = fma(tau, v, kin), hm = tau * carry, hp = tau * o;
            carry = o;
            const double2 xp = (i + 1 < M) ? x[i + 1 < M ? i + 1 : i] : xr;
            const double2 hx = cmk(fma(hm, prev.x, fma(h, x[i].x, hp * xp.x)), fma(hm, prev.y, fma(h, x[i].y, hp * xp.y)));
            prev = x[i];
            x[i] = cmk(x[i].x + hx.y, x[i].y - hx.x);  // x - i hx
        }
    }
#pragma unroll
    for (int i = 0; i < M; ++i) st2(gl, cyl_at(i, 0, npz), x[i]);
}
