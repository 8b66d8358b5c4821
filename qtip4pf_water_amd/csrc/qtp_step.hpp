// qtp_step.hpp -- Suzuki-Chin combination, propagation and thermostat, neighbour
// lists, classical step, observables.
#pragma once
#include "qtp_pair.hpp"

namespace qtp {
// ---------------------------------------------------------------------------
// Suzuki-Chin combination (forces.cpp:698-789)
// ---------------------------------------------------------------------------
struct SCArgs {
    int P, n_atoms, NAP;
    double omega_psq, epsilonsc, halfdt;
};

// After the physical-force phase.  grid: P, 256 threads.
//  even b: F_sc = 2 f / 3; tot_b = 2V; vop_b = V
//  odd  b: tot_b = 4V, fsq_b = sum f^2/m / (3 w^2); delta and the displaced
//          positions q +- eps f/m for the finite-difference phase.
// Suzuki-Chin combination, first half (forces.cpp:738-775), one 1024-thread
// block per bead: bead energy; even beads F_sc = 2f/3; odd beads |f|^2_M,
// the finite-difference step eps / sqrt(sum (f/m)^2 / (n_atoms P)) and the
// displaced positions q +- step f/m of the second force phase.
constexpr int SC_THREADS = 1024;
// f2 (may be null): the second half of split k-space forces, added into fph
// first (the sum stays in fph for the later kernels).
__global__ __launch_bounds__(SC_THREADS) void k_sc1(SCArgs a, const double *__restrict__ q,
                                                    double *__restrict__ fph,
                                                    const double *__restrict__ f2,
                                                    const double *__restrict__ epart, int ep_stride,
                                                    int ep_n, double eself,
                                                    double *__restrict__ Vout,
                                                    const double *__restrict__ m_atom,
                                                    double *__restrict__ Fsc,
                                                    double *__restrict__ qpm,
                                                    double *__restrict__ scal /*[P][4]*/)
{
    __shared__ double sh[16];
    __shared__ double s_scale;
    __shared__ double s_V;
    const int b = blockIdx.x;
    const long o = (long)b * 3 * a.NAP;
    if (f2) {
        for (int t = threadIdx.x; t < 3 * a.NAP; t += SC_THREADS) fph[o + t] += f2[o + t];
        __syncthreads();
    }
    // this thread's dofs t = threadIdx.x + SC_THREADS r: forces, masses and
    // positions loaded once, before the energy sum (one memory latency)
    constexpr int SC_RUN = 4;
    const int nt = 3 * a.NAP;
    const bool odd = b & 1;
    double fv[SC_RUN], mv[SC_RUN], qv[SC_RUN];
    const bool fits = nt <= SC_RUN * SC_THREADS;
    if (fits) {
#pragma unroll
        for (int r = 0; r < SC_RUN; ++r) {
            const int t = threadIdx.x + r * SC_THREADS;
            if (t < nt) {
                fv[r] = fph[o + t];
                if (odd) {
                    mv[r] = m_atom[t % a.NAP];
                    qv[r] = q[o + t];
                }
            }
        }
    }
    if (threadIdx.x < 64) {
        const double v = eval_energy(epart, b, ep_stride, ep_n, eself);
        if (threadIdx.x == 0) {
            s_V = v;
            Vout[b] = v;
        }
    }
    if (!odd) {
        if (fits) {
#pragma unroll
            for (int r = 0; r < SC_RUN; ++r) {
                const int t = threadIdx.x + r * SC_THREADS;
                if (t < nt) Fsc[o + t] = 2.0 * fv[r] / 3.0;
            }
        } else {
            // larger beads: the same dofs in runs of SC_RUN, each run's loads
            // issued together
            for (int t0 = threadIdx.x; t0 < nt; t0 += SC_RUN * SC_THREADS) {
                double fb[SC_RUN];
#pragma unroll
                for (int r = 0; r < SC_RUN; ++r) {
                    const int t = t0 + r * SC_THREADS;
                    if (t < nt) fb[r] = fph[o + t];
                }
#pragma unroll
                for (int r = 0; r < SC_RUN; ++r) {
                    const int t = t0 + r * SC_THREADS;
                    if (t < nt) Fsc[o + t] = 2.0 * fb[r] / 3.0;
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            const double V = s_V;
            scal[b * 4 + 0] = 2.0 * V;
            scal[b * 4 + 1] = V;
            scal[b * 4 + 2] = 0.0;
            scal[b * 4 + 3] = 0.0;
        }
        return;
    }
    // |f|^2 / m and (f / m)^2 over the real atoms: per thread in dof order,
    // then the block sum
    double fsq = 0.0, del = 0.0;
    if (fits) {
#pragma unroll
        for (int r = 0; r < SC_RUN; ++r) {
            const int t = threadIdx.x + r * SC_THREADS;
            if (t < nt && t % a.NAP < a.n_atoms) {
                const double f = fv[r], m = mv[r];
                fsq += f * f / m;
                const double fm = f / m;
                del += fm * fm;
            }
        }
    } else {
        // runs of SC_RUN dofs, loads first, sums in the same dof order
        for (int t0 = threadIdx.x; t0 < nt; t0 += SC_RUN * SC_THREADS) {
            double fb[SC_RUN], mb[SC_RUN];
#pragma unroll
            for (int r = 0; r < SC_RUN; ++r) {
                const int t = t0 + r * SC_THREADS;
                if (t < nt) {
                    fb[r] = fph[o + t];
                    mb[r] = m_atom[t % a.NAP];
                }
            }
#pragma unroll
            for (int r = 0; r < SC_RUN; ++r) {
                const int t = t0 + r * SC_THREADS;
                if (t < nt && t % a.NAP < a.n_atoms) {
                    const double f = fb[r], m = mb[r];
                    fsq += f * f / m;
                    const double fm = f / m;
                    del += fm * fm;
                }
            }
        }
    }
    fsq = block_sum(fsq, sh);
    del = block_sum(del, sh);
    if (threadIdx.x == 0) {
        const double V = s_V;
        fsq /= 3.0 * a.omega_psq;
        del /= (double)(a.n_atoms * a.P);
        del = 1.0 / sqrt(del);
        const double sc_scale = a.epsilonsc * del;
        scal[b * 4 + 0] = 4.0 * V;
        scal[b * 4 + 1] = 0.0;
        scal[b * 4 + 2] = fsq;
        scal[b * 4 + 3] = 1.0 / (9.0 * a.omega_psq * sc_scale);
        s_scale = sc_scale;
    }
    __syncthreads();
    const double sc_scale = s_scale;
    const int k = b >> 1;
    double *Pp = qpm + (long)(2 * k) * 3 * a.NAP;
    double *Pm = qpm + (long)(2 * k + 1) * 3 * a.NAP;
    if (fits) {
#pragma unroll
        for (int r = 0; r < SC_RUN; ++r) {
            const int t = threadIdx.x + r * SC_THREADS;
            if (t < nt) {
                const double dq = sc_scale * fv[r] / mv[r];
                Pp[t] = qv[r] + dq;
                Pm[t] = qv[r] - dq;
            }
        }
    } else {
        for (int t0 = threadIdx.x; t0 < nt; t0 += SC_RUN * SC_THREADS) {
            double fb[SC_RUN], mb[SC_RUN], qb[SC_RUN];
#pragma unroll
            for (int r = 0; r < SC_RUN; ++r) {
                const int t = t0 + r * SC_THREADS;
                if (t < nt) {
                    fb[r] = fph[o + t];
                    mb[r] = m_atom[t % a.NAP];
                    qb[r] = q[o + t];
                }
            }
#pragma unroll
            for (int r = 0; r < SC_RUN; ++r) {
                const int t = t0 + r * SC_THREADS;
                if (t < nt) {
                    const double dq = sc_scale * fb[r] / mb[r];
                    Pp[t] = qb[r] + dq;
                    Pm[t] = qb[r] - dq;
                }
            }
        }
    }
}
// Second half (forces.cpp:776-789): odd beads F_sc = 4f/3 - (f+ - f-) / (9 w^2
// step); the half-step kick p += dt/2 F_sc when requested; an extra last
// block sums the SC potential and sc_pot in bead order (beside the others).
// grid: P * nch + 1, SC_THREADS threads: nch blocks per bead, each taking
// every nch-th run of SC_THREADS dofs (nch > 1 for large systems).
// f2 (may be null): the second half of the split k-space forces of the
// phase-2 evaluations, added to fpm here.
__global__ __launch_bounds__(SC_THREADS) void k_sc2(SCArgs a, const double *__restrict__ fph,
                                                    const double *__restrict__ fpm,
                                                    const double *__restrict__ f2,
                                                    const double *__restrict__ scal,
                                                    double *__restrict__ Fsc, double *__restrict__ p,
                                                    int kick, double *__restrict__ out,
                                                    unsigned long long *__restrict__ step_ctr,
                                                    int nch)
{
    const int b = blockIdx.x / nch, c = blockIdx.x - b * nch;
    const long o = (long)b * 3 * a.NAP;
    const int t0 = c * SC_THREADS + threadIdx.x, dt = nch * SC_THREADS;
    if (b == a.P) {
        if (threadIdx.x == 0) {
            double tot = 0.0, vop = 0.0;
            for (int bb = 0; bb < a.P; ++bb) {
                if ((bb & 1) == 0) {
                    tot += scal[bb * 4 + 0];
                    vop += scal[bb * 4 + 1];
                } else {
                    tot += scal[bb * 4 + 0];
                    tot += scal[bb * 4 + 2];
                }
            }
            tot /= 3.0;
            out[0] = tot;
            out[1] = 2.0 * vop / a.P;
            if (step_ctr) step_ctr[0] += 1ull;
        }
        return;
    }
    // runs of four dofs per thread: the loads of a run are issued together
    const int nt = 3 * a.NAP;
    if (b & 1) {
        const int k = b >> 1;
        const double fscale = scal[b * 4 + 3];
        const long op = (long)(2 * k) * 3 * a.NAP, om = (long)(2 * k + 1) * 3 * a.NAP;
        for (int tr = t0; tr < nt; tr += 4 * dt) {
            double F[4], pv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = tr + r * dt;
                if (t < nt) {
                    F[r] = 4.0 * fph[o + t] / 3.0;
                    const double fp = f2 ? fpm[op + t] + f2[op + t] : fpm[op + t];
                    const double fm = f2 ? fpm[om + t] + f2[om + t] : fpm[om + t];
                    F[r] -= fscale * (fp - fm);
                    if (kick) pv[r] = p[o + t];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = tr + r * dt;
                if (t < nt) {
                    Fsc[o + t] = F[r];
                    if (kick) p[o + t] = pv[r] + a.halfdt * F[r];
                }
            }
        }
    } else if (kick) {
        for (int tr = t0; tr < nt; tr += 4 * dt) {
            double F[4], pv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = tr + r * dt;
                if (t < nt) {
                    F[r] = Fsc[o + t];
                    pv[r] = p[o + t];
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = tr + r * dt;
                if (t < nt) p[o + t] = pv[r] + a.halfdt * F[r];
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Ring-polymer propagation (update.cpp:281-352), PILE-G (thermostat.cpp:64-133)
// ---------------------------------------------------------------------------
struct PropArgs {
    int P, n_atoms, NAP, ntile;
    double halfdt, dt, beta_n;
    int nvt, host_dev, n_dof;  // host_dev: deviates from the host buffer
    uint64_t seed;
    // centroid: cmode 0 free (PIMD / PA-CMD), 2 held fixed (its momentum is
    // zeroed after the kick, no thermostat); cthermo 0 = PILE-G, the Bussi
    // rescale with c = exp(-dt/tau) (c = 0: thermostat.cpp:88-111), 1 =
    // PILE-L, Langevin c1_0 = exp(-dt/tau), c2_0 = sqrt(1 - c1_0^2)
    int cmode, cthermo;
    double cbussi, c1_0, c2_0;
};

// Per-mode constants: mode[k] = {scale_k, wsq_k, c1_k, c2_k}
// (update.cpp:302-304, thermostat.cpp:119-121)

// sqrt-Cayley half step of one normal mode (update.cpp:307-317)
__device__ __forceinline__ void cayley_half(double &uq, double &up, double m, double halfdt,
                                            double4 md)
{
    double temp = halfdt * up / m + uq;
    temp *= md.x;
    up = up - halfdt * md.y * uq * m;
    up *= md.x;
    uq = temp;
}

// The heat of a step is summed over groups of HP_DOFS dofs, HP_PARTS of them
// in a 64-dof tile: per mode over the group (heat_group), then over the modes
// (k_prop_dofs in LDS, k_prop_inv from k_prop_fwd's sums), in the same order in
// both forms of the propagation.  hpart[tile * HP_PARTS + group] is that sum;
// behind these, at [(tile * HP_PARTS + group) * P + k], are the sums per mode of
// the two-launch form.  A partial per mode and group left k_heat's one block
// 73 728 to read at 4096 x 32, 22.5 us; these 2304 take 5.2, and the propagation
// as long as before.
constexpr int HP_DOFS = 16, HP_PARTS = 64 / HP_DOFS;
__host__ __device__ inline size_t heat_doubles(int P, int ntile)
{
    return (size_t)(P + 1) * ntile * HP_PARTS;
}
__device__ __forceinline__ double heat_group(double h)
{
    for (int o = HP_DOFS / 2; o > 0; o >>= 1) h += __shfl_xor(h, o, 64);
    return h;
}
__device__ __forceinline__ void heat_part(double h, double *hpart, int k, int P, int tile, int ntile)
{
    const int lane = threadIdx.x & 63;
    h = heat_group(h);
    if (lane % HP_DOFS == 0)
        hpart[(long)ntile * HP_PARTS + ((long)tile * HP_PARTS + lane / HP_DOFS) * P + k] = h;
}
// A lane's share of the sum over the modes, by the HP_DOFS lanes of a group:
// lane i the modes k = i mod HP_DOFS (then heat_group).
__device__ __forceinline__ double heat_modes(int i, int P, const double *h)
{
    double s = 0.0;
    for (int k = i; k < P; k += HP_DOFS) s += h[k];
    return s;
}

// Kick, forward normal-mode transform and first half step for mode k of 64
// planar dofs; modes k >= 1 also get their Langevin step and second half
// step here (they do not wait for the centroid).  One wavefront per
// (dof tile, mode); the transform rows are wave-uniform (scalar loads).
// grid: ntile * P (tile-major, XCD-remapped), 64 threads.
// part[tile] = centroid KE after the first half step (tile partial);
// part[ntile + tile] = chi-square partial (device random numbers);
// hpart: KE before - KE after of mode k's Langevin step, per mode (heat_part).
__global__ __launch_bounds__(64) void k_prop_fwd(PropArgs A, const double *__restrict__ Cm,
                                                 const double4 *__restrict__ mode,
                                                 const double2 *__restrict__ mscale,
                                                 const double *__restrict__ q,
                                                 const double *__restrict__ p,
                                                 const double *__restrict__ F,
                                                 const double *__restrict__ m_atom,
                                                 const double *__restrict__ sqm_atom,
                                                 const double *__restrict__ dev,
                                                 double *__restrict__ nq, double *__restrict__ np,
                                                 double *__restrict__ part,
                                                 double *__restrict__ hpart,
                                                 const unsigned long long *__restrict__ step_ctr)
{
    const int P = A.P, lb = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = lb / P, k = lb - tile * P, lane = threadIdx.x;
    const long N3 = 3L * A.NAP;
    const int f = tile * 64 + lane;
    const int at = f % A.NAP, d = f / A.NAP;
    const bool va = at < A.n_atoms;
    // propagation mass of mode k: the physical mass, times (w_k / W)^2 for
    // the non-centroid modes of partially adiabatic CMD
    const double m = va ? m_atom[at] * mscale[k].x : 1.0;
    const double *cr = Cm + (long)k * P;
    double uq = 0.0, up = 0.0;
#pragma unroll 8
    for (int b = 0; b < P; ++b) {
        const double c = cr[b];
        const long idx = b * N3 + f;
        const double pk = p[idx] + A.halfdt * F[idx];  // update.cpp:281-287
        uq = fma(c, q[idx], uq);
        up = fma(c, pk, up);
    }
    const double4 md = mode[k];
    if (k == 0) {
        if (A.cmode == 2) up = 0.0;   // centroid held fixed
        cayley_half(uq, up, m, A.halfdt, md);
        const bool pile_g = A.nvt && A.cthermo == 0 && A.cmode != 2;
        double ke0 = (va && pile_g) ? 0.5 * up * up / m : 0.0;
        double chi = 0.0, h = 0.0;
        if (pile_g && !A.host_dev && va) {
            const int ridx = 3 * at + d;
            if (ridx >= 1) {
                const double z = philox_normal(A.seed, *step_ctr, (uint32_t)(P + 1), (uint32_t)ridx);
                chi = z * z;
            }
        }
        if (A.nvt && A.cthermo == 1 && A.cmode != 2 && va) {
            // PILE-L: Langevin on the centroid (random stream 0)
            h = 0.5 * up * up / m;
            const double xi = philox_normal(A.seed, *step_ctr, 0u, (uint32_t)(3 * at + d));
            up = A.c1_0 * up + sqm_atom[at] * A.c2_0 * xi;
            h -= 0.5 * up * up / m;
        }
        nq[f] = uq;
        np[f] = up;
        ke0 = wave_sum(ke0);
        chi = wave_sum(chi);
        if (lane == 0) {
            part[tile] = ke0;
            part[A.ntile + tile] = chi;
        }
        // the centroid's heat: PILE-L's here, PILE-G's in k_prop_inv
        if (A.nvt && !pile_g) heat_part(h, hpart, 0, P, tile, A.ntile);
        return;
    }
    cayley_half(uq, up, m, A.halfdt, md);
    if (A.nvt) {
        double h = 0.0;
        if (va) {
            h += 0.5 * up * up / m;
            const int ridx = 3 * at + d;
            const double xi = A.host_dev ? dev[3 + (long)(k - 1) * A.n_dof + ridx]
                                         : philox_normal(A.seed, *step_ctr, (uint32_t)k, (uint32_t)ridx);
            up = md.z * up + sqm_atom[at] * md.w * xi;
            h -= 0.5 * up * up / m;
        }
        heat_part(h, hpart, k, P, tile, A.ntile);
    }
    cayley_half(uq, up, m, A.halfdt, md);
    nq[k * N3 + f] = uq;
    np[k * N3 + f] = up;
}

// Centroid rescale (Bussi, tau -> 0), its second half step, inverse
// transform to bead b and displacement tracking.  One wavefront per
// (dof tile, bead).   grid: ntile * P (tile-major, XCD-remapped), 64 threads.
// The bead-0 waves sum the tile's heat over the modes; with the rescale the
// centroid's is - KE after it.
__global__ __launch_bounds__(64) void k_prop_inv(PropArgs A, const double *__restrict__ Cm,
                                                 const double4 *__restrict__ mode,
                                                 const double *__restrict__ nq,
                                                 const double *__restrict__ np,
                                                 const double *__restrict__ m_atom,
                                                 const double *__restrict__ part,
                                                 const double *__restrict__ dev,
                                                 double *__restrict__ q, double *__restrict__ p,
                                                 double *__restrict__ disp, int NMP,
                                                 double *__restrict__ hpart,
                                                 const unsigned long long *__restrict__ step_ctr)
{
    const int P = A.P, lb = xcd_remap(blockIdx.x, gridDim.x);
    const int tile = lb / P, b = lb - tile * P, lane = threadIdx.x;
    const long N3 = 3L * A.NAP;
    const int f = tile * 64 + lane;
    const int at = f % A.NAP, d = f / A.NAP;
    const bool va = at < A.n_atoms;
    const double m = va ? m_atom[at] : 1.0;
    double u0q = nq[f], u0p = np[f];
    const bool pile_g = A.nvt && A.cthermo == 0 && A.cmode != 2;
    // the sums per mode are loaded here and added up behind the stores
    const int i16 = lane % HP_DOFS, group = tile * HP_PARTS + lane / HP_DOFS;
    double h0 = 0.0, hm = 0.0;
    if (A.nvt && b == 0) {
        const double *H = hpart + (long)A.ntile * HP_PARTS + (long)group * P;
        hm = pile_g && i16 == 0 ? heat_modes(HP_DOFS, P, H) : heat_modes(i16, P, H);
    }
    if (pile_g) {
        const double ke = wave_sum_array(part, A.ntile);
        double R, g2;
        if (A.host_dev) {
            R = dev[0];
            g2 = (A.n_dof % 2 == 0) ? 2.0 * dev[2] + dev[1] * dev[1] : 2.0 * dev[2];
        } else {
            g2 = wave_sum_array(part + A.ntile, A.ntile);
            R = philox_normal(A.seed, *step_ctr, (uint32_t)P, 0u);
        }
        double alpha;
        if (A.cbussi == 0.0) {
            alpha = sqrt((R * R + g2) / (2.0 * A.beta_n * ke));   // thermostat.cpp:99-104
        } else {
            // Bussi, Donadio, Parrinello, J. Chem. Phys. 126, 014101 (2007),
            // eq. (A7): relaxation towards the canonical KE with time constant tau
            const double c = A.cbussi, x = 1.0 / (2.0 * A.beta_n * ke);
            alpha = sqrt(c + (1.0 - c) * (R * R + g2) * x + 2.0 * R * sqrt(c * (1.0 - c) * x));
            if (R + sqrt(c / ((1.0 - c) * x)) < 0.0) alpha = -alpha;
        }
        u0p *= alpha;
        if (b == 0) h0 = va ? -0.5 * u0p * u0p / m : 0.0;
    }
    cayley_half(u0q, u0p, m, A.halfdt, mode[0]);
    double xq = Cm[b] * u0q, xp = Cm[b] * u0p;
#pragma unroll 8
    for (int k = 1; k < P; ++k) {
        const double c = Cm[(long)k * P + b];
        xq = fma(c, nq[k * N3 + f], xq);
        xp = fma(c, np[k * N3 + f], xp);
    }
    const long idx = b * N3 + f;
    const double qold = q[idx];
    q[idx] = xq;
    p[idx] = xp;
    if (va && (at % 3) == 0) disp[((long)b * 3 + d) * NMP + at / 3] += xq - qold;
    if (A.nvt && b == 0) {
        const double h = heat_group(pile_g ? h0 + hm : hm);
        if (i16 == 0) hpart[group] = h;
    }
}

// The whole propagation of a step in one launch when the centroid needs no
// global rescale (NVE, PILE-L, or the centroid held fixed): kick, forward
// normal-mode transform, sqrt-Cayley half steps around the Langevin steps of
// every mode, inverse transform, displacement tracking (update.cpp:281-352,
// thermostat.cpp:114-129).  HP_DOFS dofs per block, a thread per (mode, dof),
// then per (bead, dof); the beads' positions and kicked momenta and the matrix
// are staged in LDS, so that HBM is read and written once.  Bound by the chain
// of load, P multiply-adds, random numbers, P multiply-adds and store.  The
// arithmetic and its order are k_prop_fwd's and k_prop_inv's.  us, k_prop_fwd +
// k_prop_inv -> this: 216 x 32 7.7 + 6.9 -> 7.5, 512 x 32 13.4 + 11.1 -> 13.1,
// 990 x 16 8.7 + 8.8 -> 8.4, 4096 x 32 64 + 44 -> 38 (a block of 64 dofs and
// 512 threads, eight modes a thread: 84).  With 64-byte pieces (eight dofs)
// instead of 128 a block would share its cache lines with the next.
// grid: HP_PARTS * ntile (XCD-remapped), HP_DOFS * P threads,
// prop_dofs_lds(P); P <= PD_MAX_BEADS.
constexpr int PD_MAX_BEADS = 64;
inline size_t prop_dofs_lds(int P) { return (size_t)(2 * P * HP_DOFS + P * (P + 1) + P) * sizeof(double); }
__global__ __launch_bounds__(HP_DOFS * PD_MAX_BEADS) void k_prop_dofs(
    PropArgs A, const double *__restrict__ Cm, const double4 *__restrict__ mode,
    const double2 *__restrict__ mscale, double *__restrict__ q, double *__restrict__ p,
    const double *__restrict__ F, const double *__restrict__ m_atom,
    const double *__restrict__ sqm_atom, double *__restrict__ part, double *__restrict__ hpart,
    double *__restrict__ disp, int NMP, const unsigned long long *__restrict__ step_ctr)
{
    extern __shared__ double S[];
    const int P = A.P, CP = P + 1;
    double *SQ = S, *SP = S + P * HP_DOFS, *C = S + 2 * P * HP_DOFS;  // C: [P][P + 1]
    double *H = C + P * CP;                                           // heat per mode
    const int blk = xcd_remap(blockIdx.x, gridDim.x);
    const int tid = threadIdx.x, k = tid / HP_DOFS, i = tid % HP_DOFS;  // mode or bead, dof
    const int tile = blk / HP_PARTS, group = blk % HP_PARTS;
    const long N3 = 3L * A.NAP;
    const int f = blk * HP_DOFS + i;
    const int at = f % A.NAP, d = f / A.NAP;
    const bool va = at < A.n_atoms;
    const long idx = k * N3 + f;
    const double qold = q[idx];
    const double pk = p[idx] + A.halfdt * F[idx];  // update.cpp:281-287
    const double m0 = va ? m_atom[at] : 1.0, sqm = va ? sqm_atom[at] : 0.0;
    const double m = va ? m0 * mscale[k].x : 1.0;
    const double4 md = mode[k];
    for (int t = tid; t < P * P; t += HP_DOFS * P) C[t / P * CP + t % P] = Cm[t];
    SQ[tid] = qold;
    SP[tid] = pk;
    __syncthreads();
    double uq = 0.0, up = 0.0;
#pragma unroll 8
    for (int b = 0; b < P; ++b) {
        const double c = C[k * CP + b];
        uq = fma(c, SQ[b * HP_DOFS + i], uq);
        up = fma(c, SP[b * HP_DOFS + i], up);
    }
    if (k == 0 && A.cmode == 2) up = 0.0;  // centroid held fixed
    cayley_half(uq, up, m, A.halfdt, md);
    if (A.nvt) {
        double h = 0.0;
        if (va && !(k == 0 && (A.cthermo != 1 || A.cmode == 2))) {
            // random stream k; the centroid: PILE-L
            h += 0.5 * up * up / m;
            const double xi = philox_normal(A.seed, *step_ctr, (uint32_t)k, (uint32_t)(3 * at + d));
            up = k == 0 ? A.c1_0 * up + sqm * A.c2_0 * xi : md.z * up + sqm * md.w * xi;
            h -= 0.5 * up * up / m;
        }
        h = heat_group(h);
        if (i == 0) H[k] = h;
    }
    if (tid == 0 && group == 0) {
        part[tile] = 0.0;
        part[A.ntile + tile] = 0.0;
    }
    cayley_half(uq, up, k == 0 ? m0 : m, A.halfdt, md);
    __syncthreads();
    SQ[tid] = uq;
    SP[tid] = up;
    __syncthreads();
    double xq = C[k] * SQ[i], xp = C[k] * SP[i];
#pragma unroll 8
    for (int kk = 1; kk < P; ++kk) {
        const double c = C[kk * CP + k];
        xq = fma(c, SQ[kk * HP_DOFS + i], xq);
        xp = fma(c, SP[kk * HP_DOFS + i], xp);
    }
    q[idx] = xq;
    p[idx] = xp;
    if (va && (at % 3) == 0) disp[((long)k * 3 + d) * NMP + at / 3] += xq - qold;
    if (A.nvt && k == 0) {
        const double h = heat_group(heat_modes(i, P, H));
        if (i == 0) hpart[blk] = h;
    }
}

// The thermostat's heat for one step: pile_g's return value (KE before -
// KE after, thermostat.cpp:86-129); heat_acc -= it (update.cpp:325).
__global__ __launch_bounds__(1024) void k_heat(int ntile, int nh, const double *__restrict__ part,
                                               const double *__restrict__ hpart,
                                               double *__restrict__ heat_acc,
                                               double *__restrict__ heat_step)
{
    __shared__ double sh[16];
    double ke = 0.0, h = 0.0;
    for (int i = threadIdx.x; i < ntile; i += blockDim.x) ke += part[i];
    for (int i = threadIdx.x; i < nh; i += blockDim.x) h += hpart[i];
    ke = block_sum(ke, sh);
    h = block_sum(h, sh);
    if (threadIdx.x == 0) {
        const double ret = ke + h;
        if (heat_step) heat_step[0] = ret;
        if (heat_acc) heat_acc[0] -= ret;
    }
}

// Generic orthonormal transform along the bead axis of a[P][len] (fourier.cpp:12-69).
// grid: ceil(len/64), 256 threads, nm_generic_lds(P) bytes of LDS (the
// block's 64 columns of all P beads; the matrix entries are wave-uniform
// loads from global memory).  fwd: u_k = sum_b C[k][b] x_b, else the transpose.
inline size_t nm_generic_lds(int P) { return (size_t)P * 64 * sizeof(double); }
__global__ __launch_bounds__(256) void k_nm_generic(int P, int len, const double *__restrict__ Cm,
                                                    double *__restrict__ a, int fwd)
{
    extern __shared__ double X[];
    const int lane = threadIdx.x & 63, kg = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    for (int b = kg; b < P; b += 4) X[b * 64 + lane] = c < len ? a[(long)b * len + c] : 0.0;
    __syncthreads();
    for (int k = kg; k < P; k += 4) {
        double u = 0.0;
        for (int b = 0; b < P; ++b) {
            const double cf = fwd ? Cm[k * P + b] : Cm[b * P + k];
            u = fma(cf, X[b * 64 + lane], u);
        }
        if (c < len) a[(long)k * len + c] = u;
    }
}

// PILE-G on normal-mode momenta in planar layout (drop-in pile_g).
// Pass 1: centroid KE partials.  grid: ntile, 256 threads.
__global__ __launch_bounds__(256) void k_pile_a(int n_atoms, int NAP, int ntile,
                                                const double *__restrict__ pnm,
                                                const double *__restrict__ m_atom,
                                                double *__restrict__ part)
{
    __shared__ double sh[16];
    const int f = blockIdx.x * 256 + threadIdx.x;
    double ke = 0.0;
    if (f < 3 * NAP) {
        const int at = f % NAP;
        if (at < n_atoms) ke = 0.5 * pnm[f] * pnm[f] / m_atom[at];
    }
    ke = block_sum(ke, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = ke;
}

// Pass 2: rescale the centroid, Langevin on modes 1..P-1 with host deviates.
// grid: ntile, 256 threads (same tiling as pass 1).
__global__ __launch_bounds__(256) void k_pile_b(int P, int n_atoms, int NAP, int n_dof, int ntile,
                                                double beta_n, const double4 *__restrict__ mode,
                                                const double *__restrict__ m_atom,
                                                const double *__restrict__ sqm_atom,
                                                const double *__restrict__ part,
                                                const double *__restrict__ dev,
                                                double *__restrict__ pnm,
                                                double *__restrict__ hpart)
{
    __shared__ double sh[16];
    __shared__ double s_alpha;
    if (threadIdx.x == 0) {
        double ke = 0.0;
        for (int t = 0; t < ntile; ++t) ke += part[t];
        const double R = dev[0];
        const double g2 = (n_dof % 2 == 0) ? 2.0 * dev[2] + dev[1] * dev[1] : 2.0 * dev[2];
        s_alpha = sqrt((R * R + g2) / (2.0 * beta_n * ke));
    }
    __syncthreads();
    const int f = blockIdx.x * 256 + threadIdx.x;
    double heat = 0.0;
    if (f < 3 * NAP) {
        const int at = f % NAP, d = f / NAP;
        if (at < n_atoms) {
            const double m = m_atom[at], sq = sqm_atom[at];
            const int ridx = 3 * at + d;
            double up = pnm[f] * s_alpha;
            pnm[f] = up;
            heat -= 0.5 * up * up / m;
            for (int k = 1; k < P; ++k) {
                const double4 md = mode[k];
                const long idx = (long)k * 3 * NAP + f;
                double v = pnm[idx];
                heat += 0.5 * v * v / m;
                v = md.z * v + sq * md.w * dev[3 + (long)(k - 1) * n_dof + ridx];
                heat -= 0.5 * v * v / m;
                pnm[idx] = v;
            }
        }
    }
    heat = block_sum(heat, sh);
    if (threadIdx.x == 0) hpart[blockIdx.x] = heat;
}

// ---------------------------------------------------------------------------
// Verlet lists (neighbour.cpp:12-62) and the rebuild test (update.cpp:356-385)
// ---------------------------------------------------------------------------

// Per bead: two largest O displacement norms; flag = d1 + d2 > r_skin - r_cut,
// or forced (force_all; or every > 0 and the step about to complete, step_ctr
// + 1, a multiple of every).
// grid: P, 256 threads.
__global__ __launch_bounds__(256) void k_check(int n_mols, int NMP, const double *__restrict__ disp,
                                               double skin, int force_all, int every,
                                               const unsigned long long *__restrict__ step_ctr,
                                               int *__restrict__ flag, double *__restrict__ nreb)
{
    __shared__ double s1[256], s2[256];
    const int b = blockIdx.x;
    double m1 = 0.0, m2 = 0.0;
    for (int i = threadIdx.x; i < n_mols; i += 256) {
        const double *D = disp + (long)b * 3 * NMP;
        const double dx = D[i], dy = D[NMP + i], dz = D[2 * NMP + i];
        const double d2 = dx * dx + dy * dy + dz * dz;
        if (d2 > m1) {
            m2 = m1;
            m1 = d2;
        } else if (d2 > m2) {
            m2 = d2;
        }
    }
    s1[threadIdx.x] = m1;
    s2[threadIdx.x] = m2;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            const double a1 = s1[threadIdx.x], a2 = s2[threadIdx.x];
            const double b1 = s1[threadIdx.x + o], b2 = s2[threadIdx.x + o];
            // top two of {a1 >= a2, b1 >= b2}
            double t1, t2;
            if (a1 >= b1) {
                t1 = a1;
                t2 = a2 >= b1 ? a2 : b1;
            } else {
                t1 = b1;
                t2 = b2 >= a1 ? b2 : a1;
            }
            s1[threadIdx.x] = t1;
            s2[threadIdx.x] = t2;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        int f = force_all || (sqrt(s1[0]) + sqrt(s2[0]) > skin);
        if (every > 0 && step_ctr && (step_ctr[0] + 1ull) % (unsigned long long)every == 0ull)
            f = 1;
        flag[b] = f;
        if (f && nreb) nreb[b] += 1.0;
    }
}

// Count O-O pairs within r_skin per row (half: j > i; full: j != i).
// The distance test is bit-for-bit neighbour.cpp:42-53.
// grid: P * ceil(n_mols/4), 256 threads (one row per wavefront).
__global__ __launch_bounds__(256) void k_nl_count(int n_mols, int NAP, const double *__restrict__ q,
                                                  Box box, double r_skin_sq,
                                                  const int *__restrict__ flag,
                                                  int *__restrict__ cnt /*[P][2][n_mols]*/)
{
    const int nrb = (n_mols + 3) / 4;
    const int b = blockIdx.x / nrb;
    if (!flag[b]) return;
    const int i = (blockIdx.x - b * nrb) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n_mols) return;
    const double *Q = q + (long)b * 3 * NAP;
    const double xi = Q[3 * i], yi = Q[NAP + 3 * i], zi = Q[2 * NAP + 3 * i];
    int nh = 0, nf = 0;
    for (int j0 = 0; j0 < n_mols; j0 += 64) {
        const int j = j0 + lane;
        bool in = false;
        if (j < n_mols && j != i) {
            const double rx = mimg_exact(xi - Q[3 * j], box.L[0]);
            const double ry = mimg_exact(yi - Q[NAP + 3 * j], box.L[1]);
            const double rz = mimg_exact(zi - Q[2 * NAP + 3 * j], box.L[2]);
            const double rsq = rx * rx + ry * ry + rz * rz;
            in = rsq < r_skin_sq;
        }
        const unsigned long long bf = __ballot(in);
        const unsigned long long bh = __ballot(in && j > i);
        nf += __popcll(bf);
        nh += __popcll(bh);
    }
    if (lane == 0) {
        cnt[((long)b * 2 + 0) * n_mols + i] = nh;
        cnt[((long)b * 2 + 1) * n_mols + i] = nf;
    }
}

// Exclusive scans -> point (reference layout) and fpoint; zero the bead's
// displacements and the unused tail of its half list (neighbour.cpp:23-32).
// grid: P, 1024 threads.
__global__ __launch_bounds__(1024) void k_nl_scan(int n_mols, int list_size, long fcap,
                                                  const int *__restrict__ flag,
                                                  const int *__restrict__ cnt,
                                                  int *__restrict__ point, int *__restrict__ fpoint,
                                                  int *__restrict__ list, double *__restrict__ disp,
                                                  int NMP, int *__restrict__ status)
{
    const int b = blockIdx.x;
    if (!flag[b]) return;
    __shared__ int sh[1024];
    __shared__ int carry[2];
    if (threadIdx.x < 2) carry[threadIdx.x] = 0;
    __syncthreads();
    for (int which = 0; which < 2; ++which) {
        const int *c = cnt + ((long)b * 2 + which) * n_mols;
        int *outp = which == 0 ? point + (long)b * n_mols : fpoint + (long)b * (n_mols + 1);
        for (int i0 = 0; i0 < n_mols; i0 += 1024) {
            const int i = i0 + threadIdx.x;
            const int v = i < n_mols ? c[i] : 0;
            sh[threadIdx.x] = v;
            __syncthreads();
            for (int o = 1; o < 1024; o <<= 1) {
                const int add = threadIdx.x >= o ? sh[threadIdx.x - o] : 0;
                __syncthreads();
                sh[threadIdx.x] += add;
                __syncthreads();
            }
            const int incl = sh[threadIdx.x];
            const int base = carry[which];
            if (i < n_mols) outp[i] = base + incl - v;
            __syncthreads();
            if (threadIdx.x == 1023) carry[which] = base + incl;
            __syncthreads();
        }
        if (which == 1 && threadIdx.x == 0) outp[n_mols] = carry[1];
    }
    __syncthreads();
    const int nh = carry[0], nf = carry[1];
    if (threadIdx.x == 0) {
        if (nh > list_size || (long)nf > fcap) atomicOr(status, 1);
    }
    int *L = list + (long)b * list_size;
    for (int k = nh + threadIdx.x; k < list_size; k += 1024) L[k] = 0;
    for (int t = threadIdx.x; t < 3 * NMP; t += 1024) disp[(long)b * 3 * NMP + t] = 0.0;
}

// Write the list entries in ascending j with ballot + prefix popcount.
// grid: as k_nl_count.
__global__ __launch_bounds__(256) void k_nl_fill(int n_mols, int NAP, const double *__restrict__ q,
                                                 Box box, double r_skin_sq, int list_size, long fcap,
                                                 const int *__restrict__ flag,
                                                 const int *__restrict__ point,
                                                 const int *__restrict__ fpoint,
                                                 int *__restrict__ list, int *__restrict__ flist)
{
    const int nrb = (n_mols + 3) / 4;
    const int b = blockIdx.x / nrb;
    if (!flag[b]) return;
    const int i = (blockIdx.x - b * nrb) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (i >= n_mols) return;
    const double *Q = q + (long)b * 3 * NAP;
    const double xi = Q[3 * i], yi = Q[NAP + 3 * i], zi = Q[2 * NAP + 3 * i];
    int kh = point[(long)b * n_mols + i];
    long kf = fpoint[(long)b * (n_mols + 1) + i];
    int *L = list + (long)b * list_size;
    int *FL = flist + (long)b * fcap;
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int j0 = 0; j0 < n_mols; j0 += 64) {
        const int j = j0 + lane;
        bool in = false;
        if (j < n_mols && j != i) {
            const double rx = mimg_exact(xi - Q[3 * j], box.L[0]);
            const double ry = mimg_exact(yi - Q[NAP + 3 * j], box.L[1]);
            const double rz = mimg_exact(zi - Q[2 * NAP + 3 * j], box.L[2]);
            const double rsq = rx * rx + ry * ry + rz * rz;
            in = rsq < r_skin_sq;
        }
        const bool inh = in && j > i;
        const unsigned long long bf = __ballot(in);
        const unsigned long long bh = __ballot(inh);
        if (in) {
            const long pos = kf + __popcll(bf & below);
            if (pos < fcap) FL[pos] = j;
        }
        if (inh) {
            const int pos = kh + __popcll(bh & below);
            if (pos < list_size) L[pos] = j;
        }
        kf += __popcll(bf);
        kh += __popcll(bh);
    }
}

// Rebuild test (update.cpp:356-385) and, when it fires, the bead's Verlet
// lists (neighbour.cpp:12-62) in one launch: one block of 1024 threads per
// bead.  Row counts live in LDS (n_mols <= NL_FUSED_MAXMOL), rows are handled one
// per wavefront with ballot + prefix-popcount compaction; the distance test
// is bit-for-bit neighbour.cpp:42-53.   grid: P.
// (a1, a2) <- the two largest of {a1 >= a2} and {b1 >= b2}
__device__ __forceinline__ void top2_merge(double &a1, double &a2, double b1, double b2)
{
    if (a1 >= b1) {
        a2 = a2 >= b1 ? a2 : b1;
    } else {
        a2 = b2 >= a1 ? b2 : a1;
        a1 = b1;
    }
}
// Above this size the rebuild runs on the four-kernel path (k_check,
// k_nl_count, k_nl_scan, k_nl_fill: a wavefront per molecule row instead of
// one block per bead), whose rebuild steps are far shorter at thousands of
// molecules; below it the single fused launch costs less per step.
constexpr int NL_FUSED_MAXMOL = 1024;
// Optional heat sum of a thermostatted step (k_heat's work), done by wave 0
// of block 0 here so that it costs no launch of its own.
struct HeatArgs {
    const double *part;  // centroid KE partials (ntile) then chi partials
    const double *hpart; // heat partials of the dofs (nh)
    double *heat_acc, *heat_step;
    int ntile, nh;
};
struct NlArgs {
    int n_mols, NAP, NMP;
    const double *q;
    Box box;
    double r_skin_sq, skin;
    int force_all, every;
    const unsigned long long *step_ctr;
    int list_size;
    long fcap;
    double *disp;
    int *flag;
    double *nreb;
    int *point, *fpoint, *list, *flist, *status;
    unsigned long long *bm;  // one-stream form: row bitmaps and counts of rebuilt beads
    int *cnt;
    HeatArgs heat;
};
struct NlLds {
    double s1[16], s2[16];
    int ch[NL_FUSED_MAXMOL], cf[NL_FUSED_MAXMOL];
    int flag, tot[2];
};
// Whether bead b's lists are rebuilt this step: its two largest O
// displacements (update.cpp:356-385), or forced.  By a block of NT threads;
// the same value in every thread.  k_phase_pairs asks in several blocks (the
// list blocks and the LJ blocks) and relies on one answer: the library is built
// without FMA contraction, so every copy rounds the same.
template <int NT>
__device__ __forceinline__ int list_flag(double *s1, double *s2, int *flag, int b, const NlArgs &A)
{
    const double *D = A.disp + (long)b * 3 * A.NMP;
    const int tid = threadIdx.x;
    double m1 = 0.0, m2 = 0.0;
    for (int i = tid; i < A.n_mols; i += NT) {
        const double dx = D[i], dy = D[A.NMP + i], dz = D[2 * A.NMP + i];
        const double d2 = dx * dx + dy * dy + dz * dz;
        if (d2 > m1) {
            m2 = m1;
            m1 = d2;
        } else if (d2 > m2) {
            m2 = d2;
        }
    }
    // top two of the block: within each wave by shuffles, then over the waves
    for (int o = 32; o > 0; o >>= 1) {
        const double b1 = __shfl_xor(m1, o, 64), b2 = __shfl_xor(m2, o, 64);
        top2_merge(m1, m2, b1, b2);
    }
    if ((tid & 63) == 0) {
        s1[tid >> 6] = m1;
        s2[tid >> 6] = m2;
    }
    __syncthreads();
    if (tid == 0) {
        double t1 = s1[0], t2 = s2[0];
        for (int ww = 1; ww < NT / 64; ++ww) top2_merge(t1, t2, s1[ww], s2[ww]);
        int f = A.force_all || (sqrt(t1) + sqrt(t2) > A.skin);
        if (A.every > 0 && A.step_ctr && (A.step_ctr[0] + 1ull) % (unsigned long long)A.every == 0ull)
            f = 1;
        *flag = f;
    }
    __syncthreads();
    return *flag;
}
// The heat sum of a thermostatted step, by the first wave of a block.
__device__ __forceinline__ void list_heat(const HeatArgs &heat)
{
    if (threadIdx.x >= 64) return;
    const double ke = wave_sum_array(heat.part, heat.ntile);
    const double h = wave_sum_array(heat.hpart, heat.nh);
    if (threadIdx.x == 0) {
        const double ret = ke + h;
        heat.heat_step[0] = ret;
        heat.heat_acc[0] -= ret;
    }
}
__global__ __launch_bounds__(1024) void k_nlist_bead(const NlArgs A)
{
    __shared__ NlLds S;
    constexpr int NT = 1024;
    const int n_mols = A.n_mols, NAP = A.NAP, NMP = A.NMP, list_size = A.list_size;
    const double *__restrict__ q = A.q;
    const Box &box = A.box;
    const double r_skin_sq = A.r_skin_sq;
    const long fcap = A.fcap;
    double *__restrict__ disp = A.disp;
    int *__restrict__ flag = A.flag;
    double *__restrict__ nreb = A.nreb;
    int *__restrict__ point = A.point;
    int *__restrict__ fpoint = A.fpoint;
    int *__restrict__ list = A.list;
    int *__restrict__ flist = A.flist;
    int *__restrict__ status = A.status;
    const int b = blockIdx.x, tid = threadIdx.x;
    if (A.heat.part && b == (int)gridDim.x - 1) {  // the extra last block: the heat sum only
        list_heat(A.heat);
        return;
    }
    double *D = disp + (long)b * 3 * NMP;
    const int f = list_flag<NT>(S.s1, S.s2, &S.flag, b, A);
    if (tid == 0) {
        flag[b] = f;
        if (f && nreb) nreb[b] += 1.0;
    }
    if (!f) return;
    // --- counts
    const double *Q = q + (long)b * 3 * NAP;
    const int lane = tid & 63, w = tid >> 6;
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int i = w; i < n_mols; i += NT / 64) {
        const double xi = Q[3 * i], yi = Q[NAP + 3 * i], zi = Q[2 * NAP + 3 * i];
        int nh = 0, nf = 0;
        for (int j0 = 0; j0 < n_mols; j0 += 64) {
            const int j = j0 + lane;
            bool in = false;
            if (j < n_mols && j != i) {
                const double rx = mimg_exact(xi - Q[3 * j], box.L[0]);
                const double ry = mimg_exact(yi - Q[NAP + 3 * j], box.L[1]);
                const double rz = mimg_exact(zi - Q[2 * NAP + 3 * j], box.L[2]);
                in = rx * rx + ry * ry + rz * rz < r_skin_sq;
            }
            nf += __popcll(__ballot(in));
            nh += __popcll(__ballot(in && j > i));
        }
        if (lane == 0) {
            S.ch[i] = nh;
            S.cf[i] = nf;
        }
    }
    __syncthreads();
    // --- exclusive scans (wave 0: chunks of 64 with a running carry)
    if (w == 0) {
        int carry_h = 0, carry_f = 0;
        for (int i0 = 0; i0 < n_mols; i0 += 64) {
            const int i = i0 + lane;
            const int vh = i < n_mols ? S.ch[i] : 0, vf = i < n_mols ? S.cf[i] : 0;
            int ih = vh, iff = vf;
            for (int o = 1; o < 64; o <<= 1) {
                const int th = __shfl_up(ih, o, 64), tf = __shfl_up(iff, o, 64);
                if (lane >= o) {
                    ih += th;
                    iff += tf;
                }
            }
            if (i < n_mols) {
                S.ch[i] = carry_h + ih - vh;
                S.cf[i] = carry_f + iff - vf;
            }
            carry_h += __shfl(ih, 63, 64);
            carry_f += __shfl(iff, 63, 64);
        }
        if (lane == 0) {
            S.tot[0] = carry_h;
            S.tot[1] = carry_f;
        }
    }
    __syncthreads();
    const int nh_tot = S.tot[0], nf_tot = S.tot[1];
    if (tid == 0 && (nh_tot > list_size || (long)nf_tot > fcap)) atomicOr(status, 1);
    for (int i = tid; i < n_mols; i += NT) {
        point[(long)b * n_mols + i] = S.ch[i];
        fpoint[(long)b * (n_mols + 1) + i] = S.cf[i];
    }
    if (tid == 0) fpoint[(long)b * (n_mols + 1) + n_mols] = nf_tot;
    int *L = list + (long)b * list_size;
    int *FL = flist + (long)b * fcap;
    for (int k = nh_tot + tid; k < list_size; k += NT) L[k] = 0;
    for (int t = tid; t < 3 * NMP; t += NT) D[t] = 0.0;
    // --- fill
    for (int i = w; i < n_mols; i += NT / 64) {
        const double xi = Q[3 * i], yi = Q[NAP + 3 * i], zi = Q[2 * NAP + 3 * i];
        int kh = S.ch[i];
        long kf = S.cf[i];
        for (int j0 = 0; j0 < n_mols; j0 += 64) {
            const int j = j0 + lane;
            bool in = false;
            if (j < n_mols && j != i) {
                const double rx = mimg_exact(xi - Q[3 * j], box.L[0]);
                const double ry = mimg_exact(yi - Q[NAP + 3 * j], box.L[1]);
                const double rz = mimg_exact(zi - Q[2 * NAP + 3 * j], box.L[2]);
                in = rx * rx + ry * ry + rz * rz < r_skin_sq;
            }
            const bool inh = in && j > i;
            const unsigned long long bf = __ballot(in), bh = __ballot(inh);
            if (in) {
                const long pos = kf + __popcll(bf & below);
                if (pos < fcap) FL[pos] = j;
            }
            if (inh) {
                const int pos = kh + __popcll(bh & below);
                if (pos < list_size) L[pos] = j;
            }
            kf += __popcll(bf);
            kh += __popcll(bh);
        }
    }
}

// The same rebuild in the launches of the one-stream phase, spread over the
// chip: list_rows leaves a flagged bead's row bitmaps and counts, NL_ROWS rows
// a block; list_fill, in the block of the next launch that needs the rows,
// their offsets and entries.  A step that rebuilds lists took this much longer
// with one block of 256 threads a bead: 2.4 ms at 990 molecules (k_nlist_bead,
// 1024 threads: 1.4), 110 us at 216.  Now 21 and 13 us.
constexpr int NL_ROWS = 64;
struct NlRowLds {
    double s1[4], s2[4];
    int flag;
};
// grid share: P * ceil(n_mols / NL_ROWS) blocks of 256 threads, and one more
// with a heat sum.
__device__ __forceinline__ void list_rows(NlRowLds &S, int block, int nblocks, const NlArgs &A)
{
    if (A.heat.part && block == nblocks - 1) {
        list_heat(A.heat);
        return;
    }
    const int n = A.n_mols, NAP = A.NAP, nw = (n + 63) >> 6;
    const int nsub = (n + NL_ROWS - 1) / NL_ROWS;
    const int b = block / nsub, sub = block - b * nsub;
    const int f = list_flag<256>(S.s1, S.s2, &S.flag, b, A);
    if (sub == 0 && threadIdx.x == 0) {
        A.flag[b] = f;
        if (f && A.nreb) A.nreb[b] += 1.0;
    }
    if (!f) return;
    const double *Q = A.q + (long)b * 3 * NAP;
    const double Lx = A.box.L[0], Ly = A.box.L[1], Lz = A.box.L[2];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // one row at a time: four that share their partners' loads raise the
    // kernel's register use, and all its other roles slow down by 4 %
    for (int i = sub * NL_ROWS + w; i < min(n, (sub + 1) * NL_ROWS); i += 4) {
        const double x = Q[3 * i], y = Q[NAP + 3 * i], z = Q[2 * NAP + 3 * i];
        unsigned long long word = 0ull;
        int nh = 0, nf = 0;
        for (int k = 0; k < nw; ++k) {
            const int j = 64 * k + lane, jj = min(j, n - 1);
            const double rx = mimg_exact(x - Q[3 * jj], Lx);
            const double ry = mimg_exact(y - Q[NAP + 3 * jj], Ly);
            const double rz = mimg_exact(z - Q[2 * NAP + 3 * jj], Lz);
            const bool in = rx * rx + ry * ry + rz * rz < A.r_skin_sq && j < n && j != i;
            const unsigned long long m = __ballot(in);
            if (lane == k) word = m;
            nf += __popcll(m);
            nh += __popcll(__ballot(in && j > i));
        }
        if (lane < nw) A.bm[((long)b * n + i) * nw + lane] = word;
        if (lane == 0) {
            A.cnt[2L * b * n + i] = nh;
            A.cnt[(2L * b + 1) * n + i] = nf;
        }
    }
}
// Rows m0 ... m0 + nrow - 1 of rebuilt bead b from the bitmaps: offsets,
// entries and the bead's share part / nparts of the unused tail of its half
// list.  256 threads; the block may read its rows afterwards.
__device__ __forceinline__ void list_fill(int (*sh)[4], int b, int m0, int nrow, int part, int nparts,
                                          const NlArgs &A)
{
    const int n = A.n_mols, nw = (n + 63) >> 6, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int *ch = A.cnt + (2L * b) * n, *cf = ch + n;
    // rows before m0 and all rows: half, full
    int v[4] = {0, 0, 0, 0};
    for (int i = tid; i < n; i += 256) {
        const int h = ch[i], f = cf[i];
        v[2] += h;
        v[3] += f;
        if (i < m0) {
            v[0] += h;
            v[1] += f;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
        if (lane == 0) sh[w][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = sh[0][k] + sh[1][k] + sh[2][k] + sh[3][k];
    int *PT = A.point + (long)b * n, *FP = A.fpoint + (long)b * (n + 1);
    int *L = A.list + (long)b * A.list_size, *FL = A.flist + (long)b * A.fcap;
    const unsigned long long below = lane == 0 ? 0ull : ~0ull >> (64 - lane);
    for (int r = w; r < nrow; r += 4) {
        const int i = m0 + r;
        // this row's offsets and, lane r, its counts
        int h = lane <= r ? ch[m0 + lane] : 0, f = lane <= r ? cf[m0 + lane] : 0;
        const int nhr = __shfl(h, r, 64), nfr = __shfl(f, r, 64);
        for (int o = 32; o > 0; o >>= 1) {
            h += __shfl_xor(h, o, 64);
            f += __shfl_xor(f, o, 64);
        }
        int kh = v[0] + h - nhr;
        long kf = v[1] + f - nfr;
        if (lane == 0) {
            PT[i] = kh;
            FP[i] = (int)kf;
            FP[i + 1] = (int)kf + nfr;  // the next row's block writes the same
        }
        const unsigned long long *bm = A.bm + ((long)b * n + i) * nw;
        for (int k = 0; k < nw; ++k) {
            const unsigned long long m = bm[k];
            const unsigned long long mh =
                64 * k > i ? m : 64 * k + 63 <= i ? 0ull : m & ~((2ull << (i & 63)) - 1ull);
            if ((m >> lane) & 1ull) {
                const long pos = kf + __popcll(m & below);
                if (pos < A.fcap) FL[pos] = 64 * k + lane;
            }
            if ((mh >> lane) & 1ull) {
                const int pos = kh + __popcll(mh & below);
                if (pos < A.list_size) L[pos] = 64 * k + lane;
            }
            kf += __popcll(m);
            kh += __popcll(mh);
        }
    }
    for (int k = v[2] + part * 256 + tid; k < A.list_size; k += nparts * 256) L[k] = 0;
    if (part == 0 && tid == 0 && (v[2] > A.list_size || (long)v[3] > A.fcap)) atomicOr(A.status, 1);
    __syncthreads();
}

// ---------------------------------------------------------------------------
// A force phase in three launches on one stream (the third is k_kforce_mf).
// With the k-space and LJ kernels on a second stream a phase spent 5 us on the
// fork and 9 us on the join (a kernel starts that long after the last event of
// another queue; 0-1 us after its predecessor on its own queue).  The FP64
// matrix instructions and the FP64 vector instructions of different blocks
// take turns on the same units, so two launches side by side gain no
// arithmetic rate either.  us a step, two streams -> this form: 216 H2O
// classical 47 -> 37, 512 classical with the learned correction 79 -> 68, 216
// x 32 154 -> 148, 512 x 32 447 -> 409, 990 x 16 566 -> 539.
// ---------------------------------------------------------------------------
// First launch, 256 threads, LDS for the largest role: n_nl blocks of list
// checks and rebuilds of a step (and its heat sum); n_ks blocks of structure
// factors; n_lj of LJ and intramolecular terms; n_rs real-space tiles.  The
// roles with the longer latency come first when all blocks fit the chip at
// once (512 classical 68 against 70 us a step) and the fuller real-space
// blocks otherwise (512 x 32 409 against 418).
// The LJ blocks here of a step's first phase (n_nl > 0) test their bead's
// displacements themselves: a bead whose lists this launch rebuilds is left to
// k_phase_reduce, which also fills the lists and zeroes the displacements
// (nothing may change them while both roles read them).
constexpr int PH_CAP = 2;   // k_ksum_mf's CAP here: few accumulators, so that six
                            // waves fit a SIMD (four: 512 x 32 469 us a step)
constexpr int PH_SUB = 32;  // sites whose factor tables are staged at a time: about
                            // the LDS of a real-space block
constexpr int PH_RESIDENT = 256 * 6;  // blocks the chip holds at once
// With at most this many LJ blocks (two a CU: a launch of their own would be
// all latency) they run in the first launch, beside the real-space tiles;
// with more, in the second (216 x 32, 432 blocks: 148 us a step in the first,
// 152 in the second; 512 x 32, 1024 blocks: 414 and 409).
constexpr int PH_LJ_EARLY = 512;
struct LjLds {
    double sh[16], s1[16], s2[16];
    int flag;
};
template <bool VIR, int LPM>
__global__ __launch_bounds__(256, 6) void k_phase_pairs(const RsArgs rs, const KsArgs ks,
                                                        const LjArgs lj, const NlArgs nl, int n_nl,
                                                        int n_ks, int n_lj, int n_rs)
{
    extern __shared__ double smem[];
    int b = blockIdx.x;
    if (b < n_nl) {
        list_rows(*(NlRowLds *)smem, b, n_nl, nl);
        return;
    }
    b -= n_nl;
    const bool rs_last = n_ks + n_lj + n_rs <= PH_RESIDENT;
    if (rs_last ? b >= n_ks + n_lj : b < n_rs) {
        rs_tile<VIR, true, 4>(*(RsLds<4> *)smem, rs_last ? b - n_ks - n_lj : b, n_rs, rs);
        return;
    }
    if (!rs_last) b -= n_rs;
    if (b < n_ks) {
        ks_block<PH_CAP, 4>(smem, b, ks);
        return;
    }
    LjLds &L = *(LjLds *)smem;
    b -= n_ks;
    if (n_nl > 0 && list_flag<256>(L.s1, L.s2, &L.flag, lj_eval<LPM>(b, n_lj, lj), nl)) return;
    lj_block<VIR, LPM>(L.sh, b, n_lj, lj);
}
// Second launch, 256 threads: n_lj blocks for the LJ and intramolecular terms,
// of every bead or (rebuilt_only) of the beads whose lists the first launch
// rebuilt, whose rows it fills first; the rest: reduction of the structure
// factors.  n_nl > 0: a step's
// first phase, whose rebuilt beads' displacements are zeroed here.
template <bool VIR, int LPM>
__global__ __launch_bounds__(256) void k_phase_reduce(const SrArgs sr, const LjArgs lj, const NlArgs nl,
                                                      int n_nl, int n_lj, int rebuilt_only)
{
    __shared__ double sh[16];
    const int b = blockIdx.x;
    if (b >= n_lj) {
        sreduce_block(sh, b - n_lj, sr);
        return;
    }
    __shared__ int cs[4][4];
    constexpr int MPB = 256 / LPM;
    const int e = lj_eval<LPM>(b, n_lj, lj), mb = lj_eval_block<LPM>(b, n_lj, lj);
    const bool rebuilt = n_nl > 0 && nl.flag[e];
    if (rebuilt)
        list_fill(cs, e, mb * MPB, min(MPB, lj.n_mols - mb * MPB), mb, (lj.n_mols + MPB - 1) / MPB, nl);
    if (rebuilt || !rebuilt_only) lj_block<VIR, LPM>(sh, b, n_lj, lj);
    if (rebuilt && mb == 0)
        for (int t = threadIdx.x; t < 3 * nl.NMP; t += 256) nl.disp[(long)e * 3 * nl.NMP + t] = 0.0;
}

// ---------------------------------------------------------------------------
// Classical velocity Verlet (update.cpp:78-137)
// ---------------------------------------------------------------------------
// p += dt/2 F; q += p dt / m; O displacements.  grid: ceil(3 NAP / 256).
// With a thermostat (lang != 0) a Langevin step p = c1 p + sqrt(m/beta) c2 xi
// comes first (random stream 0 of the step counter; the counter advances in
// k_vv_b, so every block reads the same value here).
struct VVLang {
    int on;
    double c1, c2;
    uint64_t seed;
};
__global__ __launch_bounds__(256) void k_vv_a(int n_atoms, int NAP, int NMP, double halfdt,
                                              double dt, const double *__restrict__ m_atom,
                                              const double *__restrict__ F, double *__restrict__ q,
                                              double *__restrict__ p, double *__restrict__ disp,
                                              VVLang lang, const double *__restrict__ sqm_atom,
                                              const unsigned long long *__restrict__ step_ctr)
{
    const int f = blockIdx.x * 256 + threadIdx.x;
    if (f >= 3 * NAP) return;
    const int at = f % NAP, d = f / NAP;
    if (at >= n_atoms) return;
    double p0 = p[f];
    if (lang.on) {
        const double xi = philox_normal(lang.seed, *step_ctr, 0u, (uint32_t)(3 * at + d));
        p0 = lang.c1 * p0 + sqm_atom[at] * lang.c2 * xi;
    }
    double pp = p0 + halfdt * F[f];
    p[f] = pp;
    const double m = m_atom[at];
    q[f] += pp * dt / m;
    if (at % 3 == 0) disp[d * NMP + at / 3] += pp * dt / m;
}

// F = f_phys of the single evaluation, p += dt/2 F, energy out.
// fx, ex (may be null): forces (planar) and n_ex energy partials of a
// further term added to V (the learned correction's), summed in a fixed order.
__global__ __launch_bounds__(256) void k_vv_b(int n_atoms, int NAP, double halfdt,
                                              const double *__restrict__ fe,
                                              const double *__restrict__ epart, int ep_stride,
                                              int ep_n, double eself,
                                              double *__restrict__ F, double *__restrict__ p,
                                              double *__restrict__ out,
                                              unsigned long long *__restrict__ step_ctr,
                                              const double *__restrict__ fx,
                                              const float *__restrict__ ex, int n_ex)
{
    const int f = blockIdx.x * 256 + threadIdx.x;
    if (f < 3 * NAP) {
        const double v = fx ? fe[f] + fx[f] : fe[f];
        F[f] = v;
        const int at = f % NAP;
        if (at < n_atoms) p[f] += halfdt * v;
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        double v = eval_energy(epart, 0, ep_stride, ep_n, eself);
        if (ex) {
            double x = 0.0;
            for (int a = threadIdx.x; a < n_ex; a += 64) x += (double)ex[a];
            v += wave_sum(x);
        }
        if (threadIdx.x == 0) {
            out[0] = v;
            out[1] = 0.0;
            if (step_ctr) step_ctr[0] += 1ull;
        }
    }
}

// ---------------------------------------------------------------------------
// Observables (path_integrals.cpp:10-81)
// ---------------------------------------------------------------------------
// get_kcv: 0.5 n_dof / beta + (1/P) sum_{even b} sum_j -(q_bj - qc_j) f_bj.
// grid: ceil(3 NAP / 256); out: partials per block.
// Observables of the resident state, per 256-dof block: the centroid-virial
// sum -(q_b - qbar).f_b over even beads (path_integrals.cpp:29-48; centroid
// divided by float(P) as :21), the kinetic energy sum p^2/2m and the ring
// polymer spring energy (1/2) m w_P^2 sum_b (q_{b+1} - q_b)^2, which equals
// get_conserved's normal-mode sum (1/2) m w_k^2 q~_k^2 (path_integrals.cpp:
// 63-76) because the transform is orthonormal and w_k = 2 w_P sin(k pi / P).
// part[blk], part[nb + blk], part[2 nb + blk].   grid: nb, 256 threads.
__global__ __launch_bounds__(256) void k_obs_part(int P, int n_atoms, int NAP, double omega_psq,
                                                  const double *__restrict__ q,
                                                  const double *__restrict__ p,
                                                  const double *__restrict__ f,
                                                  const double *__restrict__ m_atom,
                                                  double *__restrict__ part)
{
    __shared__ double sh[16];
    const int t = blockIdx.x * 256 + threadIdx.x;
    double kc = 0.0, ke = 0.0, sp = 0.0;
    if (t < 3 * NAP && (t % NAP) < n_atoms) {
        const long N3 = 3L * NAP;
        const double m = m_atom[t % NAP];
        double qc = 0.0;
        for (int b = 0; b < P; ++b) qc += q[b * N3 + t];
        qc /= (double)(float)P;
        for (int b = 0; b < P; ++b) {
            const double qb = q[b * N3 + t], pb = p[b * N3 + t];
            if ((b & 1) == 0) kc -= (qb - qc) * f[b * N3 + t];
            ke += 0.5 * pb * pb / m;
            if (P > 1) {
                const double dq = q[((b + 1) % P) * N3 + t] - qb;
                sp += 0.5 * m * omega_psq * dq * dq;
            }
        }
    }
    kc = block_sum(kc, sh);
    ke = block_sum(ke, sh);
    sp = block_sum(sp, sh);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = kc;
        part[gridDim.x + blockIdx.x] = ke;
        part[2 * gridDim.x + blockIdx.x] = sp;
    }
}

// Reduce k_obs_part's partials into {K_cv, conserved, energy, sc_pot} (P > 1)
// or {kinetic energy, V + KE, V, 0} (P = 1).  With a trace, only on steps
// whose counter is a multiple of `every`, into trace[n][4], n counted in
// *ntrace (host-cleared before a run), at most cap samples.
// grid: 1, 64 threads.
__global__ __launch_bounds__(64) void k_obs_fin(int P, int nb, double half_ndof_over_beta,
                                                const double *__restrict__ part,
                                                const double *__restrict__ out,
                                                const unsigned long long *__restrict__ step_ctr,
                                                int every, int cap, int *__restrict__ ntrace,
                                                double *__restrict__ dst)
{
    if (every > 0 && (step_ctr[0] % (unsigned long long)every) != 0ull) return;
    const double kc = wave_sum_array(part, nb);
    const double ke = wave_sum_array(part + nb, nb);
    const double sp = wave_sum_array(part + 2 * nb, nb);
    if (threadIdx.x == 0) {
        double *o = dst;
        if (every > 0) {
            const int n = ntrace[0];
            if (n >= cap) return;
            o = dst + 4L * n;
            ntrace[0] = n + 1;
        }
        const double e = out[0];
        if (P > 1) {
            o[0] = half_ndof_over_beta + kc / P;
            o[1] = e + ke + sp;
            o[2] = e;
            o[3] = out[1];
        } else {
            o[0] = ke;
            o[1] = e + ke;
            o[2] = e;
            o[3] = 0.0;
        }
    }
}

__global__ __launch_bounds__(256) void k_kcv(int P, int n_atoms, int NAP,
                                             const double *__restrict__ q,
                                             const double *__restrict__ f,
                                             double *__restrict__ part)
{
    __shared__ double sh[16];
    const int t = blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    if (t < 3 * NAP && (t % NAP) < n_atoms) {
        const long N3 = 3L * NAP;
        double qc = 0.0;
        for (int b = 0; b < P; ++b) qc += q[b * N3 + t];
        qc /= (double)(float)P;
        for (int b = 0; b < P; b += 2) acc -= (q[b * N3 + t] - qc) * f[b * N3 + t];
    }
    acc = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// get_conserved on normal-mode q, p: sum_k sum_j p^2/2m + m w_k^2 q^2 / 2.
__global__ __launch_bounds__(256) void k_cons(int P, int n_atoms, int NAP,
                                              const double *__restrict__ nq,
                                              const double *__restrict__ np,
                                              const double4 *__restrict__ mode,
                                              const double *__restrict__ m_atom,
                                              double *__restrict__ part)
{
    __shared__ double sh[16];
    const int t = blockIdx.x * 256 + threadIdx.x;
    double acc = 0.0;
    if (t < 3 * NAP && (t % NAP) < n_atoms) {
        const long N3 = 3L * NAP;
        const double m = m_atom[t % NAP];
        for (int k = 0; k < P; ++k) {
            const double pv = np[k * N3 + t], qv = nq[k * N3 + t];
            acc += 0.5 * pv * pv / m + 0.5 * mode[k].y * (m * qv * qv);
        }
    }
    acc = block_sum(acc, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

// ---------------------------------------------------------------------------
// Centroid mean force, radial distribution functions (no counterpart in the
// reference; the CMD and g(r) tools its README leaves to other programs)
// ---------------------------------------------------------------------------
// acc[t] += (1/P) sum_b F[b][t]: the force on the centroid of dof t, summed
// over the steps of a run (the mean force of centroid-constrained runs).
// grid: ceil(3 NAP / 256), 256 threads.
__global__ __launch_bounds__(256) void k_cmf_acc(int P, int NAP, const double *__restrict__ F,
                                                 double *__restrict__ acc,
                                                 unsigned long long *__restrict__ n)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) n[0] += 1ull;
    if (t >= 3 * NAP) return;
    const long N3 = 3L * NAP;
    double s = 0.0;
    for (int b = 0; b < P; ++b) s += F[b * N3 + t];
    acc[t] += s / P;
}

// Centroid positions (bead average) of the planar state.  grid: ceil(3 NAP/256).
__global__ __launch_bounds__(256) void k_centroid(int P, int NAP, const double *__restrict__ q,
                                                  double *__restrict__ qc)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= 3 * NAP) return;
    const long N3 = 3L * NAP;
    double s = 0.0;
    for (int b = 0; b < P; ++b) s += q[b * N3 + t];
    qc[t] = s / P;
}

// Pair-distance histograms of the centroid positions: O-O over molecule
// pairs i < j, O-H over every (O of i, H of j) including j = i.  Bin
// floor(r / dr) of the minimum-image distance (bohr) below n_bins * dr.
// One wavefront per molecule i (lanes over j); integer counts, so the
// result does not depend on the order of the atomic adds.
// grid: ceil(n_mols / 4), 256 threads.
__global__ __launch_bounds__(256) void k_rdf(int n_mols, int NAP, const double *__restrict__ qc,
                                             Box box, double inv_dr, int n_bins,
                                             unsigned int *__restrict__ hoo,
                                             unsigned int *__restrict__ hoh)
{
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n_mols) return;
    const double xo = qc[3 * i], yo = qc[NAP + 3 * i], zo = qc[2 * NAP + 3 * i];
    for (int j = lane; j < n_mols; j += 64) {
        for (int s = 0; s < 3; ++s) {
            if (s == 0 && j <= i) continue;
            const int a = 3 * j + s;
            const double dx = mimg_exact(qc[a] - xo, box.L[0]);
            const double dy = mimg_exact(qc[NAP + a] - yo, box.L[1]);
            const double dz = mimg_exact(qc[2 * NAP + a] - zo, box.L[2]);
            const double r = sqrt(dx * dx + dy * dy + dz * dz);
            const double bf = r * inv_dr;
            if (bf < (double)n_bins) atomicAdd(s == 0 ? &hoo[(int)bf] : &hoh[(int)bf], 1u);
        }
    }
}

}  // namespace qtp
