// qtp_realspace.hpp -- real-space Ewald (forces.cpp:141-177, 586-608).
#pragma once
#include "qtp_common.hpp"

namespace qtp {
// Real-space Ewald over all site pairs i<j within r_c (forces.cpp:586-608,
// rwald :141-177).  One block of W wavefronts (W = 2 or 4) per 64x64 tile
// (I<=J) of the site pair matrix; wave w takes the 64/W j-columns
// c0 = w 64/W ... c0 + 64/W - 1 against all 64 i.
// Pass 1 (lane <-> i) tests a column per turn in fixed point (RsFix: the
// box is a power of two, so differences wrap to the minimum image by
// themselves) with a slightly larger cutoff and appends the column's pairs to
// an LDS queue (the comparison is the ballot; within a column, rows
// ascending).  Pass 2 gives every lane the same number of consecutive queue
// entries: lanes stay busy however unevenly the pairs fall.  It makes the
// exact FP64 cutoff test; the few pairs that fail it are zeroed on a branch
// that is seldom taken.  The kernel issues vector instructions in about two
// thirds of its cycles and uses the LDS in more than half: the FP64 form of
// pass 1 took a third of the instructions.  Measured alone, FP64 -> fixed
// point: 216 H2O x 32 beads 34.9 -> 31.1 us, 512 x 32 at r_c 10.9 A 105 -> 98
// us, 1000 x 16 at 12 A 153 -> 141 us.  Consecutive entries mostly share
// the column j, so a lane keeps the j reaction in registers and adds it to
// the LDS column array when j changes; i forces go to the wave's own LDS
// rows with ds_add_f64.  Columns belong to one wave and every wave has its
// own rows, and the LDS adds of a wave follow program and lane order, so
// the result is reproducible.
// Partial site forces go to slot J (block I's sites) and slot I (block J's
// sites): every (site, slot) has exactly one writer.
// grid: E * nt, 64 W threads: tiles t0 ... t0 + nt - 1 of the ntile of the
// list (a launch may take a part of the list; the parts write disjoint
// slots and partials).
// VIR: also accumulate the pair virial r_ij (x) f_ij (6 components) into
// vpart[(e*6 + c)*ep_stride + ep_off + tile].
// CARG: the special functions' coefficients come from RS_COEF (SGPRs) instead
// of literals (VGPRs); the host picks it for large grids.
// W: two waves per tile halve the block and double each lane's share of the
// queue; a launch then holds fewer waves (216 H2O x 32 beads: 4224, which
// the chip holds at once, against 8448 in two rounds with four).
constexpr int RS_WAVES = 4;  // the default W
constexpr long RS_CARG_BLOCKS = 16384;  // grids at least this large use CARG
// Boxes at least this many r_c wide use k_realspace_cull, with the two-stream
// phase around it.  Time of a step against the one-stream phase without culling
// (k_max 8):
//   molecules x beads   2.3 r_c   2.55    2.8    3.0-3.3
//   512 x 1              +78 %    +73 %   +70 %
//   512 x 32             +15 %    +12 %   +13 %   +12 %
//   1000 x 1                      +54 %   +53 %   +51 %
//   1000 x 32                      +3 %    -1 %    -7 %
//   1728 x 1                      +27 %   +26 %
//   1728 x 16                       0 %    -8 %   -13 %
// It pays where the launch fills the chip several times over; the line was
// drawn for 1000 molecules x 32 beads, before the one-stream phase, which gains
// most where the launch is small.
constexpr double RS_CULL_MIN_BOX = 2.5;

// Smallest distance between [a0, a1] and the periodic images of [b0, b1]
// (period L): the nearest image on the right is f = (b0 - a1) mod L away,
// the one a period to its left L - f - |A| - |B|; negative means overlap.
// Rounding of the mod only ever lowers the result to 0.
__device__ __forceinline__ double periodic_gap(double a0, double a1, double b0, double b1,
                                               double L, double invL)
{
    double f = b0 - a1;
    f = fma(-L, floor(f * invL), f);
    const double back = L - f - (a1 - a0) - (b1 - b0);
    return fmax(0.0, fmin(f, back));
}

// Fixed-point coordinates of pass 1.  Cubic boxes: 16 bits per coordinate in
// units of L / 2^16, the squared distance by two packed dot products (five
// instructions a pair); |d| comes out at most sqrt(3) units too large, so
// r2u is (r_c + 2 units)^2.  Other boxes: 32 bits per coordinate in units of
// L_d / 2^32, differences converted to FP32 and scaled by w (12 instructions);
// r2f is (r_c (1 + 1e-5))^2, the margin far above the FP32 rounding.  The FP64
// test took 15 plus the select of a mask bit.
struct RsFix {
    float w[3], r2f;
    unsigned r2u;
    int cubic;
};
inline RsFix rs_fix(const Box &box, double rcut)
{
    RsFix f;
    for (int d = 0; d < 3; ++d) f.w[d] = (float)(box.L[d] * (1.0 / 4294967296.0));
    const double r = rcut * (1.0 + 1e-5);
    f.r2f = (float)(r * r);
    f.cubic = box.L[0] == box.L[1] && box.L[1] == box.L[2];
    const double u = rcut / box.L[0] * 65536.0 + 2.0;
    // only used for cubic boxes, where r_c <= L / 2: below 2^31
    f.r2u = f.cubic ? (unsigned)(u * u) + 1u : 0u;
    return f;
}
typedef short rs_s16x2 __attribute__((ext_vector_type(2)));
// (x | y << 16, z) of a cubic box, or (x, y, z) of 32 bits each
__device__ __forceinline__ uint4 rs_fixed(double x, double y, double z, const Box &b, int cubic)
{
    const double fx = __builtin_amdgcn_fract(x * b.inv[0]);
    const double fy = __builtin_amdgcn_fract(y * b.inv[1]);
    const double fz = __builtin_amdgcn_fract(z * b.inv[2]);
    if (cubic) {
        const unsigned ux = (unsigned)fma(fx, 65536.0, 0.5), uy = (unsigned)fma(fy, 65536.0, 0.5),
                       uz = (unsigned)fma(fz, 65536.0, 0.5);
        return make_uint4((ux & 0xffffu) | (uy << 16), uz & 0xffffu, 0u, 0u);
    }
    return make_uint4((unsigned)(fx * 4294967296.0), (unsigned)(fy * 4294967296.0),
                      (unsigned)(fz * 4294967296.0), 0u);
}
__device__ __forceinline__ bool rs_near16(uint2 a, uint2 b, unsigned r2u)
{
    const rs_s16x2 xy = __builtin_bit_cast(rs_s16x2, a.x) - __builtin_bit_cast(rs_s16x2, b.x);
    const rs_s16x2 z = __builtin_bit_cast(rs_s16x2, a.y) - __builtin_bit_cast(rs_s16x2, b.y);
    // at most 3 * 2^30: read as unsigned
    const int r = __builtin_amdgcn_sdot2(z, z, __builtin_amdgcn_sdot2(xy, xy, 0, false), false);
    return (unsigned)r < r2u;
}
__device__ __forceinline__ bool rs_near32(uint4 a, uint4 b, const RsFix &f)
{
    const float dx = (float)(int)(a.x - b.x) * f.w[0];
    const float dy = (float)(int)(a.y - b.y) * f.w[1];
    const float dz = (float)(int)(a.z - b.z) * f.w[2];
    return fmaf(dx, dx, fmaf(dy, dy, dz * dz)) < f.r2f;
}

// Index of tile (I, J), I <= J, in the real-space tile list (I-major upper
// triangle of the nblk x nblk block matrix).
__device__ __forceinline__ int tile_index(int I, int J, int nblk)
{
    return I * nblk - (I * (I - 1)) / 2 + (J - I);
}

// Doubles per block in the CULL form's box table: the block's bounding box
// (lo xyz, hi xyz) at [0, 6), then the boxes of its eight 8-site clusters,
// component c of cluster k at [6 + 8 c + k].
constexpr int RS_BOX = 6 + 6 * 8;

// Sites of each 64-site block as (x, y, z, q) (M from O, H, H; forces.cpp:
// 558-564), the block's bounding box and those of its 8-site clusters
// (RS_BOX layout), for k_realspace_cull.  A cluster holding no
// site gets an empty box (lo > hi); k_realspace_cull never tests one.
// grid: E * nblk, 64 threads.
__global__ __launch_bounds__(64) void k_sites(const double *__restrict__ pos, long pstride,
                                              const double *__restrict__ charge, int n_atoms,
                                              int NAP, int nblk, double gamma, double half1mg,
                                              double4 *__restrict__ sites,
                                              double *__restrict__ bbox)
{
    const int e = blockIdx.x / nblk, B = blockIdx.x - e * nblk;
    const int l = threadIdx.x;
    const int s = B * 64 + l;
    const double *X = pos + (long)e * pstride;
    const bool ok = s < n_atoms;  // lane 0 always holds a site
    double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
    if (ok)
        v = make_double4(site_coord(X, NAP, s, 0, gamma, half1mg),
                         site_coord(X, NAP, s, 1, gamma, half1mg),
                         site_coord(X, NAP, s, 2, gamma, half1mg), charge[s]);
    sites[(long)e * nblk * 64 + s] = v;
    double lo[3] = {ok ? v.x : 1e300, ok ? v.y : 1e300, ok ? v.z : 1e300};
    double hi[3] = {ok ? v.x : -1e300, ok ? v.y : -1e300, ok ? v.z : -1e300};
    double *bb = bbox + ((long)e * nblk + B) * RS_BOX;
    // lanes 8k ... 8k + 7 form cluster k: the first three butterfly steps
    // stay inside it
    for (int o = 1; o < 8; o <<= 1)
        for (int d = 0; d < 3; ++d) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], o, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], o, 64));
        }
    {
        const int c = l & 7, k = l >> 3;
        if (c < 6) {
            const double vc = c == 0 ? lo[0] : c == 1 ? lo[1] : c == 2 ? lo[2]
                            : c == 3 ? hi[0] : c == 4 ? hi[1] : hi[2];
            bb[6 + 8 * c + k] = vc;
        }
    }
    for (int o = 8; o < 64; o <<= 1)
        for (int d = 0; d < 3; ++d) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], o, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], o, 64));
        }
    if (l < 3) bb[l] = l == 0 ? lo[0] : (l == 1 ? lo[1] : lo[2]);
    else if (l < 6) bb[l] = l == 3 ? hi[0] : (l == 4 ? hi[1] : hi[2]);
}

// Skip flags of the CULL form, one thread per (evaluation, tile): tile (I, J)
// is skipped (rfar = 1) when its two blocks' boxes are more than r_c apart
// under every periodic image; its energy partial (and virial partials, when
// vpart is given) are zeroed here, so k_realspace_cull only reads the
// flag.  grid: ceil(E * ntile / 256), 256 threads.
__global__ __launch_bounds__(256) void k_tilefar(const int2 *__restrict__ tiles, int ntile, int nblk,
                                                int E, const double *__restrict__ bbox, Box box,
                                                Ewald ew, unsigned char *__restrict__ rfar,
                                                double *__restrict__ epart, int ep_stride,
                                                int ep_off, double *__restrict__ vpart)
{
    const long k = (long)blockIdx.x * 256 + threadIdx.x;
    if (k >= (long)E * ntile) return;
    const int e = (int)(k / ntile), t = (int)(k - (long)e * ntile);
    const int2 ij = tiles[t];
    bool far = false;
    if (ij.x != ij.y) {
        const double *bI = bbox + ((long)e * nblk + ij.x) * RS_BOX;
        const double *bJ = bbox + ((long)e * nblk + ij.y) * RS_BOX;
        double gsq = 0.0;
        for (int d = 0; d < 3; ++d) {
            const double g =
                periodic_gap(bI[d], bI[3 + d], bJ[d], bJ[3 + d], box.L[d], box.inv[d]);
            gsq = fma(g, g, gsq);
        }
        // the margin covers the rounding of the boxes and of rsq
        far = gsq > ew.rcut_sq * (1.0 + 1e-9);
    }
    rfar[k] = far ? 1 : 0;
    if (far) {
        epart[(long)e * ep_stride + ep_off + t] = 0.0;
        if (vpart)
            for (int c = 0; c < 6; ++c) vpart[((long)e * 6 + c) * ep_stride + ep_off + t] = 0.0;
    }
}

// LDS of one tile's block.
template <int W>
struct RsLds {
    double4 sI[64], sJ[64];  // x, y, z, charge
    // fixed-point sites of J and I: 8 bytes each (cubic) or 16
    uint4 uJ[64], uI[64];
    double fj[3][64];
    double fi[W][3][64];
    double ewv[W];
    double wv[W][6];
    unsigned short qe[W][64 * (64 / W)];
};
// What a launch passes to every tile.
struct RsArgs {
    const double *pos;
    long pstride;
    const double *charge;
    int n_atoms, NAP, nblk;
    double gamma, half1mg;
    const int2 *tiles;
    int ntile, t0, nt;
    int gs;  // k_realspace_cull: tiles a block
    Box box;
    Ewald ew;
    double *rpart, *epart;
    int ep_stride, ep_off;
    double *vpart;
    const double4 *sites;
    const double *bbox;
    const unsigned char *rfar;
    RsFix fx;
};

// Pass 2 over the queue entries q0 ... q1 - 1 of this lane: rows il (site i0 +
// il) and columns jl (site j0 + jl; coordinates sJ[jl], reaction fj[.][jo +
// jl]).  Adds to fi, fj, the energy and (VIR) the virial.  near: the tile may
// hold pairs of one molecule.
template <bool VIR, bool CARG>
__device__ __forceinline__ void rs_pairs(const double4 *sI, const double4 *sJ, double (*fi)[64],
                                         double (*fj)[64], int jo, const unsigned short *qe, int q0,
                                         int q1, bool near, int i0, int j0, const RsArgs &A, double &en,
                                         double (&v6)[6])
{
    const Box &box = A.box;
    const Ewald &ew = A.ew;
    // at an offset the compiler cannot see through: loaded here, not held
    // in scalar registers by the code around
    int o = 0;
    asm volatile("" : "+s"(o));
    const RsCoef &cf = *(const RsCoef *)((const char *)&RS_COEF + o);
    double gx = 0.0, gy = 0.0, gz = 0.0;
    int jcur = -1;
    double4 b = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int q = q0; q < q1; ++q) {
        const int ent = qe[q];
        const int il = ent & 63, jl = ent >> 6;
        if (jl != jcur) {
            if (jcur >= 0) {
                atomicAdd(&fj[0][jo + jcur], gx);
                atomicAdd(&fj[1][jo + jcur], gy);
                atomicAdd(&fj[2][jo + jcur], gz);
            }
            gx = gy = gz = 0.0;
            jcur = jl;
            b = sJ[jl];
        }
        const double4 a = sI[il];
        double dx = mimg_fast(a.x - b.x, box.L[0], box.inv[0]);
        double dy = mimg_fast(a.y - b.y, box.L[1], box.inv[1]);
        double dz = mimg_fast(a.z - b.z, box.L[2], box.inv[2]);
        double rsq = fma(dx, dx, fma(dy, dy, dz * dz));
        double qq = a.w * b.w;
        // the exact cutoff: a pair of pass 1's margin (or with a NaN) adds nothing
        const bool out = !(rsq < ew.rcut_sq);
        if (__builtin_expect(__ballot(out) != 0ull, 0)) {
            if (out) {
                dx = dy = dz = qq = 0.0;
                rsq = ew.rcut_sq;
            }
        }
        const double rinv = rsqrt_pos(rsq);
        double ex, ec;
        if constexpr (CARG) {
            ex = exp_nonpos(-ew.kappa2 * rsq, cf);
            ec = erfc_via_erfcx(ew.kappa * (rsq * rinv), ex, cf);
        } else {
            constexpr LitCoef lc{};
            ex = exp_nonpos(-ew.kappa2 * rsq, lc);
            ec = erfc_via_erfcx(ew.kappa * (rsq * rinv), ex, lc);
        }
        // same molecule: -erf (forces.cpp:158-166); a molecule's three sites
        // lie in one 64-site block or two consecutive ones
        if (near && (i0 + il) / 3 == (j0 + jl) / 3) ec -= 1.0;
        const double ep = qq * rinv * ec;
        const double pf = (ep + qq * ew.pref2k * ex) * (rinv * rinv);
        en += ep;
        gx = fma(-pf, dx, gx);
        gy = fma(-pf, dy, gy);
        gz = fma(-pf, dz, gz);
        if (VIR) {
            v6[0] = fma(pf * dx, dx, v6[0]);
            v6[1] = fma(pf * dy, dy, v6[1]);
            v6[2] = fma(pf * dz, dz, v6[2]);
            v6[3] = fma(pf * dx, dy, v6[3]);
            v6[4] = fma(pf * dx, dz, v6[4]);
            v6[5] = fma(pf * dy, dz, v6[5]);
        }
        atomicAdd(&fi[0][il], pf * dx);
        atomicAdd(&fi[1][il], pf * dy);
        atomicAdd(&fi[2][il], pf * dz);
    }
    if (jcur >= 0) {
        atomicAdd(&fj[0][jo + jcur], gx);
        atomicAdd(&fj[1][jo + jcur], gy);
        atomicAdd(&fj[2][jo + jcur], gz);
    }
}

// The tile of block `block` of nblocks (XCD-remapped), by its 64 W threads.
template <bool VIR, bool CARG, int W>
__device__ __forceinline__ void rs_tile(RsLds<W> &L, int block, int nblocks, const RsArgs &A)
{
    static_assert(W == 2 || W == 4, "two or four waves per tile");
    constexpr int CPW = 64 / W;  // columns per wave
    const int n_atoms = A.n_atoms, NAP = A.NAP, nblk = A.nblk, ntile = A.ntile, t0 = A.t0, nt = A.nt;
    const int ep_stride = A.ep_stride, ep_off = A.ep_off;
    const double gamma = A.gamma, half1mg = A.half1mg;
    const Box &box = A.box;
    const Ewald &ew = A.ew;
    const RsFix &fx = A.fx;
    const double *__restrict__ charge = A.charge;
    double *__restrict__ rpart = A.rpart;
    double *__restrict__ epart = A.epart;
    double *__restrict__ vpart = A.vpart;
    auto &sI = L.sI;
    auto &sJ = L.sJ;
    auto &uJ = L.uJ;
    auto &uI = L.uI;
    auto &fj = L.fj;
    auto &fi = L.fi;
    auto &qe = L.qe;
    auto &ewv = L.ewv;
    auto &wv = L.wv;
    const int bid = xcd_remap(block, nblocks);
    const int e = bid / nt, t = t0 + (bid - e * nt);
    const int I = A.tiles[t].x, J = A.tiles[t].y;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double *X = A.pos + (long)e * A.pstride;
    const long base_e = (long)e * nblk * 3 * NAP;
    if (w < 2) {
        const int s = (w == 0 ? J : I) * 64 + l;
        double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
        if (s < n_atoms)
            v = make_double4(site_coord(X, NAP, s, 0, gamma, half1mg),
                             site_coord(X, NAP, s, 1, gamma, half1mg),
                             site_coord(X, NAP, s, 2, gamma, half1mg), charge[s]);
        (w == 0 ? sJ : sI)[l] = v;
        uint4 *us = w == 0 ? uJ : uI;
        const uint4 u = rs_fixed(v.x, v.y, v.z, box, fx.cubic);
        if (fx.cubic)
            ((uint2 *)us)[l] = make_uint2(u.x, u.y);
        else
            us[l] = u;
        if (w == 0) {
            fj[0][l] = 0.0;
            fj[1][l] = 0.0;
            fj[2][l] = 0.0;
        }
    }
    fi[w][0][l] = 0.0;
    fi[w][1][l] = 0.0;
    fi[w][2][l] = 0.0;
    __syncthreads();
    const int c0 = CPW * w;
    int total = 0;
    // append column c's pairs to the wave's queue; pass 1, column by column:
    // rows that exist, j > i in diagonal tiles
    const int nrow = min(64, n_atoms - I * 64), ncol = n_atoms - J * 64;
    auto push = [&](bool close, int c) {
        const int lim = c0 + c >= ncol ? 0 : I == J ? min(nrow, c0 + c) : nrow;
        const bool in = close && l < lim;
        const unsigned long long bal = __ballot(in);
        if (in) {
            const int r = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
            qe[w][total + r] = (unsigned short)(l | (c << 6));
        }
        total += __popcll(bal);
    };
    if (fx.cubic) {
        const uint2 a = ((const uint2 *)uI)[l];
#pragma unroll
        for (int c = 0; c < CPW; ++c) push(rs_near16(a, ((const uint2 *)uJ)[c0 + c], fx.r2u), c);
    } else {
        const uint4 a = uI[l];
#pragma unroll
        for (int c = 0; c < CPW; ++c) push(rs_near32(a, uJ[c0 + c], fx), c);
    }
    __syncthreads();
    // pass 2: lane l takes queue entries [l*S, l*S + S)
    const int S = (total + 63) >> 6;
    const int q0 = min(l * S, total), q1 = min(q0 + S, total);
    double en = 0.0, v6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    rs_pairs<VIR, CARG>(sI, sJ + c0, fi[w], fj, c0, qe[w], q0, q1, J - I <= 1, I * 64, J * 64 + c0, A, en, v6);
    en = wave_sum(en);
    if (l == 0) ewv[w] = en;
    if (VIR) {
        for (int cc = 0; cc < 6; ++cc) {
            const double v = wave_sum(v6[cc]);
            if (l == 0) wv[w][cc] = v;
        }
    }
    __syncthreads();
    if (VIR && threadIdx.x < 6) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < W; ++k) v += wv[k][threadIdx.x];
        vpart[((long)e * 6 + threadIdx.x) * ep_stride + ep_off + t] = v;
    }
    // component d of both slot entries of this tile
    for (int k = threadIdx.x; k < 192; k += 64 * W) {
        const int d = k >> 6, ll = k & 63;
        double si = 0.0;
#pragma unroll
        for (int v = 0; v < W; ++v) si += fi[v][d][ll];
        if (I == J) {
            rpart[base_e + (long)I * 3 * NAP + d * NAP + I * 64 + ll] = si + fj[d][ll];
        } else {
            rpart[base_e + (long)J * 3 * NAP + d * NAP + I * 64 + ll] = si;       // slot J
            rpart[base_e + (long)I * 3 * NAP + d * NAP + J * 64 + ll] = fj[d][ll];  // slot I
        }
    }
    if (threadIdx.x == 0) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < W; ++k) s += ewv[k];
        epart[(long)e * ep_stride + ep_off + t] = s;
    }
}

template <bool VIR, bool CARG, int W>
__global__ __launch_bounds__(64 * W) void k_realspace(const RsArgs A)
{
    __shared__ RsLds<W> L;
    rs_tile<VIR, CARG, W>(L, blockIdx.x, gridDim.x, A);
}

// The culling form.  The sites come from k_sites (x, y, z, q per site and
// bounding boxes per 64-site block and per 8-site cluster).  A tile whose two
// blocks' boxes are more than r_c apart under every periodic image holds no
// pair within the cutoff: k_tilefar marks it in rfar[e * ntile + tile] and
// zeroes its energy partial; no slot entries are written for it (k_kforce_mf
// and k_kforce read none of a tile so marked).  In the other tiles the cutoff
// test runs only over pairs of clusters whose boxes lie within r_c (4096 H2O,
// r_c 9 A: a third of the cluster pairs of the near tiles), one lane per site
// pair.  The same pairs are evaluated as by k_realspace.
// RS_CW waves take A.gs consecutive tiles of the list and work off the live
// ones, each wave its columns; the rows' sites stay in LDS while I is the same.
// Few blocks are launched for tiles that hold nothing (4096 x 32: three of
// four), and a tile's few hundred pairs (4096 H2O: 400) fill the lanes of two
// waves better than those of four.  Pass 1 takes RS_UNROLL cluster pairs at a
// time, their LDS reads in flight together; the queue is worked off, in whole
// rounds of the lanes, when it holds RS_QUEUE pairs.  RS_COEF is read after
// pass 1, whose scalars would be spilled otherwise.  Vector units and LDS are
// each busy two thirds of the time; of the 4096 x 32 launch pass 2 takes 58 %,
// pass 1 20 %.  us, a block of four waves per tile (of two) before -> now: 4096
// x 32 836 (703) -> 610, 1728 x 16 at r_c 12.9 A 323 (309) -> 301, 1000 x 32 183
// (168) -> 156, 2197 x 1 28 -> 29.  One wave a tile: 593, 324, 161, 36.
// grid: E * ceil(nt / gs), 64 RS_CW threads.
constexpr int RS_CW = 2, RS_UNROLL = 4, RS_QUEUE = 1024;
constexpr long RS_CULL_BLOCKS = 16384;  // a launch has at least this many blocks, or gs = 1
template <bool CUBIC>
struct RsU {
    using type = uint2;
};
template <>
struct RsU<false> {
    using type = uint4;
};
template <bool CUBIC>
struct RsCullLds {
    double4 sI[64], sJ[64];
    typename RsU<CUBIC>::type uI[64], uJ[64];
    double fj[3][64], fi[RS_CW][3][64];
    double ewv[RS_CW], wv[RS_CW][6];
    unsigned short qe[RS_CW][RS_QUEUE + 64 * RS_UNROLL];
};
template <bool VIR, bool CUBIC>
__global__ __launch_bounds__(64 * RS_CW, 5) void k_realspace_cull(const RsArgs A)
{
    __shared__ RsCullLds<CUBIC> L;
    constexpr int W = RS_CW, CPW = 64 / W;  // columns per wave
    using U = typename RsU<CUBIC>::type;
    const int n_atoms = A.n_atoms, NAP = A.NAP, nblk = A.nblk, ntile = A.ntile, nt = A.nt;
    const int ep_stride = A.ep_stride, ep_off = A.ep_off;
    const Box &box = A.box;
    const RsFix &fx = A.fx;
    const int ng = (nt + A.gs - 1) / A.gs;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int e = bid / ng, g0 = (bid - e * ng) * A.gs;
    const int l = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double4 *sites = A.sites + (long)e * nblk * 64;
    const double *bbox = A.bbox + (long)e * nblk * RS_BOX + 6;
    double *rp = A.rpart + (long)e * nblk * 3 * NAP;
    // the live tiles of the group (gs <= 64)
    const int tl = A.t0 + g0 + l;
    unsigned long long tiles = __ballot(l < A.gs && g0 + l < nt && !A.rfar[(long)e * ntile + min(tl, ntile - 1)]);
    int Icur = -1;
    while (tiles) {
        const int t = A.t0 + g0 + __builtin_ctzll(tiles);
        tiles &= tiles - 1ull;
        const int I = A.tiles[t].x, J = A.tiles[t].y;
        // the first wave stages the sites of J, the last those of a new I
        const bool newI = I != Icur;
        Icur = I;
        double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
        if (w == 0 || newI) v = sites[(w == 0 ? J : I) * 64 + l];
        const int ci = l & 7, cj = l >> 3;
        const double *cI = bbox + (long)I * RS_BOX, *cJ = bbox + (long)J * RS_BOX;
        double gsq = 0.0;
        for (int d = 0; d < 3; ++d) {
            const double gap = periodic_gap(cI[8 * d + ci], cI[8 * (3 + d) + ci], cJ[8 * d + cj],
                                            cJ[8 * (3 + d) + cj], box.L[d], box.inv[d]);
            gsq = fma(gap, gap, gsq);
        }
        // the live 8 x 8 cluster pairs: lane l tests row cluster l & 7 against
        // column cluster l >> 3
        unsigned long long todo = __ballot(gsq <= A.ew.rcut_sq * (1.0 + 1e-9) && I * 64 + 8 * ci < n_atoms &&
                                           J * 64 + 8 * cj < n_atoms && (I != J || cj >= ci)) &
                                  (((1ull << CPW) - 1ull) << (CPW * w));
        __syncthreads();
        auto put = [&](double4 *s4, U *u) {
            s4[l] = v;
            const uint4 x = rs_fixed(v.x, v.y, v.z, box, CUBIC);
            if constexpr (CUBIC) u[l] = make_uint2(x.x, x.y);
            else u[l] = x;
        };
        if (w == 0) {
            put(L.sJ, L.uJ);
            for (int d = 0; d < 3; ++d) L.fj[d][l] = 0.0;
        }
        if (w == W - 1 && newI) put(L.sI, L.uI);
        for (int d = 0; d < 3; ++d) L.fi[w][d][l] = 0.0;
        __syncthreads();
        double en = 0.0, v6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        unsigned short *qe = L.qe[w];
        // a tile that holds places without a pair
        const bool edge = I == J || J * 64 + 64 > n_atoms;
        int total = 0;
        do {
            // pass 1 over the live cluster pairs: each one's 64 site pairs
            // take one lane each; the queue holds a cluster pair's entries by
            // column, rows within a column
            while (todo && total < RS_QUEUE) {
                int il[RS_UNROLL], jl[RS_UNROLL];
                bool in[RS_UNROLL];
#pragma unroll
                for (int u = 0; u < RS_UNROLL; ++u) {
                    in[u] = todo != 0ull;
                    const int bit = in[u] ? __builtin_ctzll(todo) : 0;
                    todo &= todo - 1ull;
                    il[u] = 8 * (bit & 7) + (l & 7);
                    jl[u] = 8 * (bit >> 3) + (l >> 3);
                }
#pragma unroll
                for (int u = 0; u < RS_UNROLL; ++u) {
                    if constexpr (CUBIC) in[u] = in[u] && rs_near16(L.uI[il[u]], L.uJ[jl[u]], fx.r2u);
                    else in[u] = in[u] && rs_near32(L.uI[il[u]], L.uJ[jl[u]], fx);
                }
                if (edge) {
#pragma unroll
                    for (int u = 0; u < RS_UNROLL; ++u)
                        in[u] = in[u] && J * 64 + jl[u] > I * 64 + il[u] && J * 64 + jl[u] < n_atoms;
                }
#pragma unroll
                for (int u = 0; u < RS_UNROLL; ++u) {
                    const unsigned long long bal = __ballot(in[u]);
                    if (in[u]) {
                        const int r = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0u));
                        qe[total + r] = (unsigned short)(il[u] | (jl[u] << 6));
                    }
                    total += __popcll(bal);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            // all of it, or whole rounds of the lanes when more is to come
            const int n = todo ? total & ~63 : total;
            const int S = (n + 63) >> 6;
            const int q0 = min(l * S, n), q1 = min(q0 + S, n);
            rs_pairs<VIR, true>(L.sI, L.sJ, L.fi[w], L.fj, 0, qe, q0, q1, J - I <= 1, I * 64, J * 64, A, en, v6);
            total -= n;
            if (total > 0) {
                const unsigned short keep = qe[n + l];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (l < total) qe[l] = keep;
            }
        } while (todo || total > 0);
        en = wave_sum(en);
        if (l == 0) L.ewv[w] = en;
        if (VIR) {
            for (int c = 0; c < 6; ++c) {
                const double x = wave_sum(v6[c]);
                if (l == 0) L.wv[w][c] = x;
            }
        }
        __syncthreads();
        if (threadIdx.x < 6 && VIR) {
            double x = 0.0;
#pragma unroll
            for (int k = 0; k < W; ++k) x += L.wv[k][threadIdx.x];
            A.vpart[((long)e * 6 + threadIdx.x) * ep_stride + ep_off + t] = x;
        }
        if (threadIdx.x == 0) {
            double x = 0.0;
#pragma unroll
            for (int k = 0; k < W; ++k) x += L.ewv[k];
            A.epart[(long)e * ep_stride + ep_off + t] = x;
        }
        for (int k = threadIdx.x; k < 192; k += 64 * W) {
            const int d = k >> 6, ll = k & 63;
            double si = 0.0;
#pragma unroll
            for (int x = 0; x < W; ++x) si += L.fi[x][d][ll];
            const double sj = L.fj[d][ll];
            if (I == J) {
                rp[((long)I * 3 + d) * NAP + I * 64 + ll] = si + sj;
            } else {
                rp[((long)J * 3 + d) * NAP + I * 64 + ll] = si;  // slot J
                rp[((long)I * 3 + d) * NAP + J * 64 + ll] = sj;  // slot I
            }
        }
    }
}

}  // namespace qtp
