// mdg_shake_tri.h -- the SHAKE sweeps of a rigid three-site molecule, shared by
// the quad kernels (mdg_shake_w3.hip, one molecule per quad of lanes) and the
// lane kernels (mdg_shake_m3.hip, one molecule per lane).
//
// The molecule's three constraints form a ring: constraint k joins atoms k and
// k + 1 (mod 3) with the vector x_{k+1} - x_k (for k = 2 the negative of the
// reference's x_2 - x_0; the sign cancels in |d|^2, in the multiplier and in
// the corrections).  Atom k belongs to constraints k and k - 1 and moves along
// their vectors dd of the stage's start.
//
// The iterates follow the reference's loops (shake.c:262-332, 378-436) rounding by
// rounding: they feed the rounding of each moved position or velocity back into the
// next multiplier, so anything less differs by that rounding (over dt, in the
// velocities: 3e-11 A/ps at dt = 1 fs).  What a sweep leaves out is exact, the
// division up to quotients next to a rounding midpoint:
//  * the factor 1/2 of the position multiplier and the 1/nAtConst sit in the
//    atoms' factors (powers of two for the two constraints of an atom);
//  * an atom's own multiplier needs no move between lanes, and of the other
//    constraint only the multiplier moves;
//  * divisions are a reciprocal (of a constant, in stage 2) and one correction
//    by the remainder, which is exact: mdg_div64, and how far that is the
//    correctly rounded quotient.
// About 65 instructions a position sweep and 40 a velocity sweep where there
// were 110 and 80.
//
// Both layouts evaluate the same operations in the same order, so their
// results are the same bit for bit.
#pragma once
#include "mdg_shake.h"
#include "mdg_math64.h"

// The constant vector utils.c:38-80 subtracts from a bond vector: a bond (about
// an angstrom) keeps its image over the sweeps of a stage, and d - shift is
// then the reference's expression.  Triclinic boxes take the full image every
// sweep instead.
__device__ inline void tri_shift(const MdgBox &B, double dx, double dy, double dz, double &sx,
                                 double &sy, double &sz)
{
#pragma clang fp contract(off)
    sx = sy = sz = 0.;
    if (B.type == 3) return;
    const double Ly = B.type == 1 ? B.a1 : B.b2, Lz = B.type == 1 ? B.a1 : B.c3;
    const double uy = B.type == 1 ? B.u1 : B.v2, uz = B.type == 1 ? B.u1 : B.w3;
    sx = B.a1 * mdg_nint(dx * B.u1);
    sy = Ly * mdg_nint(dy * uy);
    sz = Lz * mdg_nint(dz * uz);
}

// One constraint of stage 1: shift, K = dt (dt / m_k + dt / m_{k+1}), target.
struct TriR {
    double sx, sy, sz, K, rc2, thr;
};

// From the raw bond vector d: the residual |d|^2 - rc2 (the stopping rule tests
// its absolute value, shake.c:243-258) and the multiplier.
__device__ __forceinline__ double tri_lambda(const MdgBox &B, const TriR &T, double dx, double dy,
                                             double dz, double ddx, double ddy, double ddz,
                                             double &e)
{
#pragma clang fp contract(off)
    double r2;
    if (B.type == 3) {
        r2 = mdg_dist(B, dx, dy, dz);
    } else {
        dx = dx - T.sx;
        dy = dy - T.sy;
        dz = dz - T.sz;
        r2 = dx * dx + dy * dy + dz * dz;
    }
    e = r2 - T.rc2;
    return mdg_div64(e, T.K * (ddx * dx + ddy * dy + ddz * dz));
}

// Atom k's position and velocity.
struct TriAtom {
    double x, y, z, vx, vy, vz;
};

// One sweep's corrections of atom k, once per constraint membership (two per
// atom): f its factor (0.5 dt / (m nAtConst) in stage 1, half dt / (m nAtConst)
// in stage 2), l and lp the multipliers of constraints k and k - 1, p* the
// vector of constraint k - 1.  POS moves the position too (stage 1).
template <bool POS>
__device__ __forceinline__ void tri_move(TriAtom &a, double dt, double f, double l, double lp,
                                         double ddx, double ddy, double ddz, double px, double py,
                                         double pz)
{
#pragma clang fp contract(off)
    const double u = l * f, w = lp * f;
    const double tx = ddx * u - px * w, ty = ddy * u - py * w, tz = ddz * u - pz * w;
    if (POS) {
        const double ix = dt * tx, iy = dt * ty, iz = dt * tz;
        a.x = (a.x + ix) + ix;
        a.y = (a.y + iy) + iy;
        a.z = (a.z + iz) + iz;
    }
    a.vx = (a.vx + tx) + tx;
    a.vy = (a.vy + ty) + ty;
    a.vz = (a.vz + tz) + tz;
}

// Stage 2: the multiplier of a constraint, dd . dv / K with the constant K and
// its reciprocal y.
__device__ __forceinline__ double tri_lambda_v(double K, double y, double dvx, double dvy,
                                               double dvz, double ddx, double ddy, double ddz)
{
#pragma clang fp contract(off)
    const double a = ddx * dvx + ddy * dvy + ddz * dvz;
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-K, q, a), y, q);
}

// The converged-sweep bits of one molecule (or wavefront): the current word in
// a register, flushed when it is complete or the loop ends.
struct TriBits {
    unsigned long long w[SHK_MASKW], cur;
};

__device__ __forceinline__ void tri_bits_init(TriBits &b)
{
#pragma unroll
    for (int q = 0; q < SHK_MASKW; q++) b.w[q] = 0;
    b.cur = 0;
}

__device__ __forceinline__ void tri_flush(TriBits &b, int word)
{
#pragma unroll
    for (int q = 0; q < SHK_MASKW; q++)
        if (q == word) b.w[q] = b.cur;
    b.cur = 0;
}

// The lanes whose molecules stop together with this lane's: the wavefront's, in a
// batch those of its replica (idle lanes are their own share).  One pass per replica
// in the wavefront, once a stage.
template <bool BATCH>
__device__ inline unsigned long long tri_share(const ShakeArgs &A, int g)
{
    if (!BATCH) return ~0ull;
    const int r = g < A.nGrp ? A.grep[g] : -1;
    unsigned long long share = 0, todo = __builtin_amdgcn_ballot_w64(true);
    while (todo) {
        const int lead = __builtin_amdgcn_readlane(r, __builtin_ctzll(todo));
        const unsigned long long m = __builtin_amdgcn_ballot_w64(r == lead);
        if (r == lead) share = m;
        todo &= ~m;
    }
    return share;
}

// Whether this sweep can be the stopping sweep as far as this wavefront knows: every
// molecule of the lane's share is converged.
template <bool BATCH>
__device__ __forceinline__ bool tri_all(bool bad, unsigned long long share)
{
    const unsigned long long b = __builtin_amdgcn_ballot_w64(bad);
    return BATCH ? (b & share) == 0 : b == 0;
}

// The sweeps whose states part A keeps for one share, in a ring of SHK_R slots: those
// at which the share was converged (a residual that passes through zero converges at
// a lone sweep, which can be the global stop, before it settles), up to the second of
// two in a row.  A wavefront of one system ends there; one of a batch sweeps on for its
// other replicas, and states from then on would push out the ones the stop needs (512
// replicas of 40 to 52 molecules, a molecule per lane: 298 us a step, with them 340).
struct TriRing {
    int saved[SHK_R] = {-1, -1, -1, -1}, nr = 0;
    bool prev = false, done = false;   // batch

    // Whether this sweep's state is kept.
    template <bool BATCH>
    __host__ __device__ __forceinline__ bool keep(bool all)
    {
        if (!BATCH) return all;
        const bool k = all && !done;
        done = done || (all && prev);
        prev = all;
        return k;
    }

    // The slot of the next state, and that it was sweep it's.
    __host__ __device__ __forceinline__ int slot() const { return nr & (SHK_R - 1); }
    __host__ __device__ __forceinline__ void put(int it)
    {
#pragma unroll
        for (int q = 0; q < SHK_R; q++)
            if (q == slot()) saved[q] = it;
        nr++;
    }
};

// The latest saved sweep of a ring that is not past C, and its slot; -1 when there
// is none.
__host__ __device__ inline int tri_resume(const int *ring, int C, int &slot)
{
    int at = -1;
    slot = 0;
#pragma unroll
    for (int q = 0; q < SHK_R; q++) {
        const int s = ring[q];
        if (s <= C && s > at) {
            at = s;
            slot = q;
        }
    }
    return at;
}

__device__ inline int tri_resume(const ShakeArgs &A, int g, int C, int &slot)
{
    return tri_resume(A.ring + (long)SHK_R * g, C, slot);
}

template <bool BATCH>
__device__ inline const MdgBox &tri_box(const ShakeArgs &A, int g)
{
    return BATCH ? A.boxes[A.grep[g]] : A.B;
}

template <bool BATCH>
__device__ inline const unsigned long long *tri_mask(const ShakeArgs &A, int g)
{
    return BATCH ? A.mask + (long)A.grep[g] * SHK_MASKW : A.mask;
}

template <bool BATCH>
__device__ inline void tri_publish(const ShakeArgs &A, int g, const TriBits &b, int kend,
                                   bool settled)
{
    if (BATCH) shake_publish_mask_b(A, b.w, kend, settled, g < A.nGrp ? A.grep[g] : -1);
    else shake_publish_mask(A, b.w, kend, settled);
}

// A slot's position, relative coordinates and cleared force accumulators, as
// k_slot_pos writes them (a device step without a list rebuild); d2 and rel
// collect the largest squared move and |relative coordinate|.
__device__ inline void tri_write_slot(const ShakeArgs &A, int atom, double nx, double ny,
                                      double nz, bool track, double &d2, double &rel)
{
    const int s = A.atomSlot[atom];
    if (A.spr)
        rel = fmax(rel, mdg_slot_rel(A.B, A.cO, A.ncluO, s / MDG_CL, nx, ny, nz, A.spr, s));
    if (track) {
        const double L0 = A.B.a1, L1 = A.B.type == 1 ? A.B.a1 : A.B.b2,
                     L2 = A.B.type == 1 ? A.B.a1 : A.B.c3;
        double dx = nx - A.sx[s], dy = ny - A.sy[s], dz = nz - A.sz[s];
        dx -= L0 * rint(dx / L0);
        dy -= L1 * rint(dy / L1);
        dz -= L2 * rint(dz / L2);
        const double e = dx * dx + dy * dy + dz * dz;
        d2 = fmax(d2, e <= 1e300 ? e : INFINITY);   // NaN positions: no pruning
    }
    A.sx[s] = nx;
    A.sy[s] = ny;
    A.sz[s] = nz;
    A.fix[s] = 0;
    A.fix[s + A.fstr] = 0;
    A.fix[s + 2 * A.fstr] = 0;
}

// Block partials of the stage-1 replay: the SHAKE virial and, with slotWrite,
// the largest squared move and |relative coordinate|.
__device__ inline void tri_block_out(const ShakeArgs &A, double vir, bool track, double d2,
                                     double rel)
{
    double acc[1] = {vir};
    mdg_block_partials<1>(acc, A.vir);
    if (!A.slotWrite) return;
    for (int o = 32; o > 0; o >>= 1) d2 = fmax(d2, __shfl_xor(d2, o, 64));
    __shared__ double wmax[4];
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = d2;
    __syncthreads();
    if (threadIdx.x == 0)
        A.dispPart[blockIdx.x] =
            track ? fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3])) : INFINITY;
    if (A.spr) mdg_block_max(rel, A.relPart);
}
