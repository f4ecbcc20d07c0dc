// mdg_shake_w3.hip -- VV + SHAKE kernels specialised for rigid
// three-site molecules (three atoms a0 < a1 < a2 with constraints
// (a0,a1), (a0,a2), (a1,a2) in that order, e.g. TIP3P water under
// consth), with the global stopping rule of the generic kernels of
// mdg_integrate.hip and the sweeps of mdg_shake_tri.h.
//
// One molecule per quad of lanes: lane k < 3 holds atom k and the constraint
// between atoms k and k + 1 (mod 3), lane 3 idles on a constraint that is met.
// Molecules sit on every spread-th quad, so a smaller spread packs more
// molecules per wavefront and a larger one gives the SIMDs more wavefronts to
// interleave; the autotuner picks it.  A sweep moves only the multipliers
// between lanes (DPP quad permutations).
#include "mdg_shake_tri.h"

namespace {

// quad_perm selectors: lane j of the quad reads lane sel_j
constexpr int QP_N = 0xC9;     // [1,2,0,3]: the next constraint / atom
constexpr int QP_P = 0xD2;     // [2,0,1,3]: the previous one
constexpr int QP_L0 = 0xC0;    // [0,0,0,3]
constexpr int QP_L1 = 0xD5;    // [1,1,1,3]
constexpr int QP_L2 = 0xEA;    // [2,2,2,3]

template <int CTRL>
__device__ __forceinline__ double qperm(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}

// v + t over the three live lanes in the order of the given selectors, on
// every lane.
template <int A0, int A1, int A2>
__device__ inline double q_sum3(double t)
{
#pragma clang fp contract(off)
    return (qperm<A0>(t) + qperm<A1>(t)) + qperm<A2>(t);
}

// One lane's share of a molecule.
struct Q3 {
    int k, at;              // 0..2 live, 3 idle; atom k
    TriAtom a;
    double rm, rmn, nat;    // inverse masses of atoms k, k + 1; 1 / nAtConst
    double ddx, ddy, ddz;   // constraint vector at the stage start
    double px, py, pz;      // the previous constraint's
    double f;               // the atom's factor
    TriR T;                 // stage 1
    double K, y;            // stage 2
    double vir;             // this constraint's virial sum
};

// The vector from atom k to atom k + 1; every lane takes part in the moves.
__device__ __forceinline__ void q_bond(const Q3 &Q, double &dx, double &dy, double &dz)
{
    dx = qperm<QP_N>(Q.a.x) - Q.a.x;
    dy = qperm<QP_N>(Q.a.y) - Q.a.y;
    dz = qperm<QP_N>(Q.a.z) - Q.a.z;
}

// Loads atom k (lanes without one get zeros) and forms the constraint vector
// at the stage's start (integrate.c:1536-1545).  Every group has exactly three
// atoms and constraints, so its tables start at 3 g.
__device__ inline void q_load(const ShakeArgs &A, const MdgBox &B, int g, int k, Q3 &Q)
{
    Q.k = g < A.nGrp ? k : 3;
    Q.at = -1;
    Q.a.x = Q.a.y = Q.a.z = Q.a.vx = Q.a.vy = Q.a.vz = 0.;
    Q.rm = Q.nat = Q.vir = 0.;
    if (Q.k < 3) {
        const int i = A.atoms[3 * g + k];
        Q.at = i;
        Q.a.x = A.x[i];
        Q.a.y = A.y[i];
        Q.a.z = A.z[i];
        Q.a.vx = A.vx[i];
        Q.a.vy = A.vy[i];
        Q.a.vz = A.vz[i];
        Q.rm = A.rmass[i];
        Q.nat = 1.0 / (double)A.nAtConst[i];
    }
    Q.rmn = qperm<QP_N>(Q.rm);
    q_bond(Q, Q.ddx, Q.ddy, Q.ddz);
    mdg_dist(B, Q.ddx, Q.ddy, Q.ddz);
    Q.px = qperm<QP_P>(Q.ddx);
    Q.py = qperm<QP_P>(Q.ddy);
    Q.pz = qperm<QP_P>(Q.ddz);
}

__device__ inline void q_kick(const ShakeArgs &A, Q3 &Q, double fx, double fy, double fz)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
    Q.a.vx += 0.5 * dt * fx * Q.rm;
    Q.a.vy += 0.5 * dt * fy * Q.rm;
    Q.a.vz += 0.5 * dt * fz * Q.rm;
}

__device__ inline void q_force(const ShakeArgs &A, const Q3 &Q, double &fx, double &fy, double &fz)
{
    fx = fy = fz = 0.;
    if (Q.k < 3) {
        fx = A.fx[Q.at];
        fy = A.fy[Q.at];
        fz = A.fz[Q.at];
    }
}

// The constraint of stage 1 (the image shift from the drifted positions).  In
// the reference's tables (0,1), (1,2), (0,2) are constraints 0, 2, 1 of the
// group; lane 3's has multiplier 0.
__device__ inline void q_setup_r(const ShakeArgs &A, const MdgBox &B, int g, Q3 &Q)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
    Q.T.rc2 = 0.;
    Q.T.thr = 1.;
    if (Q.k < 3) {
        const int c = A.cons[3 * g + (Q.k == 0 ? 0 : 3 - Q.k)];
        Q.T.rc2 = A.rc2[c];
        Q.T.thr = A.thr[c];
    }
    double dx, dy, dz;
    q_bond(Q, dx, dy, dz);
    tri_shift(B, dx, dy, dz, Q.T.sx, Q.T.sy, Q.T.sz);
    Q.T.K = dt * (dt * Q.rm + dt * Q.rmn);
    Q.f = 0.5 * (dt * Q.rm) * Q.nat;
}

__device__ inline void q_setup_v(const ShakeArgs &A, Q3 &Q)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
    const double tr = 0.5 * dt * Q.rm, trn = 0.5 * dt * Q.rmn;
    Q.K = Q.k < 3 ? (tr + trn) * (Q.ddx * Q.ddx + Q.ddy * Q.ddy + Q.ddz * Q.ddz) : 1.;
    Q.y = 1.0 / Q.K;
    Q.f = tr * Q.nat;
}

// The lane's residual and multiplier at the current positions.
__device__ __forceinline__ double q_lambda_r(const MdgBox &B, const Q3 &Q, double &e)
{
    double dx, dy, dz;
    q_bond(Q, dx, dy, dz);
    const double l = tri_lambda(B, Q.T, dx, dy, dz, Q.ddx, Q.ddy, Q.ddz, e);
    return Q.k < 3 ? l : 0.;
}

__device__ __forceinline__ double q_lambda_v(const Q3 &Q)
{
    return tri_lambda_v(Q.K, Q.y, qperm<QP_N>(Q.a.vx) - Q.a.vx, qperm<QP_N>(Q.a.vy) - Q.a.vy,
                        qperm<QP_N>(Q.a.vz) - Q.a.vz, Q.ddx, Q.ddy, Q.ddz);
}

template <bool POS>
__device__ __forceinline__ void q_sweep(const ShakeArgs &A, Q3 &Q, double l)
{
    tri_move<POS>(Q.a, A.P.timeStep, Q.f, l, qperm<QP_P>(l), Q.ddx, Q.ddy, Q.ddz, Q.px, Q.py,
                  Q.pz);
}

// The virial term of a sweep (shake.c:290).
__device__ __forceinline__ void q_virial(Q3 &Q, double l, double ddsq)
{
#pragma clang fp contract(off)
    Q.vir += l * ddsq;
}

__device__ __forceinline__ double q_ddsq(const Q3 &Q)
{
#pragma clang fp contract(off)
    return Q.ddx * Q.ddx + Q.ddy * Q.ddy + Q.ddz * Q.ddz;
}

__device__ inline void q_store(const ShakeArgs &A, const Q3 &Q)
{
    if (Q.k >= 3) return;
    const int i = Q.at;
    A.x[i] = Q.a.x;
    A.y[i] = Q.a.y;
    A.z[i] = Q.a.z;
    A.vx[i] = Q.a.vx;
    A.vy[i] = Q.a.vy;
    A.vz[i] = Q.a.vz;
}

// The state of a sweep at which the whole wavefront was converged, in the next
// of SHK_R slots: part B starts from one of them, or arrives there at once.
template <bool POS>
__device__ inline void q_save(const ShakeArgs &A, int g, const Q3 &Q, int slot)
{
    if (Q.k >= 3) return;
    const long n = A.P.n;
    double *s = A.scr + (long)slot * 6 * n + Q.at;
    if (POS) {
        s[0] = Q.a.x;
        s[n] = Q.a.y;
        s[2 * n] = Q.a.z;
        A.virScr[((long)slot * A.nGrp + g) * 3 + Q.k] = Q.vir;
    }
    s[3 * n] = Q.a.vx;
    s[4 * n] = Q.a.vy;
    s[5 * n] = Q.a.vz;
}

template <bool POS>
__device__ inline void q_restore(const ShakeArgs &A, int g, Q3 &Q, int slot)
{
    const long n = A.P.n;
    const double *s = A.scr + (long)slot * 6 * n + Q.at;
    if (POS) {
        Q.a.x = s[0];
        Q.a.y = s[n];
        Q.a.z = s[2 * n];
        Q.vir = A.virScr[((long)slot * A.nGrp + g) * 3 + Q.k];
    }
    Q.a.vx = s[3 * n];
    Q.a.vy = s[4 * n];
    Q.a.vz = s[5 * n];
}

// Whether every lane of this lane's quad (batch) or of the wavefront (one
// system, whose molecules share a stopping sweep) is converged, from the
// wavefront's ballot of unconverged lanes.
template <bool BATCH>
__device__ __forceinline__ bool q_conv(unsigned long long bad)
{
    return BATCH ? ((bad >> (threadIdx.x & 60)) & 15) == 0 : bad == 0;
}

}  // namespace

// Stage 1, part A: half kick, drift and SHAKE-R sweeps, recording the sweeps
// at which every molecule of the wavefront (in a batch: this molecule) was
// converged.  Blocks past S.nbMain do the previous step's record and list prune
// (mdg_side.h).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_w3_vv1_a(ShakeArgs A, SideWork S)
{
#pragma clang fp contract(off)
    if ((int)blockIdx.x >= S.nbMain) {
        side_work<BATCH>(S);
        return;
    }
    const int g = shake_w3_group(A);
    const MdgBox &B = tri_box<BATCH>(A, BATCH ? min(g, A.nGrp - 1) : 0);
    Q3 Q;
    q_load(A, B, g, threadIdx.x & 3, Q);
    double fx, fy, fz;
    q_force(A, Q, fx, fy, fz);
    q_kick(A, Q, fx, fy, fz);
    const double dt = A.P.timeStep;
    Q.a.x += dt * Q.a.vx;
    Q.a.y += dt * Q.a.vy;
    Q.a.z += dt * Q.a.vz;
    q_setup_r(A, B, g, Q);
    const double ddsq = q_ddsq(Q);
    TriBits bits;
    tri_bits_init(bits);
    const unsigned long long share = tri_share<BATCH>(A, g);
    TriRing ring;
    int it = 0;
    bool prev = false, settled = false;
    // until every molecule of the wavefront was converged at two consecutive
    // checks (the wavefront's time is its slowest molecule's)
    for (;;) {
        double e;
        const double l = q_lambda_r(B, Q, e);
        // the multiplier is formed before the vote, which it overlaps
        asm volatile("" ::"v"(l));
        const bool bad = Q.k < 3 && !(fabs(e) < Q.T.thr);
        const bool cv = q_conv<BATCH>(__builtin_amdgcn_ballot_w64(bad));
        if (cv) bits.cur |= 1ull << (it & 63);
        if (ring.keep<BATCH>(tri_all<BATCH>(bad, share))) {
            q_save<true>(A, g, Q, ring.slot());
            ring.put(it);
        }
        settled = settled || (cv && prev);
        prev = cv;
        if (BATCH ? __builtin_amdgcn_ballot_w64(!settled) == 0 : settled) break;
        if (it + 1 >= A.P.maxCycle) break;
        q_sweep<true>(A, Q, l);
        q_virial(Q, l, ddsq);
        if ((it & 63) == 63) tri_flush(bits, it >> 6);
        it++;
    }
    tri_flush(bits, it >> 6);
    if (Q.k == 0) {
        for (int q = 0; q < SHK_R; q++) A.ring[(long)SHK_R * g + q] = ring.saved[q];
    }
    tri_publish<BATCH>(A, g, bits, it, settled);
}

// Stage 1, part B: every molecule goes to the first sweep C at which all
// molecules were converged, from the latest saved state that is not past it or
// from the start.
template <bool BATCH>
__global__ void __launch_bounds__(256) k_w3_vv1_b(ShakeArgs A)
{
#pragma clang fp contract(off)
    // the stage-2 mask (beside this stage's) for this step's stage 2
    if (!BATCH && blockIdx.x == 0 && threadIdx.x < SHK_MASKW) A.mask[SHK_MASKW + threadIdx.x] = ~0ull;
    const int g = shake_w3_group(A);
    const int gb = BATCH ? min(g, A.nGrp - 1) : 0;
    const MdgBox &B = tri_box<BATCH>(A, gb);
    double vblk = 0.;   // this lane's share of the block's SHAKE virial
    Q3 Q;
    q_load(A, B, g, threadIdx.x & 3, Q);
    const int C = shake_global_stop(A, tri_mask<BATCH>(A, gb));
    if (C < 0) {
        if (Q.k == 0) atomicOr(&A.ctrl[CTRL_SHAKE_FAIL], 1);
    } else {
        // the same in every live lane of a quad; lane 3 has nothing to sweep
        int slot = 0;
        const int at = Q.k < 3 ? tri_resume(A, g, C, slot) : C;
        if (at >= 0) {
            if (Q.k < 3) q_restore<true>(A, g, Q, slot);
        } else {
            double fx, fy, fz;
            q_force(A, Q, fx, fy, fz);
            q_kick(A, Q, fx, fy, fz);
            const double dt = A.P.timeStep;
            Q.a.x += dt * Q.a.vx;
            Q.a.y += dt * Q.a.vy;
            Q.a.z += dt * Q.a.vz;
        }
        q_setup_r(A, B, g, Q);
        const double ddsq = q_ddsq(Q);
        double e;
        double l = q_lambda_r(B, Q, e);
        for (int it = max(at, 0); it < C; it++) {
            q_sweep<true>(A, Q, l);
            q_virial(Q, l, ddsq);
            l = q_lambda_r(B, Q, e);
        }
        // the state at C passes the check, unless a molecule re-diverged
        // after it was taken as settled
        if (Q.k < 3 && !(fabs(e) < Q.T.thr)) atomicOr(&A.ctrl[CTRL_SHAKE_ORDER], 1);
        // constraints in their order 0, 1, 2 (lanes 0, 2, 1)
        const double vm = q_sum3<QP_L0, QP_L2, QP_L1>(Q.vir);
        if (BATCH) {
            if (Q.k == 0) A.vir[g] = vm;   // per molecule, summed per replica
        } else if (Q.k == 0) {
            vblk = vm;
        }
        q_store(A, Q);
    }
    if (BATCH) return;
    double d2 = 0., rel = 0.;
    const bool track = A.track && A.ctrl[CTRL_PRUNE] == 1;
    if (A.slotWrite && Q.k < 3)
        tri_write_slot(A, Q.at, Q.a.x, Q.a.y, Q.a.z, track, d2, rel);
    tri_block_out(A, vblk, track, d2, rel);
}

// Stage 2, part A: half kick and SHAKE-V sweeps with the same bookkeeping.
//
// With fuse set (1 mixed, 2 FP64; one box), the kernel first assembles each
// atom's force as k_finalize does (fin_atom, mdg_side.h: the same
// arithmetic, so k_finalize is not launched), keeps the correction
// partials per block, and resets the stage-1 SHAKE mask for the next step
// (k_w3_vv1_b resets the stage-2 one).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_w3_vv2_a(ShakeArgs A, FinArgs F, int fuse)
{
    __shared__ double mean[3], red[4][3];
    double facc[2] = {0., 0.};
    if (!BATCH && fuse) {
        fin_mean(F, mean, red);
        if (blockIdx.x == 0 && threadIdx.x < SHK_MASKW) F.mask[threadIdx.x] = ~0ull;
    }
    const int g = shake_w3_group(A);
    const MdgBox &B = tri_box<BATCH>(A, BATCH ? min(g, A.nGrp - 1) : 0);
    Q3 Q;
    q_load(A, B, g, threadIdx.x & 3, Q);
    double fx, fy, fz;
    if (!BATCH && fuse) {
        fx = fy = fz = 0.;
        if (Q.k < 3) {
            const bool fr = fuse == 1 ? fin_atom<true>(F, Q.at, mean, facc, fx, fy, fz)
                                      : fin_atom<false>(F, Q.at, mean, facc, fx, fy, fz);
            if (fr) Q.a.vx = Q.a.vy = Q.a.vz = 0.;
        }
    } else {
        q_force(A, Q, fx, fy, fz);
    }
    q_kick(A, Q, fx, fy, fz);
    q_setup_v(A, Q);
    const double tolvel = A.P.tolShake * A.P.rTimeStep;
    TriBits bits;
    tri_bits_init(bits);
    const unsigned long long share = tri_share<BATCH>(A, g);
    TriRing ring;
    int it = 0;
    bool prev = false, settled = false;
    // the check is the sweep's own max |lambda| (shake.c:421); every sweep
    // that is not the last one checked is applied, because the reference's
    // global loop goes on while any group is unconverged
    for (;;) {
        const double l = q_lambda_v(Q);
        const bool bad = !(fabs(l) < tolvel);
        const bool cv = q_conv<BATCH>(__builtin_amdgcn_ballot_w64(bad));
        if (cv) bits.cur |= 1ull << (it & 63);
        if (ring.keep<BATCH>(tri_all<BATCH>(bad, share))) {
            q_save<false>(A, g, Q, ring.slot());
            ring.put(it);
        }
        settled = settled || (cv && prev);
        prev = cv;
        if (BATCH ? __builtin_amdgcn_ballot_w64(!settled) == 0 : settled) break;
        if (it + 1 >= A.P.maxCycle) break;
        q_sweep<false>(A, Q, l);
        if ((it & 63) == 63) tri_flush(bits, it >> 6);
        it++;
    }
    tri_flush(bits, it >> 6);
    if (Q.k == 0) {
        for (int q = 0; q < SHK_R; q++) A.ring[(long)SHK_R * g + q] = ring.saved[q];
    }
    tri_publish<BATCH>(A, g, bits, it, settled);
    if (!BATCH && fuse) mdg_block_partials<2>(facc, F.part);
}

// Stage 2, part B: on to the global sweep C (as stage 1), kinetic energy and stress
// partials (utils.c:502-515), wrap (utils.c:162-218).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_w3_vv2_b(ShakeArgs A)
{
#pragma clang fp contract(off)
    const int g = shake_w3_group(A);
    const int gb = BATCH ? min(g, A.nGrp - 1) : 0;
    const MdgBox &B = tri_box<BATCH>(A, gb);
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    Q3 Q;
    q_load(A, B, g, threadIdx.x & 3, Q);
    const int C = shake_global_stop(A, tri_mask<BATCH>(A, gb));
    if (C < 0) {
        if (Q.k == 0) atomicOr(&A.ctrl[CTRL_SHAKE_FAIL], 2);
    } else {
        int slot = 0;
        const int at = Q.k < 3 ? tri_resume(A, g, C, slot) : C;
        if (at >= 0) {
            if (Q.k < 3) q_restore<false>(A, g, Q, slot);
        } else {
            double fx, fy, fz;
            q_force(A, Q, fx, fy, fz);
            q_kick(A, Q, fx, fy, fz);
        }
        q_setup_v(A, Q);
        double l = q_lambda_v(Q);
        for (int it = max(at, 0); it < C; it++) {
            q_sweep<false>(A, Q, l);
            l = q_lambda_v(Q);
        }
        if (!(fabs(l) < A.P.tolShake * A.P.rTimeStep)) atomicOr(&A.ctrl[CTRL_SHAKE_ORDER], 1);
    }
    double ke = 0.;
    if (Q.k < 3) {
        const double m = A.mass[Q.at];
        const double vx = Q.a.vx, vy = Q.a.vy, vz = Q.a.vz;
        ke = m * (vx * vx + vy * vy + vz * vz);
        acc[0] = ke;
        acc[1] = m * vx * vx;
        acc[2] = m * vx * vy;
        acc[3] = m * vx * vz;
        acc[4] = m * vy * vy;
        acc[5] = m * vy * vz;
        acc[6] = m * vz * vz;
        shake_image(B, Q.a.x, Q.a.y, Q.a.z);
    }
    const double kin = q_sum3<QP_L0, QP_L1, QP_L2>(ke);   // the molecule's sum, in atom order
    q_store(A, Q);
    if (BATCH && Q.k == 0) A.grpKin[g] = kin;
    mdg_block_partials<7>(acc, A.part);
}

template __global__ void k_w3_vv1_a<false>(ShakeArgs, SideWork);
template __global__ void k_w3_vv1_a<true>(ShakeArgs, SideWork);
template __global__ void k_w3_vv1_b<false>(ShakeArgs);
template __global__ void k_w3_vv1_b<true>(ShakeArgs);
template __global__ void k_w3_vv2_a<false>(ShakeArgs, FinArgs, int);
template __global__ void k_w3_vv2_a<true>(ShakeArgs, FinArgs, int);
template __global__ void k_w3_vv2_b<false>(ShakeArgs);
template __global__ void k_w3_vv2_b<true>(ShakeArgs);
