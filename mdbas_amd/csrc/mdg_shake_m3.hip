// mdg_shake_m3.hip -- VV + SHAKE kernels for rigid three-site molecules
// with one molecule per lane (SHAKE spread 0).  Same molecules, stages, sweeps
// (mdg_shake_tri.h) and global stopping rule as mdg_shake_w3.hip, which holds
// one molecule per quad of lanes; here one lane holds the three atoms
// (a0 < a1 < a2) and the ring of constraints (0,1), (1,2), (2,0).
//
// A quad's sweep is one short dependent chain with the multipliers passing
// between its lanes; a lane's sweep has three such chains and no moves.  One
// molecule per lane takes a quarter of the wavefronts and about half the
// instructions per molecule, so it wins where the wavefronts fill the SIMDs,
// and the quads where they do not.  The results are the quad kernels' bit for
// bit.
#include "mdg_shake_tri.h"

namespace {

__device__ constexpr int M_N[3] = {1, 2, 0};   // the next atom / constraint
__device__ constexpr int M_P[3] = {2, 0, 1};   // the previous one

struct M3 {
    int at[3];
    TriAtom a[3];
    double rm[3], nat[3], f[3];
    double ddx[3], ddy[3], ddz[3];   // constraint vectors at the stage start
    TriR T[3];                       // stage 1
    double K[3], y[3];               // stage 2
    double vir[3];                   // virial sums
};

// The molecule of this lane, or nGrp for an idle lane.
__device__ inline int m_group(const ShakeArgs &A)
{
    const int g = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    return g < A.nGrp ? g : A.nGrp;
}

__device__ __forceinline__ void m_bond(const M3 &M, int c, double &dx, double &dy, double &dz)
{
    const TriAtom &a = M.a[c], &n = M.a[M_N[c]];
    dx = n.x - a.x;
    dy = n.y - a.y;
    dz = n.z - a.z;
}

__device__ inline void m_load(const ShakeArgs &A, const MdgBox &B, int g, M3 &M)
{
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int i = A.atoms[3 * g + k];
        M.at[k] = i;
        TriAtom &a = M.a[k];
        a.x = A.x[i];
        a.y = A.y[i];
        a.z = A.z[i];
        a.vx = A.vx[i];
        a.vy = A.vy[i];
        a.vz = A.vz[i];
        M.rm[k] = A.rmass[i];
        M.nat[k] = 1.0 / (double)A.nAtConst[i];
        M.vir[k] = 0.;
    }
#pragma unroll
    for (int c = 0; c < 3; c++) {
        m_bond(M, c, M.ddx[c], M.ddy[c], M.ddz[c]);
        mdg_dist(B, M.ddx[c], M.ddy[c], M.ddz[c]);
    }
}

__device__ inline void m_kick(const ShakeArgs &A, M3 &M, int k, double fx, double fy, double fz)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
    M.a[k].vx += 0.5 * dt * fx * M.rm[k];
    M.a[k].vy += 0.5 * dt * fy * M.rm[k];
    M.a[k].vz += 0.5 * dt * fz * M.rm[k];
}

__device__ inline void m_kick_stored(const ShakeArgs &A, M3 &M)
{
#pragma unroll
    for (int k = 0; k < 3; k++) m_kick(A, M, k, A.fx[M.at[k]], A.fy[M.at[k]], A.fz[M.at[k]]);
}

__device__ inline void m_drift(const ShakeArgs &A, M3 &M)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        M.a[k].x += dt * M.a[k].vx;
        M.a[k].y += dt * M.a[k].vy;
        M.a[k].z += dt * M.a[k].vz;
    }
}

__device__ inline void m_setup_r(const ShakeArgs &A, const MdgBox &B, int g, M3 &M)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int c = A.cons[3 * g + (k == 0 ? 0 : 3 - k)];
        M.T[k].rc2 = A.rc2[c];
        M.T[k].thr = A.thr[c];
        M.T[k].K = dt * (dt * M.rm[k] + dt * M.rm[M_N[k]]);
        M.f[k] = 0.5 * (dt * M.rm[k]) * M.nat[k];
        double dx, dy, dz;
        m_bond(M, k, dx, dy, dz);
        tri_shift(B, dx, dy, dz, M.T[k].sx, M.T[k].sy, M.T[k].sz);
    }
}

__device__ __forceinline__ double m_ddsq(const M3 &M, int k)
{
#pragma clang fp contract(off)
    return M.ddx[k] * M.ddx[k] + M.ddy[k] * M.ddy[k] + M.ddz[k] * M.ddz[k];
}

__device__ inline void m_setup_v(const ShakeArgs &A, M3 &M)
{
#pragma clang fp contract(off)
    const double dt = A.P.timeStep;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double tr = 0.5 * dt * M.rm[k], trn = 0.5 * dt * M.rm[M_N[k]];
        M.K[k] = (tr + trn) * m_ddsq(M, k);
        M.y[k] = 1.0 / M.K[k];
        M.f[k] = tr * M.nat[k];
    }
}

// Residuals and multipliers at the current positions; whether all three
// constraints are converged.
__device__ __forceinline__ bool m_lambda_r(const MdgBox &B, const M3 &M, double (&l)[3])
{
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        double dx, dy, dz, e;
        m_bond(M, k, dx, dy, dz);
        l[k] = tri_lambda(B, M.T[k], dx, dy, dz, M.ddx[k], M.ddy[k], M.ddz[k], e);
        ok = ok && fabs(e) < M.T[k].thr;
    }
    return ok;
}

__device__ __forceinline__ bool m_lambda_v(const M3 &M, double tolvel, double (&l)[3])
{
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const TriAtom &a = M.a[k], &n = M.a[M_N[k]];
        l[k] = tri_lambda_v(M.K[k], M.y[k], n.vx - a.vx, n.vy - a.vy, n.vz - a.vz, M.ddx[k],
                            M.ddy[k], M.ddz[k]);
        ok = ok && fabs(l[k]) < tolvel;
    }
    return ok;
}

template <bool POS>
__device__ __forceinline__ void m_sweep(const ShakeArgs &A, M3 &M, const double (&l)[3])
{
#pragma clang fp contract(off)
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int p = M_P[k];
        tri_move<POS>(M.a[k], A.P.timeStep, M.f[k], l[k], l[p], M.ddx[k], M.ddy[k], M.ddz[k],
                      M.ddx[p], M.ddy[p], M.ddz[p]);
        if (POS) M.vir[k] += l[k] * m_ddsq(M, k);
    }
}

// The state of a sweep at which the whole wavefront was converged (see q_save).
template <bool POS>
__device__ inline void m_save(const ShakeArgs &A, int g, const M3 &M, int slot)
{
    const long n = A.P.n;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        double *s = A.scr + (long)slot * 6 * n + M.at[k];
        if (POS) {
            s[0] = M.a[k].x;
            s[n] = M.a[k].y;
            s[2 * n] = M.a[k].z;
            A.virScr[((long)slot * A.nGrp + g) * 3 + k] = M.vir[k];
        }
        s[3 * n] = M.a[k].vx;
        s[4 * n] = M.a[k].vy;
        s[5 * n] = M.a[k].vz;
    }
}

template <bool POS>
__device__ inline void m_restore(const ShakeArgs &A, int g, M3 &M, int slot)
{
    const long n = A.P.n;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double *s = A.scr + (long)slot * 6 * n + M.at[k];
        if (POS) {
            M.a[k].x = s[0];
            M.a[k].y = s[n];
            M.a[k].z = s[2 * n];
            M.vir[k] = A.virScr[((long)slot * A.nGrp + g) * 3 + k];
        }
        M.a[k].vx = s[3 * n];
        M.a[k].vy = s[4 * n];
        M.a[k].vz = s[5 * n];
    }
}

__device__ inline void m_store(const ShakeArgs &A, const M3 &M)
{
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int i = M.at[k];
        A.x[i] = M.a[k].x;
        A.y[i] = M.a[k].y;
        A.z[i] = M.a[k].z;
        A.vx[i] = M.a[k].vx;
        A.vy[i] = M.a[k].vy;
        A.vz[i] = M.a[k].vz;
    }
}

}  // namespace

// Stage 1, part A (see k_w3_vv1_a).  Blocks past S.nbMain do the previous
// step's record and list prune (mdg_side.h).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_m3_vv1_a(ShakeArgs A, SideWork S)
{
    if ((int)blockIdx.x >= S.nbMain) {
        side_work<BATCH>(S);
        return;
    }
    const int g = m_group(A);
    const bool live = g < A.nGrp;
    TriBits bits;
    tri_bits_init(bits);
    int it = 0;
    bool prev = false, settled = !live;
    const MdgBox &B = tri_box<BATCH>(A, BATCH ? min(g, A.nGrp - 1) : 0);
    M3 M;
    if (live) {
        m_load(A, B, g, M);
        m_kick_stored(A, M);
        m_drift(A, M);
        m_setup_r(A, B, g, M);
    }
    const unsigned long long share = tri_share<BATCH>(A, g);
    TriRing ring;
    for (;;) {
        double l[3];
        const bool ok = live ? m_lambda_r(B, M, l) : true;
        const bool all = tri_all<BATCH>(!ok, share);
        // one system: the wavefront's molecules share a stopping sweep
        const bool cv = BATCH ? ok : all;
        if (cv) bits.cur |= 1ull << (it & 63);
        if (ring.keep<BATCH>(all)) {
            if (live) m_save<true>(A, g, M, ring.slot());
            ring.put(it);
        }
        settled = settled || (cv && prev);
        prev = cv;
        if (__builtin_amdgcn_ballot_w64(!settled) == 0) break;
        if (it + 1 >= A.P.maxCycle) break;
        if (live) m_sweep<true>(A, M, l);
        if ((it & 63) == 63) tri_flush(bits, it >> 6);
        it++;
    }
    tri_flush(bits, it >> 6);
    if (live) {
        for (int q = 0; q < SHK_R; q++) A.ring[(long)SHK_R * g + q] = ring.saved[q];
    }
    tri_publish<BATCH>(A, g, bits, it, settled);
}

// Stage 1, part B (see k_w3_vv1_b).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_m3_vv1_b(ShakeArgs A)
{
#pragma clang fp contract(off)
    // the stage-2 mask (beside this stage's) for this step's stage 2
    if (!BATCH && blockIdx.x == 0 && threadIdx.x < SHK_MASKW) A.mask[SHK_MASKW + threadIdx.x] = ~0ull;
    const int g = m_group(A);
    double vblk = 0.;   // this lane's molecule's SHAKE virial
    double d2 = 0., rel = 0.;
    const bool track = A.track && A.ctrl[CTRL_PRUNE] == 1;
    if (g < A.nGrp) {
        const MdgBox &B = tri_box<BATCH>(A, g);
        M3 M;
        m_load(A, B, g, M);
        const int C = shake_global_stop(A, tri_mask<BATCH>(A, g));
        if (C < 0) {
            atomicOr(&A.ctrl[CTRL_SHAKE_FAIL], 1);
        } else {
            int slot;
            const int at = tri_resume(A, g, C, slot);
            if (at >= 0) {
                m_restore<true>(A, g, M, slot);
            } else {
                m_kick_stored(A, M);
                m_drift(A, M);
            }
            m_setup_r(A, B, g, M);
            double l[3];
            bool ok = m_lambda_r(B, M, l);
            for (int it = max(at, 0); it < C; it++) {
                m_sweep<true>(A, M, l);
                ok = m_lambda_r(B, M, l);
            }
            if (!ok) atomicOr(&A.ctrl[CTRL_SHAKE_ORDER], 1);
            const double vm = (M.vir[0] + M.vir[2]) + M.vir[1];   // constraints 0, 1, 2
            if (BATCH) A.vir[g] = vm;   // per molecule, summed per replica
            else vblk = vm;
            m_store(A, M);
        }
        if (!BATCH && A.slotWrite) {
#pragma unroll
            for (int k = 0; k < 3; k++)
                tri_write_slot(A, M.at[k], M.a[k].x, M.a[k].y, M.a[k].z, track, d2, rel);
        }
    }
    if (!BATCH) tri_block_out(A, vblk, track, d2, rel);
}

// Stage 2, part A (see k_w3_vv2_a).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_m3_vv2_a(ShakeArgs A, FinArgs F, int fuse)
{
    __shared__ double mean[3], red[4][3];
    double facc[2] = {0., 0.};
    if (!BATCH && fuse) {
        fin_mean(F, mean, red);
        if (blockIdx.x == 0 && threadIdx.x < SHK_MASKW) F.mask[threadIdx.x] = ~0ull;
    }
    const int g = m_group(A);
    const bool live = g < A.nGrp;
    TriBits bits;
    tri_bits_init(bits);
    int it = 0;
    bool prev = false, settled = !live;
    const MdgBox &B = tri_box<BATCH>(A, BATCH ? min(g, A.nGrp - 1) : 0);
    M3 M;
    if (live) {
        m_load(A, B, g, M);
        if (!BATCH && fuse) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                double gx, gy, gz;
                const bool fr = fuse == 1 ? fin_atom<true>(F, M.at[k], mean, facc, gx, gy, gz)
                                          : fin_atom<false>(F, M.at[k], mean, facc, gx, gy, gz);
                if (fr) M.a[k].vx = M.a[k].vy = M.a[k].vz = 0.;
                m_kick(A, M, k, gx, gy, gz);
            }
        } else {
            m_kick_stored(A, M);
        }
        m_setup_v(A, M);
    }
    const double tolvel = A.P.tolShake * A.P.rTimeStep;
    const unsigned long long share = tri_share<BATCH>(A, g);
    TriRing ring;
    for (;;) {
        double l[3];
        const bool ok = live ? m_lambda_v(M, tolvel, l) : true;
        const bool all = tri_all<BATCH>(!ok, share);
        const bool cv = BATCH ? ok : all;
        if (cv) bits.cur |= 1ull << (it & 63);
        if (ring.keep<BATCH>(all)) {
            if (live) m_save<false>(A, g, M, ring.slot());
            ring.put(it);
        }
        settled = settled || (cv && prev);
        prev = cv;
        if (__builtin_amdgcn_ballot_w64(!settled) == 0) break;
        if (it + 1 >= A.P.maxCycle) break;
        if (live) m_sweep<false>(A, M, l);
        if ((it & 63) == 63) tri_flush(bits, it >> 6);
        it++;
    }
    tri_flush(bits, it >> 6);
    if (live) {
        for (int q = 0; q < SHK_R; q++) A.ring[(long)SHK_R * g + q] = ring.saved[q];
    }
    tri_publish<BATCH>(A, g, bits, it, settled);
    if (!BATCH && fuse) mdg_block_partials<2>(facc, F.part);
}

// Stage 2, part B: on to the global sweep C (as stage 1), kinetic energy and stress
// partials (utils.c:502-515), wrap (utils.c:162-218).
template <bool BATCH>
__global__ void __launch_bounds__(256) k_m3_vv2_b(ShakeArgs A)
{
#pragma clang fp contract(off)
    const int g = m_group(A);
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    if (g < A.nGrp) {
        const MdgBox &B = tri_box<BATCH>(A, g);
        M3 M;
        m_load(A, B, g, M);
        const int C = shake_global_stop(A, tri_mask<BATCH>(A, g));
        if (C < 0) {
            atomicOr(&A.ctrl[CTRL_SHAKE_FAIL], 2);
        } else {
            int slot;
            const int at = tri_resume(A, g, C, slot);
            if (at >= 0) m_restore<false>(A, g, M, slot);
            else m_kick_stored(A, M);
            m_setup_v(A, M);
            const double tolvel = A.P.tolShake * A.P.rTimeStep;
            double l[3];
            bool ok = m_lambda_v(M, tolvel, l);
            for (int it = max(at, 0); it < C; it++) {
                m_sweep<false>(A, M, l);
                ok = m_lambda_v(M, tolvel, l);
            }
            if (!ok) atomicOr(&A.ctrl[CTRL_SHAKE_ORDER], 1);
        }
        double ke[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const double m = A.mass[M.at[k]];
            const double vx = M.a[k].vx, vy = M.a[k].vy, vz = M.a[k].vz;
            ke[k] = m * (vx * vx + vy * vy + vz * vz);
            acc[0] += ke[k];
            acc[1] += m * vx * vx;
            acc[2] += m * vx * vy;
            acc[3] += m * vx * vz;
            acc[4] += m * vy * vy;
            acc[5] += m * vy * vz;
            acc[6] += m * vz * vz;
            shake_image(B, M.a[k].x, M.a[k].y, M.a[k].z);
        }
        m_store(A, M);
        if (BATCH) A.grpKin[g] = (ke[0] + ke[1]) + ke[2];   // the molecule's sum, in atom order
    }
    mdg_block_partials<7>(acc, A.part);
}

template __global__ void k_m3_vv1_a<false>(ShakeArgs, SideWork);
template __global__ void k_m3_vv1_a<true>(ShakeArgs, SideWork);
template __global__ void k_m3_vv1_b<false>(ShakeArgs);
template __global__ void k_m3_vv1_b<true>(ShakeArgs);
template __global__ void k_m3_vv2_a<false>(ShakeArgs, FinArgs, int);
template __global__ void k_m3_vv2_a<true>(ShakeArgs, FinArgs, int);
template __global__ void k_m3_vv2_b<false>(ShakeArgs);
template __global__ void k_m3_vv2_b<true>(ShakeArgs);
