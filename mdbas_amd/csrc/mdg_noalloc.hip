// mdg_noalloc.hip -- mdg_nonbond_energy_noalloc: the cutoff nonbonded
// energy and forces (nonbond_energy, energy.c:216-345, the computation of
// mdg_nonbond_energy) for callers that cannot allocate device memory: code
// under HIP graph capture, tight serving loops, harnesses that forbid
// hipMalloc.  Every array is the caller's device memory; the list offsets,
// the packed atom records and the per-block partial sums live in one fixed
// file-scope device array (scratch) of MDG_NOALLOC_MAX_ATOMS atoms' worth.
//
// Each GPU holds its own copy of scratch until the process ends; its
// address on the current device is looked up once per device
// (hipGetSymbolAddress) and kept.  Calls that overlap on one GPU share that
// copy and race; calls on one stream, or otherwise ordered, do not.  Every
// word a call reads is written by that call first (the records and segment
// sums, then the offsets, the partials by each pair block), so nothing carries
// over from the previous call and nothing is cleared.
#include <mutex>

#include "mdg_internal.h"

namespace {
constexpr int MAX_ATOMS = MDG_NOALLOC_MAX_ATOMS;
constexpr int NV = 6;   // k_pair_ref64 partials per block
constexpr int MAX_BLOCKS = MAX_ATOMS / 32 + 256;   // mdg_ref64_blocks at every size
constexpr int SEG = 1024;   // list rows a block of the offset kernels scans
constexpr int MAX_SEG = (MAX_ATOMS + SEG - 1) / SEG;
// layout: list offsets (MAX_ATOMS + 1 longs), their segment sums (MAX_SEG
// longs), partials (MAX_BLOCKS x NV doubles), packed atom records
// (MAX_ATOMS x 64 bytes): 19 MB
constexpr size_t up256(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t OFF_BYTES = up256((size_t)(MAX_ATOMS + 1) * sizeof(long));
constexpr size_t SEG_BYTES = up256((size_t)MAX_SEG * sizeof(long));
constexpr size_t PART_BYTES = up256((size_t)MAX_BLOCKS * NV * sizeof(double));
constexpr size_t SCRATCH_BYTES = OFF_BYTES + SEG_BYTES + PART_BYTES +
                                 (size_t)MAX_ATOMS * sizeof(RefAtom);
}  // namespace

static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_mu;
void *g_ptr[MAX_DEVICES];

// The address of this device's scratch (host code never uses the symbol
// itself, which is a host-side stand-in).
void *scratch_ptr(int dev)
{
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_ptr[dev] = p;
    }
    return g_ptr[dev];
}

// Per block of SEG atoms: their packed records for the pair kernel, and the
// sum of the list rows at the block's positions.
__global__ void __launch_bounds__(SEG)
k_pack_sums(int n, const double *__restrict__ x, const double *__restrict__ y,
            const double *__restrict__ z, const double *__restrict__ q,
            const double *__restrict__ eps, const double *__restrict__ sig,
            RefAtom *__restrict__ at, const int *__restrict__ neighPair,
            const int *__restrict__ order, long *__restrict__ seg)
{
    __shared__ long red[SEG / 64];
    const int l = blockIdx.x * SEG + threadIdx.x;
    long v = 0;
    if (l < n) {
        at[l].r = make_double4(x[l], y[l], z[l], q[l]);
        at[l].s = make_double4(eps[l], sig[l], 0., 0.);
        v = neighPair[order[l]];
    }
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        long t = 0;
        for (int w = 0; w < SEG / 64; w++) t += red[w];
        seg[blockIdx.x] = t;
    }
}

// off[l + 1] = sum over m <= l of neighPair[order[m]], off[0] = 0: each block
// scans its SEG rows on top of the segment sums before it (at most MAX_SEG of
// them, added by every block).  One block scanning every row took 88 us at
// 30,000 atoms, its gathers one after the other.
__global__ void __launch_bounds__(SEG)
k_list_offsets(int n, const int *__restrict__ neighPair, const int *__restrict__ order,
               const long *__restrict__ seg, long *__restrict__ off)
{
    __shared__ long wsum[SEG / 64], base[SEG / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int l = blockIdx.x * SEG + threadIdx.x;
    long before = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += SEG) before += seg[b];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    long v = l < n ? neighPair[order[l]] : 0;
    for (int o = 1; o < 64; o <<= 1) {
        const long t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    if (lane == 63) wsum[wid] = v;
    if (lane == 0) base[wid] = before;
    __syncthreads();
    for (int w = 0; w < SEG / 64; w++) {
        v += base[w];
        if (w < wid) v += wsum[w];
    }
    if (l < n) off[l + 1] = v;
    if (l == 0) off[0] = 0;
}

// ener[0..3] += elec, vdw, virelec, virvdw: wavefront k sums column k of the
// partials in a fixed order, as the reference accumulates into ENERGY
// (energy.c:337-340).
__global__ void __launch_bounds__(256)
k_add_energies(const double *__restrict__ part, int rows, double *__restrict__ ener)
{
    const int k = threadIdx.x >> 6;
    double s = 0.;
    for (int r = threadIdx.x & 63; r < rows; r += 64) s += part[(long)r * NV + k];
    s = mdg_wave_sum(s);
    if ((threadIdx.x & 63) == 0) ener[k] += s;
}

}  // namespace

extern "C" int mdg_nonbond_energy_noalloc(const MDG_CTRL *ctrl, const MDG_PARAM *param,
                                          const MDG_PBC *box, const double *x, const double *y,
                                          const double *z, double *fx, double *fy, double *fz,
                                          const double *q, const double *eps, const double *sig,
                                          const int *neighList, const int *neighPair,
                                          const int *neighOrder, double *ener, void *stream)
{
    if (!ctrl || !param || !box || !x || !y || !z || !fx || !fy || !fz || !q || !eps || !sig ||
        !neighList || !neighPair || !neighOrder || !ener)
        return MDG_EARG;
    const int n = param->nAtom;
    if (n <= 0) return MDG_EARG;
    if (n > MAX_ATOMS) {
        fprintf(stderr,
                "mdg_nonbond_energy_noalloc: %d atoms exceed the fixed scratch of %d atoms\n", n,
                MAX_ATOMS);
        return MDG_ESCRATCH;
    }
    if (box->type < 1 || box->type > 3) return MDG_EUNSUPPORTED;
    // energy.c:45-65: NOELEC and FULL evaluate no electrostatics
    int et = ctrl->elecType;
    if (et == 0) et = 1;
    if (et < 1 || et > 4) return MDG_EUNSUPPORTED;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return MDG_EHIP;
    unsigned char *base = (unsigned char *)scratch_ptr(dev);
    if (!base) return MDG_EHIP;
    long *off = (long *)base;
    long *seg = (long *)(base + OFF_BYTES);
    double *part = (double *)(base + OFF_BYTES + SEG_BYTES);
    RefAtom *at = (RefAtom *)(base + OFF_BYTES + SEG_BYTES + PART_BYTES);
    MdgParams P;
    mdg_params_from(ctrl, param, P);
    MdgBox B;
    mdg_box_from(box, B);
    hipStream_t s = (hipStream_t)stream;
    const int ns = nblk(n, SEG);
    hipLaunchKernelGGL(k_pack_sums, dim3(ns), dim3(SEG), 0, s, n, x, y, z, q, eps, sig, at,
                       neighPair, neighOrder, seg);
    if (hipGetLastError() != hipSuccess) return MDG_EHIP;
    hipLaunchKernelGGL(k_list_offsets, dim3(ns), dim3(SEG), 0, s, n, neighPair, neighOrder, seg,
                       off);
    if (hipGetLastError() != hipSuccess) return MDG_EHIP;
    const int st = mdg_pair_ref64_launch(s, P, B, et, at, neighList, off, neighOrder, fx, fy, fz,
                                         part);
    if (st) return st;
    hipLaunchKernelGGL(k_add_energies, dim3(1), dim3(256), 0, s, part, mdg_ref64_blocks(n), ener);
    return hipGetLastError() == hipSuccess ? MDG_OK : MDG_EHIP;
}
