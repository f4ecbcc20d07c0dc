// mdg_conv64.hip -- FP64 convolution of a charge mesh with the influence
// function (spme.c:505-592: forward transform, multiplication, inverse
// transform) in three launches, for meshes whose planes fit in LDS.
//
// On the meshes of small and ordinary boxes a step's FP64 SPME is a chain of
// short dependent kernels, and what it costs is their number: a general
// transform takes two or three launches each way, with the multiplication
// between them.  Here each x plane is transformed along z and y inside one
// block's LDS (k_conv_fwd), the x columns are transformed, multiplied and
// transformed back without leaving LDS (k_conv_mid), and the planes return
// (k_conv_inv).  The transforms are Stockham passes of radix 2, 3, 4, 5 and 8
// over LDS, one butterfly per lane; a real row is transformed as half as many
// complex values (even and odd elements), which needs m3 even.
//
// Bound by the latency of the passes (each an LDS round trip and a barrier; the
// data is a few hundred KB): 6, 8 and 6 us a launch at 20^3 beside 4 to 5 us for
// each of five to eight launches before.  Microseconds per FP64 step against
// rocFFT and the separate multiplication: 20^3 114 : 118, 32^3 142 : 141, 48^3
// 216 : 220 (3,645 flexible atoms), 60^3 344 : 358, 80^3 575 : 577, and a
// trajectory gradient on 32^3 21.8 : 22.1 ms.  At 80^3 the two meet (80 planes
// no longer outweigh the launches), so larger planes stay with rocFFT, and so do
// odd m3 and lengths with other primes.
#include "mdg_internal.h"
#include <cmath>
#include <vector>

#define TWOPI 6.283185307179586     // global.h:53
#define CONV_COLS 8              // x columns per block: 128-byte rows of the half spectrum
#define CONV_LDS (110 * 1024)    // both buffers of a plane: up to 80 x 80

__device__ __forceinline__ unsigned conv_div(unsigned t, unsigned d, unsigned m)
{
    return d == 1 ? t : __umulhi(t, m);
}

__device__ __forceinline__ double2 c_add(double2 a, double2 b) { return {a.x + b.x, a.y + b.y}; }
__device__ __forceinline__ double2 c_sub(double2 a, double2 b) { return {a.x - b.x, a.y - b.y}; }
__device__ __forceinline__ double2 c_mul(double2 a, double2 b)
{
    return {__builtin_fma(a.x, b.x, -a.y * b.y), __builtin_fma(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ double2 c_mni(double2 a) { return {a.y, -a.x}; }   // -i a

__device__ __forceinline__ void dft2(double2 *v)
{
    const double2 a = v[0];
    v[0] = c_add(a, v[1]);
    v[1] = c_sub(a, v[1]);
}

__device__ __forceinline__ void dft3(double2 *v)
{
    const double s = 0.86602540378443864676;   // sin(2 pi / 3)
    const double2 t = c_add(v[1], v[2]), d = c_sub(v[1], v[2]);
    const double2 c = {__builtin_fma(-0.5, t.x, v[0].x), __builtin_fma(-0.5, t.y, v[0].y)};
    v[0] = c_add(v[0], t);
    v[1] = {__builtin_fma(s, d.y, c.x), __builtin_fma(-s, d.x, c.y)};
    v[2] = {__builtin_fma(-s, d.y, c.x), __builtin_fma(s, d.x, c.y)};
}

__device__ __forceinline__ void dft4(double2 *v)
{
    const double2 a = c_add(v[0], v[2]), b = c_sub(v[0], v[2]);
    const double2 c = c_add(v[1], v[3]), d = c_mni(c_sub(v[1], v[3]));
    v[0] = c_add(a, c);
    v[1] = c_add(b, d);
    v[2] = c_sub(a, c);
    v[3] = c_sub(b, d);
}

__device__ __forceinline__ void dft5(double2 *v)
{
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;   // cos(2 pi k / 5)
    const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;    // sin(2 pi k / 5)
    const double2 p = c_add(v[1], v[4]), m = c_sub(v[1], v[4]);
    const double2 q = c_add(v[2], v[3]), n = c_sub(v[2], v[3]);
    const double2 a = {__builtin_fma(c2, q.x, __builtin_fma(c1, p.x, v[0].x)),
                       __builtin_fma(c2, q.y, __builtin_fma(c1, p.y, v[0].y))};
    const double2 b = {__builtin_fma(c1, q.x, __builtin_fma(c2, p.x, v[0].x)),
                       __builtin_fma(c1, q.y, __builtin_fma(c2, p.y, v[0].y))};
    const double2 e = c_mni({__builtin_fma(s2, n.x, s1 * m.x), __builtin_fma(s2, n.y, s1 * m.y)});
    const double2 f = c_mni({__builtin_fma(-s1, n.x, s2 * m.x), __builtin_fma(-s1, n.y, s2 * m.y)});
    v[0] = c_add(v[0], c_add(p, q));
    v[1] = c_add(a, e);
    v[4] = c_sub(a, e);
    v[2] = c_add(b, f);
    v[3] = c_sub(b, f);
}

__device__ __forceinline__ void dft8(double2 *v)
{
    const double h = 0.70710678118654752440;   // sqrt(1/2)
    double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft4(e);
    dft4(o);
    o[1] = {h * (o[1].x + o[1].y), h * (o[1].y - o[1].x)};
    o[2] = c_mni(o[2]);
    o[3] = {h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y)};
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = c_add(e[k], o[k]);
        v[k + 4] = c_sub(e[k], o[k]);
    }
}

// One pass of radix R over nfft transforms of length A.n: element i of transform
// f lies at f * fs + i * es.  With the transforms adjacent (fs = 1) they run
// fastest over the lanes, else the butterflies of a transform do.  tw holds
// exp(-2 pi i k / (A.n * ts)), so A.n's own roots are ts apart.
template <int R>
__device__ __forceinline__ void conv_pass(const double2 *src, double2 *dst, const double2 *tw,
                                          int ts, int n, int L, unsigned mL, unsigned mT, int nfft,
                                          unsigned mF, int fs, int es)
{
    const unsigned nt = n / R;
    const int step = (int)(nt / L) * ts;   // A.n / (L R), in table entries
    for (unsigned b = threadIdx.x; b < nfft * nt; b += blockDim.x) {
        unsigned f, t;
        if (fs == 1) {
            t = conv_div(b, nfft, mF);
            f = b - t * nfft;
        } else {
            f = conv_div(b, nt, mT);
            t = b - f * nt;
        }
        const unsigned jL = conv_div(t, L, mL), k = t - jL * L;
        const double2 *s = src + f * fs + t * es;
        double2 v[R];
#pragma unroll
        for (int q = 0; q < R; q++) v[q] = s[q * (int)nt * es];
        if (L > 1) {
#pragma unroll
            for (int q = 1; q < R; q++) v[q] = c_mul(v[q], tw[q * (int)k * step]);
        }
        if (R == 2) dft2(v);
        else if (R == 3) dft3(v);
        else if (R == 4) dft4(v);
        else if (R == 5) dft5(v);
        else dft8(v);
        double2 *d = dst + f * fs + (jL * L * R + k) * es;
#pragma unroll
        for (int q = 0; q < R; q++) d[q * L * es] = v[q];
    }
    __syncthreads();
}

// All passes of one axis; a and b swap after each, a ends with the result.
__device__ __forceinline__ void conv_fft(const ConvAxis &A, double2 *&a, double2 *&b,
                                         const double2 *tw, int ts, int nfft, unsigned mF, int fs,
                                         int es)
{
    int L = 1;
    for (int p = 0; p < A.np; p++) {
        const int r = A.r[p];
        switch (r) {
        case 2: conv_pass<2>(a, b, tw, ts, A.n, L, A.mL[p], A.mT[p], nfft, mF, fs, es); break;
        case 3: conv_pass<3>(a, b, tw, ts, A.n, L, A.mL[p], A.mT[p], nfft, mF, fs, es); break;
        case 4: conv_pass<4>(a, b, tw, ts, A.n, L, A.mL[p], A.mT[p], nfft, mF, fs, es); break;
        case 5: conv_pass<5>(a, b, tw, ts, A.n, L, A.mL[p], A.mT[p], nfft, mF, fs, es); break;
        default: conv_pass<8>(a, b, tw, ts, A.n, L, A.mL[p], A.mT[p], nfft, mF, fs, es);
        }
        double2 *t = a;
        a = b;
        b = t;
        L *= r;
    }
}

// One x plane: real rows along z to half spectra, then columns along y.  Also
// clears the spreading's bucket counts (nbins of them; none if null).
__global__ void __launch_bounds__(512)
k_conv_fwd(ConvPlan C, const double2 *__restrict__ tw, const double *__restrict__ grid,
           double2 *__restrict__ cg, long nbins, int *__restrict__ binCnt,
           int *__restrict__ binNOut)
{
    extern __shared__ double2 sm[];
    const int m2 = C.y.n, mh = C.mh, nz = C.z.n, plane = m2 * mh;
    double2 *a = sm, *b = sm + plane, *t2 = b + plane, *t3 = t2 + m2;
    if (binCnt) {
        for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < nbins;
             i += (long)gridDim.x * blockDim.x)
            binCnt[i] = 0;
        if (blockIdx.x == 0 && threadIdx.x == 0) binNOut[0] = 0;
    }
    for (int i = threadIdx.x; i < m2; i += blockDim.x) t2[i] = tw[C.x.n + i];
    for (int i = threadIdx.x; i < 2 * nz; i += blockDim.x) t3[i] = tw[C.x.n + m2 + i];
    const double2 *g = (const double2 *)grid + (long)blockIdx.x * m2 * nz;
    for (unsigned i = threadIdx.x; i < (unsigned)(m2 * nz); i += blockDim.x) {
        const unsigned j = conv_div(i, nz, C.mNz);
        a[j * mh + (i - j * nz)] = g[i];
    }
    __syncthreads();
    conv_fft(C.z, a, b, t3, 2, m2, 0, mh, 1);
    // X[k] = (Z[k] + conj Z[-k]) / 2 - i/2 exp(-2 pi i k / m3) (Z[k] - conj Z[-k])
    for (unsigned i = threadIdx.x; i < (unsigned)plane; i += blockDim.x) {
        const unsigned j = conv_div(i, mh, C.mMh), k = i - j * mh;
        const double2 *row = a + j * mh;
        const double2 z = row[k == (unsigned)nz ? 0 : k], w = row[k == 0 ? 0 : nz - k];
        const double2 e = {0.5 * (z.x + w.x), 0.5 * (z.y - w.y)};
        const double2 o = {0.5 * (z.y + w.y), 0.5 * (w.x - z.x)};
        const double2 p = k == (unsigned)nz ? double2{-o.x, -o.y} : c_mul(t3[k], o);
        b[i] = c_add(e, p);
    }
    __syncthreads();
    double2 *t = a;
    a = b;
    b = t;
    conv_fft(C.y, a, b, t2, 1, mh, C.mMh, 1, mh);
    double2 *o = cg + (long)blockIdx.x * plane;
    for (int i = threadIdx.x; i < plane; i += blockDim.x) o[i] = a[i];
}

// CONV_COLS x columns: transform, multiply by the influence function, transform
// back (as a forward transform of the exchanged parts).  SUMS: per block
// [sum theta |F|^2, st0..st5] with full-spectrum weights, as k_spme_influence.
template <bool SUMS>
__global__ void __launch_bounds__(128)
k_conv_mid(ConvPlan C, MdgBox B, double rAlpha2, const double2 *__restrict__ tw,
           const double *__restrict__ theta, double2 *__restrict__ cg, double *__restrict__ part)
{
    extern __shared__ double2 sm[];
    const int m1 = C.x.n, m2 = C.y.n, m3 = 2 * C.z.n, mh = C.mh, plane = m2 * mh;
    double2 *a = sm, *b = sm + m1 * CONV_COLS, *t1 = b + m1 * CONV_COLS;
    double *ths = (double *)(t1 + m1);   // the columns' influence function, loaded ahead
    for (int i = threadIdx.x; i < m1; i += blockDim.x) t1[i] = tw[i];
    // the lane's column: blockDim is a multiple of CONV_COLS
    const int c = threadIdx.x % CONV_COLS, col = blockIdx.x * CONV_COLS + c;
    const bool in = col < plane;
    for (int i = threadIdx.x; i < m1 * CONV_COLS; i += blockDim.x) {
        const long g = (long)(i / CONV_COLS) * plane + col;
        a[i] = in ? cg[g] : double2{0., 0.};
        ths[i] = in ? theta[g] : 0.;
    }
    __syncthreads();
    conv_fft(C.x, a, b, t1, 1, CONV_COLS, C.mCols, 1, CONV_COLS);
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    const int j = (int)conv_div(col, mh, C.mMh), k = col - j * mh;
    const int jj = j > m2 / 2 ? j - m2 : j, kk = k > m3 / 2 ? k - m3 : k;
    const double t2 = TWOPI * jj, t3 = TWOPI * kk;
    const double wt = (k == 0 || 2 * k == m3) ? 1.0 : 2.0;
    for (int i = threadIdx.x; i < m1 * CONV_COLS; i += blockDim.x) {
        const int ix = i / CONV_COLS;
        const double th = ths[i];
        const double2 v = a[i];
        if (SUMS && th != 0.) {
            const double e = th * (v.x * v.x + v.y * v.y);
            // spme.c:509-547 reciprocal vector for (i, j, k)
            const double t1d = TWOPI * (ix > m1 / 2 ? ix - m1 : ix);
            const double rx = t1d * B.u1 + t2 * B.v1 + t3 * B.w1;
            const double ry = t1d * B.u2 + t2 * B.v2 + t3 * B.w2;
            const double rz = t1d * B.u3 + t2 * B.v3 + t3 * B.w3;
            const double rm = rx * rx + ry * ry + rz * rz;
            const double vam = -wt * 2.0 * (1.0 / rm - rAlpha2) * e;
            acc[0] += wt * e;
            acc[1] += vam * rx * rx;
            acc[2] += vam * rx * ry;
            acc[3] += vam * rx * rz;
            acc[4] += vam * ry * ry;
            acc[5] += vam * ry * rz;
            acc[6] += vam * rz * rz;
        }
        a[i] = {v.y * th, v.x * th};
    }
    __syncthreads();
    conv_fft(C.x, a, b, t1, 1, CONV_COLS, C.mCols, 1, CONV_COLS);
    for (int i = threadIdx.x; i < m1 * CONV_COLS; i += blockDim.x)
        if (in) cg[(long)(i / CONV_COLS) * plane + col] = {a[i].y, a[i].x};
    if (SUMS) mdg_block_partials<7>(acc, part);
}

// One x plane back: columns along y, then half spectra to real rows along z
// (not normalised; both as forward transforms of the exchanged parts).
__global__ void __launch_bounds__(512)
k_conv_inv(ConvPlan C, const double2 *__restrict__ tw, const double2 *__restrict__ cg,
           double *__restrict__ grid)
{
    extern __shared__ double2 sm[];
    const int m2 = C.y.n, mh = C.mh, nz = C.z.n, plane = m2 * mh;
    double2 *a = sm, *b = sm + plane, *t2 = b + plane, *t3 = t2 + m2;
    for (int i = threadIdx.x; i < m2; i += blockDim.x) t2[i] = tw[C.x.n + i];
    for (int i = threadIdx.x; i < 2 * nz; i += blockDim.x) t3[i] = tw[C.x.n + m2 + i];
    const double2 *p = cg + (long)blockIdx.x * plane;
    for (int i = threadIdx.x; i < plane; i += blockDim.x) a[i] = {p[i].y, p[i].x};
    __syncthreads();
    conv_fft(C.y, a, b, t2, 1, mh, C.mMh, 1, mh);
    // Z[k] = X[k] + conj X[nz-k] + i exp(2 pi i k / m3) (X[k] - conj X[nz-k]);
    // X[0] and X[nz] of a real mesh are real.  In a triclinic box the influence
    // function differs between a point with an index m/2 and its negative, and their
    // imaginary parts do not cancel: they belong to the imaginary part of the mesh,
    // which the reference's complex transform carries and never reads
    // (spme.c:593-646), so they are left out
    for (unsigned i = threadIdx.x; i < (unsigned)(m2 * nz); i += blockDim.x) {
        const unsigned j = conv_div(i, nz, C.mNz), k = i - j * nz;
        const double2 u = a[j * mh + k], w = a[j * mh + nz - k];
        const double2 x = {u.y, k ? u.x : 0.}, y = {w.y, k ? -w.x : 0.};   // X[k], conj X[nz-k]
        const double2 s = c_add(x, y), d = c_sub(x, y);
        const double2 e = {t3[k].x, -t3[k].y};
        const double2 o = c_mul(e, {-d.y, d.x});
        b[j * mh + k] = {s.y + o.y, s.x + o.x};
    }
    __syncthreads();
    double2 *t = a;
    a = b;
    b = t;
    conv_fft(C.z, a, b, t3, 2, m2, 0, mh, 1);
    double2 *g = (double2 *)grid + (long)blockIdx.x * m2 * nz;
    for (unsigned i = threadIdx.x; i < (unsigned)(m2 * nz); i += blockDim.x) {
        const unsigned j = conv_div(i, nz, C.mNz);
        const double2 v = a[j * mh + (i - j * nz)];
        g[i] = {v.y, v.x};
    }
}

// ---------------------------------------------------------------- host side

static unsigned magic(unsigned d) { return d > 1 ? (unsigned)((1ull << 32) / d + 1) : 0; }

// Passes of one axis: false if n has a prime factor above 5 or needs too many.
static bool plan_axis(int n, ConvAxis &A)
{
    A.n = n;
    A.np = 0;
    int m = n, a2 = 0;
    std::vector<int> r;
    while (m % 2 == 0) {
        m /= 2;
        a2++;
    }
    if (a2 % 3 == 1) {
        if (a2 == 1) r.push_back(2), a2 = 0;
        else r.push_back(4), r.push_back(4), a2 -= 4;
    } else if (a2 % 3 == 2) r.push_back(4), a2 -= 2;
    for (; a2 > 0; a2 -= 3) r.push_back(8);
    for (; m % 3 == 0; m /= 3) r.push_back(3);
    for (; m % 5 == 0; m /= 5) r.push_back(5);
    if (m != 1 || r.empty() || r.size() > CONV_PASSES) return false;
    int L = 1;
    for (int q : r) {
        A.r[A.np] = q;
        A.mL[A.np] = magic(L);
        A.mT[A.np] = magic(n / q);
        L *= q;
        A.np++;
    }
    return true;
}

static size_t plane_lds(const ConvPlan &C)
{
    return (2 * (size_t)C.y.n * C.mh + C.y.n + 2 * C.z.n) * sizeof(double2);
}

static size_t mid_lds(int m1)
{
    return (size_t)m1 * ((2 * CONV_COLS + 1) * sizeof(double2) + CONV_COLS * sizeof(double));
}

// Plans the convolution for m3 even, no prime factor above 5 and planes up to
// CONV_LDS (see above); other meshes take rocFFT.
int mdg_conv64_setup(mdg_ctx *ctx)
{
    ConvPlan &C = ctx->conv;
    const int m1 = ctx->m1, m2 = ctx->m2, m3 = ctx->m3;
    ctx->convOn = false;
    if (m3 % 2 || m3 < 4 || !plan_axis(m1, C.x) || !plan_axis(m2, C.y) || !plan_axis(m3 / 2, C.z))
        return MDG_OK;
    C.mh = m3 / 2 + 1;
    C.mMh = magic(C.mh);
    C.mNz = magic(C.z.n);
    C.mCols = magic(CONV_COLS);
    if (plane_lds(C) > CONV_LDS || mid_lds(m1) > 60 * 1024)
        return MDG_OK;
    for (const void *k : {(const void *)k_conv_fwd, (const void *)k_conv_inv})
        HIPCHK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, CONV_LDS));
    std::vector<double2> tw;
    for (int m : {m1, m2, m3})
        for (int i = 0; i < m; i++) {
            const long double w = 2.0L * 3.14159265358979323846264338327950288L * i / m;
            tw.push_back({(double)cosl(w), (double)-sinl(w)});
        }
    HIPCHK(hipMalloc(&ctx->convTw, tw.size() * sizeof(double2)));
    HIPCHK(hipMemcpy(ctx->convTw, tw.data(), tw.size() * sizeof(double2), hipMemcpyHostToDevice));
    ctx->convOn = true;
    return MDG_OK;
}

int mdg_conv64_rows(const mdg_ctx *ctx)
{
    return nblk((long)ctx->m2 * ctx->mh, CONV_COLS);
}

// grid <- theta * grid (not normalised), through cgrid64; part (may be null):
// mdg_conv64_rows rows of 7 partial sums.  clearBins: the spreading's bucket
// counts are cleared on the way.
int mdg_conv64(mdg_ctx *ctx, double *grid, double *part, bool clearBins)
{
    const ConvPlan &C = ctx->conv;
    const double2 *tw = (const double2 *)ctx->convTw;
    double2 *cg = (double2 *)ctx->cgrid64;
    const size_t lds = plane_lds(C), ldsMid = mid_lds(ctx->m1);
    const int nb = mdg_conv64_rows(ctx);
    const double rAlpha2 = -0.25 / (ctx->P.alpha * ctx->P.alpha);
    hipLaunchKernelGGL(k_conv_fwd, dim3(ctx->m1), dim3(512), lds, ctx->stream, C, tw, grid, cg,
                       clearBins ? (long)ctx->nbx * ctx->nby * ctx->nbz : 0L,
                       clearBins ? ctx->binCnt : nullptr, ctx->binNOut);
    LAUNCHCHK();
    hipLaunchKernelGGL(part ? k_conv_mid<true> : k_conv_mid<false>, dim3(nb), dim3(128), ldsMid,
                       ctx->stream, C, ctx->B, rAlpha2, tw, ctx->theta, cg, part);
    LAUNCHCHK();
    hipLaunchKernelGGL(k_conv_inv, dim3(ctx->m1), dim3(512), lds, ctx->stream, C, tw, cg, grid);
    LAUNCHCHK();
    return MDG_OK;
}
