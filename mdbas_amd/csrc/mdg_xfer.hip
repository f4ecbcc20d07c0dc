// mdg_xfer.hip -- host arrays to and from the device for the drop-in calls.
//
// A drop-in call moves a dozen arrays each way.  As copies from and to pageable
// memory each costs 10 to 15 us whatever its size, more than the kernels between
// them on an ordinary box.  Up to XFER_MAX bytes they go through one pinned
// buffer instead: the host packs it, and one kernel reads it over the bus and
// writes the arrays (back: one kernel writes it, the host unpacks).  Above that
// the host's packing (about 10 GB/s) costs more than the copies' overhead and
// each array is copied directly, as all were before.  3,000 atoms driven by the
// drop-in calls (two integrator stages and the energies a step, lists as due):
// 25.1 ms before, 12.4 ms for the same steps with this, with one wait per call
// and with an unchanged exclusion table left in place.
#include "mdg_internal.h"
#include <cstring>

#define XFER_MAX (1u << 20)

// Segments between device arrays and the pinned buffer, 16 bytes at a time and
// the rest by words; a segment without buffer offset (all ones) is zeroed.
template <bool IN>
__global__ void __launch_bounds__(256) k_xfer(MdgXferTab T, char *buf)
{
    const MdgXferSeg s = T.s[blockIdx.y];
    const unsigned i0 = blockIdx.x * 256 + threadIdx.x, st = gridDim.x * 256, nv = s.bytes / 16;
    char *dev = (char *)s.dev, *b = buf + s.off;
    const bool zero = s.off == ~0u;
    for (unsigned i = i0; i < nv; i += st) {
        if (IN) ((uint4 *)dev)[i] = zero ? uint4{0, 0, 0, 0} : ((const uint4 *)b)[i];
        else ((uint4 *)b)[i] = ((const uint4 *)dev)[i];
    }
    const unsigned w = 4 * nv + i0;
    if (w < s.bytes / 4) {
        if (IN) ((unsigned *)dev)[w] = zero ? 0 : ((const unsigned *)b)[w];
        else ((unsigned *)b)[w] = ((const unsigned *)dev)[w];
    }
}

void MdgXfer::add(void *dev, void *host, size_t bytes)
{
    if (n == MDG_XFER_SEGS) {
        full = true;
        return;
    }
    seg[n].dev = dev;
    seg[n].host = host;
    seg[n].bytes = bytes;
    seg[n].off = total;
    n++;
    if (host || !in) total += (bytes + 15) & ~(size_t)15;
}

int MdgXfer::check(mdg_ctx *ctx) const
{
    if (full) {
        ctx->err = "too many arrays in one transfer";
        return MDG_EARG;
    }
    if (missing) {
        ctx->err = "a host array of the call is missing";
        return MDG_EARG;
    }
    return MDG_OK;
}

// Whether the segments go through the pinned buffer (else directly).
int MdgXfer::prepare(mdg_ctx *ctx)
{
    RETCHK(check(ctx));
    packed = total <= XFER_MAX;
    for (int k = 0; k < n; k++)
        if (((uintptr_t)seg[k].dev & 15) || (seg[k].bytes & 3) || seg[k].bytes > XFER_MAX)
            packed = false;
    if (!packed) return MDG_OK;
    char *&b = in ? ctx->xferUp : ctx->xferDown;
    if (!b) HIPCHK(hipHostMalloc((void **)&b, XFER_MAX, hipHostMallocDefault));
    buf = b;
    return MDG_OK;
}

int MdgXfer::launch(mdg_ctx *ctx)
{
    MdgXferTab T;
    size_t mx = 0;
    for (int k = 0; k < n; k++) {
        T.s[k].dev = seg[k].dev;
        T.s[k].off = in && !seg[k].host ? ~0u : (unsigned)seg[k].off;
        T.s[k].bytes = (unsigned)seg[k].bytes;
        mx = std::max(mx, seg[k].bytes);
    }
    const dim3 g(std::min(nblk((long)mx, 256 * 16) + 1, 64), n);
    if (in) hipLaunchKernelGGL(k_xfer<true>, g, dim3(256), 0, ctx->stream, T, buf);
    else hipLaunchKernelGGL(k_xfer<false>, g, dim3(256), 0, ctx->stream, T, buf);
    LAUNCHCHK();
    return MDG_OK;
}

// Host arrays (and cleared ones) to the device, in stream order; the host arrays
// are free again when it returns.
int MdgXfer::up(mdg_ctx *ctx)
{
    if (n == 0) return MDG_OK;
    RETCHK(prepare(ctx));
    if (packed) {
        // an earlier transfer that no fetch has waited for may still be reading
        if (ctx->xferBusy) HIPCHK(hipStreamSynchronize(ctx->stream));
        for (int k = 0; k < n; k++)
            if (seg[k].host) std::memcpy(buf + seg[k].off, seg[k].host, seg[k].bytes);
        RETCHK(launch(ctx));
        ctx->xferBusy = true;
        return MDG_OK;
    }
    for (int k = 0; k < n; k++) {
        if (!seg[k].bytes) continue;
        if (seg[k].host)
            HIPCHK(hipMemcpyAsync(seg[k].dev, seg[k].host, seg[k].bytes, hipMemcpyHostToDevice,
                                  ctx->stream));
        else
            HIPCHK(hipMemsetAsync(seg[k].dev, 0, seg[k].bytes, ctx->stream));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDG_OK;
}

// Waits for the stream with the first nfirst segments delivered; deliver() then
// fills the others (which a failed call leaves untouched).
int MdgXfer::fetch(mdg_ctx *ctx, int nfirst)
{
    first = nfirst;
    RETCHK(prepare(ctx));
    if (packed && n > 0) {
        RETCHK(launch(ctx));
    } else {
        for (int k = 0; k < first; k++)
            HIPCHK(hipMemcpyAsync(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost,
                                  ctx->stream));
    }
    HIPCHK(hipStreamSynchronize(ctx->stream));
    ctx->xferBusy = false;
    if (packed)
        for (int k = 0; k < first; k++) std::memcpy(seg[k].host, buf + seg[k].off, seg[k].bytes);
    return MDG_OK;
}

int MdgXfer::deliver(mdg_ctx *ctx)
{
    for (int k = first; k < n; k++) {
        if (packed) std::memcpy(seg[k].host, buf + seg[k].off, seg[k].bytes);
        else
            HIPCHK(hipMemcpyAsync(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost,
                                  ctx->stream));
    }
    if (!packed) HIPCHK(hipStreamSynchronize(ctx->stream));
    return MDG_OK;
}

void mdg_xfer_free(mdg_ctx *ctx)
{
    if (ctx->xferUp) (void)hipHostFree(ctx->xferUp);
    if (ctx->xferDown) (void)hipHostFree(ctx->xferDown);
    ctx->xferUp = ctx->xferDown = nullptr;
}
