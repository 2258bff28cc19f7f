// kg_copy.hip -- copies from device memory to the caller's host memory.
//
// The runtime copies to pageable memory through pages that it pins for the
// call (17 GB/s), and into an array that was just allocated takes most of its
// time in page faults (4.4 GB/s).  Here the DMA fills a pinned buffer (57 GB/s)
// in halves while the processor empties the other half, and the pages of the
// destination are asked for in one call instead of one fault each, during the
// DMA.  kg_get_phase into a new array / into one that was dropped before, us,
// the runtime's copy / this: 256 B 22 / 14, 64 kB 13 / 13 and 36 / 13, 1 MB
// 60 .. 220 / 61 .. 99 and 59 / 59, 4 MB 232 .. 680 / 206 .. 356 and 235 / 186,
// 16 MB 1650 / 1270 and 940 / 630, 64 MB 6590 / 4940.  (The other direction
// stays with the runtime: 37 GB/s, and 28 GB/s this way.)
//
// Pinned buffers are shared by all handles: at most STAGES of STAGE_MAX bytes
// (kg_stage.h), each held by one call at a time, all freed with the last
// handle.  A call that finds none, memory that the runtime knows (pinned,
// managed or device), and memory that the processor may not write copy
// directly.
#include <cstring>

#include "kg_host.h"
#include "kg_stage.h"

namespace kg {

namespace {

// Allocating is harmless to a capture that is under way elsewhere in this
// process, but the runtime refuses it in the default capture mode.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

StagePool g_stages(
    [](size_t cap) -> void * {
        const RelaxedCapture relaxed;
        void *p = nullptr;
        if (hipHostMalloc(&p, cap, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        return p;
    },
    [](void *p) {
        const RelaxedCapture relaxed;
        (void)hipHostFree(p);
    });

// Memory that the runtime does not know: pageable.
bool pageable(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

hipError_t copy_direct(hipStream_t s, const HostPiece *pieces, int count)
{
    for (int k = 0; k < count; ++k)
        if (hipError_t e = hipMemcpyAsync(pieces[k].host, pieces[k].dev, pieces[k].bytes,
                                          hipMemcpyDeviceToHost, s))
            return e;
    return hipStreamSynchronize(s);
}

hipError_t copy_staged(hipStream_t s, const HostPiece *pieces, int count, char *buf, size_t half)
{
    constexpr int PARTS = 32;
    struct Part {
        char *host;
        const char *from;
        size_t n;
    } parts[2][PARTS];
    int np[2] = {0, 0}, piece = 0;
    size_t o = 0;
    auto fill = [&](int h) -> hipError_t {
        np[h] = 0;
        for (size_t at = 0; piece < count && at < half && np[h] < PARTS;) {
            const HostPiece &p = pieces[piece];
            const size_t n = p.bytes - o < half - at ? p.bytes - o : half - at;
            char *b = buf + (size_t)h * half + at;
            if (hipError_t e = hipMemcpyAsync(b, static_cast<const char *>(p.dev) + o, n,
                                              hipMemcpyDeviceToHost, s))
                return e;
            parts[h][np[h]++] = Part{static_cast<char *>(p.host) + o, b, n};
            at += (n + 255) / 256 * 256;
            o += n;
            if (o == p.bytes) {
                o = 0;
                ++piece;
            }
        }
        return hipSuccess;
    };
    if (hipError_t e = fill(0))
        return e;
    for (int h = 0; np[h] > 0; h ^= 1) {
        bool ok = true;
        for (int k = 0; k < np[h]; ++k)
            ok = populate(parts[h][k].host, parts[h][k].n) && ok;
        if (hipError_t e = hipStreamSynchronize(s))
            return e;
        if (!ok)
            return copy_direct(s, pieces, count);  // the runtime's to copy or refuse
        if (hipError_t e = fill(h ^ 1))
            return e;
        for (int k = 0; k < np[h]; ++k)
            std::memcpy(parts[h][k].host, parts[h][k].from, parts[h][k].n);
    }
    return hipSuccess;
}

}  // namespace

hipError_t copy_to_host(hipStream_t s, const HostPiece *pieces, int count)
{
    size_t total = 0;
    bool staged = true;
    for (int k = 0; k < count; ++k) {
        total += (pieces[k].bytes + 255) / 256 * 256;
        staged = staged && pageable(pieces[k].host);
    }
    const int at = staged ? g_stages.take(total) : -1;
    if (at < 0)
        return copy_direct(s, pieces, count);
    const hipError_t e =
        copy_staged(s, pieces, count, g_stages.buffer(at), g_stages.capacity(at) / 2);
    if (e != hipSuccess)
        (void)hipStreamSynchronize(s);  // nothing writes to the buffer any more
    g_stages.give(at);
    return e;
}

void stages_retain() { g_stages.retain(); }
void stages_release() { g_stages.release(); }

}  // namespace kg
