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
// Pinned buffers are shared by all handles: at most STAGES of STAGE_MAX bytes,
// each held by one call at a time, all freed with the last handle.  A call that
// finds none, memory that the runtime knows (pinned, managed or device), and
// memory that the processor may not write copy directly.
#include <cstring>
#include <mutex>

#include "kg_host.h"
#include "kg_stage.h"

namespace kg {

namespace {

constexpr int STAGES = 8;
constexpr size_t STAGE_MIN = (size_t)512 << 10, STAGE_MAX = (size_t)4 << 20;
// The first buffer costs some 13 us, a small copy through it saves 8: it is
// made for a copy of this size, or the fourth.
constexpr size_t WORTH_A_STAGE = (size_t)256 << 10;
constexpr int WORTH_COPIES = 4;

std::mutex g_mutex;
struct Stage {
    char *p;
    size_t cap;
    bool used;
} g_stages[STAGES];
int g_handles = 0, g_copies = 0;

// Allocating is harmless to a capture that is under way elsewhere in this
// process, but the runtime refuses it in the default capture mode.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// A free buffer, of twice `bytes` if that is within the limits; -1: none.
int take_stage(size_t bytes)
{
    size_t cap = STAGE_MIN;
    while (cap < 2 * bytes && cap < STAGE_MAX)
        cap *= 2;
    std::lock_guard<std::mutex> lock(g_mutex);
    int at = -1;
    for (int k = 0; k < STAGES; ++k) {
        const Stage &g = g_stages[k];
        if (g.used)
            continue;
        if (g.cap >= cap) {
            at = k;
            break;
        }
        if (at < 0 || g.cap > g_stages[at].cap)
            at = k;  // the largest too small (or empty) one grows
    }
    if (at < 0)
        return -1;
    Stage &g = g_stages[at];
    if (g.cap < cap) {
        if (g.cap == 0 && bytes < WORTH_A_STAGE && ++g_copies < WORTH_COPIES)
            return -1;
        const RelaxedCapture relaxed;
        if (g.p)
            (void)hipHostFree(g.p);
        g = Stage{nullptr, 0, false};
        void *p = nullptr;
        if (hipHostMalloc(&p, cap, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            return -1;
        }
        g = Stage{static_cast<char *>(p), cap, false};
    }
    g.used = true;
    return at;
}

void give_stage(int at)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    g_stages[at].used = false;
}

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
    const int at = staged ? take_stage(total) : -1;
    if (at < 0)
        return copy_direct(s, pieces, count);
    const hipError_t e = copy_staged(s, pieces, count, g_stages[at].p, g_stages[at].cap / 2);
    if (e != hipSuccess)
        (void)hipStreamSynchronize(s);  // nothing writes to the buffer any more
    give_stage(at);
    return e;
}

void stages_retain()
{
    std::lock_guard<std::mutex> lock(g_mutex);
    ++g_handles;
}

void stages_release()
{
    std::lock_guard<std::mutex> lock(g_mutex);
    if (--g_handles > 0)
        return;
    const RelaxedCapture relaxed;
    for (Stage &g : g_stages) {
        if (g.p)
            (void)hipHostFree(g.p);
        g = Stage{nullptr, 0, false};
    }
    g_copies = 0;
}

}  // namespace kg
