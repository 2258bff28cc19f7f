// kg_stage.h -- host memory of kg_copy.hip's copies: the pool of buffers they
// go through, and the pages they go to.  No GPU call is made here: the pool's
// memory comes from the two functions it is given.
#pragma once

#include <sys/mman.h>
#include <unistd.h>

#include <cstddef>
#include <cstdint>
#include <mutex>

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

namespace kg {

// Pages of [p, p + n) present and writable.  false: they cannot be (an
// unmapped range, a read-only or PROT_NONE mapping, one of a device), or the
// kernel has no such call (before Linux 5.14) -- a processor's store may fault.
inline bool populate(void *p, size_t n)
{
    static const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
    const uintptr_t lo = (uintptr_t)p & ~(page - 1);
    return madvise((void *)lo, (uintptr_t)p + n - lo, MADV_POPULATE_WRITE) == 0;
}

// At most STAGES buffers of up to STAGE_MAX bytes, each held by one call at a
// time.  A buffer is allocated and freed by the call that holds it, outside
// the lock: freeing pinned memory may wait for the GPU, and a call that has
// its buffer need not.
class StagePool {
  public:
    static constexpr int STAGES = 8;
    static constexpr size_t STAGE_MIN = (size_t)512 << 10, STAGE_MAX = (size_t)4 << 20;
    // The first buffer costs some 13 us, a small copy through it saves 8: it is
    // made for a copy of this size, or the fourth.
    static constexpr size_t WORTH_A_STAGE = (size_t)256 << 10;
    static constexpr int WORTH_COPIES = 4;

    using Alloc = void *(*)(size_t);  // null: no memory
    using Release = void (*)(void *);
    StagePool(Alloc alloc, Release release) : alloc_(alloc), release_(release) {}

    // A free buffer, of twice `bytes` if that is within the limits; -1: none.
    int take(size_t bytes)
    {
        size_t cap = STAGE_MIN;
        while (cap < 2 * bytes && cap < STAGE_MAX)
            cap *= 2;
        int at = -1;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (int k = 0; k < STAGES; ++k) {
                const Stage &g = stages_[k];
                if (g.used)
                    continue;
                if (g.cap >= cap) {
                    at = k;
                    break;
                }
                if (at < 0 || g.cap > stages_[at].cap)
                    at = k;  // the largest too small (or empty) one grows
            }
            if (at < 0)
                return -1;
            const size_t have = stages_[at].cap;
            if (have == 0 && bytes < WORTH_A_STAGE && ++copies_ < WORTH_COPIES)
                return -1;
            stages_[at].used = true;
            if (have >= cap)
                return at;
        }
        // this call's alone until it is given back
        Stage &g = stages_[at];
        if (g.p)
            release_(g.p);
        g.p = static_cast<char *>(alloc_(cap));
        std::lock_guard<std::mutex> lock(mutex_);
        g.cap = g.p ? cap : 0;
        g.used = g.p != nullptr;
        return g.p ? at : -1;
    }

    void give(int at)
    {
        std::lock_guard<std::mutex> lock(mutex_);
        stages_[at].used = false;
    }

    char *buffer(int at) const { return stages_[at].p; }
    size_t capacity(int at) const { return stages_[at].cap; }

    // The pool lives while any handle does: the last one frees the buffers.
    void retain()
    {
        std::lock_guard<std::mutex> lock(mutex_);
        ++handles_;
    }
    void release()
    {
        std::lock_guard<std::mutex> lock(mutex_);
        if (--handles_ > 0)
            return;
        for (Stage &g : stages_) {
            if (g.p)
                release_(g.p);
            g = Stage{};
        }
        copies_ = 0;
    }

  private:
    struct Stage {
        char *p = nullptr;
        size_t cap = 0;
        bool used = false;
    };
    const Alloc alloc_;
    const Release release_;
    std::mutex mutex_;
    Stage stages_[STAGES];
    int handles_ = 0, copies_ = 0;
};

}  // namespace kg
