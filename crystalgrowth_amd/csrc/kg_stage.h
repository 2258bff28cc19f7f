// kg_stage.h -- the pages that kg_copy.hip's copies go to.  No GPU call is made
// here.
#pragma once

#include <sys/mman.h>
#include <unistd.h>

#include <cstddef>
#include <cstdint>

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

}  // namespace kg
