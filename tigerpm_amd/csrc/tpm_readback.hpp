// tpm_readback.hpp -- which destinations of a download one kernel may write
// (host code only, no HIP dependency).
#pragma once

#include <cstdint>

// One destination array as the runtime describes it.
struct tpm_readback_dst {
    int bytes;      // of an entry
    bool host;      // its first byte is page-locked host memory with a device address
    uintptr_t dev;  // that address
    uintptr_t base; // the allocation that holds it, in device addresses
    uint64_t size;
};

// Whether one kernel may write the n entries of all arrays: each lies in one
// page-locked allocation from its first byte to its last (two allocations may
// have pageable memory between them, which a kernel cannot write), is aligned
// to its entries, and no two overlap (copies made one after the other leave
// the last array's entries, a kernel a mixture).
inline bool tpm_readback_direct(const tpm_readback_dst* d, int count, int64_t n) {
    for (int k = 0; k < count; k++) {
        const uint64_t len = (uint64_t)d[k].bytes * (uint64_t)n;
        if (!d[k].host || d[k].dev % (uintptr_t)d[k].bytes) return false;
        if (d[k].dev < d[k].base || len > d[k].size || d[k].dev - d[k].base > d[k].size - len) return false;
        for (int j = 0; j < k; j++)
            if (d[j].dev < d[k].dev + len && d[k].dev < d[j].dev + (uint64_t)d[j].bytes * (uint64_t)n) return false;
    }
    return true;
}
