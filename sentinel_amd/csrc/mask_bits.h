// Sentinel's sparse mask for one row of a 64-wide tile, as a word with one bit per element: bit c answers for key
// (query) `first + c`.  The kernels that meet the mask's edges form the word once per lane and tile and then spend two
// instructions per element (bit field extract, and) whatever edges the tile holds; comparing positions cost two for the
// diagonal and four more for the window and the global range, and kept the forward at head_dim 128 spilling.  B4 H32 T4096 d128,
// window 512: forward 242 -> 203 us (window 128: 168 -> 129), backward 700 -> 681; B8 H12 T1024 d64, window 200 with 16 global
// tokens: 26 -> 18 and 73 -> 60 us.  Plain C++ as grid_plan.h.
#ifndef SENTINEL_HIP_MASK_BITS_H
#define SENTINEL_HIP_MASK_BITS_H

#include "grid_plan.h"

namespace sentinel_hip {

// bits 0 .. n - 1 (none for n <= 0, all from 64 on)
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) unsigned long long low_bits(int n) {
    return n <= 0 ? 0ull : ~0ull >> (64 - (n < 64 ? n : 64));
}

// keys first .. first + 63 that `query` sees: none past itself, and of the others the global ones and the last `window`
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) unsigned long long visible_keys(int query, int first, int window,
                                                                                             int global_tokens) {
    return low_bits(query + 1 - first) & (low_bits(global_tokens - first) | ~low_bits(query - window + 1 - first));
}

// queries first .. first + 63 that see `key`
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) unsigned long long seeing_queries(int key, int first, int window,
                                                                                               int global_tokens) {
    return ~low_bits(key - first) & (key < global_tokens ? ~0ull : low_bits(key + window - first));
}

}  // namespace sentinel_hip
#endif
