// The dense path's mask for one query column, and where its kernels (dense_softmax.hip) find a column's elements.  Plain C++ as
// grid_plan.h.
#ifndef SENTINEL_HIP_DENSE_MASK_H
#define SENTINEL_HIP_DENSE_MASK_H

#include "grid_plan.h"

namespace sentinel_hip {

// CudaOps::runApplySparseAttentionMaskInPlace's predicate (CudaOps.cu:257-283) for one query: keys [lo, hi] that lie before
// global_end or from window_lo on
struct AllowedKeys {
    int lo, hi, global_end, window_lo;
    SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) AllowedKeys(int query, int query_position_start, int window, int global_tokens,
                                                                              int segment_length) {
        const int base = segment_length > 0 ? query / segment_length * segment_length : 0;
        const int position = segment_length > 0 ? query - base : query_position_start + query;
        lo = base;
        hi = base + position;
        // (keys past hi do not count: the end of a later segment's global keys need not go further, whatever number of them is asked for)
        global_end = base == 0 ? global_tokens : global_tokens <= position ? base + global_tokens : hi + 1;
        window_lo = window > 0 ? hi - window + 1 : lo;
    }
    SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) bool operator()(int key) const {
        return key <= hi && key >= lo && (key < global_end || key >= window_lo);
    }
};
// No key of [first, first + count) is allowed to any query between the two (whose AllowedKeys both grow with the query)
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) bool none_allowed(const AllowedKeys& first_query, const AllowedKeys& last_query, int first,
                                                                                int count) {
    const int end = first + count - 1;
    return first > last_query.hi || end < first_query.lo || (end < first_query.window_lo && first >= last_query.global_end);
}

// Byte offset of element (key, query) of a keys x queries matrix of fewer than 2^31 bytes; past the end for keys and queries past the
// last (the offset such a key would have may wrap around: one to three keys and 1.5e8 queries)
constexpr int kDeadElement = 0x7ffffff0;
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) int element_offset(int key, int query, int key_count, int query_count) {
    return key < key_count && query < query_count ? (key * query_count + query) * 4 : kDeadElement;
}

}  // namespace sentinel_hip
#endif
