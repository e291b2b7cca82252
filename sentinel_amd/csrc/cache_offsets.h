// Where the cache kernel (decode_attention.hip) reads one K/V head, fp32 [head_dim][stride]: wavefront w loads rows of head dims
// 16 w .., four positions per lane and load.  A load's address is a scalar offset plus the lane's.  The hardware takes the scalar offset
// off the head's size and checks the lane's against the rest: lanes may point past the end (and get zeros), a scalar offset may not, for
// no capacity however small.  Offsets in elements.  Plain C++ as grid_plan.h.
#ifndef SENTINEL_HIP_CACHE_OFFSETS_H
#define SENTINEL_HIP_CACHE_OFFSETS_H

#include "grid_plan.h"

namespace sentinel_hip {

struct CacheOffset {
    unsigned scalar, lane;
};

// K, load s (0 .. 3): positions p0 + 4 (lane % 16) .. + 3 of row 16 w + 4 s + lane / 16; row0 = 16 w < head_dim, p0 < stride.
// (head dims past the last: past the end)
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) CacheOffset key_offset(int row0, int s, int p0, int lane, int head_dim, unsigned stride) {
    if (row0 + 4 * s >= head_dim) return CacheOffset{(unsigned)row0 * stride + (unsigned)p0, (unsigned)head_dim * stride};
    return CacheOffset{(unsigned)(row0 + 4 * s) * stride + (unsigned)p0, (unsigned)(lane / 16) * stride + 4u * (unsigned)(lane % 16)};
}

// V, load x (0 .. 3): positions p0 + 16 x + 4 (lane / 16) .. + 3 of row 16 w + lane % 16 (past the last: the last)
SENTINEL_HIP_HOST_DEVICE inline __attribute__((always_inline)) CacheOffset value_offset(int row0, int x, int p0, int lane, int head_dim, unsigned stride) {
    const int more = lane % 16 < head_dim - 1 - row0 ? lane % 16 : head_dim - 1 - row0;
    return CacheOffset{(unsigned)row0 * stride + (unsigned)p0, (unsigned)more * stride + 4u * (unsigned)(lane / 16) + 16u * (unsigned)x};
}

}  // namespace sentinel_hip
#endif
