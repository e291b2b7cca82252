// Host-side check of the cache kernel's addresses (sentinel_amd/csrc/cache_offsets.h): every scalar offset lies inside the head, and with
// loads past the end giving zeros every value that is used comes from its own row and position.  Plain C++.
#include "../../sentinel_amd/csrc/cache_offsets.h"

#include <cstdio>

using namespace sentinel_hip;

int main() {
    int failures = 0;
    for (int d : {8, 16, 24, 32, 40, 64, 72, 80, 96, 104, 120, 128})
        for (int stride = 1; stride <= 300; stride += stride < 140 ? 1 : 53)
            for (int row0 = 0; row0 < d; row0 += 16)
                for (int p0 = 0; p0 < stride; p0 += 64)
                    for (int i = 0; i < 4; ++i)
                        for (int lane = 0; lane < 64; ++lane) {
                            const unsigned size = (unsigned)d * (unsigned)stride;
                            const CacheOffset k = key_offset(row0, i, p0, lane, d, (unsigned)stride);
                            const CacheOffset v = value_offset(row0, i, p0, lane, d, (unsigned)stride);
                            if (k.scalar >= size || v.scalar >= size) ++failures;
                            if (row0 + 4 * i >= d && k.scalar + k.lane < size) ++failures;  // (zeros)
                            const int k_row = row0 + 4 * i + lane / 16, k_position = p0 + 4 * (lane % 16);
                            if (k_row < d && k_position < stride && k.scalar + k.lane != (unsigned)(k_row * stride + k_position)) ++failures;
                            const int v_row = row0 + lane % 16, v_position = p0 + 16 * i + 4 * (lane / 16);
                            if (v_row < d && v_position < stride && v.scalar + v.lane != (unsigned)(v_row * stride + v_position)) ++failures;
                        }
    std::printf(failures ? "%d failures\n" : "cache offsets ok\n", failures);
    return failures ? 1 : 0;
}
