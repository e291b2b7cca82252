// Host-side check of the sparse mask's bit words (sentinel_amd/csrc/mask_bits.h) against the mask rule itself.  Plain C++.
#include "../../sentinel_amd/csrc/mask_bits.h"

#include <cstdio>

using namespace sentinel_hip;

// the layer's rule (Layers/CausalSelfAttention.cpp:95-100)
static bool allows(int query, int key, int window, int global_tokens) {
    return key <= query && (key < global_tokens || query - key < window);
}

int main() {
    int failures = 0;
    const int seq_len = 200;
    for (int window : {1, 2, 31, 63, 64, 65, 128, 150, 199})
        for (int global_tokens : {0, 1, 30, 63, 64, 65, 130, 200})
            for (int row = 0; row < seq_len; ++row)
                for (int first = 0; first < seq_len; first += 64) {
                    const unsigned long long keys = visible_keys(row, first, window, global_tokens);
                    const unsigned long long queries = seeing_queries(row, first, window, global_tokens);
                    for (int c = 0; c < 64; ++c) {
                        if ((keys >> c & 1) != allows(row, first + c, window, global_tokens)) ++failures;
                        if ((queries >> c & 1) != allows(first + c, row, window, global_tokens)) ++failures;
                    }
                }
    // the largest positions a call can have
    const int last = 0x7fffffff - 64;
    if (visible_keys(last, 0, last, last) != ~0ull || visible_keys(last, 0, 1, 0) != 0) ++failures;
    if (seeing_queries(0, last, 1, 1) != ~0ull || seeing_queries(0, last, 1, 0) != 0) ++failures;
    std::printf(failures ? "%d failures\n" : "mask bits ok\n", failures);
    return failures ? 1 : 0;
}
