// Host-side check of the dense path's mask (sentinel_amd/csrc/dense_mask.h) against the rule stated on positions inside a
// segment, with counts up to the largest int, and of its elements' offsets.  Plain C++.
#include "../../sentinel_amd/csrc/dense_mask.h"

#include <cstdio>

using namespace sentinel_hip;

static bool allowed_pair(long long key, long long query, long long start, long long window, long long global_tokens, long long segment) {
    long long key_position = key, query_position = start + query;
    if (segment > 0) {
        if (key / segment != query / segment) return false;
        key_position = key % segment;
        query_position = query % segment;
    }
    return key_position <= query_position && (key_position < global_tokens || window <= 0 || key_position >= query_position - window + 1);
}

int main() {
    constexpr int kMost = 0x7fffffff, kKeys = 80, kQueries = 80;
    int failures = 0;
    for (int segment : {0, 1, 7, 32, 33, 70, kMost})
        for (int window : {0, 1, 5, 40, kMost})
            for (int global_tokens : {0, 1, 9, 64, kMost - 70, kMost})
                for (int start : {0, 40}) {
                    for (int query = 0; query < kQueries; ++query) {
                        const AllowedKeys allowed(query, start, window, global_tokens, segment);
                        for (int key = 0; key < kKeys; ++key)
                            if (allowed(key) != allowed_pair(key, query, start, window, global_tokens, segment)) ++failures;
                    }
                    // a group of keys is left out for a group of queries only if none of its pairs is allowed
                    for (int query0 = 0; query0 < kQueries; query0 += 32) {
                        const int last = query0 + 31 < kQueries ? query0 + 31 : kQueries - 1;
                        const AllowedKeys first_query(query0, start, window, global_tokens, segment), last_query(last, start, window, global_tokens, segment);
                        for (int key0 = 0; key0 < kKeys; key0 += 8) {
                            if (!none_allowed(first_query, last_query, key0, 8)) continue;
                            for (int key = key0; key < key0 + 8; ++key)
                                for (int query = query0; query <= last; ++query) failures += allowed_pair(key, query, start, window, global_tokens, segment);
                        }
                    }
                }
    // an element's own offset, or one past the end of the largest matrix the kernels take, for every key a workgroup has a thread for
    for (int key_count : {1, 2, 3, 4, 31, 33, 1024}) {
        const int most = (kDeadElement - 1) / 4 / key_count;
        for (int query_count : {1, 33, most / 2, most - 1, most})
            for (int key = 0; key < 32; ++key)
                for (long long query : {0ll, 1ll, query_count - 1ll, (long long)query_count, query_count + 31ll}) {
                    const unsigned offset = (unsigned)element_offset(key, (int)query, key_count, query_count);
                    const bool inside = key < key_count && query < query_count;
                    if (inside ? offset != (unsigned long long)(key * (long long)query_count + query) * 4 : offset < (unsigned long long)key_count * query_count * 4)
                        ++failures;
                }
    }
    std::printf(failures ? "%d failures\n" : "dense mask ok\n", failures);
    return failures ? 1 : 0;
}
