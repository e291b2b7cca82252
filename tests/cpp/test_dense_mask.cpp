// Host-side check of the dense path's mask (sentinel_amd/csrc/dense_mask.h) against the rule stated on positions inside a
// segment, with counts up to the largest int.  Plain C++.
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
    std::printf(failures ? "%d failures\n" : "dense mask ok\n", failures);
    return failures ? 1 : 0;
}
