// Device sort of records by long keys, and the candidate join of match.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

struct gp_ctx;
struct gp_stats;

namespace gp {

// Records in sorted order: first key words and record numbers, in buffers of the
// context that the next sort of the same name uses again.
struct MergeSorted {
    const uint64_t* key;
    const uint32_t* idx;
};
// Key words of a sort as they turn out on the device: `words` of each record (the
// first one and the rest), of which all records share those before the last `live`.
struct MergeShape {
    uint32_t words, live;
};
// Sorts n records on the context's stream by keys[i], then by the nrest words at
// rest + i * nrest, then by i.  With `shape` (device memory, words <= nrest + 1) the rest
// words lie at rest + i * (words - 1), and the shared ones are passed over: the sorted
// keys are the words that come first after them.
MergeSorted merge_sort(gp_ctx* ctx, const std::string& name, const uint64_t* keys, int64_t n,
                       const uint64_t* rest = nullptr, int nrest = 0, const MergeShape* shape = nullptr);

// Sort + uniq of m candidate records (int8 words of n, uint8 keys of K = n/2)
// held on the device, in the byte order of their text lines; the kept records
// go to out_words / out_keys (not aliasing the inputs).  Returns their number.
int64_t sort_uniq_cands(gp_ctx* ctx, const int8_t* d_words, const uint8_t* d_keys, int64_t m, int n, int K,
                        int8_t* d_out_words, uint8_t* d_out_keys);

// Join of two candidate sets on equal key tuples (nkey bytes per record,
// row stride kstride) followed by the exact integer PAF check
//   PAF_a(s) + PAF_b(s) == paf_target  for s = 1..n/2   (golay.cpp:27-44).
// Words are int8 rows of stride wstride.  Returns the accepted (ia, ib)
// index pairs sorted lexicographically.  All pointers are device memory.
struct JoinResult {
    std::vector<uint32_t> ia, ib;
    uint64_t checks = 0;
};
JoinResult join_pairs(gp_ctx* ctx, const int8_t* d_wa, const uint8_t* d_ka, int64_t na, const int8_t* d_wb,
                      const uint8_t* d_kb, int64_t nb, int n, int nkey, int wstride, int kstride, int paf_target,
                      gp_stats* stats);

}  // namespace gp
