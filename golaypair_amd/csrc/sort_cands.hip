// Device sort + uniq of candidate records in the byte order of their text lines
// (`sort | uniq` under LC_ALL=C, src/core/sort/sort.cpp:7-23, of the lines that
// src/utils/io.cpp:14-36 writes: "PSD" d_1 .. d_{n-1} " " v_0 " " .. v_{n-1} " ").
//
// Line order without the text.  Each record gets a fixed-width key of symbols,
// packed most significant first into W 64-bit words (the first in a column of its
// own, the others together per record):
//   3 (n - 1) text symbols of 4 bits: the key digits' decimal text with '0'..'9'
//       as 1..10, followed by zeros up to the full width;
//   n letter symbols of 8 bits: each letter's rank among all letters, ordered as
//       their token strings "v " compare bytewise.
// Comparing keys word by word compares the lines bytewise: where one key text
// is a proper prefix of the other, that line has ' ' (below every digit) where
// the other has a digit, as the zero symbol is below every digit symbol; with
// equal texts both lines continue with " " and then the tokens, which are
// prefix-free (each ends in its only space), so the lines compare as the
// sequences of the tokens' ranks.  Equal keys are equal lines.
//
// A call: keys, merge sort (runs and rounds), flags of the records that differ
// from their predecessor with their count per block, compaction.
//
// HBM traffic (algorithmic, 2 N R in the sense of one read and one write of
// each record; R = n + n/2 bytes here): the key build reads each record once
// and writes W words; each merge round reads and writes 12 B per record; the
// compaction reads and writes each kept record once.
#include <algorithm>

#include "gp_internal.hpp"
#include "gp_sort.hpp"

namespace gp {

// Rank of each letter (byte) among all 256 by its token string "v ".
struct LetterRanks {
    uint8_t r[256] = {};
    // token of v as a number that compares as its text does: up to five bytes, left aligned
    static constexpr uint64_t token(int v) {
        uint64_t t = 0;
        int len = 0;
        auto put = [&](int c) {
            t = t << 8 | (uint64_t)c;
            ++len;
        };
        int a = v;
        if (a < 0) {
            put('-');
            a = -a;
        }
        if (a >= 100) put('0' + a / 100);
        if (a >= 10) put('0' + a / 10 % 10);
        put('0' + a % 10);
        put(' ');
        return t << (8 * (5 - len));
    }
    constexpr LetterRanks() {
        uint64_t t[256] = {};
        for (int x = 0; x < 256; ++x) t[x] = token((int8_t)x);
        for (int x = 0; x < 256; ++x)
            for (int y = 0; y < x; ++y) ++r[t[x] < t[y] ? y : x];
    }
};
__device__ constexpr LetterRanks kLetterRanks{};

// One record per thread: the key words of record i, the first to first[i], the
// others to rest + i (W - 1).  The symbols of a word collect in a register.
__global__ void __launch_bounds__(256) k_cand_keys(const int8_t* __restrict__ words, const uint8_t* __restrict__ keys,
                                                   int64_t m, int n, int K, int W, uint64_t* __restrict__ first,
                                                   uint64_t* __restrict__ rest) {
    __shared__ uint8_t rank[256];
    rank[threadIdx.x] = kLetterRanks.r[threadIdx.x];
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    uint64_t cur = 0;
    int used = 0, w = 0;  // nibbles in cur, words written
    uint64_t* const r = rest + i * (W - 1) - 1;
    auto flush = [&]() {
        if (w == 0) first[i] = cur;
        else r[w] = cur;
        ++w;
        cur = 0;
        used = 0;
    };
    auto put = [&](uint32_t nibble) {
        cur = cur << 4 | nibble;
        if (++used == 16) flush();
    };
    const uint8_t* kd = keys + i * K;
    int nsym = 0;
    for (int k = 1; k < n; ++k) {
        const uint32_t d = kd[(k <= K ? k : n - k) - 1], h = d / 100u, t = d / 10u % 10u;
        if (d >= 100) put(h + 1);
        if (d >= 10) put(t + 1);
        put(d % 10u + 1);
        nsym += 1 + (d >= 10) + (d >= 100);
    }
    for (; nsym < 3 * (n - 1); ++nsym) put(0);
    const int8_t* wd = words + i * n;
    for (int p = 0; p < n; ++p) {
        const uint32_t x = rank[(uint8_t)wd[p]];
        put(x >> 4);
        put(x & 15);
    }
    if (used > 0) {
        cur <<= 4 * (16 - used);
        flush();
    }
}

// Sum of v over the block's 256 threads, in every thread; `part` is 4 words of LDS.
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* part) {
    for (int o = 32; o; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    return part[0] + part[1] + part[2] + part[3];
}

// flag[i] = 1 when sorted record i differs from record i - 1 (or i == 0), and
// the number of them in each block's `chunk` records.
__global__ void __launch_bounds__(256) k_sort_uniq(MergeSorted s, const uint64_t* __restrict__ rest, int nrest,
                                                   int64_t m, int64_t chunk, uint8_t* __restrict__ flag,
                                                   uint32_t* __restrict__ counts) {
    __shared__ uint32_t part[4];
    const int64_t end = min(((int64_t)blockIdx.x + 1) * chunk, m);
    uint32_t mine = 0;
    for (int64_t i = (int64_t)blockIdx.x * chunk + threadIdx.x; i < end; i += 256) {
        bool f = i == 0 || s.key[i] != s.key[i - 1];
        if (!f) {
            const uint64_t* a = rest + (int64_t)s.idx[i] * nrest;
            const uint64_t* b = rest + (int64_t)s.idx[i - 1] * nrest;
            for (int w = 0; w < nrest && !f; w += 4) {
                uint64_t x = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) x |= a[min(w + j, nrest - 1)] ^ b[min(w + j, nrest - 1)];
                f = x != 0;
            }
        }
        flag[i] = f;
        mine += f;
    }
    const uint32_t sum = block_sum(mine, part);
    if (threadIdx.x == 0) counts[blockIdx.x] = sum;
}

// The flagged records to their places, the sum of the blocks before plus the
// place in the block: 256 records at a time, their bytes written by consecutive
// threads.  counts[gridDim.x] is set to the number of records kept.
__global__ void __launch_bounds__(256) k_sort_compact(const int8_t* __restrict__ words,
                                                      const uint8_t* __restrict__ keys, int n, int K, int64_t m,
                                                      int64_t chunk, const uint32_t* __restrict__ idx,
                                                      const uint8_t* __restrict__ flag, uint32_t* counts,
                                                      int8_t* __restrict__ out_w, uint8_t* __restrict__ out_k) {
    __shared__ uint32_t part[4], src[256];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    uint32_t before = 0;
    for (int b = t; b < (int)blockIdx.x; b += 256) before += counts[b];
    uint32_t out = block_sum(before, part);
    const int64_t end = min(((int64_t)blockIdx.x + 1) * chunk, m);
    auto rows = [&](uint32_t cnt, int len, const auto* __restrict__ from, auto* __restrict__ to) {
        const uint32_t step_r = 256u / (uint32_t)len, step_c = 256u % (uint32_t)len;
        uint32_t r = (uint32_t)t / (uint32_t)len, c = (uint32_t)t % (uint32_t)len;
        for (uint32_t j = t; j < cnt * (uint32_t)len; j += 256) {
            to[(int64_t)out * len + j] = from[(int64_t)src[r] * len + c];
            r += step_r;
            c += step_c;
            if (c >= (uint32_t)len) {
                c -= (uint32_t)len;
                ++r;
            }
        }
    };
    for (int64_t i0 = (int64_t)blockIdx.x * chunk; i0 < end; i0 += 256) {
        const bool f = i0 + t < end && flag[i0 + t];
        const unsigned long long b = __ballot(f);
        __syncthreads();  // the reads of src and part of the records before are done
        if (lane == 0) part[wave] = (uint32_t)__popcll(b);
        __syncthreads();
        uint32_t at = (uint32_t)__popcll(b & ((1ull << lane) - 1ull)), cnt = 0;
        for (int w = 0; w < 4; ++w) {
            if (w < wave) at += part[w];
            cnt += part[w];
        }
        if (f) src[at] = idx[i0 + t];
        __syncthreads();
        rows(cnt, n, words, out_w);
        rows(cnt, K, keys, out_k);
        out += cnt;
    }
    if (t == 0 && blockIdx.x + 1 == gridDim.x) counts[gridDim.x] = out;
}

// Sorts and uniqs the m records (words n bytes, keys K bytes each) held in
// d_words / d_keys on the context's stream; writes the kept records in line
// order to d_out_words / d_out_keys and returns their number.
int64_t sort_uniq_cands(gp_ctx* ctx, const int8_t* d_words, const uint8_t* d_keys, int64_t m, int n, int K,
                        int8_t* d_out_words, uint8_t* d_out_keys) {
    if (m <= 0) return 0;
    if (m > 0xFFFFFFFFll) throw ArgError("gp_sort_candidates: more than 2^32 records");
    if (n < 2 || n > kMaxN || K != n / 2) throw ArgError("gp_sort_candidates: bad record shape");
    hipStream_t st = ctx->stream;
    const int W = (4 * 3 * (n - 1) + 8 * n + 63) / 64;
    uint64_t* first = ctx->dev<uint64_t>("s_first", (size_t)m);
    uint64_t* rest = ctx->dev<uint64_t>("s_rest", (size_t)(W - 1) * m + 1);
    hipLaunchKernelGGL(k_cand_keys, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, d_words, d_keys, m, n, K, W,
                       first, rest);
    GP_HIP(hipGetLastError());
    const MergeSorted s = merge_sort(ctx, "s_sort", first, m, rest, W - 1);
    // at most 2048 blocks, so that each can add up the counts of those before it
    const int64_t chunk = std::max<int64_t>(256, (m + 2047) / 2048);
    const unsigned blocks = (unsigned)((m + chunk - 1) / chunk);
    uint8_t* flag = ctx->dev<uint8_t>("s_flag", (size_t)m);
    uint32_t* counts = ctx->dev<uint32_t>("s_counts", (size_t)blocks + 1);
    hipLaunchKernelGGL(k_sort_uniq, dim3(blocks), dim3(256), 0, st, s, rest, W - 1, m, chunk, flag, counts);
    GP_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sort_compact, dim3(blocks), dim3(256), 0, st, d_words, d_keys, n, K, m, chunk, s.idx, flag,
                       counts, d_out_words, d_out_keys);
    GP_HIP(hipGetLastError());
    uint32_t kept = 0;
    GP_HIP(hipMemcpyAsync(&kept, counts + blocks, 4, hipMemcpyDeviceToHost, st));
    GP_HIP(hipStreamSynchronize(st));
    return (int64_t)kept;
}

}  // namespace gp
