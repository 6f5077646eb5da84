// Device sort + uniq of candidate records in the byte order of their text lines
// (`sort | uniq` under LC_ALL=C, src/core/sort/sort.cpp:7-23, of the lines that
// src/utils/io.cpp:14-36 writes: "PSD" d_1 .. d_{n-1} " " v_0 " " .. v_{n-1} " ").
//
// Line order without the text.  Each record gets a fixed-width key of symbols,
// packed most significant first into 64-bit words (the first in a column of its
// own, the others together per record):
//   3 (n - 1) text symbols of 4 bits: the key digits' decimal text with '0'..'9'
//       as 1..10, followed by zeros up to the full width;
//   n letter symbols of 8 bits: each letter's rank among all letters, ordered as
//       their token strings "v " compare bytewise (of many records: its rank among the
//       letters that occur, in as many bits as their number needs).
// Comparing keys word by word compares the lines bytewise: where one key text
// is a proper prefix of the other, that line has ' ' (below every digit) where
// the other has a digit, as the zero symbol is below every digit symbol; with
// equal texts both lines continue with " " and then the tokens, which are
// prefix-free (each ends in its only space), so the lines compare as the
// sequences of the tokens' ranks.  Equal keys are equal lines.
//
// A call: keys, merge sort (runs and rounds), flags of the records that differ from
// their predecessor with their count per block, compaction.
//
// Comparing records whose first words are equal reads their other words, at random, in
// every round.  Words before the first one in which some record differs from record 0 are
// passed over, so that records that share their digits, or are all the same, cost no more
// than others: 61000 equal records of 50 letters take 355 us (1200 with all words, 435
// with a radix sort of the varying bytes).  Beyond 2^18 records the letters' few bits also
// let one word decide between records that share their digits: 4e6 records of 15 letters
// 5.3 ms (13.9 and 9.7 ms).  (One record apart from 4e6 that share their digits still
// costs what no shared words do.)
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

// What the keys of a call have in common: the letters that occur, by their ranks among
// all 256 (bit by bit), and the shape of the key words.
struct SortCtl {
    unsigned long long present[4];
    MergeShape shape;
};

// Letters that occur among `count` bytes.
__global__ void __launch_bounds__(256) k_sort_letters(const int8_t* __restrict__ words, int64_t count, SortCtl* ctl) {
    __shared__ unsigned long long bits[4];
    if (threadIdx.x < 4) bits[threadIdx.x] = 0;
    __syncthreads();
    unsigned long long small = 0;  // letters v = bit - 32
    auto take = [&](int v) {
        if ((unsigned)(v + 32) < 64u) {
            small |= 1ull << (v + 32);
        } else {
            const uint32_t r = kLetterRanks.r[(uint8_t)v];
            atomicOr(&bits[r >> 6], 1ull << (r & 63));
        }
    };
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
    for (int64_t i = t; i < count / 16; i += step) {  // (allocations are aligned)
        const uint4 x = reinterpret_cast<const uint4*>(words)[i];
        for (const uint32_t y : {x.x, x.y, x.z, x.w}) {
            take((int8_t)y);
            take((int8_t)(y >> 8));
            take((int8_t)(y >> 16));
            take((int8_t)(y >> 24));
        }
    }
    for (int64_t i = count / 16 * 16 + t; i < count; i += step) take(words[i]);
    for (int o = 32; o; o >>= 1) small |= __shfl_xor(small, o);
    if ((threadIdx.x & 63) == 0)
        for (; small; small &= small - 1) {
            const uint32_t r = kLetterRanks.r[(uint8_t)(__ffsll((long long)small) - 33)];
            atomicOr(&bits[r >> 6], 1ull << (r & 63));
        }
    __syncthreads();
    if (threadIdx.x < 4 && bits[threadIdx.x]) {
        unsigned long long* p = &ctl->present[threadIdx.x];
        const unsigned long long b = bits[threadIdx.x];
        if ((__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & b) != b) atomicOr(p, b);
    }
}

// Records beyond which sort_letters runs: it costs 12 us at 61000 records, of 290.
constexpr int64_t kSortDense = 1 << 18;

// One record per thread: the key words of record i, the first to first[i], the
// others to rest + i (words - 1).  The symbols of a word collect in a register; the
// records' bytes come through LDS, the digits' text from a table: 10.3 us for 61000
// records (11.1 with bytes read in place and decimals made by division).
template <bool DENSE>
__global__ void __launch_bounds__(256) k_cand_keys(const int8_t* __restrict__ words, const uint8_t* __restrict__ keys,
                                                   int64_t m, int n, int K, SortCtl* ctl, uint64_t* __restrict__ first,
                                                   uint64_t* __restrict__ rest) {
    __shared__ uint8_t rank[256], ref[kMaxN + kMaxN / 2];
    __shared__ uint16_t digits[256];  // the text of a key digit: its symbols, and their bits << 12
    __shared__ uint4 rows[256 * (kMaxN + kMaxN / 2) / 16];  // the block's words, then its keys
    const int64_t i0 = (int64_t)blockIdx.x * 256, i = i0 + threadIdx.x;
    const int held = (int)min<int64_t>(256, m - i0), nw = (held * n + 15) / 16, nk = (held * K + 15) / 16;
    for (int x = threadIdx.x; x < nw + nk; x += 256)  // (i0 n and i0 K are multiples of 16; allocations have slack)
        rows[x] = x < nw ? reinterpret_cast<const uint4*>(words + i0 * n)[x]
                         : reinterpret_cast<const uint4*>(keys + i0 * K)[x - nw];
    if ((int)threadIdx.x < n + K) ref[threadIdx.x] = (int)threadIdx.x < n ? (uint8_t)words[threadIdx.x] : keys[threadIdx.x - n];
    {
        const uint32_t d = threadIdx.x, t = d / 10u;
        digits[d] = (uint16_t)(d < 10 ? 4u << 12 | (d + 1)
                               : d < 100 ? 8u << 12 | (t + 1) << 4 | (d % 10u + 1)
                                         : 12u << 12 | (d / 100u + 1) << 8 | (t % 10u + 1) << 4 | (d % 10u + 1));
    }
    int lbits = 8;
    if (DENSE) {
        const int r = kLetterRanks.r[threadIdx.x];
        int letters = 0, below = 0;
        for (int w = 0; w < 4; ++w) {
            const unsigned long long b = ctl->present[w];
            letters += __popcll(b);
            below += __popcll(w < r >> 6 ? b : w == r >> 6 ? b & ((1ull << (r & 63)) - 1ull) : 0ull);
        }
        rank[threadIdx.x] = (uint8_t)below;
        lbits = letters > 1 ? 32 - __clz(letters - 1) : 1;
    } else {
        rank[threadIdx.x] = kLetterRanks.r[threadIdx.x];
    }
    __syncthreads();
    const int text = 4 * 3 * (n - 1), W = (text + n * lbits + 63) / 64;
    if (i == 0) ctl->shape.words = (uint32_t)W;
    int differ = 64 * W;  // first bit of the symbol in which the record differs from record 0
    if (i < m) {
        uint64_t cur = 0;
        int used = 0, w = 0;  // bits in cur, words written
        uint64_t* const r = rest + i * (W - 1) - 1;
        auto flush = [&]() {
            if (w == 0) first[i] = cur;
            else r[w] = cur;
            ++w;
            cur = 0;
            used = 0;
        };
        auto put = [&](uint32_t x, int bits) {  // 0 < bits <= 12
            const int over = used + bits - 64;
            if (over < 0) {
                cur = cur << bits | x;
                used += bits;
                return;
            }
            cur = cur << (bits - over) | x >> over;
            flush();
            cur = x & ((1u << over) - 1u);
            used = over;
        };
        const uint8_t* wd = reinterpret_cast<const uint8_t*>(rows) + threadIdx.x * n;
        const uint8_t* kd = reinterpret_cast<const uint8_t*>(rows + nw) + threadIdx.x * K;
        int at = 0;
        for (int k = 1; k < n; ++k) {
            const int q = (k <= K ? k : n - k) - 1;
            const uint32_t d = kd[q], x = digits[d];
            if (d != ref[n + q]) differ = min(differ, at);
            put(x & 0xFFFu, (int)(x >> 12));
            at += (int)(x >> 12);
        }
        for (int pad; (pad = min(text - at, 12)) > 0; at += pad) put(0, pad);
        for (int p = 0; p < n; ++p, at += lbits) {
            if (wd[p] != ref[p]) differ = min(differ, at);
            put(rank[wd[p]], lbits);
        }
        if (used > 0) {
            cur <<= 64 - used;
            flush();
        }
    }
    __shared__ int wave_differ[4];
    for (int o = 32; o; o >>= 1) differ = min(differ, __shfl_xor(differ, o));
    if ((threadIdx.x & 63) == 0) wave_differ[threadIdx.x >> 6] = differ;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (const int d : wave_differ) differ = min(differ, d);
        const uint32_t live = (uint32_t)(W - differ / 64);
        if (__hip_atomic_load(&ctl->shape.live, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < live)
            atomicMax(&ctl->shape.live, live);
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
__global__ void __launch_bounds__(256) k_sort_uniq(MergeSorted s, const uint64_t* __restrict__ rest,
                                                   const SortCtl* __restrict__ ctl, int64_t m, int64_t chunk, uint8_t* __restrict__ flag,
                                                   uint32_t* __restrict__ counts) {
    __shared__ uint32_t part[4];
    const int nrest = (int)ctl->shape.words - 1, from = (int)(ctl->shape.words - ctl->shape.live);
    const int64_t end = min(((int64_t)blockIdx.x + 1) * chunk, m);
    uint32_t mine = 0;
    for (int64_t i = (int64_t)blockIdx.x * chunk + threadIdx.x; i < end; i += 256) {
        bool f = i == 0 || s.key[i] != s.key[i - 1];
        if (!f) {
            const uint64_t* a = rest + (int64_t)s.idx[i] * nrest;
            const uint64_t* b = rest + (int64_t)s.idx[i - 1] * nrest;
            for (int w = from; w < nrest && !f; w += 4) {
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
                                                      int8_t* __restrict__ out_w, uint8_t* __restrict__ out_k,
                                                      SortCtl* ctl) {
    __shared__ uint32_t part[4], src[256];
    if (blockIdx.x == 0 && threadIdx.x == 0) *ctl = SortCtl{};  // for the next call
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
    // (the letters take at most 8 bits; how many, the device knows)
    const int W = (4 * 3 * (n - 1) + 8 * n + 63) / 64;
    uint64_t* first = ctx->dev<uint64_t>("s_first", (size_t)m);
    uint64_t* rest = ctx->dev<uint64_t>("s_rest", (size_t)(W - 1) * m + 1);
    SortCtl* ctl = ctx->dev<SortCtl>("s_ctl", 1);
    if (!ctx->sort_ctl_clear) GP_HIP(hipMemsetAsync(ctl, 0, sizeof(SortCtl), st));
    ctx->sort_ctl_clear = false;
    const bool dense = m > kSortDense;
    if (dense)
        hipLaunchKernelGGL(k_sort_letters, dim3((unsigned)ctx->num_cus * 4), dim3(256), 0, st, d_words, m * n, ctl);
    hipLaunchKernelGGL(dense ? k_cand_keys<true> : k_cand_keys<false>, dim3((unsigned)((m + 255) / 256)), dim3(256), 0,
                       st, d_words, d_keys, m, n, K, ctl, first, rest);
    GP_HIP(hipGetLastError());
    const MergeSorted s = merge_sort(ctx, "s_sort", first, m, rest, W - 1, &ctl->shape);
    // at most 2048 blocks, so that each can add up the counts of those before it
    const int64_t chunk = std::max<int64_t>(256, (m + 2047) / 2048);
    const unsigned blocks = (unsigned)((m + chunk - 1) / chunk);
    uint8_t* flag = ctx->dev<uint8_t>("s_flag", (size_t)m);
    uint32_t* counts = ctx->dev<uint32_t>("s_counts", (size_t)blocks + 1);
    hipLaunchKernelGGL(k_sort_uniq, dim3(blocks), dim3(256), 0, st, s, rest, ctl, m, chunk, flag, counts);
    GP_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_sort_compact, dim3(blocks), dim3(256), 0, st, d_words, d_keys, n, K, m, chunk, s.idx, flag,
                       counts, d_out_words, d_out_keys, ctl);
    GP_HIP(hipGetLastError());
    uint32_t kept = 0;
    GP_HIP(hipMemcpyAsync(&kept, counts + blocks, 4, hipMemcpyDeviceToHost, st));
    GP_HIP(hipStreamSynchronize(st));
    ctx->sort_ctl_clear = true;
    return (int64_t)kept;
}

}  // namespace gp
