// Merge sort of records by a first key word (uint64) and, where two first words
// are equal, by `nrest` further words per record and then by record number.
//   k_ms_block  runs of one tile of records, sorted in LDS
//   k_ms_rank   places of all records of some runs at once (up to 2^16 records, or
//               2^18 without further words), k_ms_place moves them there
//   k_ms_merge  one round of pairwise merges: a block makes one tile of
//               consecutive records of the output
// What moves is the first word and the record number (12 bytes, read and written
// once per round); the further words stay where they are and are read only for
// records whose first words are equal.
//
// Why merges and not a radix sort: candidate keys are hundreds of bits wide, of
// which 19 bytes vary in the records of order 45, 3 -> 1 (19 passes of 5 launches
// each), while the first 64 bits tell nearly all records apart, and a level's
// files hold 1e4 .. 1e5 records, where the number of launches is the time: 1 + 6
// launches and 0.12 ms for 6e4 records against 95 launches and 0.74 ms (1 + 4 with
// k_ms_rank).  The rounds
// grow with the logarithm of the records, so a large sort gains as well: 0.45 ms
// for 4e6 records against 1.4 ms.  A round is bound by its chain of dependent
// reads (the split of the two runs, the merge in LDS), at 4e6 records by memory.
#include <algorithm>

#include "gp_internal.hpp"
#include "gp_sort.hpp"

namespace gp {

constexpr int kMsThreads = 256;
// Records per thread (I) and tile: 4 and 1024 up to kMsSmall records, which is a
// block per CU, else 8 and 2048.  Each thread merges its records one after the
// other: a round of 6e4 records takes 15 us with 4 and 21 us with 8.  The larger
// tile saves a round where a round is bound by memory.
constexpr int64_t kMsSmall = 1 << 18;
// Rounds over runs of a few tiles are one step (k_ms_rank, k_ms_place): each record's
// place among `ms_rank_runs` runs, all searched at once, two per block.  A record is
// searched in every run where a round of merges passes it once, but the searches do
// not wait for each other.  Calls of gp_sort_candidates on records of n = 15 with merges
// alone, ranks of 16 and of 32 runs, in us, where the first words differ, and where all but
// one record have the same first word, so that each search reads further words:
//   32 768 records  195, 175, 177 and 315, 300, 298
//   61 000          250, 234, 234     382, 387, 455
//  100 000          360, 347, 349     516, 578, 720
//  200 000          580, 567, 581     764, 978, 1230
// Beyond 2^16 the ranks gain 3 % and lose more where first words tie.  Without
// further words an equal first word costs nothing more.
__host__ __device__ constexpr int64_t ms_rank_runs(int64_t n, bool rest) {
    return !rest || n <= 1 << 15 ? 32 : n <= 1 << 16 ? 16 : 0;
}
constexpr uint32_t kMsNone = 0xFFFFFFFFu;  // a place past the last record: after every record

struct MsRec {
    uint64_t k;
    uint32_t i;
};

// LDS slot of record x of a tile: threads that start I records apart start in
// different banks.
template <int I>
__device__ __forceinline__ int ms_at(int x) { return x + x / I; }

// The further words, and with `shape` their number and the shared ones among them.
struct MsRest {
    const uint64_t* p;
    int n;
    const MergeShape* shape;
    // the first key word after the shared ones, given the very first
    __device__ uint64_t first(const uint64_t* __restrict__ keys, int64_t x) const {
        if (!shape) return keys[x];
        const int words = (int)shape->words, skip = words - (int)shape->live;
        return skip == 0 ? keys[x] : skip < words ? p[x * (words - 1) + skip - 1] : 0;
    }
};

template <bool REST>
__device__ __forceinline__ bool ms_less(const MsRec& a, const MsRec& b, const MsRest& rest) {
    if (a.k != b.k) return a.k < b.k;
    if (REST && a.i != kMsNone && b.i != kMsNone) {
        int n = rest.n, from = 0;
        if (rest.shape) {  // (read here: most comparisons do not come this far)
            n = (int)rest.shape->words - 1;
            from = (int)(rest.shape->words - rest.shape->live);
        }
        const uint64_t* x = rest.p + (int64_t)a.i * n;
        const uint64_t* y = rest.p + (int64_t)b.i * n;
        for (int w = from; w < n; w += 4) {  // four words at a time: their reads do not wait for each other
            uint64_t u[4], v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int at = min(w + j, n - 1);
                u[j] = x[at];
                v[j] = y[at];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (u[j] != v[j]) return u[j] < v[j];
        }
    }
    return a.i < b.i;
}

// Records d .. d + I - 1 of the merge of the sorted LDS ranges [a0, a1) and
// [b0, b1) (fewer at the end: the others get kMsNone).
template <bool REST, int I>
__device__ __forceinline__ void ms_merge_items(const uint64_t* sk, const uint32_t* si, int a0, int a1, int b0, int b1,
                                               int d, const MsRest& rest, MsRec (&out)[I]) {
    auto rec = [&](int x) { return MsRec{sk[ms_at<I>(x)], si[ms_at<I>(x)]}; };
    const int na = a1 - a0, nb = b1 - b0;
    int lo = max(0, d - nb), hi = min(d, na);
    while (lo < hi) {  // records of the first range among the first d
        const int mid = (lo + hi) >> 1;
        if (!ms_less<REST>(rec(b0 + d - 1 - mid), rec(a0 + mid), rest)) lo = mid + 1;
        else hi = mid;
    }
    int a = a0 + min(lo, na), b = b0 + min(max(d - lo, 0), nb);
    const MsRec none{~0ull, kMsNone};
    MsRec x = a < a1 ? rec(a) : none, y = b < b1 ? rec(b) : none;
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const bool first = b >= b1 || (a < a1 && !ms_less<REST>(y, x, rest));
        out[j] = first ? x : y;
        if (first) {
            ++a;
            x = a < a1 ? rec(a) : none;
        } else {
            ++b;
            y = b < b1 ? rec(b) : none;
        }
    }
}

template <bool REST, int I>
__global__ void __launch_bounds__(kMsThreads) k_ms_block(const uint64_t* __restrict__ keys, int64_t n,
                                                         const uint64_t* __restrict__ restp, int nrest,
                                                         const MergeShape* shape, uint64_t* __restrict__ kout,
                                                         uint32_t* __restrict__ iout) {
    constexpr int kTile = kMsThreads * I;
    __shared__ uint64_t sk[kTile + kMsThreads];
    __shared__ uint32_t si[kTile + kMsThreads];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kTile;
    const MsRest rest{restp, nrest, shape};
    MsRec r[I];
#pragma unroll
    for (int j = 0; j < I; ++j) {  // any I records: the loads of a wave are consecutive
        const int64_t x = base + j * kMsThreads + t;
        r[j] = x < n ? MsRec{REST ? rest.first(keys, x) : keys[x], (uint32_t)x} : MsRec{~0ull, kMsNone};
    }
    // a thread's records: Batcher's networks of 5 and 19 exchanges
    auto exchange = [&](int x, int y) {
        if (ms_less<REST>(r[y], r[x], rest)) {
            const MsRec z = r[x];
            r[x] = r[y];
            r[y] = z;
        }
    };
    static_assert(I == 4 || I == 8, "the networks below");
#pragma unroll
    for (int q = 0; q < I; q += 4) {
        exchange(q, q + 1); exchange(q + 2, q + 3);
        exchange(q, q + 2); exchange(q + 1, q + 3);
        exchange(q + 1, q + 2);
    }
    if constexpr (I == 8) {
        exchange(0, 4); exchange(1, 5); exchange(2, 6); exchange(3, 7);
        exchange(2, 4); exchange(3, 5);
        exchange(1, 2); exchange(3, 4); exchange(5, 6);
    }
    for (int run = I; run < kTile; run *= 2) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < I; ++j) {
            sk[ms_at<I>(t * I + j)] = r[j].k;
            si[ms_at<I>(t * I + j)] = r[j].i;
        }
        __syncthreads();
        const int o = t * I, a0 = o & ~(2 * run - 1);
        ms_merge_items<REST, I>(sk, si, a0, a0 + run, a0 + run, a0 + 2 * run, o - a0, rest, r);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < I; ++j) {
        sk[ms_at<I>(t * I + j)] = r[j].k;
        si[ms_at<I>(t * I + j)] = r[j].i;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const int x = j * kMsThreads + t;
        if (base + x < n) {
            kout[base + x] = sk[ms_at<I>(x)];
            iout[base + x] = si[ms_at<I>(x)];
        }
    }
}

// Records of [a0, a0 + na) among the first d of its merge with [b0, b0 + nb), by a
// whole wave: 64 places are tried at a time, so that three dependent reads of
// memory find the place in 2^18 records.
template <bool REST>
__device__ __forceinline__ int64_t ms_split(const uint64_t* __restrict__ k, const uint32_t* __restrict__ i, int64_t a0,
                                            int64_t na, int64_t b0, int64_t nb, int64_t d, const MsRest& rest,
                                            int lane) {
    int64_t lo = max<int64_t>(0, d - nb), hi = min(d, na);
    while (lo < hi) {
        const int64_t step = (hi - lo + 63) / 64, at = lo + lane * step;
        bool first = false;  // the record at a0 + at comes before the one at b0 + d - 1 - at
        if (at < hi) {
            const int64_t b = b0 + d - 1 - at;
            first = !ms_less<REST>(MsRec{k[b], i[b]}, MsRec{k[a0 + at], i[a0 + at]}, rest);
        }
        const int c = __popcll(__ballot(first));  // true for the first places, then false
        if (c == 0) return lo;
        hi = min(hi, lo + c * step);
        lo = lo + (c - 1) * step + 1;
    }
    return lo;
}

template <bool REST, int I>
__global__ void __launch_bounds__(kMsThreads) k_ms_merge(const uint64_t* __restrict__ kin,
                                                         const uint32_t* __restrict__ iin, int64_t n, int64_t run,
                                                         const uint64_t* __restrict__ restp, int nrest,
                                                         const MergeShape* shape, uint64_t* __restrict__ kout,
                                                         uint32_t* __restrict__ iout) {
    constexpr int kTile = kMsThreads * I;
    __shared__ uint64_t sk[kTile + kMsThreads];
    __shared__ uint32_t si[kTile + kMsThreads];
    __shared__ int64_t split[2];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const MsRest rest{restp, nrest, shape};
    const int64_t out0 = (int64_t)blockIdx.x * kTile, base = out0 / (2 * run) * (2 * run);
    const int64_t amax = min(base + run, n), bmax = min(base + 2 * run, n);
    const int64_t d0 = out0 - base, d1 = min(d0 + kTile, bmax - base);
    if (wave < 2) {
        const int64_t s = ms_split<REST>(kin, iin, base, amax - base, amax, bmax - amax, wave ? d1 : d0, rest, lane);
        if (lane == 0) split[wave] = s;
    }
    __syncthreads();
    const int64_t a = base + split[0], b = amax + (d0 - split[0]);
    const int na = (int)(split[1] - split[0]), total = (int)(d1 - d0);
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const int x = j * kMsThreads + t;
        if (x < total) {
            const int64_t src = x < na ? a + x : b + (x - na);
            sk[ms_at<I>(x)] = kin[src];
            si[ms_at<I>(x)] = iin[src];
        }
    }
    __syncthreads();
    MsRec r[I];
    const int d = min(t * I, total);
    ms_merge_items<REST, I>(sk, si, 0, na, na, total, d, rest, r);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < I; ++j) {
        sk[ms_at<I>(t * I + j)] = r[j].k;
        si[ms_at<I>(t * I + j)] = r[j].i;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const int x = j * kMsThreads + t;
        if (x < total) {
            kout[out0 + x] = sk[ms_at<I>(x)];
            iout[out0 + x] = si[ms_at<I>(x)];
        }
    }
}

// Places of the records of a tile (blockIdx.x) in the sort of all tiles, as far as
// the runs blockIdx.y, blockIdx.y + gridDim.y, ... decide them: how many of their
// records come before each, into part[blockIdx.y][record].  A run is searched in
// LDS, by first words; the records of a first word that the run has too are
// searched by all words.  The next run's loads are in flight during the search.
template <bool REST, int I>
__global__ void __launch_bounds__(kMsThreads) k_ms_rank(const uint64_t* __restrict__ kin,
                                                        const uint32_t* __restrict__ iin, int64_t n,
                                                        const uint64_t* __restrict__ restp, int nrest,
                                                        const MergeShape* shape, int runs,
                                                        uint32_t* __restrict__ part) {
    constexpr int kTile = kMsThreads * I;
    __shared__ uint64_t sk[kTile];
    __shared__ uint32_t si[kTile];
    const int t = threadIdx.x, own = blockIdx.x, seg = own / runs * runs, run0 = seg + blockIdx.y;
    const MsRest rest{restp, nrest, shape};
    const int tiles = min((int)((n + kTile - 1) / kTile), seg + runs);
    MsRec r[I], next[I];
    uint32_t place[I] = {};
    auto load = [&](int tile, MsRec (&v)[I]) {
#pragma unroll
        for (int j = 0; j < I; ++j) {
            const int64_t x = (int64_t)tile * kTile + j * kMsThreads + t;
            v[j] = x < n ? MsRec{kin[x], iin[x]} : MsRec{~0ull, kMsNone};
        }
    };
    load(own, r);
    load(run0, next);
    for (int run = run0; run < tiles; run += gridDim.y) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < I; ++j) {
            sk[j * kMsThreads + t] = next[j].k;
            si[j * kMsThreads + t] = next[j].i;
        }
        __syncthreads();
        if (run + (int)gridDim.y < tiles) load(run + gridDim.y, next);
        if (run == own) {
#pragma unroll
            for (int j = 0; j < I; ++j) place[j] += j * kMsThreads + t;
            continue;
        }
        const int len = (int)min<int64_t>(kTile, n - (int64_t)run * kTile);
        int lo[I] = {};
#pragma unroll
        for (int step = kTile / 2; step; step /= 2)
#pragma unroll
            for (int j = 0; j < I; ++j)
                if (sk[lo[j] + step - 1] < r[j].k) lo[j] += step;
#pragma unroll
        for (int j = 0; j < I; ++j) {
            if (sk[lo[j]] < r[j].k) ++lo[j];
            int a = lo[j];
            if (a < len && sk[a] == r[j].k && r[j].i != kMsNone) {
                int b = len;
                while (a < b) {  // records after a of a larger first word compare as such
                    const int mid = (a + b) >> 1;
                    if (ms_less<REST>(MsRec{sk[mid], si[mid]}, r[j], rest)) a = mid + 1;
                    else b = mid;
                }
            }
            place[j] += (uint32_t)a;
        }
    }
#pragma unroll
    for (int j = 0; j < I; ++j) {
        const int64_t x = (int64_t)own * kTile + j * kMsThreads + t;
        if (x < n) part[(int64_t)blockIdx.y * n + x] = place[j];
    }
}

__global__ void k_ms_place(const uint64_t* __restrict__ kin, const uint32_t* __restrict__ iin, int64_t n,
                           const uint32_t* __restrict__ part, int groups, int64_t seg, uint64_t* __restrict__ kout,
                           uint32_t* __restrict__ iout) {
    const int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n) return;
    int64_t at = x / seg * seg;
#pragma unroll 8
    for (int g = 0; g < groups; ++g) at += part[(int64_t)g * n + x];
    kout[at] = kin[x];
    iout[at] = iin[x];
}

namespace {

template <bool REST, int I>
MergeSorted run_merge_sort(hipStream_t st, const uint64_t* keys, int64_t n, const uint64_t* rest, int nrest,
                           const MergeShape* shape, uint64_t* const (&kb)[2], uint32_t* const (&ib)[2], uint32_t* part) {
    constexpr int64_t kTile = kMsThreads * I;
    const dim3 grid((unsigned)((n + kTile - 1) / kTile));
    hipLaunchKernelGGL((k_ms_block<REST, I>), grid, dim3(kMsThreads), 0, st, keys, n, rest, nrest, shape, kb[0],
                       ib[0]);
    int at = 0;
    int64_t run = kTile;
    if constexpr (I == 4) {
        if (part) {
            const int runs = (int)ms_rank_runs(n, REST);
            hipLaunchKernelGGL((k_ms_rank<REST, I>), dim3(grid.x, runs / 2), dim3(kMsThreads), 0, st, kb[0], ib[0], n, rest,
                               nrest, shape, runs, part);
            run *= runs;
            hipLaunchKernelGGL(k_ms_place, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, kb[0], ib[0], n, part,
                               runs / 2, run, kb[1], ib[1]);
            at = 1;
        }
    }
    for (; run < n; run *= 2, at ^= 1)
        hipLaunchKernelGGL((k_ms_merge<REST, I>), grid, dim3(kMsThreads), 0, st, kb[at], ib[at], n, run, rest, nrest,
                           shape, kb[at ^ 1], ib[at ^ 1]);
    GP_HIP(hipGetLastError());
    return MergeSorted{kb[at], ib[at]};
}

}  // namespace

MergeSorted merge_sort(gp_ctx* ctx, const std::string& name, const uint64_t* keys, int64_t n, const uint64_t* rest,
                       int nrest, const MergeShape* shape) {
    if (n > 0xFFFFFFFFll) throw ArgError("sort: more than 2^32 records");
    if (n <= 0) return MergeSorted{nullptr, nullptr};
    uint64_t* const kb[2] = {ctx->dev<uint64_t>(name + ".k0", (size_t)n), ctx->dev<uint64_t>(name + ".k1", (size_t)n)};
    uint32_t* const ib[2] = {ctx->dev<uint32_t>(name + ".i0", (size_t)n), ctx->dev<uint32_t>(name + ".i1", (size_t)n)};
    const int64_t runs = n > 2 * kMsThreads * 4 && n <= kMsSmall ? ms_rank_runs(n, nrest > 0) : 0;  // two tiles: a merge
    uint32_t* const part = runs ? ctx->dev<uint32_t>(name + ".rank", (size_t)(n * runs / 2)) : nullptr;
    if (n <= kMsSmall)
        return nrest > 0 ? run_merge_sort<true, 4>(ctx->stream, keys, n, rest, nrest, shape, kb, ib, part)
                         : run_merge_sort<false, 4>(ctx->stream, keys, n, rest, nrest, shape, kb, ib, part);
    return nrest > 0 ? run_merge_sort<true, 8>(ctx->stream, keys, n, rest, nrest, shape, kb, ib, part)
                     : run_merge_sort<false, 8>(ctx->stream, keys, n, rest, nrest, shape, kb, ib, part);
}

}  // namespace gp
