// Candidate join + exact PAF check (replaces the merge-join of match_pairs,
// src/core/match/match_pairs.cpp:15-121, and check_if_pair, golay.cpp:27-44).
//
// The reference merge-joins two files sorted on the key text and runs
// check_if_pair on every (A, B) with equal key text.  Key text equality and
// key tuple equality select the same PAF-passing pairs: if (A, B) passes the
// PAF check, PSD_A(k) + PSD_B(k) = Q for all k != 0 with Q an integer, so the
// inverted B key is the A key shifted by the constant BOUND - Q, and two
// digit strings of tuples that differ by a nonzero constant shift cannot be
// equal (the first component keeps or changes its decimal length, and either
// way the strings differ).  The join therefore hashes the key tuples:
//   k_join_insert  B records into a hash table, a chain per key
//   k_join_probe   for every A its key's chain: equal tuples
//   k_join_check   the integer PAF condition of the candidate pairs
// (or, of many candidates, k_join_slots, k_join_runs, k_join_scan: see there)
// and the accepted pairs are sorted into the reference's emission order.
// Bound by launches and the copies of the four input buffers.  The files of order
// 45, 3 -> 1 (at most 53000 records each) take 214-221 us, against 775 us with B radix
// sorted by hash (40 launches) and the pairs sorted on the host.
#include <algorithm>

#include "gp_internal.hpp"
#include "gp_sort.hpp"
#include "psd_core.hpp"

namespace gp {

__device__ __forceinline__ uint64_t key_hash(const uint8_t* __restrict__ k, int nkey) {
    uint64_t h = 0x243F6A8885A308D3ull;
    for (int i = 0; i < nkey; i += 8) {
        uint64_t v = 0;
        for (int j = 0; j < 8 && i + j < nkey; ++j) v |= (uint64_t)k[i + j] << (8 * j);
        h = splitmix64(h ^ v);
    }
    return h;
}

// A slot of the hash table: the tag of the keys it holds (0: free) and the first of
// their B records, numbered from 1 (0: none).  Records of one key are chained in one
// slot, others in the slots after it, so that an A record walks the records of its own
// key only (tags that collide apart): chains of all that share a slot index made 2e5 A
// records beside 1e5 B records of one other key take 21 ms, the longest chain's walk.
struct JoinSlot {
    uint32_t tag, head;
};

__device__ __forceinline__ uint32_t join_tag(uint64_t h) { return (uint32_t)(h >> 32) | 1u; }

// The slot of a key of hash h, or a free one where the table lacks it.
__device__ __forceinline__ uint64_t join_find(const JoinSlot* __restrict__ slot, uint64_t mask, uint64_t h) {
    uint64_t s = h & mask;
    for (uint32_t t; (t = slot[s].tag) != 0 && t != join_tag(h);) s = (s + 1) & mask;
    return s;
}

// B record i in front of the chain of its key.  Of the lanes with the hash of the
// wave's first one, which link up among themselves, that one alone goes to the table
// (atomics on one address are applied one at a time).
__global__ void k_join_insert(const uint8_t* __restrict__ keys, int64_t m, int nkey, int kstride,
                              uint32_t* __restrict__ next, JoinSlot* slot, uint64_t mask) {
    const int lane = threadIdx.x & 63;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t h = key_hash(keys + i * kstride, nkey);
        const uint64_t h0 = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(h >> 32)) << 32 |
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)h);
        const unsigned long long same = __ballot(h == h0), mine = h == h0 ? same : 1ull << lane;
        const int first = __ffsll((long long)mine) - 1, last = 63 - __clzll((long long)mine);
        const unsigned long long after = mine >> lane >> 1;
        if (after) next[i] = (uint32_t)i + (uint32_t)__ffsll((long long)after) + 1;  // (lanes hold records in a row)
        if (lane != first) continue;
        uint64_t s = h & mask;
        for (;; s = (s + 1) & mask) {  // (the table is at most half full)
            uint32_t t = __hip_atomic_load(&slot[s].tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (t == 0) t = atomicCAS(&slot[s].tag, 0u, join_tag(h));
            if (t == 0 || t == join_tag(h)) break;
        }
        next[i + last - first] = atomicExch(&slot[s].head, (uint32_t)i + 1);
    }
}

struct JoinCtl {
    unsigned long long out;
    unsigned long long cand;
};

// Entries that a wave appends to a list (at most cap kept), collected in LDS so that
// about 200 take one atomic: atomics on one address are applied one at a time, and
// one per step of a wave made the probe of 2^21 records a side with 2^20 candidates
// take 1.63 ms instead of 0.20 ms.  Every lane of the wave must call push, and every
// thread of the block finish, which takes one atomic for what the 4 waves still hold.
struct WaveQueue {
    static constexpr int kCap = 256;
    uint64_t* q;
    unsigned long long* count;
    uint64_t* list;
    int64_t cap;
    int n = 0;
    bool full = false;  // the list had no room for some of the last entries
    __device__ void push(bool have, uint64_t x) {
        const unsigned long long b = __ballot(have);
        if (have) q[n + __popcll(b & ((1ull << (threadIdx.x & 63)) - 1ull))] = x;
        n += __popcll(b);
        if (n > kCap - 64) flush();
    }
    __device__ void flush() {
        if (n == 0) return;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the other lanes' writes
        __builtin_amdgcn_wave_barrier();
        const int lane = threadIdx.x & 63;
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(count, (unsigned long long)n);
        base = __shfl(base, 0);
        for (int x = lane; x < n; x += 64)
            if ((int64_t)(base + x) < cap) list[base + x] = q[x];
        full = (int64_t)base + n > cap;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        n = 0;
    }
    __device__ void finish() {
        __shared__ int held[4];
        __shared__ unsigned long long base;
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        if (lane == 0) held[wave] = n;
        __syncthreads();
        if (threadIdx.x == 0) {
            const int sum = held[0] + held[1] + held[2] + held[3];
            base = sum ? atomicAdd(count, (unsigned long long)sum) : 0ull;
        }
        __syncthreads();
        unsigned long long at = base;
        for (int w = 0; w < wave; ++w) at += (unsigned long long)held[w];
        for (int x = lane; x < n; x += 64)
            if ((int64_t)(at + x) < cap) list[at + x] = q[x];
        n = 0;
    }
};

__device__ __forceinline__ bool same_keys(const uint8_t* __restrict__ x, const uint8_t* __restrict__ y, int nkey) {
    uint32_t d = 0;
    for (int q = 0; q < nkey; ++q) d |= x[q] ^ y[q];  // (a loop that ends early waits for each byte)
    return d == 0;
}

// Candidate pairs A << 32 | B with equal key tuples, one A record per lane.  A wave
// that finds the list full stops: ctl->cand is above cap then.
__global__ void __launch_bounds__(256) k_join_probe(const uint8_t* __restrict__ ka, int64_t na,
                                                    const uint8_t* __restrict__ kb, int nkey, int kstride,
                                                    const uint32_t* __restrict__ next,
                                                    const JoinSlot* __restrict__ slot, uint64_t mask,
                                                    uint64_t* __restrict__ cand, int64_t cap, JoinCtl* ctl) {
    __shared__ uint64_t queue[4][WaveQueue::kCap];
    WaveQueue out{queue[threadIdx.x >> 6], &ctl->cand, cand, cap};
    for (int64_t i0 = (int64_t)blockIdx.x * 256; i0 < na && !out.full; i0 += (int64_t)gridDim.x * 256) {
        const int64_t i = i0 + threadIdx.x;
        const uint8_t* k = ka + i * kstride;
        uint32_t j = 0;
        if (i < na) j = slot[join_find(slot, mask, key_hash(k, nkey))].head;
        while (__any(j != 0) && !out.full) {
            bool eq = j != 0;
            const uint32_t at = j - 1;
            if (eq) {
                j = next[at];
                eq = same_keys(k, kb + (int64_t)at * kstride, nkey);
            }
            out.push(eq, (uint64_t)i << 32 | at);
        }
    }
    out.finish();
}

// The PAF condition of each candidate by 8 lanes, which take the shifts in turn
// (a lane that checked its candidate alone had a chain of n^2 / 2 dependent
// adds, and each accepted pair its own atomic).
__global__ void __launch_bounds__(256) k_join_check(const int8_t* __restrict__ wa, const int8_t* __restrict__ wb, int n,
                                                    int wstride, int target, const uint64_t* __restrict__ cand,
                                                    int64_t cap, uint64_t* __restrict__ out, JoinCtl* ctl) {
    __shared__ uint64_t queue[4][WaveQueue::kCap];
    WaveQueue pairs{queue[threadIdx.x >> 6], &ctl->out, out, cap};
    const int64_t m = min((int64_t)ctl->cand, cap);
    const int lane = threadIdx.x & 63, sub = lane & 7;
    for (int64_t c0 = (int64_t)blockIdx.x * 32; c0 < m; c0 += (int64_t)gridDim.x * 32) {
        const int64_t c = c0 + (threadIdx.x >> 3);
        const uint64_t x = c < m ? cand[c] : 0;
        bool ok = c < m;
        if (ok) {
            const int8_t* a = wa + (int64_t)(x >> 32) * wstride;
            const int8_t* b = wb + (int64_t)(uint32_t)x * wstride;
            for (int s = 1 + sub; s <= n / 2; s += 8) {
                int acc = 0, j = s;
                for (int p = 0; p < n; ++p) {
                    acc += (int)a[p] * (int)a[j] + (int)b[p] * (int)b[j];
                    if (++j == n) j = 0;
                }
                ok = ok && acc == target;
            }
        }
        const unsigned long long all = __ballot(ok);
        const bool pass = (all >> (lane & 56) & 255ull) == 255ull;
        pairs.push(pass && sub == 0, x);
    }
    pairs.finish();
}

// Where there are more candidates than the list holds (a few per record), none are
// listed: the B records are sorted by slot, and a wave checks an A record's run of them,
// one per lane.  3000 records of one key on either side: 0.59 ms, against 13.3 ms with a
// list of all 9e6 candidates, made in a second walk of the chains.
__global__ void k_join_slots(const uint8_t* __restrict__ keys, int64_t m, int nkey, int kstride,
                             const JoinSlot* __restrict__ slot, uint64_t mask, uint64_t* __restrict__ at) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
        at[i] = join_find(slot, mask, key_hash(keys + i * kstride, nkey));
}

// A slot's run of the sorted records: its first place, from 1, as the slot's head, and
// the place after its last as `next` of the first.
__global__ void k_join_runs(const uint64_t* __restrict__ at, int64_t m, uint32_t* __restrict__ next,
                            JoinSlot* __restrict__ slot) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < m; p += (int64_t)gridDim.x * blockDim.x)
        if (p == 0 || at[p - 1] != at[p]) {
            slot[at[p]].head = (uint32_t)p + 1;
            int64_t lo = p + 1, hi = m;
            while (lo < hi) {
                const int64_t mid = (lo + hi) >> 1;
                if (at[mid] > at[p]) hi = mid;
                else lo = mid + 1;
            }
            next[p] = (uint32_t)lo;
        }
}

__global__ void __launch_bounds__(256) k_join_scan(const int8_t* __restrict__ wa, const uint8_t* __restrict__ ka,
                                                   int64_t na, const int8_t* __restrict__ wb,
                                                   const uint8_t* __restrict__ kb, int n, int nkey, int wstride,
                                                   int kstride, int target, const uint32_t* __restrict__ idx,
                                                   const uint32_t* __restrict__ next,
                                                   const JoinSlot* __restrict__ slot, uint64_t mask,
                                                   uint64_t* __restrict__ out, int64_t cap, JoinCtl* ctl) {
    __shared__ uint64_t queue[4][WaveQueue::kCap];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    WaveQueue pairs{queue[wave], &ctl->out, out, cap};
    unsigned long long checks = 0;
    for (int64_t i = (int64_t)blockIdx.x * 4 + wave; i < na; i += (int64_t)gridDim.x * 4) {
        const uint8_t* k = ka + i * kstride;
        const int8_t* a = wa + i * wstride;
        const uint32_t head = slot[join_find(slot, mask, key_hash(k, nkey))].head;
        const int64_t end = head ? next[head - 1] : 0;
        for (int64_t p0 = (int64_t)head - 1; head && p0 < end; p0 += 64) {
            bool ok = p0 + lane < end;
            uint32_t j = 0;
            if (ok) {
                j = idx[p0 + lane];
                ok = same_keys(k, kb + (int64_t)j * kstride, nkey);
            }
            checks += ok;
            if (ok) {
                const int8_t* b = wb + (int64_t)j * wstride;
                for (int s = 1; s <= n / 2 && ok; ++s) {
                    int acc = 0, q = s;
                    for (int p = 0; p < n; ++p) {
                        acc += (int)a[p] * (int)a[q] + (int)b[p] * (int)b[q];
                        if (++q == n) q = 0;
                    }
                    ok = acc == target;
                }
            }
            pairs.push(ok, (uint64_t)i << 32 | j);
        }
    }
    pairs.finish();
    block_atomic_add(&ctl->cand, checks);
}

JoinResult join_pairs(gp_ctx* ctx, const int8_t* d_wa, const uint8_t* d_ka, int64_t na, const int8_t* d_wb,
                      const uint8_t* d_kb, int64_t nb, int n, int nkey, int wstride, int kstride, int paf_target,
                      gp_stats* stats) {
    JoinResult res;
    if (na <= 0 || nb <= 0) return res;
    if (na > 0xFFFFFFFFll || nb > 0xFFFFFFFFll) throw ArgError("join: more than 2^32 candidates");
    hipStream_t st = ctx->stream;
    uint64_t slots = 64;  // two slots per B record or more
    while (slots < 2 * (uint64_t)nb) slots <<= 1;
    const uint64_t mask = slots - 1;
    uint32_t* next = ctx->dev<uint32_t>("j_next", nb);
    JoinSlot* slot = ctx->dev<JoinSlot>("j_slot", slots);
    JoinCtl* ctl = ctx->dev<JoinCtl>("j_ctl", 1);
    if (stats) GP_HIP(hipEventRecord(ctx->ev2, st));
    GP_HIP(hipMemsetAsync(slot, 0, slots * sizeof(JoinSlot), st));
    const auto blocks = [&](int64_t n_) { return dim3((unsigned)std::min<int64_t>((n_ + 255) / 256, ctx->num_cus * 8)); };
    hipLaunchKernelGGL(k_join_insert, blocks(nb), dim3(256), 0, st, d_kb, nb, nkey, kstride, next, slot, mask);
    GP_HIP(hipGetLastError());
    int64_t cap = std::max<int64_t>(1024, 2 * std::max(na, nb));
    JoinCtl h{};
    uint64_t* out = ctx->dev<uint64_t>("j_out", cap);
    uint64_t* cand = ctx->dev<uint64_t>("j_cand", cap);
    const auto read = [&]() {
        GP_HIP(hipGetLastError());
        GP_HIP(hipMemcpyAsync(&h, ctl, sizeof h, hipMemcpyDeviceToHost, st));
        GP_HIP(hipStreamSynchronize(st));
    };
    GP_HIP(hipMemsetAsync(ctl, 0, sizeof(JoinCtl), st));
    hipLaunchKernelGGL(k_join_probe, blocks(na), dim3(256), 0, st, d_ka, na, d_kb, nkey, kstride, next, slot, mask,
                       cand, cap, ctl);
    hipLaunchKernelGGL(k_join_check, blocks(8 * na), dim3(256), 0, st, d_wa, d_wb, n, wstride, paf_target, cand, cap,
                       out, ctl);
    read();
    if ((int64_t)h.cand > cap) {
        uint64_t* at = ctx->dev<uint64_t>("j_at", nb);
        hipLaunchKernelGGL(k_join_slots, blocks(nb), dim3(256), 0, st, d_kb, nb, nkey, kstride, slot, mask, at);
        const MergeSorted s = merge_sort(ctx, "j_runs", at, nb);
        hipLaunchKernelGGL(k_join_runs, blocks(nb), dim3(256), 0, st, s.key, nb, next, slot);
        for (int attempt = 0; attempt < 2; ++attempt) {
            GP_HIP(hipMemsetAsync(ctl, 0, sizeof(JoinCtl), st));
            hipLaunchKernelGGL(k_join_scan, blocks(64 * na), dim3(256), 0, st, d_wa, d_ka, na, d_wb, d_kb, n, nkey,
                               wstride, kstride, paf_target, s.idx, next, slot, mask, out, cap, ctl);
            read();
            if ((int64_t)h.out <= cap) break;
            cap = (int64_t)h.out;
            out = ctx->dev<uint64_t>("j_out", cap);
        }
    }
    // emission order of the reference: A position outer, B position inner
    std::vector<uint64_t> pairs(h.out);
    if (h.out > 0xFFFFFFFFull) {  // (more than the device sort numbers)
        GP_HIP(hipMemcpyAsync(pairs.data(), out, h.out * 8, hipMemcpyDeviceToHost, st));
        GP_HIP(hipStreamSynchronize(st));
        std::sort(pairs.begin(), pairs.end());
    } else if (h.out) {
        const MergeSorted s = merge_sort(ctx, "j_sort", out, (int64_t)h.out);
        GP_HIP(hipMemcpyAsync(pairs.data(), s.key, h.out * 8, hipMemcpyDeviceToHost, st));
    }
    if (stats) GP_HIP(hipEventRecord(ctx->ev3, st));
    GP_HIP(hipStreamSynchronize(st));
    res.checks = h.cand;
    if (stats) {
        float ms = 0;
        GP_HIP(hipEventElapsedTime(&ms, ctx->ev2, ctx->ev3));
        stats->pair_checks += h.cand;
        stats->kernel_ms += ms;
    }
    res.ia.resize(h.out);
    res.ib.resize(h.out);
    for (size_t i = 0; i < pairs.size(); ++i) {
        res.ia[i] = (uint32_t)(pairs[i] >> 32);
        res.ib[i] = (uint32_t)pairs[i];
    }
    return res;
}

}  // namespace gp
