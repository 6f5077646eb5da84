// Equivalence filter (replaces cache_filter, src/core/filter/filter.cpp:18-163).
//
// The reference builds the pair group as the closure of an index template under
// shift_pair (rotate b), swap_pair, reverse_pair (reverse b), decimate_pair (the
// same unit on a and b) and, when COMPRESS == 1 and LEN is even, altnegative_pair
// (negate the odd positions of a and b) (equivalence.cpp:46-95,146-267,
// filter.cpp:80-87).  Every element of that closure acts as
//   (X, Y) = swap ? (b, a) : (a, b)
//   a'[i] = sa * (-1)^(kappa i) * X[(u i + ta) mod n]
//   b'[i] = sb * (-1)^(kappa i) * Y[(e u i + tb) mod n]
// with u a unit mod n, e = +-1, ta, tb in Z_n, and (kappa, sa, sb) = (0, +1, +1)
// without altnegative, free in {0,1} x {+-1}^2 with it; the set of transforms the
// reference applies in generateClassPairs (equivalence.cpp:97-144, including
// its swapped-template branch) is this whole group, so its classes are orbits.
// Walking the pairs in (a, b) order and erasing each survivor's class
// (filter.cpp:117-144) therefore keeps the lexicographically smallest input
// member of every orbit.  Here, on the GPU,
//   k_value_range   the range of the values, which gives the bits per value
//   k_orbit_bits    every pair's orbit minimum, one pair per wave, with whole
//   k_orbit_min     words as integers where they fit in 128 bits, else by letters
//   k_class_insert  a hash table of the minima, each slot with its least pair
//   k_class_keep    the pairs in the table
// and the kept pairs are sorted by (a, b) and gathered.
#include <algorithm>
#include <cstring>
#include <functional>
#include <numeric>
#include <vector>

#include "gp_host.hpp"
#include "gp_internal.hpp"
#include "gp_sort.hpp"

namespace gp {

struct FilterParams {
    int32_t n;
    int32_t alt;
    int32_t nunits;
    int32_t units[64];
    int32_t mx, sh, B, E;  // value v packs as (v + mx) >> sh in B bits, E = 64 / B values per word
};

template <int W>
__device__ __forceinline__ bool key_less(const uint64_t (&x)[W], const uint64_t (&y)[W]) {
#pragma unroll
    for (int w = 0; w < W; ++w)
        if (x[w] != y[w]) return x[w] < y[w];
    return false;
}

template <int W>
__device__ __forceinline__ bool key_eq(const uint64_t (&x)[W], const uint64_t (&y)[W]) {
    bool e = true;
#pragma unroll
    for (int w = 0; w < W; ++w) e = e && x[w] == y[w];
    return e;
}

// minimum over the 64 lanes of the wave, returned to every lane
template <int W>
__device__ __forceinline__ void wave_min(uint64_t (&k)[W]) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        uint64_t o[W];
#pragma unroll
        for (int w = 0; w < W; ++w) o[w] = __shfl_xor(k[w], off);
        if (key_less(o, k))
#pragma unroll
            for (int w = 0; w < W; ++w) k[w] = o[w];
    }
}

// Least rotation (the start r of the lexicographically smallest rotation) of
// the lane's sequence z[0..n) held in LDS at z[j * 64] (signed order); the
// two-pointer minimum-expression method, O(n).
__device__ __forceinline__ int least_rotation(const int8_t* z, int n) {
    int i = 0, j = 1, k = 0;
    while (i < n && j < n && k < n) {
        int x = i + k, y = j + k;
        if (x >= n) x -= n;
        if (y >= n) y -= n;
        const int a = z[x * 64], b = z[y * 64];
        if (a == b) {
            ++k;
            continue;
        }
        if (a > b) i += k + 1;
        else j += k + 1;
        if (i == j) ++j;
        k = 0;
    }
    return i < j ? i : j;
}

// Writes z[j] = sigma * (-1)^(kappa j) * X[(u j) mod n] (lane's column of the
// LDS sequence area); kappa is used only for even n (altnegative).
__device__ __forceinline__ void decimated(const int8_t* X, int n, int u, int kappa, int sigma, int8_t* z) {
    int idx = 0;
    for (int j = 0; j < n; ++j) {
        int v = X[idx] * sigma;
        if (kappa & j & 1) v = -v;
        z[j * 64] = (int8_t)v;
        idx += u;
        if (idx >= n) idx -= n;
    }
}

// Packed key of the rotation of z starting at r (layout of img_key).
template <int W>
__device__ __forceinline__ void rot_key(const int8_t* z, const FilterParams& P, int r, uint64_t (&k)[W]) {
    const int n = P.n;
    int idx = r, i = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        uint64_t acc = 0;
        const int iend = min(n, (w + 1) * P.E);
        const int cnt = max(0, iend - i);
        for (; i < iend; ++i) {
            acc = (acc << P.B) | (uint64_t)((z[idx * 64] + P.mx) >> P.sh);
            if (++idx == n) idx = 0;
        }
        k[w] = cnt ? acc << (P.B * (P.E - cnt)) : 0ull;
    }
}

// One pair per wave; the orbit minimum by construction.  Every transform acts
// as image[i] = s (-1)^(kappa i) X[(u i + t) mod n] on each half.  With
// t = u s' this is a rotation by s' of z[j] = (-1)^(kappa j) X[(u j) mod n]
// (for kappa = 1, n is even and (-1)^(kappa i) = (-1)^(s') (-1)^(kappa (i + s')),
// so the rotation's sign is s (-1)^(s'), both signs reachable since s is free
// whenever kappa is).  So for each (swap, u, kappa, sign) the minimum over t
// is the least rotation of +-z.  Phase 1: lanes over the a-part variants
// (swap, u, kappa, sign); the wave minimum is the a key.  Phase 2: every lane
// whose variant reaches it takes the least rotations of its b-part variants
// (unit e u with e = +-1, the same kappa, sign free with altnegative), which
// do not depend on the a-part's shift or sign; the wave minimum is the b key.
// canon[q] = (a key, b key), as the minimum over the whole group.
template <int W>
__global__ void __launch_bounds__(256) k_orbit_min(FilterParams P, const int8_t* __restrict__ pa,
                                                   const int8_t* __restrict__ pb, int64_t m,
                                                   uint64_t* __restrict__ canon) {
    __shared__ int8_t sx[4][2][kMaxN];
    __shared__ int8_t zs[4][kMaxN * 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int n = P.n;
    const int nk = P.alt ? 2 : 1, ns = P.alt ? 2 : 1;
    const int nvar = 2 * P.nunits * nk * ns;
    int8_t* z = &zs[wv][lane];
    for (int64_t q = (int64_t)blockIdx.x * 4 + wv; q < m; q += (int64_t)gridDim.x * 4) {
        if (lane < n) {
            sx[wv][0][lane] = pa[q * n + lane];
            sx[wv][1][lane] = pb[q * n + lane];
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // variant c -> (swap, unit index, kappa, sign)
        auto decode = [&](int c, int& sw, int& ui, int& kappa, int& sg) {
            sg = (c % ns) ? -1 : 1;
            c /= ns;
            kappa = c % nk;
            c /= nk;
            ui = c % P.nunits;
            sw = c / P.nunits;
        };
        uint64_t ka[W], kb[W], lmin[W];
#pragma unroll
        for (int w = 0; w < W; ++w) ka[w] = kb[w] = ~0ull;
        for (int c = lane; c < nvar; c += 64) {
            int sw, ui, kappa, sg;
            decode(c, sw, ui, kappa, sg);
            decimated(sx[wv][sw], n, P.units[ui], kappa, sg, z);
            uint64_t k[W];
            rot_key<W>(z, P, least_rotation(z, n), k);
            if (key_less(k, ka))
#pragma unroll
                for (int w = 0; w < W; ++w) ka[w] = k[w];
        }
#pragma unroll
        for (int w = 0; w < W; ++w) lmin[w] = ka[w];
        wave_min<W>(ka);
        const bool mine = key_eq(lmin, ka);
        // phase 2: the lanes holding a minimising variant (re-found by recomputing)
        for (int c = lane; c < nvar && mine; c += 64) {
            int sw, ui, kappa, sg;
            decode(c, sw, ui, kappa, sg);
            decimated(sx[wv][sw], n, P.units[ui], kappa, sg, z);
            uint64_t k[W];
            rot_key<W>(z, P, least_rotation(z, n), k);
            if (!key_eq(k, ka)) continue;
            const int u = P.units[ui];
            for (int e = 0; e < 2; ++e) {
                const int ub = e ? (n - u) % n : u;
                for (int sb = 0; sb < ns; ++sb) {
                    decimated(sx[wv][sw ? 0 : 1], n, n == 1 ? 0 : ub, kappa, sb ? -1 : 1, z);
                    rot_key<W>(z, P, least_rotation(z, n), k);
                    if (key_less(k, kb))
#pragma unroll
                        for (int w = 0; w < W; ++w) kb[w] = k[w];
                }
            }
        }
        wave_min<W>(kb);
        if (lane == 0) {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                canon[q * 2 * W + w] = ka[w];
                canon[q * 2 * W + W + w] = kb[w];
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

typedef unsigned __int128 u128;

template <class T>
__device__ __forceinline__ T wave_min_bits(T v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        T o;
        if constexpr (sizeof(T) == 16)
            o = (T)__shfl_xor((unsigned long long)(v >> 64), off) << 64 | __shfl_xor((unsigned long long)v, off);
        else if constexpr (sizeof(T) == 8)
            o = __shfl_xor((unsigned long long)v, off);
        else
            o = (T)__shfl_xor((int)v, off);
        v = o < v ? o : v;
    }
    return v;
}

// k_orbit_min for words of n * B bits that fit in T (first letter in the highest
// field): a rotation is two shifts, a negated word a subtraction from the word of
// largest fields, and the least rotation the minimum of all n.
//   The words decimated by every unit, of a and of b, one per lane, go to LDS.
//   Phase 1: variants (swap, unit, kappa, sign) over the lanes; the wave's least
//   rotation is the a key.  Phase 2, for each variant that reaches it: the lanes
//   share the rotations of its b-part words, which are in LDS already.
// Bound by VALU: about 150 rotation steps of 9 operations per pair at n = 50.
// 120011 pairs of n = 50 with altnegative take 0.39 ms against 4.95 ms by letters (a
// least rotation by comparing letters in LDS, one after the other), 18645 pairs of
// n = 45 0.04 ms against 0.31 ms.
template <class T>
__global__ void __launch_bounds__(256) k_orbit_bits(FilterParams P, const int8_t* __restrict__ pa,
                                                    const int8_t* __restrict__ pb, int64_t m,
                                                    uint64_t* __restrict__ canon) {
    constexpr int W = sizeof(T) == 16 ? 2 : 1;
    __shared__ uint8_t fld[4][2][kMaxN];
    __shared__ T zl[4][2 * kMaxN];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int n = P.n, B = P.B, nb = n * B, nu = P.nunits;
    const int nk = P.alt ? 2 : 1, ns = nk, per = nk * ns;
    T mask = 0, all = 0, odd = 0;  // all bits; the largest value in every field; the fields of odd letters
    for (int j = 0; j < n; ++j) {
        const T f = (T)((1u << B) - 1u);
        mask = mask << B | f;
        all = all << B | (T)((2 * P.mx) >> P.sh);
        odd = odd << B | (j & 1 ? f : (T)0);
    }
    auto variant = [&](T y, int kappa, int sg) {
        if (kappa) y = (y & ~odd) | ((all & odd) - (y & odd));
        return sg ? all - y : y;
    };
    for (int64_t q = (int64_t)blockIdx.x * 4 + wv; q < m; q += (int64_t)gridDim.x * 4) {
        if (lane < n) {
            fld[wv][0][lane] = (uint8_t)((pa[q * n + lane] + P.mx) >> P.sh);
            fld[wv][1][lane] = (uint8_t)((pb[q * n + lane] + P.mx) >> P.sh);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int c = lane; c < 2 * nu; c += 64) {
            const uint8_t* x = fld[wv][c >= nu];
            const int u = P.units[c >= nu ? c - nu : c];
            T z = 0;
            int idx = 0;
            for (int j = 0; j < n; ++j) {
                z = z << B | x[idx];
                idx += u;
                if (idx >= n) idx -= n;
            }
            zl[wv][c] = z;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        T best = ~(T)0;
        uint32_t bits = 0;  // the lane's variants (c = lane + 64 bit) that reach `best`
        int round = 0;
        for (int c = lane; c < 2 * nu * per; c += 64, ++round) {
            T y = variant(zl[wv][c / per], c % per / ns, c % ns), mn = y;
            for (int r = 1; r < n; ++r) {
                y = (y << B | y >> (nb - B)) & mask;
                mn = y < mn ? y : mn;
            }
            if (mn < best) {
                best = mn;
                bits = 0;
            }
            if (mn == best) bits |= 1u << round;
        }
        const T ka = wave_min_bits(best);
        if (best != ka) bits = 0;
        T kb = ~(T)0;
        for (unsigned long long reach; (reach = __ballot(bits != 0)) != 0;) {
            const int l = __ffsll((long long)reach) - 1;
            const uint32_t lb = (uint32_t)__builtin_amdgcn_readlane((int)bits, l);
            const int c = l + 64 * (__ffs((int)lb) - 1);
            if (lane == l) bits &= bits - 1;
            const int v = c / per, kappa = c % per / ns, ui = v < nu ? v : v - nu;
            // candidates (unit u or -u, sign): 64 / (2 ns) lanes each; -u has index nu - 1 - ui
            const int share = 32 / ns, cand = lane / share;
            const T y = variant(zl[wv][(v < nu ? nu : 0) + (cand & 1 ? nu - 1 - ui : ui)], kappa, cand >> 1);
            for (int r = lane % share; r < n; r += share) {
                const T x = r ? (y << (r * B) | y >> (nb - r * B)) & mask : y;
                kb = x < kb ? x : kb;
            }
        }
        kb = wave_min_bits(kb);
        if (lane == 0) {
            if constexpr (W == 2) {
                canon[q * 4] = (uint64_t)(ka >> 64);
                canon[q * 4 + 1] = (uint64_t)ka;
                canon[q * 4 + 2] = (uint64_t)(kb >> 64);
                canon[q * 4 + 3] = (uint64_t)kb;
            } else {
                canon[q * 2] = (uint64_t)ka;
                canon[q * 2 + 1] = (uint64_t)kb;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// What the packing needs of the values of a call, and its count of kept pairs.
struct FilterCtl {
    uint32_t mx;      // max |v|
    uint32_t parity;  // bit 0: some value is even, bit 1: some is odd
    uint32_t kept;
    uint32_t pad;
};

__global__ void __launch_bounds__(256) k_value_range(const int8_t* __restrict__ a, const int8_t* __restrict__ b,
                                                     int64_t count, FilterCtl* ctl) {
    uint32_t mx = 0, par = 0;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    auto take = [&](int v) {
        mx = max(mx, (uint32_t)abs(v));
        par |= v & 1 ? 2u : 1u;
    };
    for (int64_t i = t; i < count / 4; i += step) {  // (allocations are aligned)
        const char4 x = reinterpret_cast<const char4*>(a)[i], y = reinterpret_cast<const char4*>(b)[i];
        take(x.x); take(x.y); take(x.z); take(x.w);
        take(y.x); take(y.y); take(y.z); take(y.w);
    }
    for (int64_t i = count / 4 * 4 + t; i < count; i += step) {
        take(a[i]);
        take(b[i]);
    }
    // one atomic of each kind per block (they are applied one at a time, 10 ns apart)
    __shared__ uint32_t part[2][4];
    for (int o = 32; o; o >>= 1) {
        mx = max(mx, (uint32_t)__shfl_xor((int)mx, o));
        par |= (uint32_t)__shfl_xor((int)par, o);
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = mx;
        part[1][threadIdx.x >> 6] = par;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(&ctl->mx, max(max(part[0][0], part[0][1]), max(part[0][2], part[0][3])));
        atomicOr(&ctl->parity, part[1][0] | part[1][1] | part[1][2] | part[1][3]);
    }
}

constexpr uint32_t kNoPair = 0xFFFFFFFFu;

// Pair i before pair j in (a, b) order (golay.h:25-31)?
__device__ __forceinline__ bool pair_before(const int8_t* __restrict__ pa, const int8_t* __restrict__ pb, int n,
                                            uint32_t i, uint32_t j) {
    for (int p = 0; p < n; ++p) {
        const int x = pa[(int64_t)i * n + p], y = pa[(int64_t)j * n + p];
        if (x != y) return x < y;
    }
    for (int p = 0; p < n; ++p) {
        const int x = pb[(int64_t)i * n + p], y = pb[(int64_t)j * n + p];
        if (x != y) return x < y;
    }
    return false;
}

// Open addressing over the CW words of the orbit minimum (at most half full).  A
// slot once taken stays with its class, and holds the class's least pair so far.
__global__ void __launch_bounds__(256) k_class_insert(const uint64_t* __restrict__ canon, int CW,
                                                      const int8_t* __restrict__ pa, const int8_t* __restrict__ pb,
                                                      int n, int64_t m, uint32_t* slot, uint64_t mask) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t* k = canon + i * CW;
        uint64_t h = 0x9e3779b97f4a7c15ull;
        for (int w = 0; w < CW; ++w) h = splitmix64(h ^ k[w]);
        for (uint64_t s = h & mask;; s = (s + 1) & mask) {
            uint32_t j = __hip_atomic_load(&slot[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (j == kNoPair) j = atomicCAS(&slot[s], kNoPair, (uint32_t)i);
            if (j == kNoPair) break;
            bool same = true;
            for (int w = 0; w < CW && same; ++w) same = canon[(int64_t)j * CW + w] == k[w];
            if (!same) continue;
            while (pair_before(pa, pb, n, (uint32_t)i, j)) {
                const uint32_t was = atomicCAS(&slot[s], j, (uint32_t)i);
                if (was == j) break;
                j = was;
            }
            break;
        }
    }
}

// One block per kKeepSlots slots, with one atomic.
constexpr int kKeepSlots = 1024;
__global__ void __launch_bounds__(256) k_class_keep(const uint32_t* __restrict__ slot, uint32_t* __restrict__ keep,
                                                    FilterCtl* ctl) {
    __shared__ uint32_t part[4], base;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint4 x = reinterpret_cast<const uint4*>(slot)[(int64_t)blockIdx.x * (kKeepSlots / 4) + t];
    const uint32_t v[4] = {x.x, x.y, x.z, x.w};
    uint32_t mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) mine += v[j] != kNoPair;
    uint32_t incl = mine;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d);
        if (lane >= d) incl += y;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    if (t == 0) base = atomicAdd(&ctl->kept, part[0] + part[1] + part[2] + part[3]);
    __syncthreads();
    uint32_t at = base + incl - mine;
    for (int w = 0; w < wave; ++w) at += part[w];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (v[j] != kNoPair) keep[at++] = v[j];
}

// Key words of the kept pairs, a then b, as packed for the orbit minima (E values
// a word, the first one highest): the first word of each pair in a column, the
// other 2 wn - 1 together.
__global__ void __launch_bounds__(256) k_keep_keys(FilterParams P, const int8_t* __restrict__ pa,
                                                   const int8_t* __restrict__ pb, const uint32_t* __restrict__ keep,
                                                   int64_t kept, int wn, uint64_t* __restrict__ first,
                                                   uint64_t* __restrict__ rest) {
    for (int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; x < kept * 2 * wn;
         x += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = x / (2 * wn);
        const int w = (int)(x - i * 2 * wn), j0 = (w < wn ? w : w - wn) * P.E, j1 = min(j0 + P.E, P.n);
        const int8_t* v = (w < wn ? pa : pb) + (int64_t)keep[i] * P.n;
        uint64_t acc = 0;
        for (int j = j0; j < j1; ++j) acc = acc << P.B | (uint64_t)((v[j] + P.mx) >> P.sh);
        if (w == 0) first[i] = acc;
        else rest[i * (2 * wn - 1) + w - 1] = acc;
    }
}

__global__ void __launch_bounds__(256) k_keep_rows(const int8_t* __restrict__ pa, const int8_t* __restrict__ pb, int n,
                                                   const uint32_t* __restrict__ keep,
                                                   const uint32_t* __restrict__ order, int64_t kept,
                                                   int8_t* __restrict__ oa, int8_t* __restrict__ ob) {
    for (int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; x < kept * n;
         x += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = x / n, src = (int64_t)keep[order[i]] * n + (x - i * n);
        oa[x] = pa[src];
        ob[x] = pb[src];
    }
}

int filter_pairs(gp_ctx* ctx, int order, int compress, const gp_pairs& in, PairSet& out, gp_stats* stats) {
    const int n = order / compress;
    out.n = n;
    out.a.clear();
    out.b.clear();
    if (in.count < 0 || (in.count > 0 && (!in.a || !in.b))) throw ArgError("bad pair set");
    const int64_t m = in.n == 0 ? 0 : in.count;  // (pairs of no letters: none)
    if (m == 0) return GP_OK;
    if (in.n != n) throw ArgError("filter: pair length != order/compress");
    if (n > kMaxN) throw ArgError("filter: length above 64");
    // (pair numbers are 32 bits, all ones an empty slot)
    if (m >= (int64_t)kNoPair) throw ArgError("filter: more than 2^32 - 2 pairs");
    FilterParams P{};
    P.n = n;
    P.alt = !(compress > 1 || n % 2 == 1);  // filter.cpp:83-87
    for (int u = 1; u < n || (n == 1 && u == 1); ++u)
        if (std::gcd(u, n) == 1) P.units[P.nunits++] = u;
    if (n == 1) { P.nunits = 1; P.units[0] = 0; }
    hipStream_t st = ctx->stream;
    Phase ph("filter: upload");
    int8_t* da = ctx->dev<int8_t>("f_a", (size_t)m * n);
    int8_t* db = ctx->dev<int8_t>("f_b", (size_t)m * n);
    FilterCtl* ctl = ctx->dev<FilterCtl>("f_ctl", 1);
    GP_HIP(hipMemsetAsync(ctl, 0, sizeof(FilterCtl), st));
    copy_to_device(ctx, da, in.a, (size_t)m * n);
    copy_to_device(ctx, db, in.b, (size_t)m * n);
    const auto blocks = [&](int64_t threads, int per_cu) {
        return dim3((unsigned)std::min<int64_t>((threads + 255) / 256, (int64_t)ctx->num_cus * per_cu));
    };
    hipLaunchKernelGGL(k_value_range, blocks((m * n + 15) / 16, 2), dim3(256), 0, st, da, db, m * n, ctl);
    GP_HIP(hipGetLastError());
    FilterCtl h{};
    GP_HIP(hipMemcpyAsync(&h, ctl, sizeof h, hipMemcpyDeviceToHost, st));
    GP_HIP(hipStreamSynchronize(st));
    ph.next("filter: device");
    // key packing: the values and their negations lie in [-mx, mx]; halve when all
    // have mx's parity (every v + mx even)
    const int mx = (int)h.mx;
    P.mx = mx;
    P.sh = h.parity == (mx & 1 ? 2u : 1u) ? 1 : 0;
    const int range = (2 * mx) >> P.sh;
    P.B = range <= 1 ? 1 : range <= 3 ? 2 : range <= 15 ? 4 : 8;
    P.E = 64 / P.B;
    const int wneed = (n + P.E - 1) / P.E;
    // (the letter -128 has no negative in a byte: by letters)
    const int W = mx > 127 || wneed > 2 ? (wneed <= 4 ? 4 : 8) : wneed <= 1 ? 1 : 2, CW = 2 * W;
    uint64_t* dc = ctx->dev<uint64_t>("f_c", (size_t)m * CW);
    uint64_t slots = kKeepSlots;
    while (slots < 2 * (uint64_t)m) slots <<= 1;
    uint32_t* slot = ctx->dev<uint32_t>("f_slot", slots);
    uint32_t* keep = ctx->dev<uint32_t>("f_keep", (size_t)m);
    if (stats) GP_HIP(hipEventRecord(ctx->ev0, st));  // (the look at the values, 3 us, is not counted)
    const dim3 grid((unsigned)std::min<int64_t>((m + 3) / 4, (int64_t)ctx->num_cus * 16));
    const auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, P, da, db, m, dc); };
    if (W == 1 && n * P.B <= 32) launch(k_orbit_bits<uint32_t>);
    else if (W == 1) launch(k_orbit_bits<uint64_t>);
    else if (W == 2) launch(k_orbit_bits<u128>);
    else if (W == 4) launch(k_orbit_min<4>);
    else launch(k_orbit_min<8>);
    GP_HIP(hipGetLastError());
    GP_HIP(hipMemsetAsync(slot, 0xFF, slots * 4, st));
    hipLaunchKernelGGL(k_class_insert, blocks(m, 8), dim3(256), 0, st, dc, CW, da, db, n, m, slot, slots - 1);
    hipLaunchKernelGGL(k_class_keep, dim3((unsigned)(slots / kKeepSlots)), dim3(256), 0, st, slot, keep, ctl);
    GP_HIP(hipGetLastError());
    if (stats) GP_HIP(hipEventRecord(ctx->ev1, st));
    GP_HIP(hipMemcpyAsync(&h, ctl, sizeof h, hipMemcpyDeviceToHost, st));
    GP_HIP(hipStreamSynchronize(st));
    ph.next("filter: order");
    const int64_t kept = h.kept;
    uint64_t* first = ctx->dev<uint64_t>("f_first", (size_t)kept);
    uint64_t* rest = ctx->dev<uint64_t>("f_rest", (size_t)kept * (2 * wneed - 1));
    if (stats) GP_HIP(hipEventRecord(ctx->ev2, st));
    hipLaunchKernelGGL(k_keep_keys, blocks(kept * 2 * wneed, 8), dim3(256), 0, st, P, da, db, keep, kept, wneed, first,
                       rest);
    GP_HIP(hipGetLastError());
    const MergeSorted s = merge_sort(ctx, "f_sort", first, kept, rest, 2 * wneed - 1);
    int8_t* oa = ctx->dev<int8_t>("f_oa", (size_t)kept * n);
    int8_t* ob = ctx->dev<int8_t>("f_ob", (size_t)kept * n);
    hipLaunchKernelGGL(k_keep_rows, blocks(kept * n, 8), dim3(256), 0, st, da, db, n, keep, s.idx, kept, oa, ob);
    GP_HIP(hipGetLastError());
    if (stats) GP_HIP(hipEventRecord(ctx->ev3, st));
    out.a.resize((size_t)kept * n);
    out.b.resize((size_t)kept * n);
    copy_to_host(ctx, out.a.data(), oa, out.a.size());
    copy_to_host(ctx, out.b.data(), ob, out.b.size());
    GP_HIP(hipStreamSynchronize(st));
    if (stats) {
        float ms = 0, ms_order = 0;
        GP_HIP(hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        GP_HIP(hipEventElapsedTime(&ms_order, ctx->ev2, ctx->ev3));
        stats->kernel_ms += ms + ms_order;
        stats->pairs += (uint64_t)kept;
    }
    return GP_OK;
}

}  // namespace gp

using namespace gp;
namespace gp {
int guarded_call(gp_ctx* ctx, const std::function<int()>& f);
}

extern "C" int gp_filter(gp_ctx* ctx, int order, int compress, const gp_pairs* in, gp_pairs* out, gp_stats* stats) {
    if (!ctx) return GP_ERR_ARG;
    return guarded_call(ctx, [&] {
        GP_HIP(hipSetDevice(ctx->device));
        if (!in || !out || order <= 0 || compress <= 0) throw ArgError("gp_filter: bad arguments");
        PairSet o;
        int rc = filter_pairs(ctx, order, compress, *in, o, stats);
        if (rc != GP_OK) return rc;
        return export_pairs(o, out, false);
    });
}
