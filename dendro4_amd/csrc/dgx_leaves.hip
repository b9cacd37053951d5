// dgx_leaves.hip -- the textbook leaves of points2Octree from the sorted point
// keys (step 3 and 4 of dgx_octree.hip): which points begin a leaf, the leaf's
// level, and the empty leaves in the gaps.
//
// Everything about a leaf is local: its level is one more than the longest
// common prefix of the pairs (p_i, p_{i+m}) around a point, and the gap before it
// follows from the leaf of the previous point.  So two passes over the keys do it,
// in tiles of 512 points: one counts the octants of each tile, and after a scan of
// the tiles' counts one writes them, one lane per octant.  Bound: HBM (keys read twice, octants written once).  Levels, leaf
// keys, heads, their scan and compaction, gap counts and their scan were passes of
// their own over arrays of n keys or words: 3.18 ms of kernels on 64M points and
// 199 us on 4M, now 1.15 ms and 85 us.
#include "dgx_octree.h"

namespace {

constexpr uint32_t LB = 256;
// A tile is PER points for each of NT threads.  Below kSmallN points tiles of 512
// leave most of the chip idle (k_leaf_emit on 4096 points: 13.2 us with 8 tiles,
// 8.4 with 64); above it they read less halo per point.
constexpr size_t kSmallN = size_t(1) << 16;
struct LargeTile {
    static constexpr uint32_t NT = 256, PER = 2, N = NT * PER;
};
struct SmallTile {
    static constexpr uint32_t NT = 64, PER = 1, N = NT * PER;
};

// Sum of the digits of levels t0 and up of a key whose digits past its level are 0.
__device__ __forceinline__ uint32_t digit_sum(const Key &k, uint32_t t0) {
    constexpr uint64_t M = 0x1249249249249249ull;  // the lowest bit of each digit
    const uint64_t hi = t0 <= 21 ? k.hi & ((1ull << (66 - 3 * t0)) - 1ull) : 0ull,
                   lo = (t0 <= 22 ? k.lo : k.lo & ((1ull << (66 - 3 * (t0 - 21))) - 1ull)) & ~31ull;
    return (uint32_t)(__popcll(hi & M) + __popcll(lo & M) + 2 * (__popcll(hi & (M << 1)) + __popcll(lo & (M << 1))) +
                      4 * (__popcll(hi & (M << 2)) + __popcll(lo & (M << 2))));
}
// Octants of the coarsest completion after A, and strictly between A and B (A < B
// disjoint, k levels in common); before B it is digit_sum(B, 1).
__device__ __forceinline__ uint32_t gap_after(const Key &A) { return 7 * key_level(A) - digit_sum(A, 1); }
__device__ __forceinline__ uint32_t gap_between(const Key &A, const Key &B, uint32_t k) {
    return key_digit(B, k + 1) - key_digit(A, k + 1) - 1 + 7 * (key_level(A) - k - 1) - digit_sum(A, k + 2) +
           digit_sum(B, k + 2);
}
// Octants that point j emits: for the first point of a leaf the gap before it and
// the leaf, for the last point of all the gap after it as well.  Consecutive
// leaves must be disjoint and increasing; otherwise *err is raised (the host then
// refuses the result).
__device__ __forceinline__ uint32_t point_count(size_t j, size_t n, const Key &A, const Key &B, uint32_t *err) {
    uint32_t c = 0;
    if (j == 0) {
        c = 1 + digit_sum(B, 1);
    } else if (!key_eq(A, B)) {
        const uint32_t k = key_common_levels(A, B);
        if (k >= min(key_level(A), key_level(B)) || key_digit(B, k + 1) <= key_digit(A, k + 1)) {
            if (err) atomicOr(err, 1u);
            return 0;
        }
        c = 1 + gap_between(A, B, k);
    }
    return j + 1 == n ? c + gap_after(B) : c;
}

// The workgroup's exclusive prefix of v and the total.
template <typename TL>
__device__ __forceinline__ uint32_t tile_scan(uint32_t v, uint32_t *s, uint32_t &total) {
    uint32_t wt;
    const uint32_t ex = wave_excl_sum(v, wt), w = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0) s[w] = wt;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t i = 0; i < TL::NT / 64; ++i) {
        before += i < w ? s[i] : 0u;
        total += s[i];
    }
    __syncthreads();
    return ex + before;
}

// For maxNumPts above kLeafWindow: common levels of (p_i, p_{i+m}), then the leaf
// level of each point, by passes over global memory.
__global__ void __launch_bounds__(LB) k_leaf_pairs(const Key *__restrict__ pk, size_t n, uint32_t m, uint32_t md,
                                                   uint8_t *__restrict__ lev) {
    const size_t i = (size_t)blockIdx.x * LB + threadIdx.x;
    if (i + m < n) lev[i] = (uint8_t)min(key_common_levels(pk[i], pk[i + m]), md - 1);
}
__global__ void __launch_bounds__(LB) k_leaf_levels(size_t n, uint32_t m, const uint8_t *__restrict__ lev,
                                                    uint8_t *__restrict__ leaf) {
    const size_t j = (size_t)blockIdx.x * LB + threadIdx.x;
    if (j >= n) return;
    const size_t lo = j >= m ? j - m : 0, hi = min(j, n - m - 1);
    uint32_t L = 0;
    for (size_t i = lo; i <= hi; ++i) L = max(L, (uint32_t)lev[i]);
    leaf[j] = (uint8_t)(L + 1);
}

// Points whose windows of m pairs are read from LDS (one tile and m points on
// either side).  Beyond it the halo would cost more than the extra passes.
constexpr uint32_t kLeafWindow = 64;

// Octants of each tile; leaf[j], the level of point j's leaf, is made here (WINDOW)
// or read.  *sat is raised by a leaf at level md.
template <bool WINDOW, typename TL>
__global__ void __launch_bounds__(TL::NT) k_leaf_count(const Key *__restrict__ pk, size_t n, uint32_t m, uint32_t md,
                                                   uint8_t *__restrict__ leaf, uint32_t *__restrict__ cnt,
                                                   uint32_t *err, uint32_t *sat, const uint32_t *unsorted) {
    __shared__ Key sk[TL::N + 1 + (WINDOW ? 2 * kLeafWindow : 0)];  // points base - 1 - m ... with a window
    __shared__ uint8_t sp[WINDOW ? TL::N + 1 + kLeafWindow : 1], sl[TL::N + 1];
    __shared__ uint32_t s_scan[TL::NT / 64];
    const size_t base = (size_t)blockIdx.x * TL::N;
    const uint32_t h = WINDOW ? m : 0, none = *unsorted;
    // index q of sk is point base - 1 - h + q
    for (uint32_t q = threadIdx.x; q < TL::N + 1 + 2 * h; q += TL::NT) {
        const size_t g = base + q;  // one more than the point, plus h
        if (g > h && g - 1 - h < n) sk[q] = pk[g - 1 - h];
    }
    if (!WINDOW)
        for (uint32_t q = threadIdx.x; q < TL::N + 1; q += TL::NT)
            if (base + q > 0 && base + q - 1 < n) sl[q] = leaf[base + q - 1];
    __syncthreads();
    if (none) return;  // set by a launch before: the same for every thread
    if (WINDOW) {
        for (uint32_t q = threadIdx.x; q < TL::N + 1 + m; q += TL::NT) {  // pair (q, q + m)
            const size_t g = base + q;
            sp[q] = g > m && g - 1 < n ? (uint8_t)min(key_common_levels(sk[q], sk[q + m]), md - 1) : (uint8_t)0;
        }
        __syncthreads();
        for (uint32_t q = threadIdx.x; q < TL::N + 1; q += TL::NT) {
            uint32_t L = 0;
            for (uint32_t i = 0; i <= m; ++i) L = max(L, (uint32_t)sp[q + i]);
            sl[q] = (uint8_t)(L + 1);
            if (q && base + q - 1 < n) leaf[base + q - 1] = (uint8_t)(L + 1);
        }
        __syncthreads();
    }
    uint32_t c = 0;
    bool full = false;
#pragma unroll
    for (uint32_t r = 0; r < TL::PER; ++r) {
        const uint32_t q = threadIdx.x * TL::PER + r + 1;
        const size_t j = base + q - 1;
        if (j >= n) continue;
        const Key Bk = key_truncate(sk[q + h], sl[q]);
        c += point_count(j, n, j ? key_truncate(sk[q + h - 1], sl[q - 1]) : Bk, Bk, err);
        full = full || sl[q] == md;
    }
    uint32_t total;
    tile_scan<TL>(c, s_scan, total);
    if (threadIdx.x == 0) cnt[blockIdx.x] = total;
    if (__ballot(full) && (threadIdx.x & 63u) == 0) atomicOr(sat, 1u);
}

__device__ __forceinline__ Key with_digit(const Key &base, uint32_t t, uint32_t r) {
    Key k = key_truncate(base, t);
    key_set_digit(k, t, r);
    return k;
}
// The octants of each tile, at off[tile].  A lane makes one octant at a time: its
// point by binary search in the points' prefix counts, its level and digit by
// running through the gap's levels (7 - digit octants after A at a level, digit
// octants before B).  Stores are whole lines; a lane per point emitting its
// octants in turn took 915 us for 64M points instead of 683.  SAT (some leaf is at
// level md): also each octant's first point tb, and the number of points tc of the
// leaves at level md (0 for other octants; nothing reads theirs).
template <bool SAT, typename TL>
__global__ void __launch_bounds__(TL::NT) k_leaf_emit(const Key *__restrict__ pk, size_t n, uint32_t md,
                                                  const uint8_t *__restrict__ leaf, const uint32_t *__restrict__ off,
                                                  Key *__restrict__ T, uint32_t *__restrict__ tb,
                                                  uint32_t *__restrict__ tc) {
    __shared__ Key sk[TL::N + 1];
    __shared__ uint8_t sl[TL::N + 1];
    __shared__ uint32_t s_scan[TL::NT / 64], s_pre[TL::N];
    const size_t base = (size_t)blockIdx.x * TL::N;
    for (uint32_t q = threadIdx.x; q < TL::N + 1; q += TL::NT)
        if (base + q > 0 && base + q - 1 < n) {
            sl[q] = leaf[base + q - 1];
            sk[q] = key_truncate(pk[base + q - 1], sl[q]);
        }
    __syncthreads();
    uint32_t c[TL::PER], sum = 0;
#pragma unroll
    for (uint32_t r = 0; r < TL::PER; ++r) {
        const uint32_t q = threadIdx.x * TL::PER + r + 1;
        const size_t j = base + q - 1;
        c[r] = j < n ? point_count(j, n, sk[j ? q - 1 : q], sk[q], nullptr) : 0u;
        sum += c[r];
    }
    uint32_t total;
    uint32_t pre = tile_scan<TL>(sum, s_scan, total);
#pragma unroll
    for (uint32_t r = 0; r < TL::PER; ++r) {
        s_pre[threadIdx.x * TL::PER + r] = pre;
        pre += c[r];
    }
    __syncthreads();
    const size_t o0 = off[blockIdx.x];
    for (uint32_t o = threadIdx.x; o < total; o += TL::NT) {
        uint32_t q = 0;  // the last point with a prefix <= o
#pragma unroll
        for (uint32_t step = TL::N / 2; step; step >>= 1)
            if (s_pre[q + step] <= o) q += step;
        uint32_t r = o - s_pre[q];
        const size_t j = base + q;
        const Key Bk = sk[q + 1], A = sk[j ? q : q + 1];
        const uint32_t lb = key_level(Bk);
        uint32_t b0 = (uint32_t)j, cn = 0;
        Key out = Bk;
        // octant r of those after P, the deepest level first
        auto after = [&](const Key &P, uint32_t r_) {
            uint32_t t = key_level(P), w;
            while ((w = 7u - key_digit(P, t)) <= r_) {
                r_ -= w;
                --t;
            }
            return with_digit(P, t, key_digit(P, t) + 1 + r_);
        };
        bool tail = true;
        if (j == 0 || !key_eq(A, Bk)) {
            uint32_t t0 = 1, na = 0, nm = 0;
            if (j) {
                const uint32_t k = key_common_levels(A, Bk);
                na = 7 * (key_level(A) - k - 1) - digit_sum(A, k + 2);
                nm = key_digit(Bk, k + 1) - key_digit(A, k + 1) - 1;
                t0 = k + 2;
            }
            const uint32_t nb = digit_sum(Bk, t0);
            tail = false;
            if (r < na) {
                out = after(A, r);
            } else if (r < na + nm) {
                out = with_digit(A, t0 - 1, key_digit(A, t0 - 1) + 1 + (r - na));
            } else if (r < na + nm + nb) {
                r -= na + nm;
                uint32_t t = t0, w;
                while ((w = key_digit(Bk, t)) <= r) {
                    r -= w;
                    ++t;
                }
                out = with_digit(Bk, t, r);
            } else if (r == na + nm + nb) {
                if (SAT && lb == md) {  // the points of the cell are the equal keys from j on
                    const Key P = pk[j];
                    size_t lo = j + 1, step = 1, hi = j + 1;
                    while (hi < n && key_eq(pk[hi], P)) {
                        lo = hi + 1;
                        hi = min(n, hi + step);
                        step *= 2;
                    }
                    while (lo < hi) {
                        const size_t mid = lo + (hi - lo) / 2;
                        if (key_eq(pk[mid], P)) lo = mid + 1;
                        else hi = mid;
                    }
                    cn = (uint32_t)(lo - j);
                }
            } else {
                tail = true;
                r -= na + nm + nb + 1;
            }
        }
        if (tail) {  // behind the last point
            out = after(Bk, r);
            b0 = (uint32_t)n;
        }
        T[o0 + o] = out;
        if (SAT) {
            tb[o0 + o] = b0;
            tc[o0 + o] = cn;
        }
    }
}

}  // namespace

LeafTiles::LeafTiles(size_t n, hipStream_t s)
    : tiles(grid_for(n, n < kSmallN ? SmallTile::N : LargeTile::N)), leaf(n, s), cnt(tiles, s), off(tiles, s) {}

template <typename TL>
static void leaf_count(LeafTiles &w, const Key *pk, size_t n, uint32_t m, uint32_t md, uint32_t *err, uint32_t *sat,
                       const uint32_t *unsorted, hipStream_t s) {
    if (m <= kLeafWindow) {
        k_leaf_count<true, TL><<<w.tiles, TL::NT, 0, s>>>(pk, n, m, md, w.leaf.p, w.cnt.p, err, sat, unsorted);
    } else {
        DevBuf<uint8_t> lev(n - m, s);
        k_leaf_pairs<<<grid_for(n - m, LB), LB, 0, s>>>(pk, n, m, md, lev.p);
        k_leaf_levels<<<grid_for(n, LB), LB, 0, s>>>(n, m, lev.p, w.leaf.p);
        k_leaf_count<false, TL><<<w.tiles, TL::NT, 0, s>>>(pk, n, m, md, w.leaf.p, w.cnt.p, err, sat, unsorted);
    }
    HIP_OK(hipGetLastError());
}
template <typename TL>
static void leaf_emit(const LeafTiles &w, const Key *pk, size_t n, uint32_t md, Key *T, uint32_t *tb, uint32_t *tc,
                      hipStream_t s) {
    if (tb) k_leaf_emit<true, TL><<<w.tiles, TL::NT, 0, s>>>(pk, n, md, w.leaf.p, w.off.p, T, tb, tc);
    else k_leaf_emit<false, TL><<<w.tiles, TL::NT, 0, s>>>(pk, n, md, w.leaf.p, w.off.p, T, nullptr, nullptr);
    HIP_OK(hipGetLastError());
}
void p2o_leaf_count(LeafTiles &w, const Key *pk, size_t n, uint32_t m, uint32_t md, uint32_t *total, uint32_t *err,
                    uint32_t *sat, const uint32_t *unsorted, hipStream_t s) {
    if (n < kSmallN) leaf_count<SmallTile>(w, pk, n, m, md, err, sat, unsorted, s);
    else leaf_count<LargeTile>(w, pk, n, m, md, err, sat, unsorted, s);
    scan_exclusive_u32_async(w.cnt.p, w.off.p, w.tiles, total, s);
}
void p2o_leaf_emit(const LeafTiles &w, const Key *pk, size_t n, uint32_t md, Key *T, uint32_t *tb, uint32_t *tc,
                   hipStream_t s) {
    if (n < kSmallN) leaf_emit<SmallTile>(w, pk, n, md, T, tb, tc, s);
    else leaf_emit<LargeTile>(w, pk, n, md, T, tb, tc, s);
}
