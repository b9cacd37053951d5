// dgx_balance.hip -- 2:1 balance of a complete linear octree by searching
// (ot::balanceOctree, src/balance.cpp:55-64 -> comboRipple; one rank).
//
// The balanced octree is the closure of one rule: when an octant is split, the
// parents of its 26 neighbours are split too.  A complete sorted octree already
// holds almost all of those splits, so this path looks for the ones it lacks
// instead of rebuilding every level:
//   1. k_bal_check tests that the input is complete, sorted and linear (each
//      leaf begins where the one before it ends) and fills a table of where
//      each coarse cell begins in the leaves;
//   2. k_bal_find lists the split octants of the input (ancestors, each at its
//      first leaf), takes the up-to-7 neighbour parents of each and finds the
//      leaf that holds it: a leaf no finer than the parent means a missing
//      split.  Missing splits go into a hash set, and each new one is treated
//      like a split octant in turn, in the workgroup that found it;
//   3. k_bal_emit copies the leaves and refines, in place in the order of the
//      curve, those that hold missing splits.
// One host read (the number of new splits) lies between 2 and 3, and 3 is waited
// for.  Where 1 or 2 find that this path cannot answer, its other workgroups stop
// and the levels are rebuilt.  The rule's closure does not depend on the order in
// which splits are found, so the result is the level-by-level step's, octant for
// octant.
//
// Bound: the chains of dependent reads of the searches (about log2 of a cell's
// leaves) and of the curve encodes, hidden by many waves; 32 B per leaf of
// traffic.  It sorts nothing: the level-by-level step of balance_build sorts
// every level's seeds (about two per leaf) and then all leaves.
// Measured on MI355X, kernel time level by level -> here: 1.87M leaves
// (4,194,304 log-normal points) 1.37 -> 0.11 ms, 56M leaves (67,108,864 points
// of 16 Gaussians) 14.2 -> 2.8 ms, 8K leaves (4,096 uniform points) 0.41 ->
// 0.06 ms with 90 launches and 8 host reads fewer.
#include "dgx_octree.h"

#include <algorithm>

namespace {

constexpr uint32_t FB = 256;

struct BalFast {
    uint32_t flags;     // why this path cannot answer (BF_*); 0: it can
    uint32_t nnew;      // splits the input lacks
    uint32_t ntail;     // new splits that did not fit their workgroup's queue
    uint32_t lmax, lup;        // finest level; 31 minus the coarsest
    uint32_t ndense;           // workgroups that found many new splits
    unsigned long long seeds;  // what the level-by-level step counts as its seeds
    uint32_t spread[64][16];   // levels beside leaf 0's (BS_*): 64 copies, each in a line of its own
};
enum : uint32_t {
    BF_INCOMPLETE = 1,  // not a complete, sorted, linear octree
    BF_HASH = 2,        // the hash set or the overflow list is full
    BF_DEEP = 4,        // a missing split more than kMaxRel levels below its leaf
    BF_WIDE = 8,        // a leaf with more than kMaxSplits missing splits
    BF_MANY = 16        // the octree would grow several times over
};
enum : uint32_t { BS_FAR = 1, BS_FINER = 2, BS_COARSER = 4 };  // two levels or more, one finer, one coarser
// A missing split is a 64-bit word: the leaf that holds it, and below it a 1
// followed by its digits from the leaf's level on (3 bits a level).
constexpr uint32_t kMaxRel = 10;
// k_bal_emit refines a leaf on one wave, in time quadratic in its splits; more
// (a deep cluster against a coarse octant) are left to the level-by-level step.
constexpr uint32_t kMaxSplits = 512;
// Leaves per workgroup of k_bal_emit, and log2 of it, by leaves per thread.
constexpr uint32_t blk_shift(uint32_t lpt) { return lpt == 1 ? 8 : 10; }
constexpr uint32_t kQueue = 512;  // new splits a workgroup holds per round
constexpr uint32_t kProbes = 128;

struct Axes {
    uint32_t x, y, z, lev;
};

// Position where the octant after k on the curve begins, as digits (levels
// 1..21 in hi, 22..31 in the upper bits of lo); hi = 2^63 past the last one.
__device__ __forceinline__ void cell_end(const Key &k, uint64_t &hi, uint64_t &lo) {
    const uint32_t L = key_level(k);
    if (L <= 21) {
        hi = k.hi + (1ull << (63 - 3 * L));
        lo = 0;
    } else {
        const uint64_t v = (k.lo & ~31ull) + (1ull << (63 - 3 * (L - 21)));
        hi = k.hi + (v >> 63);
        lo = v & ~(1ull << 63);
    }
}

// Thread i: leaf i and its successor must share an end; cell i of the level-cl
// table gets the first leaf whose high word reaches it.  Also zeroes the
// counts of new splits per leaf (extra) and per workgroup of k_bal_emit (blk).
// The level range of a workgroup goes to levels[] (finest << 8 | coarsest) for
// k_bal_find_tail: an atomic per wave on one word took 95 us of 109 on 1.9M leaves.
// Whether there are leaves two levels apart at all is in st->spread, where most
// workgroups find their bits set (with 8 copies for 64 this cost 20 us on 1.9M leaves).
__global__ void __launch_bounds__(FB) k_bal_check(const Key *__restrict__ k, size_t n, uint32_t md, uint32_t cl, uint32_t bsh,
                                                  uint32_t *__restrict__ cstart, uint16_t *__restrict__ extra,
                                                  uint32_t *__restrict__ blk, uint16_t *__restrict__ levels,
                                                  BalFast *__restrict__ st) {
    __shared__ uint32_t s_lv[FB / 64][2];
    const size_t i = (size_t)blockIdx.x * FB + threadIdx.x;
    const uint32_t ncell = 1u << (3 * cl);
    bool bad = false;
    uint32_t lmax = 0, lmin = 31, l0 = 0, had = 0;
    uint32_t *sp = st->spread[blockIdx.x % 64];
    if (threadIdx.x == 0) {
        l0 = key_level(k[0]);
        had = __hip_atomic_load(sp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (i < n) {
        const Key a = k[i];
        uint64_t eh, el;
        cell_end(a, eh, el);
        uint64_t bh = 1ull << 63, bl = 0;
        if (i + 1 < n) {
            const Key b = k[i + 1];
            bh = b.hi;
            bl = b.lo & ~31ull;
        }
        lmax = lmin = key_level(a);
        bad = bh != eh || bl != el || lmax > md || (i == 0 && (a.hi | (a.lo & ~31ull)));
        extra[i] = 0;
        if ((i & ((size_t(1) << bsh) - 1)) == 0) blk[i >> bsh] = 0;
    }
    for (int o = 32; o > 0; o >>= 1) {
        lmax = max(lmax, (uint32_t)__shfl_xor(lmax, o, 64));
        lmin = min(lmin, (uint32_t)__shfl_xor(lmin, o, 64));
    }
    const uint64_t anybad = __ballot(bad);
    if ((threadIdx.x & 63u) == 0) {
        if (anybad) atomicOr(&st->flags, (uint32_t)BF_INCOMPLETE);
        s_lv[threadIdx.x >> 6][0] = lmax;
        s_lv[threadIdx.x >> 6][1] = lmin;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < FB / 64; ++w) {
            lmax = max(lmax, s_lv[w][0]);
            lmin = min(lmin, s_lv[w][1]);
        }
        levels[blockIdx.x] = (uint16_t)(lmax << 8 | lmin);
        const uint32_t bits = (max(lmax, l0) - min(lmin, l0) >= 2 ? BS_FAR : 0u) | (lmax > l0 ? BS_FINER : 0u) |
                              (lmin < l0 ? BS_COARSER : 0u);
        if (i < n && (bits & ~had)) atomicOr(sp, bits);
    }
    if (i < ncell) {
        const uint64_t h = (uint64_t)i << (63 - 3 * cl);
        size_t lo = 0, hi = n;
        while (lo < hi) {
            const size_t mid = lo + (hi - lo) / 2;
            if (k[mid].hi < h) lo = mid + 1;
            else hi = mid;
        }
        cstart[i] = (uint32_t)lo;
        if (i == 0) cstart[ncell] = (uint32_t)n;
    }
}

__device__ __forceinline__ uint64_t hash_of(uint64_t v) {
    v ^= v >> 31;
    v *= 0x9e3779b97f4a7c15ull;
    v ^= v >> 29;
    v *= 0xbf58476d1ce4e5b9ull;
    return v ^ (v >> 32);
}
// 1: inserted, 0: was there, -1: no room
__device__ __forceinline__ int hash_insert(unsigned long long *tab, uint64_t mask, uint64_t v) {
    uint64_t s = hash_of(v) & mask;
#pragma unroll 1
    for (uint32_t p = 0; p < kProbes; ++p, s = (s + 1) & mask) {
        const unsigned long long old = atomicCAS(&tab[s], 0ull, (unsigned long long)v);
        if (old == 0) return 1;
        if (old == v) return 0;
    }
    return -1;
}
__device__ __forceinline__ bool hash_has(const unsigned long long *tab, uint64_t mask, uint64_t v) {
    uint64_t s = hash_of(v) & mask;
#pragma unroll 1
    for (uint32_t p = 0; p < kProbes; ++p, s = (s + 1) & mask) {
        const unsigned long long w = tab[s];
        if (w == v) return true;
        if (w == 0) return false;
    }
    return false;
}

// Key of the octant with `path` (1, then digits) below leaf f.
__device__ __forceinline__ Key key_below(const Key &f, uint64_t path) {
    const uint32_t r = (63 - (uint32_t)__clzll(path)) / 3, l0 = key_level(f);
    Key k = f;
    for (uint32_t t = 1; t <= r; ++t) key_set_digit(k, l0 + t, (uint32_t)(path >> (3 * (r - t))) & 7u);
    k.lo = (k.lo & ~31ull) | (l0 + r);
    return k;
}

// Orders this wave's LDS accesses before and after the call.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct FindArgs {
    const Key *k;
    const uint32_t *cstart;
    uint16_t *extra;
    uint32_t *blk;
    unsigned long long *tab;
    uint64_t mask;
    unsigned long long *tail;  // overflow list of new splits
    uint32_t tail_cap, dense_cap;
    BalFast *st;
    uint32_t md, cl, bsh;
};

__device__ __forceinline__ uint32_t flags_now(const FindArgs &A) {
    return __hip_atomic_load(&A.st->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Parent t (bit a: the neighbouring one along axis a) of the neighbours of the
// split octant q.  False when it lies outside the domain.
__device__ __forceinline__ bool nbr_parent(const Axes &q, uint32_t t, uint32_t md, uint32_t c[3]) {
    const uint32_t sh = md - q.lev + 1;  // log2 of the parent's length
    const uint32_t p[3] = {q.x, q.y, q.z};
    bool ok = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const uint64_t lo = (uint64_t)(p[a] >> sh) << sh, len = 1ull << sh;
        const bool upper = (p[a] & (uint32_t)(len - 1)) != 0;
        if ((t >> a) & 1u) {
            ok = ok && (upper ? lo + len < (1ull << md) : lo >= len);
            c[a] = (uint32_t)(upper ? lo + len : lo - len);
        } else {
            c[a] = (uint32_t)lo;
        }
    }
    return ok;
}

// The octant at level lev anchored at c is required to be split.  Returns its
// word when it was not and this call is the first to record it, else 0.
// stop is set when this path cannot answer.
__device__ __forceinline__ uint64_t require_split(const FindArgs &A, const uint16_t *rc2, const uint8_t *rc,
                                                  const uint32_t c[3], uint32_t lev, volatile uint32_t &stop) {
    uint32_t rot;
    const Key pk = morton_to_curve_rot(rc2, rc, morton_encode(c[0], c[1], c[2], lev, A.md), rot);
    // the leaf that holds its first cell: the last one not after it
    const Key top{pk.hi, pk.lo | 31ull};
    const uint32_t cell = (uint32_t)(pk.hi >> (63 - 3 * A.cl));
    uint32_t lo = A.cstart[cell], hi = A.cstart[cell + 1];
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (key_le(A.k[mid], top)) lo = mid + 1;
        else hi = mid;
    }
    const uint32_t f = lo - 1;  // leaf 0 begins at 0: lo >= 1
    const uint32_t lf = key_level(A.k[f]);
    if (lf > lev) return 0;  // the input splits it
    const uint32_t r = lev - lf;
    if (r > kMaxRel) {
        atomicOr(&A.st->flags, (uint32_t)BF_DEEP);
        stop = 1;
        return 0;
    }
    uint32_t path = 1;
    for (uint32_t t = lf + 1; t <= lev; ++t) path = path << 3 | key_digit(pk, t);
    const uint64_t word = (uint64_t)f << 32 | path;
    const int got = hash_insert(A.tab, A.mask, word);
    if (got <= 0) {
        if (got < 0) {
            atomicOr(&A.st->flags, (uint32_t)BF_HASH);
            stop = 1;
        }
        return 0;
    }
    if (flags_now(A)) {
        stop = 1;
        return 0;
    }
    // One 16-bit count per leaf, two to a word.  The lanes that name the first one's
    // leaf or workgroup add together: a fine surface against one coarse leaf counts
    // all its splits on one word (8.5M leaves, 9.5 ms until each was counted).
    const uint32_t f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)f), b0 = f0 >> A.bsh;
    const uint64_t leaf = __ballot(f == f0), group = __ballot(f >> A.bsh == b0), lt = (1ull << __lane_id()) - 1ull;
    if (f != f0 || !(leaf & lt)) {
        const uint32_t sh = 16 * (f & 1u), add = f == f0 ? (uint32_t)__popcll(leaf) : 1u;
        const uint32_t was = atomicAdd((uint32_t *)A.extra + (f >> 1), add << sh) >> sh & 0xffffu;
        if (was + add > kMaxSplits) {
            atomicOr(&A.st->flags, (uint32_t)BF_WIDE);
            stop = 1;
        }
    }
    if (f >> A.bsh != b0 || !(group & lt)) atomicAdd(&A.blk[f >> A.bsh], f >> A.bsh == b0 ? (uint32_t)__popcll(group) : 1u);
    return word;
}

// Shared state of a workgroup that works through split octants.
struct FindShared {
    uint8_t rc[192], mc[192];
    uint16_t rc2[24 * 64];
    Axes q[FB];                   // the split octants of this round
    unsigned long long queue[2][kQueue];
    uint32_t nnext, seeds, nnew, dense;
    uint32_t stop;           // read between barriers only
    volatile uint32_t halt;  // set at any time: look-ups are pointless
};

// New splits that make a workgroup dense.  When one in 8 is, the octree would grow
// to several times its size, on which sorting whole levels is the faster way (a
// million points along a line, 9 times: 34 ms here before the hash set was full,
// 35 ms there); the others then stop.
constexpr uint32_t dense_splits(uint32_t leaves) { return leaves / 2; }

__device__ __forceinline__ void find_init(FindShared &S, const SfcPacked &tab) {
    for (uint32_t i = threadIdx.x; i < 192; i += FB) {
        S.rc[i] = tab.rc[i];
        S.mc[i] = tab.mc[i];
    }
    for (uint32_t i = threadIdx.x; i < 24 * 64; i += FB) S.rc2[i] = rc2_entry(tab.rc, i);
    if (threadIdx.x == 0) {
        S.nnext = S.seeds = S.nnew = S.dense = 0;
        S.stop = S.halt = 0;
    }
}

// A new split (0: none) goes to queue[dst] or, past its end, to the overflow list.
__device__ __forceinline__ void find_push(FindShared &S, const FindArgs &A, uint64_t w, uint32_t dst) {
    if (!w) return;
    atomicAdd(&S.nnew, 1u);
    const uint32_t p = atomicAdd(&S.nnext, 1u);
    if (p < kQueue) {
        S.queue[dst][p] = w;
    } else {
        const uint32_t g = atomicAdd(&A.st->ntail, 1u);
        if (g < A.tail_cap) A.tail[g] = w;
        else atomicOr(&A.st->flags, (uint32_t)BF_HASH);
    }
}

// Requires the parents and neighbour parents of the n octants in S.q (level >= 1).
// Counts those inside the domain (the seeds of the level-by-level step).
__device__ void find_round(FindShared &S, const FindArgs &A, uint32_t n, uint32_t dst) {
    uint32_t seeds = 0;
    for (uint32_t j = threadIdx.x; j < n * 8 && !S.halt; j += FB) {
        const Axes q = S.q[j / 8];
        uint32_t c[3];
        if (!nbr_parent(q, j % 8, A.md, c)) continue;
        ++seeds;
        if (q.lev < 2) continue;  // the parent is the root
        find_push(S, A, require_split(A, S.rc2, S.rc, c, q.lev - 1, S.halt), dst);
    }
    for (int o = 32; o > 0; o >>= 1) seeds += (uint32_t)__shfl_xor(seeds, o, 64);
    if ((threadIdx.x & 63u) == 0 && seeds) atomicAdd(&S.seeds, seeds);
}

// Works through the new splits in queue[cur] until no more follow from them, or
// some workgroup has found that this path cannot answer.  many: dense_splits.
__device__ void find_drain(FindShared &S, const FindArgs &A, uint32_t cur, uint32_t many) {
    for (;;) {
        __syncthreads();
        const uint32_t n = S.stop ? 0u : min(S.nnext, kQueue);
        __syncthreads();
        if (!n) break;
        if (threadIdx.x == 0) {
            S.nnext = 0;
            S.stop = flags_now(A);
            if (S.nnew > many && !S.dense) {
                S.dense = 1;
                if (atomicAdd(&A.st->ndense, 1u) + 1 == A.dense_cap) atomicOr(&A.st->flags, (uint32_t)BF_MANY);
            }
        }
        for (uint32_t b = 0; b < n; b += FB) {
            const uint32_t m = min(n - b, FB);
            __syncthreads();
            if (threadIdx.x < m) {
                const uint64_t w = S.queue[cur][b + threadIdx.x];
                Axes q;
                dev_decode(S.mc, key_below(A.k[w >> 32], (uint32_t)w), A.md, q.x, q.y, q.z, q.lev);
                S.q[threadIdx.x] = q;
            }
            __syncthreads();
            // a new split's own parent may be missing too; level 0 cannot be new
            find_round(S, A, m, cur ^ 1u);
        }
        cur ^= 1u;
    }
}
// The first round of a workgroup: the octants' own parents are split (they hold
// them), and neighbour parents that several of its split octants share are looked up once.  Some 140
// split octants of 1024 leaves name 1000 neighbour parents, about 100 of them
// different, and a look-up (key on the curve, binary search in memory) costs far
// more than finding out: a parent's place relative to the first one, in its own
// size, and its level are one word of an LDS hash table.  A parent too far away
// for the word, or that finds no slot, is looked up as it is.  With one look-up per
// name, and 36 KB of LDS instead of 20, k_bal_find took 1986 us on the leaves of 64M
// points instead of 979, 70 us instead of 39 on those of 4M.
constexpr uint32_t kSeen = kQueue, kSeenProbes = 8;
__device__ void find_first(FindShared &S, const FindArgs &A, uint32_t n, uint16_t *todo, uint32_t *ntodo) {
    unsigned long long *seen = S.queue[1];  // not in use yet
    for (uint32_t i = threadIdx.x; i < kSeen; i += FB) seen[i] = 0;
    if (threadIdx.x == 0) *ntodo = 0;
    __syncthreads();
    uint32_t seeds = threadIdx.x < n ? 1u : 0u;  // the octant's own parent
    const Axes o = S.q[0];
    for (uint32_t j = threadIdx.x; j < n * 7; j += FB) {
        const Axes q = S.q[j / 7];
        uint32_t c[3];
        if (!nbr_parent(q, 1 + j % 7, A.md, c)) continue;
        ++seeds;
        if (q.lev < 2) continue;  // the parent is the root
        const uint32_t sh = A.md - q.lev + 1, ref[3] = {o.x, o.y, o.z};
        uint64_t w = 1ull << 62 | (uint64_t)q.lev << 57;
        bool near = true;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const uint32_t d = (c[a] >> sh) - (ref[a] >> sh) + (1u << 18);
            near = near && d < (1u << 19);
            w |= (uint64_t)(d & 0x7ffffu) << (19 * a);
        }
        bool mine = !near;
        if (near) {
            uint32_t s = (((uint32_t)w * 0x9e3779b1u ^ (uint32_t)(w >> 32) * 0x85ebca6bu) >> 20) & (kSeen - 1);
            uint32_t p = 0;
            for (; p < kSeenProbes; ++p, s = (s + 1) & (kSeen - 1)) {
                const unsigned long long was = atomicCAS(&seen[s], 0ull, (unsigned long long)w);
                if (was == 0ull) mine = true;
                if (was == 0ull || was == w) break;
            }
            mine = mine || p == kSeenProbes;
        }
        if (mine) todo[atomicAdd(ntodo, 1u)] = (uint16_t)j;
    }
    for (int k = 32; k > 0; k >>= 1) seeds += (uint32_t)__shfl_xor(seeds, k, 64);
    if ((threadIdx.x & 63u) == 0 && seeds) atomicAdd(&S.seeds, seeds);
    __syncthreads();
    const uint32_t m = *ntodo;
    for (uint32_t i = threadIdx.x; i < m && !S.halt; i += FB) {
        const uint32_t j = todo[i];
        const Axes q = S.q[j / 7];
        uint32_t c[3];
        nbr_parent(q, 1 + j % 7, A.md, c);
        find_push(S, A, require_split(A, S.rc2, S.rc, c, q.lev - 1, S.halt), 0);
    }
}
// LPT leaves per thread.  The split octants whose first leaf lies in the
// workgroup's FB * LPT leaves: at most (FB LPT - 1) / 7 inside it and a chain
// of 31 that reach past it.  One leaf per thread while that leaves CUs idle.
template <uint32_t LPT>
__global__ void __launch_bounds__(FB) k_bal_find(FindArgs A, size_t n, SfcPacked tab, uint32_t *__restrict__ seeds) {
    constexpr uint32_t NL = FB * LPT;
    __shared__ FindShared S;
    __shared__ uint16_t s_int[FB];  // leaf in the workgroup << 5 | level of the ancestor
    __shared__ uint32_t s_nint;
    __shared__ uint16_t s_todo[7 * FB];
    static_assert((NL - 1) / 7 + 31 < FB, "split octants of one workgroup fit one round");
    uint32_t sp = threadIdx.x < 64 ? A.st->spread[threadIdx.x][0] : 0u, fl = threadIdx.x == 0 ? flags_now(A) : 0u;
    find_init(S, tab);
    for (int o = 32; o > 0; o >>= 1) sp |= (uint32_t)__shfl_xor((int)sp, o, 64);
    if (threadIdx.x == 0) {
        s_nint = 0;
        // leaves of two neighbouring levels lack nothing
        if (fl || (!(sp & BS_FAR) && (sp & (BS_FINER | BS_COARSER)) != (BS_FINER | BS_COARSER))) S.stop = 1;
        if (S.stop) seeds[2 * (size_t)blockIdx.x] = seeds[2 * (size_t)blockIdx.x + 1] = 0;
    }
    __syncthreads();
    if (S.stop) return;
    const size_t i0 = (size_t)blockIdx.x * NL;
    for (uint32_t e = 0; e < LPT; ++e) {
        const uint32_t j = e * FB + threadIdx.x;
        if (i0 + j >= n) break;
        const Key k = A.k[i0 + j];
        // ancestors whose first leaf this is: one per trailing zero digit
        const uint32_t L = key_level(k);
        for (uint32_t t = L; t >= 2 && key_digit(k, t) == 0; --t) {
            const uint32_t p = atomicAdd(&s_nint, 1u);
            if (p < FB) s_int[p] = (uint16_t)(j << 5 | (t - 1));
        }
    }
    __syncthreads();
    const uint32_t ni = min(s_nint, FB);
    if (threadIdx.x < ni) {
        const uint32_t v = s_int[threadIdx.x];
        Axes q;
        dev_decode(S.mc, key_truncate(A.k[i0 + (v >> 5)], v & 31u), A.md, q.x, q.y, q.z, q.lev);
        S.q[threadIdx.x] = q;
    }
    __syncthreads();
    find_first(S, A, ni, s_todo, &s_nint);
    find_drain(S, A, 0, dense_splits(NL));
    if (threadIdx.x == 0) {
        seeds[2 * (size_t)blockIdx.x] = S.seeds;
        seeds[2 * (size_t)blockIdx.x + 1] = S.nnew;
    }
}

__device__ __forceinline__ unsigned long long block_sum(unsigned long long v, unsigned long long *lds) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63u) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0;
    for (uint32_t w = 0; w < FB / 64; ++w) v += lds[w];
    return v;
}

// The new splits that found no room in their workgroup's queue, by the first
// workgroup; those it adds itself past its own queue follow in the list.  And the
// sums over the launches before, a share per workgroup: nfind counts of seeds and
// new splits, ncheck level ranges.
__global__ void __launch_bounds__(FB) k_bal_find_tail(FindArgs A, SfcPacked tab, const uint32_t *seeds, uint32_t nfind,
                                                      const uint16_t *levels, uint32_t ncheck) {
    __shared__ FindShared S;
    __shared__ uint32_t s_end;
    __shared__ unsigned long long s_sum[FB / 64];
    if (threadIdx.x == 0) {
        S.seeds = S.nnew = 0;
        S.stop = flags_now(A);
    }
    __syncthreads();
    if (S.stop) return;
    if (blockIdx.x == 0 && A.st->ntail) {
        find_init(S, tab);
        uint32_t at = 0;
        for (;;) {
            __syncthreads();
            if (threadIdx.x == 0)
                s_end = min(__hip_atomic_load(&A.st->ntail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), A.tail_cap);
            __syncthreads();
            const uint32_t m = min(s_end - at, kQueue);
            if (!m || S.stop) break;
            for (uint32_t j = threadIdx.x; j < m; j += FB) S.queue[0][j] = A.tail[at + j];
            if (threadIdx.x == 0) S.nnext = m;
            at += m;
            find_drain(S, A, 0, ~0u);
        }
    }
    __syncthreads();
    const uint32_t i0 = blockIdx.x * FB + threadIdx.x, step = gridDim.x * FB;
    unsigned long long nnew = 0, nseed = 0;
    uint32_t lmax = 0, lup = 0;
#pragma unroll 8
    for (uint32_t b = i0; b < nfind; b += step) {
        const uint2 v = reinterpret_cast<const uint2 *>(seeds)[b];
        nseed += v.x;
        nnew += v.y;
    }
#pragma unroll 8
    for (uint32_t b = i0; b < ncheck; b += step) {
        const uint32_t v = levels[b];
        lmax = max(lmax, v >> 8);
        lup = max(lup, 31u - (v & 255u));
    }
    nnew = block_sum(nnew, s_sum);
    nseed = block_sum(nseed, s_sum);
    for (int o = 32; o > 0; o >>= 1) {
        lmax = max(lmax, (uint32_t)__shfl_xor(lmax, o, 64));
        lup = max(lup, (uint32_t)__shfl_xor(lup, o, 64));
    }
    if ((threadIdx.x & 63u) == 0) {
        atomicMax(&A.st->lmax, lmax);
        atomicMax(&A.st->lup, lup);
    }
    if (threadIdx.x == 0) {
        atomicAdd(&A.st->nnew, (uint32_t)nnew + S.nnew);
        atomicAdd(&A.st->seeds, nseed + S.seeds);
    }
}

// Output of the leaves, LPT per thread: 4, or 1 where that leaves CUs idle (4,096
// uniform points 21.9 us with 9 workgroups, 9.0 with 36).  base[b] (nullptr: summed
// here) counts the new splits in the workgroups before b; each adds 7 octants.
// A leaf with one new split is split itself and nothing below it: its thread
// stores the 8 children.  A leaf with more is a wave's: it finds the leaf's
// splits breadth first, 8 splits' children per round of hash reads, until it
// has them all, and then stores every unsplit child at its place, which
// follows from counting the splits before it:
//   place of octant o = sum of o's digits below the leaf
//                       + 7 (splits that begin before o and do not hold o).
// One thread per leaf, depth first, waited for one hash read per octant:
// 113 us on the octree of 4,096 uniform points against 21 us, 162 against
// 29 us on the levels of a hierarchy of 3,000,000 points.
template <uint32_t LPT>
__global__ void __launch_bounds__(FB) k_bal_emit(const Key *__restrict__ k, size_t n, const uint16_t *__restrict__ extra,
                                                 const uint32_t *__restrict__ blk, const uint32_t *__restrict__ base,
                                                 const unsigned long long *__restrict__ tab, uint64_t mask,
                                                 Key *__restrict__ out) {
    static_assert(FB * LPT == 1u << blk_shift(LPT), "the counts are per workgroup");
    __shared__ uint32_t tmp[FB / 64 + 1], s_base;
    __shared__ uint32_t s_many[FB];  // leaves with several splits: leaf in the workgroup << 16 | splits
    __shared__ uint32_t s_off[FB];   // ... and the splits before it in the workgroup
    __shared__ uint32_t s_nmany;
    __shared__ uint32_t s_path[FB / 64][kMaxSplits];   // a wave's splits
    __shared__ uint32_t s_start[FB / 64][kMaxSplits];  // where they begin: digits of kMaxRel levels
    __shared__ uint8_t s_kids[FB / 64][kMaxSplits];    // which children are split
    const size_t i0 = (size_t)blockIdx.x * (FB * LPT);
    if (base) {
        if (threadIdx.x == 0) s_base = base[blockIdx.x];
    } else {
        uint32_t sum = 0, total;
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += FB) sum += blk[b];
        (void)block_excl_scan_u32(sum, tmp, total);
        if (threadIdx.x == 0) s_base = total;
    }
    __syncthreads();
    const size_t o0 = i0 + 7ull * s_base;
    if (blk[blockIdx.x] == 0) {  // nothing to refine here
#pragma unroll
        for (uint32_t e = 0; e < LPT; ++e) {
            const size_t i = i0 + e * FB + threadIdx.x;
            if (i < n) out[o0 + e * FB + threadIdx.x] = k[i];
        }
        return;
    }
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    uint32_t *path = s_path[wid], *start = s_start[wid];
    uint8_t *kids = s_kids[wid];
    uint32_t done = 0;  // new splits in the rounds before
    for (uint32_t e = 0; e < LPT; ++e) {
        const uint32_t j = e * FB + threadIdx.x;
        const size_t i = i0 + j;
        const uint32_t x = i < n ? extra[i] : 0u;
        if (threadIdx.x == 0) s_nmany = 0;
        uint32_t total;
        const uint32_t ex = done + block_excl_scan_u32(x, tmp, total);
        if (i < n) {
            const size_t o = o0 + j + 7ull * ex;
            const Key f = k[i];
            if (x == 0) {
                out[o] = f;
            } else if (x == 1) {
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c) out[o + c] = key_below(f, 8 + c);
            } else {
                const uint32_t p = atomicAdd(&s_nmany, 1u);
                s_many[p] = j << 16 | x;
                s_off[p] = ex;
            }
        }
        done += total;
        __syncthreads();
        const uint32_t nmany = s_nmany;
        for (uint32_t m = wid; m < nmany; m += FB / 64) {
            const uint32_t lj = s_many[m] >> 16, lx = s_many[m] & 0xffffu;
            const uint64_t leaf = (uint64_t)(i0 + lj) << 32;
            const Key f = k[i0 + lj];
            if (lane == 0) {
                path[0] = 1;
                start[0] = 0;
            }
            for (uint32_t q = lane; q < lx; q += 64) kids[q] = 0;
            wave_order();
            uint32_t head = 0, tail = 1;
            while (tail < lx && head < tail) {
                const uint32_t g = head + (lane >> 3);
                bool has = false;
                uint32_t pc = 0;
                if (g < tail) {
                    const uint32_t pp = path[g];
                    pc = pp << 3 | (lane & 7u);
                    has = pp < (1u << (3 * kMaxRel)) && hash_has(tab, mask, leaf | pc);
                }
                const uint64_t found = __ballot(has);
                if (g < tail && (lane & 7u) == 0) kids[g] = (uint8_t)(found >> lane);
                if (has) {
                    const uint32_t at = tail + (uint32_t)__popcll(found & ((1ull << lane) - 1ull));
                    if (at < lx) {
                        const uint32_t r = (31 - (uint32_t)__clz(pc)) / 3;
                        path[at] = pc;
                        start[at] = (pc ^ (1u << (3 * r))) << (3 * (kMaxRel - r));
                    }
                }
                head = min(head + 8, tail);
                tail = min(tail + (uint32_t)__popcll(found), lx);
                wave_order();
            }
            const size_t o = o0 + lj + 7ull * s_off[m];
            for (uint32_t q = lane; q < 8 * tail; q += 64) {
                const uint32_t g = q >> 3, c = q & 7u;
                if ((kids[g] >> c) & 1u) continue;
                const uint32_t pp = path[g], r = (31 - (uint32_t)__clz(pp)) / 3 + 1;
                // digits of the octant: their sum, and the zeros at the end
                uint32_t sum = c, tz = c == 0 ? 1u : 0u;
                bool run = c == 0;
                for (uint32_t t = pp; t > 1; t >>= 3) {
                    sum += t & 7u;
                    run = run && (t & 7u) == 0;
                    tz += run ? 1u : 0u;
                }
                // splits that begin before it; of the r octants that hold it, r - tz do
                const uint32_t lim =
                    start[g] + (c ? 1u + (uint32_t)((((uint64_t)c << (3 * (kMaxRel + 1 - r))) - 1u) >> 3) : 0u);
                uint32_t before = 0;
                for (uint32_t t = 0; t < tail; ++t) before += start[t] < lim ? 1u : 0u;
                out[o + sum + 7 * (before - (r - tz))] = key_below(f, (uint64_t)pp << 3 | c);
            }
            wave_order();
        }
        __syncthreads();
    }
}

}  // namespace

bool balance_search(const Key *in, size_t n, uint32_t md, int curve, hipStream_t s, BalStats *stats,
                    DevBuf<Key> &out) {
    if (n < 8 || n > 0x7fffffffull) return false;
    const SfcPacked tab = make_packed(curve);
    uint32_t cl = 1;  // cells of the search table: about 8 leaves each, 2^18 at most
    while (cl < 6 && cl < md && (64ull << (3 * cl)) <= n) ++cl;
    const uint32_t ncell = 1u << (3 * cl);
    // 2^18 leaves at one per thread are four workgroups a CU
    const bool small = n < (size_t(1) << 18);
    const uint32_t bsh = blk_shift(small ? 1 : 4);
    const size_t nblk = (n + (size_t(1) << bsh) - 1) >> bsh;
    // Twice as many slots as half the leaves could fill: up to n / 4 new
    // splits (the octree nearly triples) stay under half load.  Small octrees get
    // room for up to n: the other step takes some 20 launches a level whatever their size.
    uint64_t slots = 16384;
    while (slots < (small ? 2 * n : n / 2)) slots <<= 1;
    const uint32_t tail_cap = (uint32_t)(slots / 4);
    const size_t zero = sizeof(BalFast) + slots * 8;
    DevBuf<uint8_t> ws(zero + (size_t)tail_cap * 8, s);
    BalFast *st = (BalFast *)ws.p;
    unsigned long long *hash = (unsigned long long *)(ws.p + sizeof(BalFast));
    unsigned long long *tail = hash + slots;
    const uint32_t ncheck = grid_for(std::max<size_t>(n, ncell), FB), nfind = grid_for(n, small ? FB : FB * 4);
    DevBuf<uint32_t> cstart(ncell + 1, s), blk(nblk, s), seeds(2 * (size_t)nfind, s);
    DevBuf<uint16_t> extra(n + (n & 1), s), levels(ncheck, s);
    HIP_OK(hipMemsetAsync(ws.p, 0, zero, s));
    k_bal_check<<<ncheck, FB, 0, s>>>(in, n, md, cl, bsh, cstart.p, extra.p, blk.p, levels.p, st);
    const FindArgs A{in, cstart.p, extra.p, blk.p, hash, slots - 1, tail, tail_cap, small ? ~0u : nfind / 8,
                     st, md,       cl,      bsh};
    if (small) k_bal_find<1><<<nfind, FB, 0, s>>>(A, n, tab, seeds.p);
    else k_bal_find<4><<<nfind, FB, 0, s>>>(A, n, tab, seeds.p);
    k_bal_find_tail<<<std::min(64u, 1 + nfind / 1024), FB, 0, s>>>(A, tab, seeds.p, nfind, levels.p, ncheck);
    HIP_OK(hipGetLastError());
    BalFast h;
    dgx_read_back(&h, st, offsetof(BalFast, spread), s);
    if (h.flags) return false;
    BalStats bs{};
    if (h.lmax + h.lup >= 31 + 2) {  // else the octree is returned as it is (TreeNode.cpp:929-947)
        bs.levels = h.lmax;
        bs.seeds = n + h.seeds;
    }
    const size_t total = n + 7ull * h.nnew;
    out.alloc(total, s);
    if (!h.nnew) {
        HIP_OK(hipMemcpyAsync(out.p, in, n * sizeof(Key), hipMemcpyDeviceToDevice, s));
    } else {
        // each workgroup sums the counts before its own; past 4096 workgroups a scan does
        DevBuf<uint32_t> base;
        if (nblk > 4096) {
            base.alloc(nblk, s);
            scan_exclusive_u32_async(blk.p, base.p, nblk, nullptr, s);
        }
        if (small) k_bal_emit<1><<<(unsigned)nblk, FB, 0, s>>>(in, n, extra.p, blk.p, base.p, hash, slots - 1, out.p);
        else k_bal_emit<4><<<(unsigned)nblk, FB, 0, s>>>(in, n, extra.p, blk.p, base.p, hash, slots - 1, out.p);
        HIP_OK(hipGetLastError());
    }
    // the result exists when the call returns: a hierarchy's set-up reads it on another stream
    HIP_OK(hipStreamSynchronize(s));
    if (bs.levels) bs.leaves = total;
    if (stats) *stats = bs;
    return true;
}
