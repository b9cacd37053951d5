// dgx_da_nodes.hip -- hanging anchors and element node lists of the DA, one
// workgroup per 512 octants (flagNodesType3, octFunctions.cpp:1556-2168;
// buildNodeList, odaBuildNlist.cpp:47-934; dgx_da.hip has the whole build).
//
// Both are searches in the sorted local keys, bound by the dependent reads of
// a binary search and of the curve encodes.  Neighbouring octants ask for the
// same points, so a workgroup first finds out which distinct ones its 512
// octants need, answers what lies among its own octants from LDS, and searches
// for the rest:
//   * anchors: octants of one parent share its neighbours; a probe whose key
//     falls between the workgroup's first and last key is looked up in LDS.
//     13.8M elements: 2.44 ms with a search per probe, 0.36 ms here.
//   * node lists: the 4096 vertices of 512 elements are some 800 points, and
//     most of those are anchors of elements of the workgroup.  A hash table of
//     points in LDS holds the owner of each; the used ones, sorted, are the
//     block's node list of the matvec, so no sort of all vertices is needed.
//     13.8M elements: 6.9 ms as per-element searches, a mark of every entry,
//     an ordering and a sort per block, 1.31 ms here (0.3 of it waiting for LDS,
//     the rest for the reads of some 450 searches per block).
#include "dgx_da.h"

#include <algorithm>

namespace {

constexpr uint32_t NB = kElemBlock;  // octants, and threads, per workgroup
constexpr uint8_t F_NODE = 128;

__device__ __forceinline__ uint32_t cell_of(const Key &k) { return (uint32_t)(k.hi >> kCellShift); }

struct CurveTables {
    uint8_t rc[192];
    uint16_t rc2[24 * 64];
};
__device__ __forceinline__ void load_tables(CurveTables &T, const SfcPacked &tab) {
    for (uint32_t i = threadIdx.x; i < 192; i += NB) T.rc[i] = tab.rc[i];
    for (uint32_t i = threadIdx.x; i < 24 * 64; i += NB) T.rc2[i] = rc2_entry(tab.rc, i);
}
__device__ __forceinline__ Key curve_key(const CurveTables &T, uint32_t x, uint32_t y, uint32_t z, uint32_t lev,
                                         uint32_t md) {
    uint32_t rot;
    return morton_to_curve_rot(T.rc2, T.rc, morton_encode(x, y, z, lev, md), rot);
}

// First index in k[lo, hi) whose key is not before p.  Three keys are read per
// step, so a range of 10,000 takes 7 dependent reads, not 14: the anchors'
// few probes wait for their reads (402 -> 363 us on 13.8M elements).  The node
// lists' many searches are bound by the number of reads instead (1.31 ms
// with two-way steps, 1.45 ms with these).
__device__ __forceinline__ uint32_t lower_bound4(const Key *__restrict__ k, uint32_t lo, uint32_t hi, const Key &p) {
    while (hi - lo > 3) {
        const uint32_t q = (hi - lo) >> 2, m1 = lo + q, m2 = m1 + q, m3 = m2 + q;
        const bool b1 = key_lt(k[m1], p), b2 = key_lt(k[m2], p), b3 = key_lt(k[m3], p);
        lo = b3 ? m3 + 1 : b2 ? m2 + 1 : b1 ? m1 + 1 : lo;
        hi = b3 ? hi : b2 ? m3 : b1 ? m2 : m1;
    }
    const uint32_t n = hi - lo;  // 0..3 keys left
    const bool c0 = n > 0 && key_lt(k[lo], p), c1 = n > 1 && key_lt(k[lo + 1], p), c2 = n > 2 && key_lt(k[lo + 2], p);
    return lo + (c0 ? 1u : 0u) + (c1 ? 1u : 0u) + (c2 ? 1u : 0u);
}

// NODE flags: an anchor hangs iff one of the parents of the -x/-y/-z
// neighbours that its child number selects is an octant itself.  Those are the
// parent's own neighbours at its level, in up to 6 directions: -x, -y, -z, -x-y,
// -x-z, -y-z (bits 0..5).  Consecutive octants of one parent are a run (cut at
// wave borders); one task per run and direction any of its octants needs.
__global__ void __launch_bounds__(NB) k_da_flag_nodes(const Key *__restrict__ k, size_t n,
                                                      const uint32_t *__restrict__ cstart, uint32_t md, SfcPacked tab,
                                                      const uint32_t *__restrict__ xs, const uint32_t *__restrict__ ys,
                                                      const uint32_t *__restrict__ zs, uint8_t *flags) {
    constexpr uint32_t kFar = 512;
    __shared__ CurveTables T;
    __shared__ Key sk[NB];
    __shared__ uint32_t s_res[NB];           // per run (its first octant): directions found
    __shared__ uint16_t s_task[3 * NB];      // first octant << 3 | direction; an octant needs at most 3
    __shared__ Key s_far[kFar];              // probes outside the workgroup's keys
    __shared__ uint16_t s_fartask[kFar];
    __shared__ uint32_t s_nt, s_nfar;
    const uint32_t t = threadIdx.x, lane = t & 63u;
    const size_t i0 = (size_t)blockIdx.x * NB, i = i0 + t;
    const uint32_t nb = (uint32_t)min((size_t)NB, n - i0);
    load_tables(T, tab);
    if (t == 0) s_nt = s_nfar = 0;
    s_res[t] = 0;
    Key key{~0ull, ~0ull};
    uint32_t need = 0, lev = 0, fl = 0;
    if (t < nb) {
        key = k[i];
        fl = flags[i];
        lev = fl & 31u;
        const uint32_t X = xs[i], Y = ys[i], Z = zs[i], b = md - lev;
        const uint32_t cn = (((Z >> b) & 1u) << 2) | (((Y >> b) & 1u) << 1) | ((X >> b) & 1u);
        const bool bx = X != 0, by = Y != 0, bz = Z != 0;
        if (lev != 1) switch (cn) {
            case 1: need = (by ? 2u : 0u) | (bz ? 4u : 0u) | (by && bz ? 32u : 0u); break;
            case 2: need = (bx ? 1u : 0u) | (bz ? 4u : 0u) | (bx && bz ? 16u : 0u); break;
            case 3: need = bz ? 4u : 0u; break;
            case 4: need = (bx ? 1u : 0u) | (by ? 2u : 0u) | (bx && by ? 8u : 0u); break;
            case 5: need = by ? 2u : 0u; break;
            case 6: need = bx ? 1u : 0u; break;
            default: break;
        }
    }
    sk[t] = key;
    __syncthreads();
    const bool head = lane == 0 || t >= nb || !key_eq(key_parent(sk[t - 1]), key_parent(key));
    const uint64_t heads = __ballot(head), upto = ~0ull >> (63 - lane);
    const uint32_t first = 63 - (uint32_t)__clzll(heads & upto);  // lane of this run's first octant
    const uint64_t after = lane == 63 ? 0ull : heads & ~upto;
    const uint64_t mine = (after ? ((1ull << (__ffsll((unsigned long long)after) - 1)) - 1) : ~0ull) & ~(upto >> 1);
    uint32_t want = 0;
#pragma unroll
    for (uint32_t d = 0; d < 6; ++d)
        if (__ballot((need >> d) & 1u) & mine) want |= 1u << d;
    if (!head) want = 0;
    uint32_t total;
    const uint32_t ex = wave_excl_sum((uint32_t)__popc(want), total);
    uint32_t at = 0;
    if (lane == 0 && total) at = atomicAdd(&s_nt, total);
    at = __shfl(at, 0) + ex;
    for (uint32_t d = 0; d < 6; ++d)
        if ((want >> d) & 1u) s_task[at++] = (uint16_t)(t << 3 | d);
    __syncthreads();
    const uint32_t nt = s_nt;
    const Key kfirst = sk[0], klast = sk[nb - 1];
    auto search = [&](const Key &p) {
        const uint32_t c = cell_of(p), lo = lower_bound4(k, cstart[c], cstart[c + 1], p);
        return lo < n && key_eq(k[lo], p);
    };
    for (uint32_t q = t; q < nt; q += NB) {
        const uint32_t task = s_task[q], o = task >> 3, d = task & 7u;
        const uint32_t lp = key_level(sk[o]) - 1, ps = md - lp, len = 1u << ps;
        const uint32_t X = (xs[i0 + o] >> ps) << ps, Y = (ys[i0 + o] >> ps) << ps, Z = (zs[i0 + o] >> ps) << ps;
        const uint32_t ax = (0x19u >> d) & 1u, ay = (0x2au >> d) & 1u, az = (0x34u >> d) & 1u;
        const Key p = curve_key(T, X - ax * len, Y - ay * len, Z - az * len, lp, md);
        if (!key_lt(p, kfirst) && !key_lt(klast, p)) {
            uint32_t lo = 0, hi = nb;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (key_lt(sk[mid], p)) lo = mid + 1;
                else hi = mid;
            }
            if (lo < nb && key_eq(sk[lo], p)) atomicOr(&s_res[o], 1u << d);
        } else {
            const uint32_t f = atomicAdd(&s_nfar, 1u);
            if (f < kFar) {
                s_far[f] = p;
                s_fartask[f] = (uint16_t)task;
            } else if (search(p)) {
                atomicOr(&s_res[o], 1u << d);
            }
        }
    }
    __syncthreads();
    const uint32_t nfar = min(s_nfar, kFar);
    for (uint32_t q = t; q < nfar; q += NB)
        if (search(s_far[q])) atomicOr(&s_res[s_fartask[q] >> 3], 1u << (s_fartask[q] & 7u));
    __syncthreads();
    if (t < nb && !(s_res[(t & ~63u) + first] & need)) flags[i] = (uint8_t)(fl | F_NODE);
}

struct NodeArgs {
    const Key *k;
    size_t n, ne;
    const uint32_t *cstart, *xs, *ys, *zs;
    const uint8_t *flags;
    uint32_t md;
    uint32_t *nlist;
    uint8_t *mask;
    uint16_t *meta;
    uint32_t *ulist, *ucount;
    uint32_t nblk;
    uint16_t *lconn, *cmeta;
    uint8_t *isnode;
    uint32_t *bad, *nbad;  // the blocks left to k_da_nodes_general
};

// The records of one element, stored by its workgroup once the block's local
// indices are known: node list, hanging mask, element meta, and at the
// element's slot the local indices and the mask in the child frame.
__device__ __forceinline__ void store_element(const NodeArgs &A, uint32_t b, uint32_t slot, size_t e, uint32_t lev,
                                              uint32_t cn, uint32_t mask, const uint32_t *nl, const uint16_t *loc) {
    uint4 *o = reinterpret_cast<uint4 *>(A.nlist + 8 * e);
    o[0] = make_uint4(nl[0], nl[1], nl[2], nl[3]);
    o[1] = make_uint4(nl[4], nl[5], nl[6], nl[7]);
    A.mask[e] = (uint8_t)mask;
    A.meta[e] = (uint16_t)(mask | cn << 8 | (lev - 1) << 11);
    uint32_t v[8];  // local indices as byte offsets, and the mask, in the child frame
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) v[j] = (uint32_t)loc[j] * 8u | ((mask >> j) & 1u) << 31;
    child_frame(v, cn);
    uint32_t cm = 0;
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
        cm |= (v[j] >> 31) << j;
        v[j] &= 0xffffu;
    }
    reinterpret_cast<uint4 *>(A.lconn)[(size_t)b * NB + slot] =
        make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
    A.cmeta[(size_t)b * NB + slot] = (uint16_t)(cm | (lev - 1) << 8);
}

// Slot of each element inside its block: elements without hanging vertices
// first, then the others, so that most waves are uniform; inside each class the
// SFC order is spread by spread8.  wf, wh: one counter per wave.
__device__ __forceinline__ uint32_t element_slot(bool valid, bool hang, uint32_t nb, uint32_t *wf, uint32_t *wh) {
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    const uint64_t bf = __ballot(valid && !hang), bh = __ballot(valid && hang);
    if (lane == 0) {
        wf[wid] = (uint32_t)__popcll(bf);
        wh[wid] = (uint32_t)__popcll(bh);
    }
    __syncthreads();
    uint32_t pf = 0, ph = 0, nflat = 0;
    for (uint32_t w = 0; w < NB / 64; ++w) {
        if (w < wid) {
            pf += wf[w];
            ph += wh[w];
        }
        nflat += wf[w];
    }
    const uint64_t lt = (1ull << lane) - 1ull;
    return hang ? nflat + spread8(ph + (uint32_t)__popcll(bh & lt), nb - nflat)
                : spread8(pf + (uint32_t)__popcll(bf & lt), nflat);
}

__device__ __forceinline__ void lds_wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// Bitonic sort of a[0..P) (P a power of two) by the workgroup.  Compare-exchange
// c of a stage with partner distance <= 64 touches only the 128 elements of
// its wave, so such stages follow each other without a workgroup barrier.
template <typename V>
__device__ void block_bitonic(V *a, uint32_t P) {
    bool prev_local = false;
    for (uint32_t kk = 2; kk <= P; kk <<= 1)
        for (uint32_t j = kk >> 1; j > 0; j >>= 1) {
            const bool local = j <= 64;
            if (local && prev_local) lds_wave_order();
            else __syncthreads();
            const uint32_t lj = __ffs(j) - 1;
            for (uint32_t c = threadIdx.x; c < (P >> 1); c += NB) {
                const uint32_t i = ((c >> lj) << (lj + 1)) | (c & (j - 1)), o = i + j;
                const V x = a[i], y = a[o];
                if ((i & kk) == 0 ? y < x : x < y) {
                    a[i] = y;
                    a[o] = x;
                }
            }
            prev_local = local;
        }
    __syncthreads();
}

// Node lists of one block.  Points are packed 21 bits per axis in units of
// level 21, which holds for octants down to that level.  Vertex j of an element
// resolves to the octant anchored there if that is a NODE; otherwise it hangs
// and takes corner j of the parent, resolved the same way (odaBuildNlist.cpp:
// 531-566).  Blocks with deeper octants, with more points than the table
// takes, or with a vertex that resolves neither way (the reference's forward
// ghost scan) go to the list bad[] and are left to k_da_nodes_general.
constexpr uint32_t HS = 2048, kProbes = 64;
constexpr uint64_t kEmpty = ~0ull;
constexpr uint32_t kPending = 0xfffffffeu, kNone = 0xffffffffu;
// The octants are read four at a time, 16 bytes that have to lie on a multiple of 16.
union PointTable {
    unsigned long long point[HS];
    uint32_t octant[2 * HS];
    uint4 octant4[HS / 2];
};
static_assert(alignof(PointTable) == 16 && sizeof(PointTable) == 8 * HS, "one table of HS slots");
__global__ void __launch_bounds__(NB) k_da_nodes(NodeArgs A, SfcPacked tab) {
    __shared__ CurveTables T;
    __shared__ PointTable table;             // points; then the octants outside the block that they refer to
    unsigned long long *hkey = table.point;
    __shared__ uint32_t hown[HS];            // local index of the NODE octant anchored there
    __shared__ uint16_t hloc[HS];            // used; then the local index in the block's list
    __shared__ uint16_t plist[HS];           // slots to be searched for; then those of the octants
    __shared__ uint32_t wf[NB / 64], wh[NB / 64], s_n, s_below, s_bad;
    const uint32_t t = threadIdx.x, lane = t & 63u, b = blockIdx.x;
    const size_t e0 = (size_t)b * NB, e = e0 + t;
    const uint32_t nb = (uint32_t)min((size_t)NB, A.ne - e0), md = A.md;
    const bool valid = t < nb;
    load_tables(T, tab);
    for (uint32_t i = t; i < HS; i += NB) {
        hkey[i] = kEmpty;
        hown[i] = kPending;
        hloc[i] = 0;
    }
    uint32_t d = 1, x = 0, y = 0, z = 0, fl = 0;
    if (valid) {
        fl = A.flags[e];
        d = fl & 31u;
        x = A.xs[e];
        y = A.ys[e];
        z = A.zs[e];
    }
    if (t == 0) {
        s_bad = 0;
        if (b == 0) A.ucount[A.nblk] = 0;  // so that the exclusive scan ends with the total
    }
    const uint32_t sh = md > 21 ? md - 21 : 0;
    if (__syncthreads_or(d > 21)) {
        if (t == 0) A.bad[atomicAdd(A.nbad, 1u)] = b;
        return;
    }
    const uint32_t sz = 1u << (md - d), ps = md - d + 1;
    const uint32_t px = (x >> ps) << ps, py = (y >> ps) << ps, pz = (z >> ps) << ps;
    auto pack = [&](uint32_t vx, uint32_t vy, uint32_t vz) {
        return (uint64_t)(vx >> sh) | (uint64_t)(vy >> sh) << 21 | (uint64_t)(vz >> sh) << 42;
    };
    // The three fields are mixed before the top bits are taken: coarse octants
    // leave the low bits of each field zero, and one product of the whole word
    // clustered so that one block in 30 ran out of probes.  The fields' products
    // are shared by the vertices of an element: with three multiplies per vertex,
    // and eight rounds for the hanging ones, the kernel took 1.47 ms instead of
    // 1.25 on 13.8M elements.
    auto hx = [&](uint32_t vx) { return (vx >> sh) * 0x9e3779b1u; };
    auto hy = [&](uint32_t vy) { return (vy >> sh) * 0x85ebca77u; };
    auto hz = [&](uint32_t vz) { return (vz >> sh) * 0xc2b2ae3du; };
    auto hash = [](uint32_t h) {  // of the exclusive or of the three
        h ^= h >> 16;
        h *= 0x7feb352du;
        return h >> 21;
    };
    auto probe_on = [&](uint64_t key, uint32_t h, uint64_t old) {  // the rest of an insertion whose first probe gave old
#pragma unroll 1
        for (uint32_t p = 1; old != kEmpty && old != key; ++p) {
            if (p == kProbes) {
                s_bad = 1;
                return 0u;
            }
            h = (h + 1) & (HS - 1);
            old = atomicCAS(&hkey[h], kEmpty, (unsigned long long)key);
        }
        return h;
    };
    static_assert(HS == 1u << 11, "hash gives 11 bits");
    uint32_t slot[8];
    if (valid) {
        uint64_t key[8], old[8];
        const uint64_t k0 = pack(x, y, z), s0 = sz >> sh;  // a level above 21: sz is a multiple of the unit
        const uint32_t mx[2] = {hx(x), hx(x + sz)}, my[2] = {hy(y), hy(y + sz)}, mz[2] = {hz(z), hz(z + sz)};
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            key[j] = k0 + ((j & 1) ? s0 : 0) + ((j & 2) ? s0 << 21 : 0) + ((j & 4) ? s0 << 42 : 0);
            slot[j] = hash(mx[j & 1] ^ my[(j >> 1) & 1] ^ mz[j >> 2]);
            old[j] = atomicCAS(&hkey[slot[j]], kEmpty, (unsigned long long)key[j]);
        }
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) slot[j] = probe_on(key[j], slot[j], old[j]);
        // the octant anchored at vertex 0 is the element itself
        if (atomicCAS(&hown[slot[0]], kPending, (fl & F_NODE) ? (uint32_t)e : kNone) != kPending) s_bad = 1;
    }
    auto resolve = [&]() {  // finds the owners of the points that have none yet
        __syncthreads();
        if (t == 0) s_n = 0;
        __syncthreads();
        for (uint32_t q = 0; q < HS / NB; ++q) {
            const uint32_t s = q * NB + t;
            const bool p = hkey[s] != kEmpty && hown[s] == kPending;
            const uint64_t m = __ballot(p);
            uint32_t at = 0;
            if (lane == 0 && m) at = atomicAdd(&s_n, (uint32_t)__popcll(m));
            at = __shfl(at, 0);
            if (p) plist[at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)s;
        }
        __syncthreads();
        for (uint32_t q = t; q < s_n; q += NB) {
            const uint32_t s = plist[q];
            const uint64_t key = hkey[s];
            const uint32_t vx = (uint32_t)(key & 0x1fffffu) << sh, vy = (uint32_t)((key >> 21) & 0x1fffffu) << sh,
                           vz = (uint32_t)(key >> 42) << sh;
            const Key p = curve_key(T, vx, vy, vz, md, md);
            const uint32_t c = cell_of(p);  // the octant that holds the point: the last one not after it
            uint32_t lo = A.cstart[c], hi = A.cstart[c + 1];
            while (lo < hi) {
                const uint32_t mid = lo + ((hi - lo) >> 1);
                if (key_le(A.k[mid], p)) lo = mid + 1;
                else hi = mid;
            }
            uint32_t own = kNone;
            if (lo) {
                // it is anchored at the point iff it holds the point's cell and
                // the point is a multiple of its size
                const Key f = A.k[lo - 1];
                const uint32_t l = key_level(f), off = (vx | vy | vz) & ((1u << (md - l)) - 1u);
                if (!off && key_eq(key_truncate(p, l), f) && (A.flags[lo - 1] & F_NODE)) own = lo - 1;
            }
            hown[s] = own;
        }
        __syncthreads();
    };
    resolve();
    const uint32_t anchor = valid ? slot[0] : 0u;
    uint32_t hang = 0;
    bool fresh = false;
    if (valid) {
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
            if (hown[slot[j]] == kNone) hang |= 1u << j;
        // each lane its own next vertex: as many rounds as some element has hanging ones
        for (uint32_t left = hang; left; left &= left - 1) {
            const uint32_t j = (uint32_t)__ffs(left) - 1u;
            const uint32_t vx = px + (j & 1) * 2 * sz, vy = py + ((j >> 1) & 1) * 2 * sz, vz = pz + (j >> 2) * 2 * sz;
            const uint64_t key = pack(vx, vy, vz);
            const uint32_t h = hash(hx(vx) ^ hy(vy) ^ hz(vz));
            const uint32_t s = probe_on(key, h, atomicCAS(&hkey[h], kEmpty, (unsigned long long)key));
            fresh = fresh || hown[s] == kPending;  // owners are settled for the points that were there
#pragma unroll
            for (uint32_t q = 0; q < 8; ++q)
                if (q == j) slot[q] = s;
        }
    }
    if (__syncthreads_or(fresh)) resolve();
    uint32_t nl[8];
    if (valid) {
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            nl[j] = hown[slot[j]];
            if (nl[j] >= kPending) s_bad = 1;
            hloc[slot[j]] = 1;
        }
    }
    if (t == 0) s_n = s_below = 0;
    __syncthreads();
    if (s_bad) {
        if (t == 0) A.bad[atomicAdd(A.nbad, 1u)] = b;
        return;
    }
    // The octants the elements refer to, in order: those of the block follow
    // their elements; the others, which lie before or after the block, are
    // ranked by counting (a bitonic sort of all took 13 us of a workgroup's 53).
    uint32_t *own_l = table.octant;  // the points are no longer needed
    const bool in = valid && hloc[anchor] && hown[anchor] == (uint32_t)e;
    const uint64_t bin = __ballot(in);
    if (lane == 0) wf[t >> 6] = (uint32_t)__popcll(bin);
    for (uint32_t q = 0; q < HS / NB; ++q) {
        const uint32_t s = q * NB + t, o = hown[s];
        const bool p = hloc[s] != 0 && (size_t)o - e0 >= nb;  // unsigned: before the block wraps
        const uint64_t m = __ballot(p), below = __ballot(p && o < e0);
        uint32_t at = 0;
        if (lane == 0 && m) {
            at = atomicAdd(&s_n, (uint32_t)__popcll(m));
            if (below) atomicAdd(&s_below, (uint32_t)__popcll(below));
        }
        at = __shfl(at, 0);
        if (p) {
            const uint32_t i = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            own_l[i] = o;
            plist[i] = (uint16_t)s;
        }
    }
    __syncthreads();
    const uint32_t nout = s_n, nbelow = s_below, npad = (nout + 7) & ~7u;
    uint32_t pin = 0, nin = 0;
    for (uint32_t w = 0; w < NB / 64; ++w) {
        if (w < t >> 6) pin += wf[w];
        nin += wf[w];
    }
    if (t < npad - nout) own_l[nout + t] = kNone;
    __syncthreads();
    uint32_t *ul = A.ulist + (size_t)b * 8 * NB;
    auto place = [&](uint32_t r, uint32_t s, uint32_t o) {
        hloc[s] = (uint16_t)r;
        ul[r] = o;
        A.isnode[o] = 1;
    };
    // two threads per octant, each against half of the list
    for (uint32_t i0 = 0; i0 < nout; i0 += NB / 2) {
        const uint32_t i = i0 + (t >> 1);
        const uint32_t o = i < nout ? own_l[i] : 0u;
        uint32_t r = 0;
        const uint4 *l4 = table.octant4;
        for (uint32_t q = t & 1u; q < npad / 4; q += 2) {
            const uint4 v = l4[q];
            r += (v.x < o ? 1u : 0u) + (v.y < o ? 1u : 0u) + (v.z < o ? 1u : 0u) + (v.w < o ? 1u : 0u);
        }
        r += (uint32_t)__shfl_xor((int)r, 1, 64);
        if (i < nout && (t & 1u) == 0) place(o < e0 ? r : r + nin, plist[i], o);
    }
    if (in) place(nbelow + pin + (uint32_t)__popcll(bin & ((1ull << lane) - 1ull)), anchor, (uint32_t)e);
    if (t == 0) A.ucount[b] = nout + nin;
    __syncthreads();  // wf is used again
    const uint32_t es = element_slot(valid, hang != 0, nb, wf, wh);  // its barrier publishes hloc
    if (valid) {
        uint16_t loc[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) loc[j] = hloc[slot[j]];
        const uint32_t bt = md - d;
        store_element(A, b, es, e, d, (((z >> bt) & 1u) << 2) | (((y >> bt) & 1u) << 1) | ((x >> bt) & 1u), hang, nl,
                      loc);
    }
}

// greatest k[i] <= p
__device__ __forceinline__ bool max_lower_bound(const NodeArgs &A, const Key &p, size_t &idx) {
    const uint32_t c = cell_of(p);
    size_t lo = A.cstart[c], hi = A.cstart[c + 1];
    while (lo < hi) {
        const size_t mid = lo + (hi - lo) / 2;
        if (key_le(A.k[mid], p)) lo = mid + 1;
        else hi = mid;
    }
    if (lo == 0) {
        idx = 0;
        return false;
    }
    idx = lo - 1;
    return true;
}

// The same for the blocks marked bad, as the reference does it: per element a
// search for each vertex, then for the parent's corner, then the forward ghost
// scan (odaBuildNlist.cpp:531-934 on one rank); the block's list is a sort of
// all its entries.  counters: [0] unresolved entries, [1] ghost scans.
__global__ void __launch_bounds__(NB) k_da_nodes_general(NodeArgs A, SfcPacked tab, uint32_t *counters) {
    const uint32_t nbad = *A.nbad;
    if (!nbad) return;
    __shared__ uint8_t s_rc[192];
    __shared__ uint8_t s_rot[kTailCols * NB];  // rotation states of each thread's path, levels 1..32
    __shared__ Key s_tail[24 * kTailCols];
    __shared__ uint32_t v[8 * NB];             // the block's entries, sorted; then the distinct ones
    __shared__ uint32_t tmp[NB / 64 + 1], wf[NB / 64], wh[NB / 64];
    const uint32_t t = threadIdx.x, md = A.md;
    for (uint32_t q = t; q < 192; q += NB) s_rc[q] = tab.rc[q];
    __syncthreads();
    for (uint32_t q = t; q < 24 * kTailCols; q += NB) s_tail[q] = zero_tail(s_rc, q / kTailCols, q % kTailCols, md);
    for (uint32_t bi = blockIdx.x; bi < nbad; bi += gridDim.x) {
        const uint32_t b = A.bad[bi];
        const size_t e0 = (size_t)b * NB, i = e0 + t, n = A.n;
        const uint32_t nb = (uint32_t)min((size_t)NB, A.ne - e0);
        const bool valid = t < nb;
        __syncthreads();  // the tables; the LDS of the block before
        uint32_t nl[8], mask = 0, d = 1, cn = 0;
        if (valid) {
            d = A.flags[i] & 31u;
            const uint32_t x = A.xs[i], y = A.ys[i], z = A.zs[i];
            uint8_t *rots = s_rot + t;
            const Key kref = path_walk(s_rc, x, y, z, d, md, rots, NB);
            const bool inode = A.flags[i] & F_NODE;
            const uint32_t ps = md - d + 1, parX = (x >> ps) << ps, parY = (y >> ps) << ps, parZ = (z >> ps) << ps;
            const uint32_t sz = 1u << (md - d);
            cn = (((z >> (md - d)) & 1u) << 2) | (((y >> (md - d)) & 1u) << 1) | ((x >> (md - d)) & 1u);
            auto anchored = [&](bool found, size_t idx, uint32_t ax, uint32_t ay, uint32_t az) {
                return found && A.xs[idx] == ax && A.ys[idx] == ay && A.zs[idx] == az && (A.flags[idx] & F_NODE);
            };
            for (uint32_t j = 0; j < 8; ++j) {
                const uint32_t bx = j & 1, by = (j >> 1) & 1, bz = j >> 2;
                const uint32_t vx = x + bx * sz, vy = y + by * sz, vz = z + bz * sz;
                const uint32_t wx = parX + bx * (sz << 1), wy = parY + by * (sz << 1), wz = parZ + bz * (sz << 1);
                size_t idx = 0;
                uint32_t r = 0;
                bool done = false;
                if (j == 0) {
                    r = (uint32_t)i;
                    done = true;
                    if (!inode) {
                        const Key pk =
                            key_from_path(s_rc, kref, rots, NB, x, y, z, wx, wy, wz, d - 1, md, md, s_tail);
                        if (anchored(max_lower_bound(A, pk, idx), idx, wx, wy, wz)) r = (uint32_t)idx;
                    }
                } else {
                    const Key sk = key_from_path(s_rc, kref, rots, NB, x, y, z, vx, vy, vz, d, md, md, s_tail);
                    bool found = max_lower_bound(A, sk, idx);
                    if (found && !(key_is_ancestor(A.k[idx], sk) || key_eq(A.k[idx], sk))) found = false;
                    done = anchored(found, idx, vx, vy, vz);
                    if (!done) {
                        const Key pk =
                            key_from_path(s_rc, kref, rots, NB, x, y, z, wx, wy, wz, d - 1, md, md, s_tail);
                        done = anchored(max_lower_bound(A, pk, idx), idx, wx, wy, wz);
                    }
                    r = (uint32_t)idx;
                }
                if (!done) {
                    // forward ghost scan (odaBuildNlist.cpp:566-600)
                    atomicAdd(&counters[1], 1u);
                    const Key nk = dev_encode(s_rc, wx, wy, wz, d - 1, md);
                    Key dld = nk;  // last cell of nk
                    for (uint32_t l = d; l <= md; ++l) key_set_digit(dld, l, 7);
                    dld.lo = (dld.lo & ~31ull) | md;
                    r = (uint32_t)n;
                    for (size_t kk = 1; idx + kk < n; ++kk) {
                        const Key &c = A.k[idx + kk];
                        if (key_eq(key_parent(c), nk)) {
                            if (A.flags[idx + kk] & F_NODE) continue;
                            r = (uint32_t)(idx + kk);
                            break;
                        }
                        if (key_lt(dld, c)) break;
                    }
                }
#pragma unroll
                for (uint32_t q = 0; q < 8; ++q)
                    if (q == j) nl[q] = r;
                if (r >= n) {
                    atomicAdd(&counters[0], 1u);
                    continue;
                }
                uint32_t ox = A.xs[r], oy = A.ys[r], oz = A.zs[r];
                if (!(A.flags[r] & F_NODE)) {
                    const uint32_t s2 = md - (A.flags[r] & 31u) + 1;
                    ox = (ox >> s2) << s2;
                    oy = (oy >> s2) << s2;
                    oz = (oz >> s2) << s2;
                }
                if (j == 0 ? !inode : (vx != ox || vy != oy || vz != oz)) mask |= 1u << j;
            }
        }
        const uint32_t m = 8 * nb;
        uint32_t P = 64;
        while (P < m) P <<= 1;
        for (uint32_t q = m + t; q < P; q += NB) v[q] = 0xffffffffu;
        if (valid)
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) v[8 * t + j] = nl[j];
        block_bitonic(v, P);
        // distinct entries, in place: a thread's 8 entries and the one before them
        // go to registers before the scan's barriers
        uint32_t r[8], f = 0, cnt = 0;
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) {
            r[q] = valid ? v[8 * t + q] : 0u;
            const uint32_t before = q ? r[q - 1] : (t && valid ? v[8 * t - 1] : ~r[0]);
            if (valid && r[q] != before) {
                f |= 1u << q;
                ++cnt;
            }
        }
        uint32_t nu;
        uint32_t w = block_excl_scan_u32(cnt, tmp, nu);
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q)
            if ((f >> q) & 1u) v[w++] = r[q];
        __syncthreads();
        for (uint32_t q = t; q < nu; q += NB) {
            A.ulist[(size_t)b * 8 * NB + q] = v[q];
            if (v[q] < n) A.isnode[v[q]] = 1;
        }
        if (t == 0) A.ucount[b] = nu;
        const uint32_t es = element_slot(valid, mask != 0, nb, wf, wh);
        if (valid) {
            uint16_t loc[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                uint32_t lo = 0, hi = nu;
                while (lo < hi) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (v[mid] < nl[j]) lo = mid + 1;
                    else hi = mid;
                }
                loc[j] = (uint16_t)lo;
            }
            store_element(A, b, es, i, d, cn, mask, nl, loc);
        }
    }
}

}  // namespace

void da_flag_nodes(DaDevice &da, const uint32_t *cstart, hipStream_t s) {
    k_da_flag_nodes<<<grid_for(da.n_local, NB), NB, 0, s>>>(da.key.p, da.n_local, cstart, da.md, make_packed(da.curve),
                                                           da.x.p, da.y.p, da.z.p, da.flags.p);
    HIP_OK(hipGetLastError());
}

void da_node_lists(DaDevice &da, const uint32_t *cstart, uint8_t *isnode, const NodeCounters &nc, BlockLists &bl,
                   hipStream_t s) {
    const uint32_t nblk = grid_for(da.n_elem, NB);
    da.nlist.alloc(8 * da.n_elem, s);
    da.mask.alloc(da.n_elem, s);
    da.meta.alloc(da.n_elem, s);
    da.lconn.alloc((size_t)nblk * 8 * NB, s);
    da.cmeta.alloc((size_t)nblk * NB, s);  // whole blocks, like lconn
    bl.ulist.alloc((size_t)nblk * 8 * NB, s);
    bl.ucount.alloc(nblk + 1, s);
    DevBuf<uint32_t> bad(nblk, s);
    const NodeArgs A{da.key.p,   da.n_local, da.n_elem,  cstart,      da.x.p,     da.y.p,  da.z.p,
                     da.flags.p, da.md,      da.nlist.p, da.mask.p,   da.meta.p,  bl.ulist.p, bl.ucount.p,
                     nblk,       da.lconn.p, da.cmeta.p, isnode,      bad.p,      nc.nbad};
    const SfcPacked tab = make_packed(da.curve);
    k_da_nodes<<<nblk, NB, 0, s>>>(A, tab);
    k_da_nodes_general<<<std::min(nblk, 512u), NB, 0, s>>>(A, tab, nc.unresolved_ghost);
    HIP_OK(hipGetLastError());
}
