// dgx_da.hip -- ot::DA construction on one rank (MPI_COMM_SELF) for gfx950.
//
// Follows the reference factory (src/oda/private/odaFactory.cpp:102-923):
//   Part1 (:150-205): embed every octant one level deeper in a 2^(D+1) domain and
//         add the positive-boundary pseudo-octants (octFunctions.cpp:681-770),
//         then re-sort on the curve.  The original domain is Morton child 0 of
//         the embedded root, so its octants precede all pseudo-octants.
//   Part2 (:207-220): NODE flags (flagNodesType3, octFunctions.cpp:1556-2168):
//         an anchor is hanging iff the parent of one of the -x/-y/-z neighbours
//         selected by the child number is itself an octant.
//   Part3: one rank has no ghosts, so the local buffer is [elements | pseudo-
//         octants] and buildNodeList (odaBuildNlist.cpp:47-934, 3010-3095)
//         resolves each element's 8 vertices (dgx_da_nodes.hip): the vertex's owner (maxLowerBound at the
//         vertex cell) if it is a NODE anchored there, else the owner of the
//         parent's vertex, else the forward ghost scan.
// Node vectors are compacted in local-buffer order over NODE octants
// (DA::vecGetBuffer, oda.cpp:863-882).
#include "dgx_da.h"

#include <algorithm>
#include <type_traits>
#include <cstdlib>
#include <vector>

namespace {

constexpr int B = 256;
constexpr uint8_t F_BOUNDARY = 64, F_NODE = 128;

// Device counters of a build.
enum : uint32_t {
    C_NPSEUDO,              // pseudo-octants
    C_FAIL_E, C_FAIL_P,     // what TopSort left undone: elements (or they came unsorted), pseudo-octants
    C_UNRESOLVED, C_GHOST,  // node-list entries unresolved, found by the ghost scan
    C_REF_E, C_REF_P,       // octants referred to: elements, pseudo-octants
    C_NODES,                // NODE octants
    C_PAIRS, C_MAXN,        // (block, node) pairs, largest block
    C_SHARED, C_SLOTS,      // shared nodes, their partial slots
    C_BAD,                  // blocks left to k_da_nodes_general
    C_FILL,                 // pseudo-octants placed so far
    C_COUNT
};

__device__ inline uint32_t n_pseudo(uint32_t f) {
    // +x, +y, +z, +x+y, +x+z, +y+z, +x+y+z (octFunctions.cpp:702-757)
    uint32_t c = __popc(f);
    return c == 3 ? 7u : (c == 2 ? 3u : c);
}

// The octants' keys in the embedded domain (counted for the sort on the way):
// the curve's digits become Morton digits, and those the digits below child 0
// of the embedded root, both two levels per table read.  An octant touches the
// positive x boundary iff the x bit of all its Morton digits is 1 (TreeNode::
// isBoundaryOctant(POSITIVE), TreeNode.cpp:247-269); bflag[i] gets the three
// axes, ctr the number of pseudo-octants that follow.  With
// unsorted, *unsorted is raised by an octant that comes before its predecessor.
// Bound: LDS latency, 8 waves a SIMD.
__global__ void __launch_bounds__(B) k_da_embed(const Key *in, size_t n, SfcPacked tab, Key *dkey, uint8_t *bflag,
                                                uint32_t *ctr, uint32_t *unsorted, TopHist th) {
    __shared__ uint8_t s_rc[192], s_mc[192];
    __shared__ uint16_t s_rc2[24 * 64], s_mc2[24 * 64];
    __shared__ uint32_t h[kTopWords], s_np;
    for (uint32_t i = threadIdx.x; i < 192; i += B) {
        s_rc[i] = tab.rc[i];
        s_mc[i] = tab.mc[i];
    }
    for (uint32_t i = threadIdx.x; i < 24 * 64; i += B) {
        s_rc2[i] = rc2_entry(tab.rc, i);
        s_mc2[i] = rc2_entry(tab.mc, i);  // the same composition of two table steps
    }
    for (uint32_t i = threadIdx.x; i < top_hist_words(th); i += B) h[i] = 0;
    if (threadIdx.x == 0) s_np = 0;
    __syncthreads();
    const uint32_t root = s_rc[0];  // child 0 of the embedded root: rank | rotation << 3
    uint32_t np = 0;
    const size_t stride = (size_t)gridDim.x * B, nround = (n + stride - 1) / stride * stride;  // whole waves stay in the loop
    for (size_t i = (size_t)blockIdx.x * B + threadIdx.x; i < nround; i += stride) {
        Key k{0ull, 0ull};
        if (i < n) {
            const Key o = in[i];
            const uint32_t l = key_level(o);
            k.hi = (uint64_t)(root & 7u) << 60;
            uint32_t r1 = 0, r2 = root >> 3, all = 7, t = 1;
            for (; t + 1 <= l && t + 2 <= 21; t += 2) {  // the pair's new place is inside the high word
                const uint32_t v = s_mc2[r1 * 64 + ((uint32_t)(o.hi >> (60 - 3 * t)) & 63u)], m = v & 63u;
                const uint32_t w = s_rc2[r2 * 64 + m];
                r1 = v >> 6;
                r2 = w >> 6;
                all &= m & (m >> 3);
                k.hi |= (uint64_t)(w & 63u) << (57 - 3 * t);
            }
            for (; t <= l; ++t) {
                const uint32_t v = s_mc[r1 * 8 + key_digit(o, t)], m = v & 7u, w = s_rc[r2 * 8 + m];
                r1 = v >> 3;
                r2 = w >> 3;
                all &= m;
                key_set_digit(k, t + 1, w & 7u);
            }
            k.lo |= l + 1;
            dkey[i] = k;
            bflag[i] = (uint8_t)all;
            if (unsorted && i && key_lt(o, in[i - 1])) atomicOr(unsorted, 1u);
            np += n_pseudo(all);
        }
        top_hist_add(h, th, k.hi, i < n);
    }
    for (int o = 32; o > 0; o >>= 1) np += (uint32_t)__shfl_xor(np, o, 64);
    if (__lane_id() == 0 && np) atomicAdd(&s_np, np);
    __syncthreads();
    if (threadIdx.x == 0 && s_np) atomicAdd(&ctr[C_NPSEUDO], s_np);
    top_hist_flush(h, th);
}

// The pseudo-octants of the octants on the positive boundary, in any order
// (they are sorted next): places by one atomic per workgroup that has any.  In
// Morton digits an axis moved to the boundary has its bits cleared below a 1 at
// the embedded root; both conversions take two levels per table read (one level
// per step, for every pseudo-octant, took 17.7 us for a 30,000-point octree
// instead of 12.2).
constexpr uint32_t BE_ITEMS = 4;
__global__ void __launch_bounds__(B) k_da_bdy_emit(const Key *in, const uint8_t *bflag, size_t n, SfcPacked tab,
                                                   uint32_t *ctr, Key *bkey) {
    __shared__ uint8_t s_rc[192], s_mc[192];
    __shared__ uint16_t s_rc2[24 * 64], s_mc2[24 * 64];
    __shared__ uint32_t red[B / 64 + 1];
    const size_t i0 = (size_t)blockIdx.x * B * BE_ITEMS + threadIdx.x;
    uint32_t f[BE_ITEMS], cnt = 0;
#pragma unroll
    for (uint32_t r = 0; r < BE_ITEMS; ++r) {
        const size_t i = i0 + (size_t)r * B;
        f[r] = i < n ? bflag[i] : 0u;
        cnt += n_pseudo(f[r]);
    }
    if (!__syncthreads_or(cnt != 0)) return;
    for (uint32_t i = threadIdx.x; i < 192; i += B) {
        s_rc[i] = tab.rc[i];
        s_mc[i] = tab.mc[i];
    }
    for (uint32_t i = threadIdx.x; i < 24 * 64; i += B) {
        s_rc2[i] = rc2_entry(tab.rc, i);
        s_mc2[i] = rc2_entry(tab.mc, i);
    }
    uint32_t o = block_reserve(&ctr[C_FILL], cnt, red);  // its barriers publish the tables
#pragma unroll 1
    for (uint32_t r = 0; r < BE_ITEMS; ++r) {
        if (!f[r]) continue;
        uint32_t rot;
        const Key m = morton_to_curve_rot(s_mc2, s_mc, in[i0 + (size_t)r * B], rot);  // curve to Morton
        // one level down, below child 0 of the embedded root
        const uint64_t hi = m.hi >> 3, lo = (m.lo & ~31ull) >> 3 | (m.hi & 7u) << 60;
        constexpr uint64_t X = 0x1249249249249249ull;  // the x bit of each digit
#pragma unroll 1
        for (uint32_t a = 1; a < 8; ++a) {  // the axes moved to the boundary
            if (a & ~f[r]) continue;
            const uint64_t clear = (a & 1u ? X : 0ull) | (a & 2u ? X << 1 : 0ull) | (a & 4u ? X << 2 : 0ull);
            const Key p{(hi & ~clear) | (uint64_t)a << 60, (lo & ~clear & ~31ull) | (key_level(m) + 1)};
            bkey[o++] = morton_to_curve_rot(s_rc2, s_rc, p, rot);
        }
    }
}

// The local buffer: the sorted elements, then the sorted pseudo-octants; keys,
// anchors, levels.  Thread c of the first 2^18 + 1 also finds where cell c
// begins.  Clears the marks of referred octants.
__global__ void __launch_bounds__(B) k_da_decode(const Key *ekey, const Key *bkey, size_t nelem, size_t n, uint32_t md,
                                                 SfcPacked tab, Key *key, uint32_t *xs, uint32_t *ys, uint32_t *zs,
                                                 uint8_t *flags, uint8_t *isnode, uint32_t *cstart) {
    __shared__ uint8_t s_mc[192];
    for (uint32_t i = threadIdx.x; i < 192; i += B) s_mc[i] = tab.mc[i];
    __syncthreads();
    const size_t i = (size_t)blockIdx.x * B + threadIdx.x;
    if (i < n) {
        const Key k = i < nelem ? ekey[i] : bkey[i - nelem];
        uint32_t x, y, z, l;
        dev_decode(s_mc, k, md, x, y, z, l);
        key[i] = k;
        xs[i] = x;
        ys[i] = y;
        zs[i] = z;
        flags[i] = (uint8_t)(l | (i >= nelem ? F_BOUNDARY : 0));
        isnode[i] = 0;
    }
    if (i <= (1u << kCellBits)) {
        size_t lo = 0, hi = n;
        if (i == (1u << kCellBits)) {
            lo = n;  // past every key (bit 63 of the high word is 0)
        } else {
            const uint64_t h = (uint64_t)i << kCellShift;  // first key whose high word is at least h
            while (lo < hi) {
                const size_t mid = lo + (hi - lo) / 2;
                if ((mid < nelem ? ekey[mid] : bkey[mid - nelem]).hi < h) lo = mid + 1;
                else hi = mid;
            }
        }
        cstart[i] = (uint32_t)lo;
    }
}

// Numbering of the nodes, over tiles of 16 octants per thread: the octants an
// element refers to become NODEs and each tile's NODEs are counted; one
// workgroup turns the counts into offsets; the last pass numbers them.  No
// array of flags or positions lies in between.
constexpr uint32_t NI = 16, NTILE = B * NI;
struct TileCount {
    uint32_t nodes, ref_e, ref_p;
};
__global__ void __launch_bounds__(B) k_node_count(const uint8_t *isnode, size_t n, size_t nelem, uint8_t *flags,
                                                  TileCount *tile) {
    __shared__ uint32_t s_c[3];
    if (threadIdx.x < 3) s_c[threadIdx.x] = 0;
    __syncthreads();
    const size_t i0 = (size_t)blockIdx.x * NTILE + (size_t)threadIdx.x * NI;
    uint32_t c[3] = {0, 0, 0};
    auto one = [&](size_t i, uint32_t ref, uint32_t &f) {
        if (ref) {
            f |= F_NODE;
            c[i < nelem ? 1 : 2] += 1;
        }
        c[0] += (f & F_NODE) ? 1u : 0u;
    };
    if (i0 + NI <= n) {
        const uint4 r = *reinterpret_cast<const uint4 *>(isnode + i0);
        uint4 f = *reinterpret_cast<const uint4 *>(flags + i0);
        const uint32_t rw[4] = {r.x, r.y, r.z, r.w};
        uint32_t fw[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (uint32_t q = 0; q < NI; ++q) {
            uint32_t v = (fw[q >> 2] >> (8 * (q & 3u))) & 255u;
            one(i0 + q, (rw[q >> 2] >> (8 * (q & 3u))) & 255u, v);
            fw[q >> 2] |= v << (8 * (q & 3u));
        }
        *reinterpret_cast<uint4 *>(flags + i0) = make_uint4(fw[0], fw[1], fw[2], fw[3]);
    } else {
        for (size_t i = i0; i < n; ++i) {
            uint32_t v = flags[i];
            one(i, isnode[i], v);
            flags[i] = (uint8_t)v;
        }
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        for (int o = 32; o > 0; o >>= 1) c[q] += (uint32_t)__shfl_xor(c[q], o, 64);
        if (__lane_id() == 0 && c[q]) atomicAdd(&s_c[q], c[q]);
    }
    __syncthreads();
    if (threadIdx.x == 0) tile[blockIdx.x] = TileCount{s_c[0], s_c[1], s_c[2]};
}
// Also adds up the blocks' octants and takes the most of one (ucount; an atomic
// per block on two words cost k_da_nodes 0.9 ms on 26,965 blocks).
__global__ void __launch_bounds__(1024) k_node_offsets(TileCount *tile, uint32_t nt, const uint32_t *ucount,
                                                       uint32_t nblk, uint32_t *ctr) {
    __shared__ uint32_t tmp[1024 / 64 + 1];
    uint32_t carry = 0, re = 0, rp = 0, np = 0, mx = 0;
#pragma unroll 4
    for (uint32_t b = threadIdx.x; b < nblk; b += 1024) {
        const uint32_t u = ucount[b];
        np += u;
        mx = max(mx, u);
    }
    for (uint32_t b = 0; b < nt; b += 1024) {
        const uint32_t t = b + threadIdx.x;
        const TileCount v = t < nt ? tile[t] : TileCount{0, 0, 0};
        uint32_t total;
        const uint32_t ex = block_excl_scan_u32(v.nodes, tmp, total);
        if (t < nt) tile[t].nodes = carry + ex;
        carry += total;
        re += v.ref_e;
        rp += v.ref_p;
    }
    for (int o = 32; o > 0; o >>= 1) {
        re += (uint32_t)__shfl_xor(re, o, 64);
        rp += (uint32_t)__shfl_xor(rp, o, 64);
        np += (uint32_t)__shfl_xor(np, o, 64);
        mx = max(mx, (uint32_t)__shfl_xor(mx, o, 64));
    }
    if (__lane_id() == 0) {
        if (re) atomicAdd(&ctr[C_REF_E], re);
        if (rp) atomicAdd(&ctr[C_REF_P], rp);
        if (np) atomicAdd(&ctr[C_PAIRS], np);
        atomicMax(&ctr[C_MAXN], mx);
    }
    if (threadIdx.x == 0) ctr[C_NODES] = carry;
}
// Local index <-> node id, whether a node lies on the boundary of the unit cube
// (anchor coordinate 0 or 2^(md-1)), and a cleared count of blocks per node.
__global__ void __launch_bounds__(B) k_node_number(const uint8_t *flags, size_t n, const TileCount *tile,
                                                   const uint32_t *xs, const uint32_t *ys, const uint32_t *zs,
                                                   uint32_t md, uint32_t *l2n, uint32_t *n2l, uint8_t *bdy,
                                                   uint32_t *ncount) {
    __shared__ uint32_t tmp[B / 64 + 1], s_pos[B];
    __shared__ uint16_t s_m[B];
    const size_t t0 = (size_t)blockIdx.x * NTILE, i0 = t0 + (size_t)threadIdx.x * NI;
    uint32_t m = 0;
    if (i0 + NI <= n) {
        const uint4 f = *reinterpret_cast<const uint4 *>(flags + i0);
        const uint32_t fw[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (uint32_t q = 0; q < NI; ++q) m |= ((fw[q >> 2] >> (8 * (q & 3u) + 7)) & 1u) << q;
    } else {
        for (uint32_t q = 0; i0 + q < n; ++q) m |= (flags[i0 + q] & F_NODE) ? 1u << q : 0u;
    }
    uint32_t total;
    s_pos[threadIdx.x] = tile[blockIdx.x].nodes + block_excl_scan_u32((uint32_t)__popc(m), tmp, total);
    s_m[threadIdx.x] = (uint16_t)m;
    __syncthreads();
    // the counts are per 16 octants of a thread, the accesses a row of B octants
    // at a time (16 of one thread at a time: 558 us instead of 57 for 14M)
    const uint32_t D = 1u << (md - 1);
#pragma unroll 4
    for (uint32_t r = 0; r < NI; ++r) {
        const uint32_t k = r * B + threadIdx.x, q = k % NI;
        const size_t i = t0 + k;
        if (i >= n) break;
        const uint32_t mk = s_m[k / NI], pos = s_pos[k / NI] + (uint32_t)__popc(mk & ((1u << q) - 1u));
        const bool node = (mk >> q) & 1u;
        l2n[i] = node ? pos : 0xffffffffu;
        if (!node) continue;
        const uint32_t x = xs[i], y = ys[i], z = zs[i];
        n2l[pos] = (uint32_t)i;
        bdy[pos] = x == 0 || y == 0 || z == 0 || x == D || y == D || z == D ? 1 : 0;
        ncount[pos] = 0;
    }
}

}  // namespace

DaDevice::~DaDevice() {}

static void da_build_blocks(DaDevice &da, BlockLists &bl, DevBuf<uint32_t> &ncount, uint32_t *ctr, hipStream_t s,
                            bool colour);

std::unique_ptr<DaDevice> da_build(const Key *oct, size_t n, uint32_t md0, int curve, hipStream_t s, bool colour,
                                   bool keep_cells) {
    if (n <= 8) {  // blockPartStage1 asserts nodes.size() > 2^dim (blockPart.cpp:583)
        dgx_set_error("ot::DA needs more than 8 octants (got %zu)", n);
        throw DgxError();
    }
    std::unique_ptr<DaDevice> da(new DaDevice());
    da->md = md0 + 1;
    da->curve = curve;
    const uint32_t md = md0 + 1;
    SfcPacked tab = make_packed(curve);
    // Part1
    DevBuf<uint32_t> ctr(C_COUNT, s);
    HIP_OK(hipMemsetAsync(ctr.p, 0, C_COUNT * 4, s));
    uint32_t hc[C_COUNT];
    DevBuf<Key> ekey(n, s);
    DevBuf<uint8_t> bflag(n, s);
    const unsigned eg = std::min(grid_for(n, B), n < (size_t(1) << 23) ? 2048u : 4096u);
    if (tab.rc[0] >> 3 == 0) {
        // The curve inside child 0 of the embedded root is the octree's own
        // (Morton), so a sorted octree's keys stay sorted and only an octree
        // imported unsorted needs the sort: 67 us of kernels in eight launches for
        // a 30,000-point octree.
        k_da_embed<<<eg, B, 0, s>>>(oct, n, tab, ekey.p, bflag.p, ctr.p, ctr.p + C_FAIL_E, TopHist{nullptr, 0, 0, 0});
        HIP_OK(hipGetLastError());
    } else {
        TopSort top(ekey.p, n, s);
        k_da_embed<<<eg, B, 0, s>>>(oct, n, tab, top.input(), bflag.p, ctr.p, nullptr, top.hist());
        HIP_OK(hipGetLastError());
        top.sort(true, ctr.p + C_FAIL_E);
    }
    dgx_read_back(hc, ctr.p, sizeof hc, s);
    if (hc[C_FAIL_E]) sort_keys_again(ekey.p, n, s, 0, hc[C_FAIL_E]);
    const size_t nbd = hc[C_NPSEUDO], N = n + nbd;
    DevBuf<Key> bkey(nbd, s);
    if (nbd) {
        TopSort top(bkey.p, nbd, s);
        k_da_bdy_emit<<<grid_for(n, B * BE_ITEMS), B, 0, s>>>(oct, bflag.p, n, tab, ctr.p, top.input());
        HIP_OK(hipGetLastError());
        // the steps up to the next host read need the order of the cells: no may_skip
        top.sort(false, ctr.p + C_FAIL_P);
    }
    bflag.release();
    da->n_local = N;
    da->n_elem = n;
    da->key.alloc(N, s);
    da->x.alloc(N, s);
    da->y.alloc(N, s);
    da->z.alloc(N, s);
    da->flags.alloc(N, s);
    const uint32_t ntile = grid_for(N, NTILE);
    DevBuf<uint32_t> &cstart = da->cstart;
    cstart.alloc((1u << kCellBits) + 1, s);
    DevBuf<uint8_t> isnode(N, s);
    DevBuf<TileCount> tile(ntile, s);
    BlockLists bl;
    for (;;) {
        k_da_decode<<<grid_for(std::max<size_t>(N, (1u << kCellBits) + 1), B), B, 0, s>>>(
            ekey.p, bkey.p, n, N, md, tab, da->key.p, da->x.p, da->y.p, da->z.p, da->flags.p, isnode.p, cstart.p);
        // Part2
        da_flag_nodes(*da, cstart.p, s);
        // Part3: node lists
        da_node_lists(*da, cstart.p, isnode.p, NodeCounters{ctr.p + C_UNRESOLVED, ctr.p + C_BAD}, bl, s);
        k_node_count<<<ntile, B, 0, s>>>(isnode.p, N, n, da->flags.p, tile.p);
        k_node_offsets<<<1, 1024, 0, s>>>(tile.p, ntile, bl.ucount.p, grid_for(n, kElemBlock), ctr.p);
        HIP_OK(hipGetLastError());
        dgx_read_back(hc, ctr.p, sizeof hc, s);
        if (!hc[C_FAIL_P]) break;
        // a cell of the boundary holds more pseudo-octants than TopSort orders:
        // sort them again and redo the steps
        sort_keys_again(bkey.p, nbd, s, 0, hc[C_FAIL_P]);
        HIP_OK(hipMemsetAsync(ctr.p, 0, C_COUNT * 4, s));
    }
    if (!keep_cells) cstart.release();
    ekey.release();
    bkey.release();
    isnode.release();
    const uint32_t nn = hc[C_NODES];
    da->n_unresolved = hc[C_UNRESOLVED];
    da->n_ghost_scans = hc[C_GHOST];
    da->node_size = hc[C_REF_E];
    da->bnd_node_size = hc[C_REF_P];
    da->n_nodes = nn;
    if (hc[C_UNRESOLVED]) {
        dgx_set_error("ot::DA: %u node-list entries unresolved on one rank", hc[C_UNRESOLVED]);
        throw DgxError();
    }
    if (hc[C_REF_E] + hc[C_REF_P] != nn) {
        dgx_set_error("ot::DA: %u NODE octants but %u referenced nodes", nn, hc[C_REF_E] + hc[C_REF_P]);
        throw DgxError();
    }
    if ((uint64_t)hc[C_MAXN] * 8 > 65535) {  // lconn holds 16-bit byte offsets of 8-byte slots
        dgx_set_error("DA: an element block touches %u nodes, more than the 8191 its records can address", hc[C_MAXN]);
        throw DgxError();
    }
    da->l2n.alloc(N, s);
    da->n2l.alloc(nn, s);
    da->bdy_node.alloc(nn, s);
    DevBuf<uint32_t> ncount(nn, s);
    k_node_number<<<ntile, B, 0, s>>>(da->flags.p, N, tile.p, da->x.p, da->y.p, da->z.p, md, da->l2n.p, da->n2l.p,
                                      da->bdy_node.p, ncount.p);
    HIP_OK(hipGetLastError());
    da->n_pairs = hc[C_PAIRS];
    da->max_block_nodes = hc[C_MAXN];
    da_build_blocks(*da, bl, ncount, ctr.p, s, colour);
    HIP_OK(hipStreamSynchronize(s));
    return da;
}

// ---------------------------------------------------------------------------
// Matvec block view.
// ---------------------------------------------------------------------------
namespace {

constexpr uint32_t ID_MASK = 0x3fffffffu, BDY_BIT = 0x40000000u, SHARED_BIT = 0x80000000u, NO_SLOT = 0xffffffffu;

// Turns the blocks' lists of octants into node ids, which follow the order of
// the octants (bit 30: a Dirichlet boundary node), counts the blocks of each
// node, and writes the elements' node ids (conn) from the block's local
// indices: one lookup in LDS per vertex instead of a read of l2n.
__global__ void __launch_bounds__(kElemBlock) k_blk_nodes(const uint32_t *ulist, const uint32_t *l2n,
                                                          const uint8_t *bdy, const uint32_t *boff, size_t ne,
                                                          const uint16_t *lconn, const uint16_t *meta, uint32_t *bnode,
                                                          uint32_t *ncount, uint32_t *conn) {
    constexpr uint32_t EB = kElemBlock;
    __shared__ uint32_t id[8 * EB];
    __shared__ uint32_t wf[EB / 64], wh[EB / 64];
    const uint32_t b = blockIdx.x, t = threadIdx.x, s0 = boff[b], n = boff[b + 1] - s0;
    const uint32_t *ul = ulist + (size_t)b * 8 * EB;
    for (uint32_t i = t; i < n; i += EB) {
        const uint32_t g = l2n[ul[i]];
        id[i] = g;
        bnode[s0 + i] = g | (bdy[g] ? BDY_BIT : 0u);
        atomicAdd(&ncount[g], 1u);
    }
    // the slot of element t, as its record was placed
    const size_t e = (size_t)b * EB + t;
    const uint32_t nb = (uint32_t)min((size_t)EB, ne - (size_t)b * EB), lane = t & 63u, wid = t >> 6;
    const bool valid = t < nb;
    const uint32_t mt = valid ? meta[e] : 0u;
    const bool hang = (mt & 255u) != 0;
    const uint64_t bf = __ballot(valid && !hang), bh = __ballot(hang);
    if (lane == 0) {
        wf[wid] = (uint32_t)__popcll(bf);
        wh[wid] = (uint32_t)__popcll(bh);
    }
    __syncthreads();
    if (!valid) return;
    uint32_t pf = 0, ph = 0, nflat = 0;
    for (uint32_t w = 0; w < EB / 64; ++w) {
        if (w < wid) {
            pf += wf[w];
            ph += wh[w];
        }
        nflat += wf[w];
    }
    const uint64_t lt = (1ull << lane) - 1ull;
    const uint32_t slot = hang ? nflat + spread8(ph + (uint32_t)__popcll(bh & lt), nb - nflat)
                               : spread8(pf + (uint32_t)__popcll(bf & lt), nflat);
    const uint4 r = *reinterpret_cast<const uint4 *>(lconn + ((size_t)b * EB + slot) * 8);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w}, c = (mt >> 8) & 7u;
    uint32_t v[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) v[q] = id[((w[q >> 1] >> (16 * (q & 1u))) & 0xffffu) >> 3];
    child_frame(v, c);
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) conn[(size_t)j * ne + e] = v[j];
}
// Shared nodes (touched by more than one block) and their node-major partial
// slots, one per block touching the node, blocks in increasing order.  Tiles
// of 16 nodes per thread count the shared nodes and their slots, one workgroup
// turns the counts into offsets, and the last pass numbers both:
//   base[g] = first slot of node g (NO_SLOT if not shared), snode, soff.
__device__ __forceinline__ void load16(const uint32_t *a, size_t i0, size_t n, uint32_t *v) {
    if (i0 + 16 <= n) {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint4 r = reinterpret_cast<const uint4 *>(a + i0)[q];
            v[4 * q] = r.x;
            v[4 * q + 1] = r.y;
            v[4 * q + 2] = r.z;
            v[4 * q + 3] = r.w;
        }
    } else {
#pragma unroll
        for (uint32_t q = 0; q < 16; ++q) v[q] = i0 + q < n ? a[i0 + q] : 0u;
    }
}
__global__ void __launch_bounds__(B) k_shared_count(const uint32_t *ncount, uint32_t nn, uint2 *tile) {
    __shared__ uint32_t s_c[2];
    if (threadIdx.x < 2) s_c[threadIdx.x] = 0;
    __syncthreads();
    uint32_t v[16], sh = 0, sl = 0;
    load16(ncount, (size_t)blockIdx.x * NTILE + threadIdx.x * 16u, nn, v);
#pragma unroll
    for (uint32_t q = 0; q < 16; ++q)
        if (v[q] > 1) {
            ++sh;
            sl += v[q];
        }
    for (int o = 32; o > 0; o >>= 1) {
        sh += (uint32_t)__shfl_xor(sh, o, 64);
        sl += (uint32_t)__shfl_xor(sl, o, 64);
    }
    if (__lane_id() == 0 && sh) {
        atomicAdd(&s_c[0], sh);
        atomicAdd(&s_c[1], sl);
    }
    __syncthreads();
    if (threadIdx.x == 0) tile[blockIdx.x] = make_uint2(s_c[0], s_c[1]);
}
__global__ void __launch_bounds__(1024) k_shared_offsets(uint2 *tile, uint32_t nt, uint32_t *ctr) {
    __shared__ uint32_t tmp[1024 / 64 + 1];
    uint32_t c0 = 0, c1 = 0;
    for (uint32_t b = 0; b < nt; b += 1024) {
        const uint32_t t = b + threadIdx.x;
        const uint2 v = t < nt ? tile[t] : make_uint2(0, 0);
        uint32_t t0, t1;
        const uint32_t e0 = block_excl_scan_u32(v.x, tmp, t0);
        const uint32_t e1 = block_excl_scan_u32(v.y, tmp, t1);
        if (t < nt) tile[t] = make_uint2(c0 + e0, c1 + e1);
        c0 += t0;
        c1 += t1;
    }
    if (threadIdx.x == 0) {
        ctr[C_SHARED] = c0;
        ctr[C_SLOTS] = c1;
    }
}
__global__ void __launch_bounds__(B) k_shared_number(const uint32_t *ncount, uint32_t nn, const uint2 *tile,
                                                     const uint8_t *bdy, uint32_t *base, uint32_t *snode,
                                                     uint32_t *soff, uint32_t nsn, uint32_t ns) {
    __shared__ uint32_t tmp[B / 64 + 1], s_a[B];
    __shared__ uint16_t s_m[B];
    __shared__ uint32_t s_o[NTILE + NTILE / 16];  // first slot per node, padded against bank conflicts
    const size_t t0 = (size_t)blockIdx.x * NTILE, i0 = t0 + threadIdx.x * 16u;
    uint32_t v[16], m = 0, sl = 0;
    load16(ncount, i0, nn, v);
#pragma unroll
    for (uint32_t q = 0; q < 16; ++q)
        if (v[q] > 1) {
            m |= 1u << q;
            sl += v[q];
        }
    uint32_t total;
    s_a[threadIdx.x] = tile[blockIdx.x].x + block_excl_scan_u32((uint32_t)__popc(m), tmp, total);
    s_m[threadIdx.x] = (uint16_t)m;
    uint32_t o = tile[blockIdx.x].y + block_excl_scan_u32(sl, tmp, total);
#pragma unroll
    for (uint32_t q = 0; q < 16; ++q) {
        s_o[threadIdx.x * 17u + q] = v[q] > 1 ? o : NO_SLOT;
        o += v[q] > 1 ? v[q] : 0u;
    }
    __syncthreads();
#pragma unroll 4
    for (uint32_t r = 0; r < 16; ++r) {
        const uint32_t k = r * B + threadIdx.x, q = k % 16u;
        const size_t g = t0 + k;
        if (g >= nn) break;
        const uint32_t first = s_o[k + k / 16u], mk = s_m[k / 16u];
        base[g] = first;
        if (first == NO_SLOT) continue;
        const uint32_t a = s_a[k / 16u] + (uint32_t)__popc(mk & ((1u << q) - 1u));
        snode[a] = (uint32_t)g | (bdy[g] ? BDY_BIT : 0u);
        soff[a] = first;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) soff[nsn] = ns;
}
// every shared pair claims a slot of its node, in any order (the counts of
// blocks are used up) ...
__global__ void k_shared_claim(uint32_t *bnode, const uint32_t *base, uint32_t np, uint32_t *ncount,
                               uint32_t *tpair) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const uint32_t v = bnode[p], g = v & ID_MASK, a = base[g];
    if (a == NO_SLOT) return;
    bnode[p] = v | SHARED_BIT;
    tpair[a + atomicSub(&ncount[g], 1u) - 1u] = p;
}
// ... and each shared node orders its pairs (few), which follow the blocks
__global__ void k_shared_order(const uint32_t *soff, uint32_t nsn, uint32_t *tpair, uint32_t *bdst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nsn) return;
    const uint32_t a = soff[i], z = soff[i + 1];
    for (uint32_t q = a + 1; q < z; ++q) {
        const uint32_t kp = tpair[q];
        uint32_t r = q;
        while (r > a && tpair[r - 1] > kp) {
            tpair[r] = tpair[r - 1];
            --r;
        }
        tpair[r] = kp;
    }
    for (uint32_t q = a; q < z; ++q) bdst[tpair[q]] = q;
}
// Node numbering inside a block against LDS bank conflicts.  The matvec adds
// element results into the block's FP64 LDS slots with ds_add_f64, which
// serves 16 lanes per pass and runs without conflicts (8 clocks per wave
// instruction on gfx950) only when their slots differ mod 16; an unordered
// numbering costs about 3x that.  The 16 lanes of one pass are 16 consecutive
// element slots of the block at one record position p, a "lane group".  The
// block's nodes are coloured greedily with 16 colours (colour = slot mod 16):
// each node takes the colour used least so far by the lane groups it appears
// in (ties rotate with the node index), colour c holding
// exactly n/16 + (c < n mod 16) nodes, so that slot = 16 x (rank inside its
// colour) + colour is again a permutation of 0..n-1.  The records and the
// node list are then renumbered.  Deterministic (the use counts are updated
// with atomics); one workgroup per block.  Blocks past this kernel's LDS tables (more than kColMaxN nodes or
// kColMaxE elements) keep the sorted numbering.
// Two waves per block colour 8 nodes per step.  Measured on the lognormal-4M
// DA (matvec back to back / multigrid set-up): one wave, 4 nodes per step,
// 29.5 us / 30.0 ms; two waves 29.7 us / 29.0 ms; four waves 30.0 us / 28.3 ms.
// The LDS tables are sized by the template: <kColSmallN, kColSmallE> (13 KB,
// twelve workgroups per CU) takes the blocks that fit it, and <kColMaxN,
// kColMaxE> (33 KB, four per CU) the rest (big = true skips the small ones).
// Both number a block identically.  The colour use counts reuse the degree
// table, and the node-list copy at the end the adjacency table, each once the
// earlier one is dead.
// With at most kColFewBlocks blocks, a few per CU, the chain of steps is what
// counts, and four waves take 16 nodes per step (G = 16): 77 -> 54 us on the
// levels of a 16,000-point hierarchy; DA build of 10,000 uniform points 313 ->
// 293 us, 30,000 351 -> 343, 120,000 492 -> 486, 250,000 (past the line) 668
// against 697; the matvecs of these DAs take the same time within 2 %.
constexpr uint32_t kColFewBlocks = 1024;
constexpr uint32_t kColMaxN = 2048, kColMaxE = 1024, kColSmallN = 1024, kColSmallE = 512;
// 12-byte element records: the 8 local indices (10 bits each, from lconn's
// byte offsets of 8-byte slots) and cmeta in the top 16 bits.
__device__ __forceinline__ void pack_record(const uint32_t v[8], uint32_t cm, uint32_t *rec) {
    rec[0] = v[0] | v[1] << 10 | v[2] << 20 | v[3] << 30;
    rec[1] = v[3] >> 2 | v[4] << 8 | v[5] << 18 | v[6] << 28;
    rec[2] = v[6] >> 4 | v[7] << 6 | cm << 16;
}
// lrec (nullptr: blocks too large for it) receives the renumbered records too.
template <uint32_t MAXN, uint32_t MAXE, bool BIG, uint32_t G>
__global__ void __launch_bounds__(16 * G) k_blk_color(uint16_t *lconn, const uint32_t *boff, uint32_t *bnode,
                                                     size_t ne, uint32_t eb, const uint16_t *cmeta, uint32_t *lrec) {
    constexpr uint32_t kCntWords = ((MAXE / 16) * 8 + 1) * 16 / 4;  // and a row that stays 0
    // degree, then fill position; then [lane group][colour] uses so far, one
    // byte each (at most 16 uses per lane group), four to a word for the
    // atomic updates
    __shared__ __align__(16) uint32_t degcnt[MAXN > kCntWords ? MAXN : kCntWords];
    uint32_t *deg = degcnt, *cnt32 = degcnt;
    uint8_t *cnt = reinterpret_cast<uint8_t *>(degcnt);
    __shared__ uint16_t ptr[MAXN + 1];  // adjacency offsets
    // lane groups of each node's uses; then the copy of the node list
    using Grp = typename std::conditional<(MAXE / 16) * 8 <= 256, uint8_t, uint16_t>::type;
    constexpr uint32_t kAdjWords = 8 * MAXE * sizeof(Grp) / 4;
    __shared__ uint32_t adjw[kAdjWords > MAXN ? kAdjWords : MAXN];
    Grp *adj = reinterpret_cast<Grp *>(adjw);
    uint32_t *tmp = adjw;
    __shared__ uint16_t newidx[MAXN];
    constexpr uint32_t NT = 16 * G, PW = G / 4;
    static_assert(G % 4 == 0 && (MAXN >> 4) + 1 < 255, "picks and colour counts are bytes of words");
    __shared__ __align__(16) uint32_t pick[2][PW];  // the groups' choices of a step, one byte each
    const uint32_t b = blockIdx.x, tid = threadIdx.x;
    const uint32_t s0 = boff[b], n = boff[b + 1] - s0;
    const size_t e0 = (size_t)b * eb;
    if (n > MAXN || eb > MAXE || e0 >= ne) return;  // uniform over the workgroup
    if (BIG && n <= kColSmallN && eb <= kColSmallE) return;  // coloured by the small variant
    const uint32_t nbe = (uint32_t)min((size_t)eb, ne - e0), nuse = 8 * nbe;
    const uint32_t ngroups = ((nbe + 15) / 16) * 8;
    uint16_t *rec = lconn + e0 * 8;
    for (uint32_t i = tid; i < n; i += NT) deg[i] = 0;
    __syncthreads();
    for (uint32_t t = tid; t < nuse; t += NT) atomicAdd(&deg[rec[t] >> 3], 1u);
    __syncthreads();
    if (tid < 64) {  // exclusive scan of the degrees, one chunk per lane of wave 0
        const uint32_t lane = tid;
        const uint32_t ch = (n + 63) / 64, i0 = min(n, lane * ch), i1 = min(n, i0 + ch);
        uint32_t sum = 0;
        for (uint32_t i = i0; i < i1; ++i) sum += deg[i];
        uint32_t incl = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(incl, o, 64);
            if ((int)lane >= o) incl += v;
        }
        uint32_t run = incl - sum;
        for (uint32_t i = i0; i < i1; ++i) {
            const uint32_t d = deg[i];
            ptr[i] = (uint16_t)run;
            deg[i] = run;
            run += d;
        }
        if (lane == 63) ptr[n] = (uint16_t)incl;
    }
    __syncthreads();
    for (uint32_t t = tid; t < nuse; t += NT) {
        const uint32_t q = atomicAdd(&deg[rec[t] >> 3], 1u);
        adj[q] = (Grp)((t >> 7) * 8 + (t & 7));  // element slot t/8, lane group (t/8)/16, position t%8
    }
    __syncthreads();
    for (uint32_t i = tid; i < ngroups * 4 + 4; i += NT) cnt32[i] = 0;  // the degrees are dead
    __syncthreads();
    const uint32_t base = n >> 4, extra = n & 15u;
    // G nodes per step, one per 16-lane group, taken from the G equal
    // parts of the list (far apart, so they rarely share lane groups); lane j
    // of a group scores colour j, ties going to the first colour from l on.  The
    // choices are then committed in order, a choice whose colour has filled up
    // in this step moving to the next colour with room.  Bound: the chain of
    // dependent LDS accesses and lane exchanges of a step (few blocks), instruction
    // issue (many).  So the uses of the next step's nodes are read ahead, the
    // minimum over a group's lanes is taken by DPP rotations, and every thread
    // commits all choices itself, comparing them byte by byte in two words, from
    // the colours' counts in registers (lane j of each group has colour j's).  On
    // the 26,965 blocks of a 13.8M-element mesh and on 250 blocks: choices committed
    // by one thread through counts in LDS 2.88 ms and 216 us; one colour count read
    // at a time and slots assigned as well 1.79 ms and 105 us; now 1.13 ms and 84
    // us.  One wave with two nodes per group and no barrier was slower.
    const uint32_t g = tid >> 4, j = tid & 15u, part = (n + G - 1) / G;
    const uint32_t cap = base + (j < extra ? 1u : 0u);
    uint32_t used = 0;  // nodes of colour j so far
    // Lane j holds use j of its group's node (kNoUse past the last one, whose
    // counts stay 0).  It reads that use's 16 colour counts at once, and the lanes
    // exchange halves of them (lane bits 3 to 0, sums in 16 bits) until lane j has
    // the sum of colour j.
    const uint32_t kNoUse = ngroups;
    struct Node {
        uint32_t l, a, z, use;
        bool has;
    } nx;
    auto fetch = [&](uint32_t t) {
        nx.l = g * part + t;
        nx.has = t < part && nx.l < n;
        nx.a = nx.has ? ptr[nx.l] : 0u;
        nx.z = nx.has ? ptr[nx.l + 1] : 0u;
        nx.use = nx.a + j < nx.z ? adj[nx.a + j] : kNoUse;
    };
    const bool b3 = j & 8u, b2 = j & 4u, b0 = j & 1u;
    const uint32_t keep = j & 2u ? 0x07060302u : 0x05040100u, send = j & 2u ? 0x05040100u : 0x07060302u;
    auto score = [&](uint32_t use) {
        const uint4 w = reinterpret_cast<const uint4 *>(cnt)[use];
        constexpr uint32_t M = 0x00ff00ffu;
#define DGX_LANE(x, ctrl) (uint32_t) __builtin_amdgcn_update_dpp(0, (int)(x), ctrl, 0xf, 0xf, false)
        const uint32_t k0 = b3 ? w.z : w.x, k1 = b3 ? w.w : w.y;
        const uint32_t r0 = DGX_LANE(b3 ? w.x : w.z, 0x128), r1 = DGX_LANE(b3 ? w.y : w.w, 0x128);  // row_ror:8
        const uint32_t a = (k0 & M) + (r0 & M), b = ((k0 >> 8) & M) + ((r0 >> 8) & M);
        const uint32_t c = (k1 & M) + (r1 & M), d = ((k1 >> 8) & M) + ((r1 >> 8) & M);
        const uint32_t e = (b2 ? c : a) + DGX_LANE(b2 ? a : c, 0x141);  // row_half_mirror
        const uint32_t f = (b2 ? d : b) + DGX_LANE(b2 ? b : d, 0x141);
        // quad_perm: lanes 2 apart, then 1 apart
        const uint32_t h = __builtin_amdgcn_perm(f, e, keep) + DGX_LANE(__builtin_amdgcn_perm(f, e, send), 0x4e);
        const uint32_t lo = h & 0xffffu, hi = h >> 16;
        return (b0 ? hi : lo) + DGX_LANE(b0 ? lo : hi, 0xb1);
#undef DGX_LANE
    };
    // bit 7 of each byte that is 0
    auto zero_bytes = [](uint32_t x) { return ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu); };
    fetch(0);
    for (uint32_t t = 0; t < part; ++t) {
        const Node nd = nx;
        uint32_t pen = score(nd.use);
        for (uint32_t q = nd.a + 16; __ballot(q < nd.z); q += 16) pen += score(q + j < nd.z ? adj[q + j] : kNoUse);
        fetch(t + 1);
        uint32_t key = nd.has && used < cap ? ((pen << 4) | ((j - nd.l) & 15u)) : 0xffffffffu;
        key = min(key, (uint32_t)__builtin_amdgcn_update_dpp((int)key, (int)key, 0x128, 0xf, 0xf, false));  // row_ror:8
        key = min(key, (uint32_t)__builtin_amdgcn_update_dpp((int)key, (int)key, 0x124, 0xf, 0xf, false));
        key = min(key, (uint32_t)__builtin_amdgcn_update_dpp((int)key, (int)key, 0x122, 0xf, 0xf, false));
        key = min(key, (uint32_t)__builtin_amdgcn_update_dpp((int)key, (int)key, 0x121, 0xf, 0xf, false));
        if (j == 0)
            reinterpret_cast<uint8_t *>(pick[t & 1])[g] =
                (uint8_t)(!nd.has ? 254u : key == 0xffffffffu ? 255u : ((key & 15u) + nd.l) & 15u);
        __syncthreads();
        uint32_t pw[PW], more = 0, none = 0;
#pragma unroll
        for (uint32_t q = 0; q < PW; ++q) pw[q] = pick[t & 1][q];
#pragma unroll
        for (uint32_t q = 0; q < PW; ++q) {
            pw[q] = (uint32_t)__builtin_amdgcn_readfirstlane((int)pw[q]);
            more += (uint32_t)__popc(zero_bytes(pw[q] ^ j * 0x01010101u));
            none |= zero_bytes(~pw[q]);
        }
        auto choice = [&](uint32_t h) {
            uint32_t w = pw[0];
#pragma unroll
            for (uint32_t q = 1; q < PW; ++q) w = (h >> 2) == q ? pw[q] : w;
            return (w >> (8 * (h & 3u))) & 255u;
        };
        uint32_t mine = choice(g);
        if (!none && !__ballot(used + more > cap)) {  // every choice has room
            used += more;
        } else {
            for (uint32_t h = 0; h < G; ++h) {
                const uint32_t lh = h * part + t;
                if (lh >= n) continue;
                uint32_t c = choice(h);
                bool room = false;
                for (uint32_t d = 0; d <= 16 && !room; ++d) {  // the choice, then the colours from lh on
                    if (d) c = (lh + d - 1) & 15u;
                    else if (c == 255u) continue;
                    room = (uint32_t)__shfl((int)used, (int)((tid & 48u) | c), 64) < base + (c < extra ? 1u : 0u);
                }
                if (h == g) mine = c;
                if (c == j) used += 1;
            }
        }
        if (nd.has) {
            if (j == 0) newidx[nd.l] = (uint16_t)mine;
            if (nd.use != kNoUse) {
                const uint32_t idx = nd.use * 16u + mine;
                atomicAdd(&cnt32[idx >> 2], 1u << (8 * (idx & 3u)));
            }
            for (uint32_t q = nd.a + j + 16; q < nd.z; q += 16) {
                const uint32_t idx = adj[q] * 16u + mine;
                atomicAdd(&cnt32[idx >> 2], 1u << (8 * (idx & 3u)));
            }
        }
        __syncthreads();
    }
    // newidx holds colours; inside each the slots follow the node order (ascending ids), so
    // that neighbouring slots hold nearby nodes and a wave's gathers and
    // stores touch fewer lines.  Thread (part p, colour c) counts its colour
    // in the p-th of G parts of the list, then renumbers it.
    {
        __shared__ uint32_t ccount[G][16];
        const uint32_t c = tid & 15u, p = tid >> 4;
        const uint32_t ch = (n + G - 1) / G, i0 = min(n, p * ch), i1 = min(n, i0 + ch);
        uint32_t k = 0;
        for (uint32_t i = i0; i < i1; ++i) k += (newidx[i] & 15u) == c ? 1u : 0u;
        ccount[p][c] = k;
        __syncthreads();
        uint32_t r = 0;
        for (uint32_t q = 0; q < p; ++q) r += ccount[q][c];
        // the colour bits of newidx[] do not change, so other threads' tests stay valid
        for (uint32_t i = i0; i < i1; ++i)
            if ((newidx[i] & 15u) == c) newidx[i] = (uint16_t)((r++) * 16u + c);
        __syncthreads();
    }
    for (uint32_t e = tid; e < nbe; e += NT) {
        uint4 *r4 = reinterpret_cast<uint4 *>(rec) + e;
        const uint4 r = *r4;
        const uint32_t w[4] = {r.x, r.y, r.z, r.w};
        uint32_t v[8];
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) v[q] = newidx[((w[q >> 1] >> (16 * (q & 1u))) & 0xffffu) >> 3];
        *r4 = make_uint4(v[0] << 3 | v[1] << 19, v[2] << 3 | v[3] << 19, v[4] << 3 | v[5] << 19, v[6] << 3 | v[7] << 19);
        if (lrec) pack_record(v, cmeta[e0 + e], lrec + 3 * (e0 + e));
    }
    for (uint32_t i = tid; i < n; i += NT) tmp[i] = bnode[s0 + i];
    __syncthreads();
    for (uint32_t i = tid; i < n; i += NT) bnode[s0 + newidx[i]] = tmp[i];
}
__global__ void k_blk_pack(const uint16_t *lconn, const uint16_t *cmeta, size_t n, uint32_t *rec) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    uint32_t v[8];
    for (int j = 0; j < 8; ++j) v[j] = (lconn[8 * e + j] >> 3) & 1023u;
    pack_record(v, cmeta[e], rec + 3 * e);
}

}  // namespace

static void da_build_blocks(DaDevice &da, BlockLists &bl, DevBuf<uint32_t> &ncount, uint32_t *ctr, hipStream_t s,
                            bool colour) {
    const size_t E = da.n_elem;
    const uint32_t eb = kElemBlock, nblk = (uint32_t)((E + eb - 1) / eb), nn = da.n_nodes;
    const uint32_t np = (uint32_t)da.n_pairs, nt = grid_for(nn, NTILE);
    const bool small = da.max_block_nodes <= kPipeMaxNodes;
    da.n_blocks = nblk;
    da.bnode_off.alloc(nblk + 1, s);
    scan_exclusive_u32_async(bl.ucount.p, da.bnode_off.p, nblk + 1, nullptr, s);
    da.bnode.alloc(np, s);
    da.conn.alloc(8 * E, s);
    k_blk_nodes<<<nblk, eb, 0, s>>>(bl.ulist.p, da.l2n.p, da.bdy_node.p, da.bnode_off.p, E, da.lconn.p, da.meta.p,
                                    da.bnode.p, ncount.p, da.conn.p);
    DevBuf<uint2> tile(nt, s);
    k_shared_count<<<nt, B, 0, s>>>(ncount.p, nn, tile.p);
    k_shared_offsets<<<1, 1024, 0, s>>>(tile.p, nt, ctr);
    HIP_OK(hipGetLastError());
    bl.ulist.release();
    bl.ucount.release();
    if (small) da.lrec.alloc(3 * (size_t)nblk * eb, s);
    if (colour) {
        if (nblk <= kColFewBlocks)
            k_blk_color<kColSmallN, kColSmallE, false, 16><<<nblk, 256, 0, s>>>(
                da.lconn.p, da.bnode_off.p, da.bnode.p, E, eb, da.cmeta.p, da.lrec.p);
        else
            k_blk_color<kColSmallN, kColSmallE, false, 8><<<nblk, 128, 0, s>>>(
                da.lconn.p, da.bnode_off.p, da.bnode.p, E, eb, da.cmeta.p, da.lrec.p);
        if (da.max_block_nodes > kColSmallN)
            k_blk_color<kColMaxN, kColMaxE, true, 8><<<nblk, 128, 0, s>>>(da.lconn.p, da.bnode_off.p, da.bnode.p, E, eb,
                                                                          da.cmeta.p, da.lrec.p);
    } else if (small) {
        k_blk_pack<<<grid_for((size_t)nblk * eb, B), B, 0, s>>>(da.lconn.p, da.cmeta.p, (size_t)nblk * eb, da.lrec.p);
    }
    HIP_OK(hipGetLastError());
    uint32_t hs[2];
    dgx_read_back(hs, ctr + C_SHARED, sizeof hs, s);
    const uint32_t nsn = hs[0], ns = hs[1];
    da.bdst.alloc(np, s);  // read for every pair, used for the shared ones
    if (ns) {
        DevBuf<uint32_t> base(nn, s), tpair(ns, s);
        da.snode.alloc(nsn, s);
        da.soff.alloc(nsn + 1, s);
        k_shared_number<<<nt, B, 0, s>>>(ncount.p, nn, tile.p, da.bdy_node.p, base.p, da.snode.p, da.soff.p, nsn, ns);
        k_shared_claim<<<grid_for(np, B), B, 0, s>>>(da.bnode.p, base.p, np, ncount.p, tpair.p);
        k_shared_order<<<grid_for(nsn, B), B, 0, s>>>(da.soff.p, nsn, tpair.p, da.bdst.p);
        HIP_OK(hipGetLastError());
        da.n_shared = nsn;
    }
    da.partial_slots = ns;
    da.partial.alloc(ns, s);
}
