// dgx_sort.hip -- device-wide primitives: exclusive scan and stable LSD radix
// sort of 128-bit SFC keys for gfx950.
//
// Radix sort (one-sweep): digits of 8 bits (9 for a large sort on top bits),
// tiles of 2048 to 8192 keys.  One up-front pass builds the global histogram
// of every candidate digit position, and one workgroup turns them into global
// digit offsets and skips positions whose digit is the same in every key, all
// on the device.  Each remaining pass is ONE kernel: a tile counts its digits,
// publishes the counts, ranks its keys stably (a ballot per bit, LDS counters
// across the waves), obtains the counts of the tiles before it
// by decoupled look-back, and writes its keys run by run.
#include "dgx_common.h"

#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <type_traits>
#include <vector>

namespace {

constexpr int SB = 256;          // threads per block
constexpr int SITEMS = kSortItems;  // keys per thread per tile

template <int RB = 8>
__device__ __forceinline__ uint32_t digit_of(const Key &k, int bit) {
    if (RB == 9) return (uint32_t)(k.hi >> (bit - 64)) & 511u;  // in the high word
    return bit >= 64 ? (uint32_t)((k.hi >> (bit - 64)) & 255u) : (uint32_t)((k.lo >> bit) & 255u);
}

// ---------------------------------------------------------------- scan ----
constexpr int SCAN_B = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_B * SCAN_ITEMS;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *lds, uint32_t &total) {
    // lds: SCAN_B/64 + 1 entries
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t acc = 0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            uint32_t t = lds[w];
            lds[w] = acc;
            acc += t;
        }
        lds[blockDim.x >> 6] = acc;
    }
    __syncthreads();
    uint32_t res = x - v + lds[wid];
    total = lds[blockDim.x >> 6];
    __syncthreads();
    return res;
}

__global__ void __launch_bounds__(SCAN_B) k_scan_reduce(const uint32_t *in, size_t n, uint32_t *partial) {
    __shared__ uint32_t lds[SCAN_B / 64 + 1];
    size_t base = (size_t)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        size_t idx = base + (size_t)i * SCAN_B + threadIdx.x;
        if (idx < n) s += in[idx];
    }
    uint32_t tot;
    block_exclusive_scan(s, lds, tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// Single block: exclusive scan of the per-tile partials (any count).
__global__ void __launch_bounds__(1024) k_scan_partials(uint32_t *partial, size_t np, uint32_t *d_total) {
    __shared__ uint32_t lds[1024 / 64 + 1];
    uint32_t carry = 0;
    for (size_t base = 0; base < np; base += 1024) {
        size_t idx = base + threadIdx.x;
        uint32_t v = idx < np ? partial[idx] : 0u;
        uint32_t tot;
        uint32_t ex = block_exclusive_scan(v, lds, tot);
        if (idx < np) partial[idx] = ex + carry;
        carry += tot;
    }
    if (threadIdx.x == 0 && d_total) *d_total = carry;
}

// The tile is staged through LDS (padded against bank conflicts), so global
// loads and stores are coalesced while each thread scans 16 consecutive items.
__device__ __forceinline__ uint32_t scan_pad(uint32_t x) { return x + (x >> 5); }
__global__ void __launch_bounds__(SCAN_B) k_scan_down(const uint32_t *in, uint32_t *out, size_t n,
                                                     const uint32_t *partial) {
    __shared__ uint32_t lds[SCAN_B / 64 + 1];
    __shared__ uint32_t t[SCAN_TILE + SCAN_TILE / 32];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE;
    const uint32_t tid = threadIdx.x;
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        const uint32_t e = (uint32_t)r * SCAN_B + tid;
        t[scan_pad(e)] = base + e < n ? in[base + e] : 0u;
    }
    __syncthreads();
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        v[i] = t[scan_pad(tid * SCAN_ITEMS + i)];
        s += v[i];
    }
    uint32_t tot;
    uint32_t ex = block_exclusive_scan(s, lds, tot) + partial[blockIdx.x];
#pragma unroll
    for (int i = 0; i < SCAN_ITEMS; ++i) {
        t[scan_pad(tid * SCAN_ITEMS + i)] = ex;
        ex += v[i];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SCAN_ITEMS; ++r) {
        const uint32_t e = (uint32_t)r * SCAN_B + tid;
        if (base + e < n) out[base + e] = t[scan_pad(e)];
    }
}

// Inclusive sum over the 64 lanes (all active), by DPP row shifts and broadcasts.
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}

// One workgroup scans any n (in place allowed): 16 waves, up to 16 rows of 64
// consecutive items each per round, carry between rounds.  Used for small
// arrays, where the three-kernel scan would be launch-bound.  Latency is all it
// takes, so rows are read whole and scanned by DPP: the scans of a 16,000-point
// request take 3.6 us on average, with 16 items per thread and shuffles 6.8.
constexpr int SS_B = 1024, SS_ITEMS = 16;
__global__ void __launch_bounds__(SS_B) k_scan_single(const uint32_t *in, uint32_t *out, size_t n,
                                                      uint32_t *d_total) {
    __shared__ uint32_t lds[2][SS_B / 64];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    uint32_t carry = 0, par = 0;
    for (size_t base = 0; base < n; base += (size_t)SS_B * SS_ITEMS, par ^= 1u) {
        const uint32_t rows = (uint32_t)min((size_t)SS_ITEMS, (n - base + SS_B - 1) / SS_B);
        const size_t b0 = base + (size_t)w * 64 * rows + lane;
        uint32_t v[SS_ITEMS], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < SS_ITEMS; ++i) v[i] = i < rows && b0 + 64 * i < n ? in[b0 + 64 * i] : 0u;
#pragma unroll
        for (uint32_t i = 0; i < SS_ITEMS; ++i) {
            if (i >= rows) continue;
            const uint32_t incl = wave_incl_sum(v[i]);
            v[i] = sum + incl - v[i];
            sum += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        if (lane == 0) lds[par][w] = sum;
        __syncthreads();
        const uint32_t ws = lane < SS_B / 64 ? lds[par][lane] : 0u, wi = wave_incl_sum(ws);
        const uint32_t ex = carry + (w ? (uint32_t)__shfl((int)wi, (int)w - 1, 64) : 0u);
        carry += (uint32_t)__builtin_amdgcn_readlane((int)wi, SS_B / 64 - 1);
#pragma unroll
        for (uint32_t i = 0; i < SS_ITEMS; ++i)
            if (i < rows && b0 + 64 * i < n) out[b0 + 64 * i] = ex + v[i];
    }
    if (threadIdx.x == 0 && d_total) *d_total = carry;
}

// --------------------------------------------------------- radix sort ----
// Sort of at most NT x KPT keys in one workgroup, whole key order: stable LSD
// passes over 8-bit digits with the keys in LDS (each wave ranks its 64 x KPT
// consecutive keys as k_onesweep does).  Only bytes that vary get a pass; if those
// are many, the leading ones with some 14 bits more than n distinct keys need,
// after which runs of keys that agree in them (neighbours, a few keys each) are
// put in order by one lane; a run past kBlockRun makes all varying bytes sorted.
// Bound: LDS latency and barriers, about 4.5 us a pass with 16 waves.  Up to 1,024
// keys take 7.1 us (a bitonic network in LDS: 15), 4,096 points 22.5 us (eight
// launches of the one-sweep sort: 45).
constexpr uint32_t kBlockRun = 16;
template <int NT, int KPT>
__global__ void __launch_bounds__(NT) k_sort_block(Key *keys, uint32_t n) {
    constexpr int NW = NT / 64, N = NT * KPT;
    __shared__ Key sk[N];
    __shared__ uint32_t wcnt[NW][256];  // keys of digit d in wave w, then the waves' exclusive prefix
    __shared__ uint32_t dbase[256];
    __shared__ uint64_t s_or[NW][2];
    __shared__ uint32_t s_sum[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6, wbase = wid * 64u * KPT;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    Key k[KPT];
    const Key k0 = keys[0];
    uint64_t xh = 0, xl = 0;
#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t p = wbase + r * 64u + lane;
        k[r] = p < n ? keys[p] : Key{~0ull, ~0ull};  // the padding stays behind the keys
        if (p < n) {
            xh |= k[r].hi ^ k0.hi;
            xl |= k[r].lo ^ k0.lo;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        xh |= __shfl_xor(xh, o, 64);
        xl |= __shfl_xor(xl, o, 64);
    }
    if (lane == 0) {
        s_or[wid][0] = xh;
        s_or[wid][1] = xl;
    }
    __syncthreads();
    for (int w = 0; w < NW; ++w) {
        xh |= s_or[w][0];
        xl |= s_or[w][1];
    }
    // bytes that vary: bit p of all for byte p (8-15: hi)
    uint32_t all = 0;
    for (uint32_t p = 0; p < 8; ++p) {
        all |= ((xl >> (8 * p)) & 255u) ? 1u << p : 0u;
        all |= ((xh >> (8 * p)) & 255u) ? 256u << p : 0u;
    }
    all = (uint32_t)__builtin_amdgcn_readfirstlane((int)all);
    uint32_t top = all;
    if (__popc(all) > 6) {  // leading bytes until they hold log2(n) + 14 varying bits
        const uint32_t need = 32 - (uint32_t)__clz(n) + 14;
        uint32_t bits = 0;
        top = 0;
        for (int p = 15; p >= 0 && bits < need; --p) {
            if (!((all >> p) & 1u)) continue;
            top |= 1u << p;
            bits += (uint32_t)__popc((uint32_t)((p >= 8 ? xh >> (8 * (p - 8)) : xl >> (8 * p)) & 255u));
        }
        top = (uint32_t)__builtin_amdgcn_readfirstlane((int)top);
    }
    auto pass = [&](int bit) {
        uint32_t *wc = wcnt[wid];
        uint32_t d[KPT], pr[KPT];
        for (uint32_t i = lane; i < 256; i += 64) wc[i] = 0;
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < KPT; ++r) {
            d[r] = digit_of(k[r], bit);
            uint64_t peers = ~0ull;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t bal = __ballot((d[r] >> b) & 1u);
                peers &= ((d[r] >> b) & 1u) ? bal : ~bal;
            }
            const uint32_t rank = __popcll(peers & lt), before = wc[d[r]];
            pr[r] = before + rank;
            __builtin_amdgcn_wave_barrier();
            if (rank == 0) wc[d[r]] = before + (uint32_t)__popcll(peers);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        uint32_t cnt = 0, incl = 0;
        if (tid < 256) {
            uint32_t c[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) c[w] = wcnt[w][tid];
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                wcnt[w][tid] = cnt;
                cnt += c[w];
            }
            incl = wave_incl_sum(cnt);
            if (lane == 63) s_sum[wid] = incl;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t b = incl - cnt;
            for (uint32_t w = 0; w < wid; ++w) b += s_sum[w];
            dbase[tid] = b;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KPT; ++r) sk[dbase[d[r]] + wc[d[r]] + pr[r]] = k[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < KPT; ++r) k[r] = sk[wbase + r * 64u + lane];
    };
    if (!all) return;  // one key, or equal ones
#pragma unroll 1
    for (int p = 0; p < 16; ++p)
        if ((top >> p) & 1u) pass(8 * p);
    if (top != all) {
        uint64_t mh = 0, ml = 0;
        for (uint32_t p = 0; p < 8; ++p) {
            if ((top >> p) & 1u) ml |= 255ull << (8 * p);
            if ((top >> (p + 8)) & 1u) mh |= 255ull << (8 * p);
        }
        auto same = [&](const Key &a, const Key &b) { return !(((a.hi ^ b.hi) & mh) | ((a.lo ^ b.lo) & ml)); };
        uint32_t run[KPT];
        bool far = false;
#pragma unroll
        for (int r = 0; r < KPT; ++r) {
            const uint32_t p = wbase + r * 64u + lane;
            run[r] = 0;
            if (p >= n || (p > 0 && same(sk[p - 1], k[r]))) continue;
            uint32_t c = 1;
            while (c <= kBlockRun && p + c < n && same(sk[p + c], k[r])) ++c;
            run[r] = c;
            far = far || c > kBlockRun;
        }
        if (__syncthreads_or(far)) {
#pragma unroll 1
            for (int p = 0; p < 16; ++p)
                if ((all >> p) & 1u) pass(8 * p);
        } else {
#pragma unroll 1
            for (int r = 0; r < KPT; ++r) {
                const uint32_t p = wbase + r * 64u + lane;
                for (uint32_t a = 1; a < run[r]; ++a) {
                    const Key v = sk[p + a];
                    uint32_t b = a;
                    for (; b > 0 && key_lt(v, sk[p + b - 1]); --b) sk[p + b] = sk[p + b - 1];
                    sk[p + b] = v;
                }
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < KPT; ++r) k[r] = sk[wbase + r * 64u + lane];
        }
    }
#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t p = wbase + r * 64u + lane;
        if (p < n) keys[p] = k[r];
    }
}
// Keys that one workgroup sorts: it is as fast as the one-sweep launches at 8,192
// (38 us against 7-8 us a pass and the launches around them), and its LDS is full.
constexpr size_t kBlockSort = 8192;
void sort_block(Key *keys, size_t n, hipStream_t s) {
    if (n <= 1024) k_sort_block<256, 4><<<1, 256, 0, s>>>(keys, (uint32_t)n);
    else if (n <= 4096) k_sort_block<1024, 4><<<1, 1024, 0, s>>>(keys, (uint32_t)n);
    else k_sort_block<1024, 8><<<1, 1024, 0, s>>>(keys, (uint32_t)n);
    HIP_OK(hipGetLastError());
}

// Global histograms of the digit positions in pmask (bit p: the byte at bit
// 8p), into 16 x 256 counters.  Four keys per thread are loaded ahead.  The
// counters have one copy per XCD (workgroup b adds into copy b % 8, the XCD
// it runs on), so the flushes of the workgroups spread over 8 places.
constexpr int GH_U = 4, GH_COPIES = 8;
__global__ void __launch_bounds__(SB) k_global_hist(const Key *keys, size_t n, uint32_t *ghist, uint32_t pmask) {
    __shared__ uint32_t h[16 * 256];
    for (int i = threadIdx.x; i < 16 * 256; i += SB) h[i] = 0;
    __syncthreads();
    const size_t stride = (size_t)gridDim.x * SB * GH_U;
    const size_t nround = (n + stride - 1) / stride * stride;  // whole waves stay in the loop
    for (size_t i0 = (size_t)blockIdx.x * SB * GH_U + threadIdx.x; i0 < nround; i0 += stride) {
        Key k[GH_U];
#pragma unroll
        for (int u = 0; u < GH_U; ++u) {
            const size_t i = i0 + (size_t)u * SB;
            k[u] = i < n ? keys[i] : Key{0ull, 0ull};
        }
#pragma unroll
        for (int u = 0; u < GH_U; ++u) {
            const bool valid = i0 + (size_t)u * SB < n;
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                if (pmask & (1u << p)) wave_hist_add(&h[p * 256], (uint32_t)((k[u].lo >> (8 * p)) & 255u), valid);
                if (pmask & (1u << (p + 8)))
                    wave_hist_add(&h[(p + 8) * 256], (uint32_t)((k[u].hi >> (8 * p)) & 255u), valid);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * 256; i += SB)
        if (h[i]) atomicAdd(&ghist[(blockIdx.x % GH_COPIES) * (16 * 256) + i], h[i]);
}

// The same for the digits of a TopSort whose keys were not counted as they were written.
__global__ void __launch_bounds__(SB) k_top_hist(const Key *keys, size_t n, TopHist th) {
    __shared__ uint32_t h[kTopWords];
    for (uint32_t i = threadIdx.x; i < top_hist_words(th); i += SB) h[i] = 0;
    __syncthreads();
    const size_t stride = (size_t)gridDim.x * SB * GH_U;
    const size_t nround = (n + stride - 1) / stride * stride;  // whole waves stay in the loop
    for (size_t i0 = (size_t)blockIdx.x * SB * GH_U + threadIdx.x; i0 < nround; i0 += stride) {
        uint64_t hi[GH_U];
#pragma unroll
        for (int u = 0; u < GH_U; ++u) hi[u] = i0 + (size_t)u * SB < n ? keys[i0 + (size_t)u * SB].hi : 0ull;
#pragma unroll
        for (int u = 0; u < GH_U; ++u) top_hist_add(h, th, hi[u], i0 + (size_t)u * SB < n);
    }
    __syncthreads();
    top_hist_flush(h, th);
}

// Look-back status of one (tile, digit) of one pass: bits 0-31 the count,
// bits 32-61 the pass's epoch (its index + 1; the words are zeroed once per
// sort), bits 62-63 what the count is: the tile's own count (AGG) or the
// count of that digit in all tiles up to and including it (INCL).
constexpr uint64_t ST_AGG = 1ull << 62, ST_INCL = 2ull << 62;
constexpr uint32_t SPIN_LIMIT = 1u << 20;  // polls of one status word before giving up

__device__ __forceinline__ uint64_t status_load(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void status_store(uint64_t *p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Candidate passes of one sort and what the plan kernel derives from the
// global histograms: whether the pass's digit varies at all, which buffer
// holds its input (0 = caller's, 1 = temporary), and the exclusive global
// offset of every digit value.
struct SortPlan {
    uint32_t skip;  // a TopSort's keys agree in too many of its bits: no pass runs
    uint32_t active[16];
    uint32_t src[17];  // src[npass]: the buffer holding the sorted result
    uint32_t gofs[16 * 256];  // of digit d in pass j: gofs[j * 256 + d], with 9-bit digits gofs[j * 512 + d]
};

// One workgroup, one wave per candidate pass j (digit position
// pos[j] = (packed >> 4j) & 15, of RB bits): a digit position is skipped when one digit
// value holds all n keys; then thread 0 assigns the buffers in pass order.
//
// With fail (a TopSort) the number of passes that run keeps its parity, so that
// the last one ends in the caller's buffer: one skipped digit gets its pass if
// need be.  With may_skip, keys whose top bits do not spread them are left
// unsorted and *fail is raised at once: the caller sorts them on more bits, and
// passes over these would come on top (points in a cell of 2^-13, or half of the
// points there).  The spread is judged by the digits' collision probabilities,
// -sum log2 sum (c / n)^2 bits if they were independent, against the log2 n that
// distinct places need.  Clouds of 20,000 to 128M points: uniform 17 to 25 bits more,
// log-normal 15 to 23, 4 and 16 Gaussians of sigma 0.005 and up 10 to 20 (each with
// hardly two keys to a run); one Gaussian of sigma 0.005 1 to 8 (up to 1.4 other
// keys in a key's run), of 0.001 -6 to 2 (up to 170), clouds with half of their
// points in a cell of 2^-13 -9 to -2 (hundreds to 400,000).  Runs of some tens of
// keys are ordered faster than more passes are made: at 0.001, 8M points (-2 bits) take
// 0.79 ms in points2Octree, skipped 1.08; in a cell of 2^-6, 4M (1 bit) 0.44 and 0.63.
constexpr float kMinSpare = -3.0f;
template <int RB>
__global__ void __launch_bounds__(1024) k_sort_plan(const uint32_t *ghist, uint32_t n, uint64_t packed, int npass,
                                                    SortPlan *plan, uint32_t *fail, bool may_skip) {
    __shared__ uint32_t act[16];
    __shared__ float s_bits[16];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (w < npass) {
        const uint32_t p = (uint32_t)(packed >> (4 * w)) & 15u;
        constexpr int Q = (1 << RB) / 64;
        uint32_t c[Q], sum = 0;
        double sq = 0.0;
        bool whole = false;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            c[q] = 0;
#pragma unroll
            for (int x = 0; x < GH_COPIES; ++x) c[q] += ghist[x * (16 * 256) + (p << RB) + lane * Q + q];
            sum += c[q];
            whole = whole || c[q] == n;
            sq += (double)c[q] * (double)c[q];
        }
        for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o, 64);
        const bool trivial = __ballot(whole) != 0;
        uint32_t total;
        uint32_t ex = wave_excl_sum(sum, total);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            plan->gofs[(w << RB) + lane * Q + q] = ex;
            ex += c[q];
        }
        if (lane == 0) {
            act[w] = trivial ? 0u : 1u;
            s_bits[w] = -log2f((float)(sq / ((double)n * (double)n)));
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t src = 0, skipped = 0;
        float bits = -log2f((float)n);
        for (int j = 0; j < npass; ++j) {
            skipped += act[j] ^ 1u;
            bits += s_bits[j];
        }
        const bool none = fail && may_skip && bits < kMinSpare;
        plan->skip = none ? 1u : 0u;
        if (none) *fail = kTopSkipped;
        for (int j = 0; j < npass; ++j) {
            if (none) {
                act[j] = 0;
            } else if (fail && (skipped & 1u) && !act[j]) {
                act[j] = 1;
                skipped = 0;
            }
        }
        for (int j = 0; j < npass; ++j) {
            plan->active[j] = act[j];
            plan->src[j] = src;
            src ^= act[j];
        }
        plan->src[npass] = src;
    }
}

// One pass of the one-sweep LSD sort over the RB-bit digit at `bit`, on tiles
// of NT x SITEMS keys.  Tiles are taken in the order of a global counter, so a
// tile only ever waits for tiles that are already running.  A tile: loads its
// keys, wave w the contiguous 64 x SITEMS keys w of the tile; ranks them
// stably within the wave without workgroup barriers (per round of 64 keys: RB
// ballots give each lane its peers of equal digit, the wave's own LDS counter
// row gives the count from its earlier rounds, and the group's first lane
// advances it); turns the waves' digit counts into per-wave offsets and the
// tile's digit counts; publishes the counts (AGG); stages the keys in digit
// order in LDS; sums the counts of the tiles before it by walking back until
// a tile that already published its inclusive count (INCL); publishes its
// own inclusive count; and writes the staged keys run by run to global digit
// offset + earlier tiles' count + position in the run.  The first 2^RB
// threads own one digit each for the counters and the look-back.
template <int NT, int RB>
__global__ void __launch_bounds__(NT) k_onesweep(Key *ka, Key *kb, uint32_t n, int bit, int j, const SortPlan *plan,
                                                 uint64_t *status, uint32_t *tile_ctr, uint32_t *fault) {
    constexpr int NW = NT / 64, TILE = NT * SITEMS, DIG = 1 << RB;
    // 16-bit counters where 32-bit ones of 512 digits would not fit beside the keys
    using Count = typename std::conditional<RB == 9, uint16_t, uint32_t>::type;
    static_assert(NT >= DIG && TILE < 65536, "one thread per digit; counts of a tile in 16 bits");
    __shared__ uint32_t run_off[DIG];   // output position of staged index 0 of digit d's run, minus its start
    __shared__ uint32_t tile_off[DIG];  // start of digit d in the staged tile
    __shared__ Count wcnt[NW][DIG];  // keys of digit d in wave w; then the waves' exclusive prefix
    __shared__ uint32_t scan_tmp[NW + 1];
    __shared__ uint32_t s_tile;
    __shared__ Key sk[TILE];
    if (!plan->active[j]) return;  // the digit is the same in every key
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const bool from_b = plan->src[j] != 0;
    const Key *kin = from_b ? kb : ka;
    Key *kout = from_b ? ka : kb;
    const uint64_t epoch = (uint64_t)(j + 1) << 32;
    if (tid == 0) s_tile = atomicAdd(&tile_ctr[j], 1u);
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t base = tile * (uint32_t)TILE, wbase = base + (uint32_t)wid * (64u * SITEMS);
    Key k[SITEMS];
    uint32_t d[SITEMS], prank[SITEMS];
#pragma unroll
    for (int r = 0; r < SITEMS; ++r) {
        const uint32_t idx = wbase + (uint32_t)(r * 64 + lane);
        const bool valid = idx < n;
        k[r] = valid ? kin[idx] : Key{0ull, 0ull};
        d[r] = digit_of<RB>(k[r], bit);
    }
    // this wave's counter row: LDS operations of one wave complete in order,
    // so the row needs no barrier between its rounds
    Count *wc = wcnt[wid];
    for (int i = lane; i < DIG; i += 64) wc[i] = 0;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int r = 0; r < SITEMS; ++r) {
        const bool valid = wbase + (uint32_t)(r * 64 + lane) < n;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const uint64_t bal = __ballot((d[r] >> b) & 1u);
            peers &= ((d[r] >> b) & 1u) ? bal : ~bal;
        }
        const uint32_t rank = __popcll(peers & lt_mask);
        const uint32_t before = wc[d[r]];
        prank[r] = before + rank;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0) wc[d[r]] = (Count)(before + (uint32_t)__popcll(peers));
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // digit tid: the waves' counts become exclusive offsets, their sum the tile's count
    uint32_t cnt = 0;
    if (tid < DIG) {
        for (int w = 0; w < NW; ++w) {
            const uint32_t c = wcnt[w][tid];
            wcnt[w][tid] = (Count)cnt;
            cnt += c;
        }
    }
    uint64_t *mine = status + (size_t)tile * DIG + (tid & (DIG - 1));
    if (tid < DIG) status_store(mine, (tile == 0 ? ST_INCL : ST_AGG) | epoch | cnt);
    uint32_t total;
    const uint32_t toff = block_exclusive_scan(cnt, scan_tmp, total);
    if (tid < DIG) tile_off[tid] = toff;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SITEMS; ++r)
        if (wbase + (uint32_t)(r * 64 + lane) < n) {
            const uint32_t pos = tile_off[d[r]] + wc[d[r]] + prank[r];
            sk[pos] = k[r];
        }
    // count of digit tid in the tiles before this one
    if (tid < DIG) {
        uint32_t excl = 0;
        if (tile > 0) {
            uint32_t t = tile - 1;
            for (;;) {
                uint64_t w = status_load(status + (size_t)t * DIG + tid);
                uint32_t spins = 0;
                while ((w & ~(3ull << 62) & ~0xffffffffull) != epoch) {
                    if (++spins > SPIN_LIMIT) {
                        __hip_atomic_store(fault, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                    w = status_load(status + (size_t)t * DIG + tid);
                }
                excl += (uint32_t)w;
                if ((w & ST_INCL) || t == 0 || spins > SPIN_LIMIT) break;
                --t;
            }
            status_store(mine, ST_INCL | epoch | (excl + cnt));
        }
        run_off[tid] = plan->gofs[j * DIG + tid] + excl - toff;
    }
    __syncthreads();
    const uint32_t tn = min((uint32_t)TILE, n - base);
    for (uint32_t i = tid; i < tn; i += NT) {
        const Key key = sk[i];
        const uint32_t pos = run_off[digit_of<RB>(key, bit)] + i;
        if (pos < n) kout[pos] = key;  // always true unless a look-back wait gave up (then the fault word is set)
    }
}

// Copies the result back into the caller's buffers when the last active pass
// wrote the temporary ones.
__global__ void k_sort_finish(Key *ka, const Key *kb, size_t n, int npass, const SortPlan *plan) {
    if (!plan->src[npass]) return;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        ka[i] = kb[i];
}

// ---- keys sorted on their top bits: runs of equal top bits -----------------
// After the passes over the top bits, the keys that agree in all of them (a
// run) are put in order of the whole key, in place.  Every position keeps its
// top bits whatever the order inside its run, so run borders are found by the
// top bits alone while other workgroups reorder theirs, and only the workgroup
// that holds a run's first key touches the run.  Where all runs are pairs inside
// a wave, their first lanes order them.  Other workgroups put their keys (and, if
// their last run goes on, the kRunCap behind) into LDS, and every key of a run
// counts the keys of it that come before.  Runs past kRunCap go to a list for
// k_sort_long_runs.
// (A network in registers for runs of up to 8 inside a wave, and a wave per longer
// run, which counted from global memory, run after run, took 1.93 ms in points2Octree
// for 8M points of a Gaussian of sigma 0.001, now 0.79, and 1.08 ms for 4M in a cell
// of 2^-6, now 0.63; 0.75 ms on 128M points of 16 Gaussians, now 0.72; 53 us on 14M
// octants of 4 Gaussians, whose runs are siblings, now 66.)
constexpr uint32_t kRunCap = 256, kLongRun = 4096;

// skip: the plan's word (nullptr: none).  When set, the keys are still in `from`,
// unsorted: they are copied to k if that is another buffer, and nothing else.
__global__ void __launch_bounds__(SB) k_sort_runs(Key *k, const Key *from, size_t n, int sh, const uint32_t *skip,
                                                  uint32_t *nlong, uint32_t *list) {
    static_assert(kRunCap == SB, "one key behind the tile per thread");
    constexpr uint32_t SPAN = SB + kRunCap, NW = SB / 64;
    __shared__ Key sk[SPAN];
    __shared__ uint64_t s_head[SPAN / 64];  // bit q: key q begins a run, or lies past the end
    __shared__ uint32_t s_over;             // the last run of the tile goes on behind it
    const size_t base = (size_t)blockIdx.x * SB, j = base + threadIdx.x;
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const bool in_range = j < n;
    if (skip && *skip) {
        if (from != k && in_range) k[j] = from[j];
        return;
    }
    // one load per key; the neighbours' top bits come from the adjacent lanes,
    // and from memory at the ends of the wave
    const Key key = in_range ? k[j] : Key{0ull, 0ull};
    const uint64_t h = key.hi >> sh;
    uint64_t hp = __shfl_up(h, 1), hn = __shfl_down(h, 1);
    if (lane == 0 && j > 0 && j <= n) hp = k[j - 1].hi >> sh;
    if (lane == 63 && j + 1 < n) hn = k[j + 1].hi >> sh;
    const bool next = j + 1 < n && hn == h, prev = in_range && j > 0 && hp == h;
    const bool start = next && !prev;
    const uint64_t eq = __ballot(next), heads = __ballot(!prev);
    const bool pair = start && lane < 63 && !((eq >> (lane + 1)) & 1ull);
    if (!__syncthreads_or(start && !pair)) {
        const Key b{__shfl_down(key.hi, 1), __shfl_down(key.lo, 1)};
        if (pair && key_lt(b, key)) {
            k[j] = b;
            k[j + 1] = key;
        }
        return;
    }
    sk[threadIdx.x] = key;
    if (lane == 0) s_head[wid] = heads;
    if (threadIdx.x == SB - 1) s_over = next ? 1u : 0u;
    __syncthreads();
    const bool over = s_over;
    const size_t jo = j + SB;
    if (over) {
        const Key o = jo < n ? k[jo] : Key{~0ull, ~0ull};
        const uint64_t ho = o.hi >> sh;
        uint64_t hq = __shfl_up(ho, 1);
        if (lane == 0) hq = k[min(jo, n) - 1].hi >> sh;
        sk[SB + threadIdx.x] = o;
        const uint64_t m = __ballot(jo >= n || hq != ho);
        if (lane == 0) s_head[NW + wid] = m;
        __syncthreads();
    }
    const uint32_t span = over ? SPAN : SB;
    for (uint32_t q = threadIdx.x; q < span; q += SB) {
        if (base + q >= n) continue;
        // the run of key q: [s, e)
        uint32_t w = q >> 6;
        uint64_t m = s_head[w] & (~0ull >> (63 - lane));
        while (!m && w > 0) m = s_head[--w];
        if (!m) continue;  // begins before the tile
        const uint32_t s0 = 64 * w + 63 - (uint32_t)__clzll(m);
        if (s0 >= SB) continue;  // begins behind it
        w = q >> 6;
        m = lane == 63 ? 0ull : s_head[w] & (~0ull << (lane + 1));
        while (!m && ++w < span / 64) m = s_head[w];
        const uint32_t e0 = m ? 64 * w + (uint32_t)__ffsll((unsigned long long)m) - 1 : span, len = e0 - s0;
        if (len > kRunCap) {  // so is one that goes on at SPAN, wherever it ends
            if (q == s0) list[atomicAdd(nlong, 1u)] = (uint32_t)(base + s0);
            continue;
        }
        if (len < 2) continue;
        const Key v = sk[q];
        uint32_t r = 0;
#pragma unroll 4
        for (uint32_t t = s0; t < e0; ++t) r += (key_lt(sk[t], v) || (key_eq(sk[t], v) && t < q)) ? 1u : 0u;
        if (s0 + r != q) k[base + s0 + r] = v;
    }
}

// Runs past kRunCap, one workgroup each (bitonic in LDS).  A run past kLongRun
// is left as it is: it is listed in huge if that is given and has room
// (*fail |= kTopHuge), else *fail |= kTopLong.  So is everything when there are so
// many runs that passes over more bits cost less.
__global__ void __launch_bounds__(1024) k_sort_long_runs(Key *k, size_t n, int sh, const uint32_t *skip,
                                                         const uint32_t *nlong, const uint32_t *list, uint32_t *fail,
                                                         HugeRuns *huge) {
    __shared__ Key sk[kLongRun];
    if (skip && *skip) return;
    const uint32_t nl = *nlong;
    if (nl > 64 && nl > n / 1024) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(fail, kTopLong);
        return;
    }
    for (uint32_t b = blockIdx.x; b < nl; b += gridDim.x) {
        const size_t j0 = list[b];
        const uint64_t h0 = k[j0].hi >> sh;
        uint32_t len = 0;
        bool whole = false;
        while (len < kLongRun && !whole) {
            const size_t i = j0 + len + threadIdx.x;
            const bool in_run = i < n && (k[i].hi >> sh) == h0;
            if (in_run) sk[len + threadIdx.x] = k[i];
            // runs are contiguous: the keys of this one come first
            const uint32_t got = (uint32_t)__syncthreads_count(in_run);
            len += got;
            whole = got < 1024;
        }
        const size_t end = j0 + len;
        if (!whole && end < n && (k[end].hi >> sh) == h0) {
            if (threadIdx.x == 0) {
                size_t lo = end + 1, hi = n;  // the run's end: the keys are in order of their top bits
                while (lo < hi) {
                    const size_t mid = lo + (hi - lo) / 2;
                    if ((k[mid].hi >> sh) <= h0) lo = mid + 1;
                    else hi = mid;
                }
                const uint32_t at = huge ? atomicAdd(&huge->count, 1u) : HugeRuns::kMax;
                if (at < HugeRuns::kMax) {
                    huge->at[at] = (uint32_t)j0;
                    huge->len[at] = (uint32_t)(lo - j0);
                }
                atomicOr(fail, at < HugeRuns::kMax ? kTopHuge : kTopLong);
            }
            __syncthreads();
            continue;
        }
        uint32_t P = 1;
        while (P < len) P <<= 1;
        for (uint32_t i = len + threadIdx.x; i < P; i += 1024) sk[i] = Key{~0ull, ~0ull};
        __syncthreads();
        for (uint32_t kk = 2; kk <= P; kk <<= 1)
            for (uint32_t jj = kk >> 1; jj > 0; jj >>= 1) {
                for (uint32_t i = threadIdx.x; i < P; i += 1024) {
                    const uint32_t l = i ^ jj;
                    if (l > i) {
                        const bool up = (i & kk) == 0;
                        const Key a = sk[i], c = sk[l];
                        if (up ? key_lt(c, a) : key_lt(a, c)) {
                            sk[i] = c;
                            sk[l] = a;
                        }
                    }
                }
                __syncthreads();
            }
        for (uint32_t i = threadIdx.x; i < len; i += 1024) k[j0 + i] = sk[i];
        __syncthreads();
    }
}

}  // namespace

void scan_exclusive_u32_async(const uint32_t *in, uint32_t *out, size_t n, uint32_t *d_total, hipStream_t s) {
    if (n == 0) {
        if (d_total) HIP_OK(hipMemsetAsync(d_total, 0, sizeof(uint32_t), s));
        return;
    }
    if (n <= (size_t)SS_B * SS_ITEMS) {  // one round of the single-workgroup scan
        k_scan_single<<<1, SS_B, 0, s>>>(in, out, n, d_total);
        HIP_OK(hipGetLastError());
        return;
    }
    size_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    DevBuf<uint32_t> partial(nb, s);
    k_scan_reduce<<<(unsigned)nb, SCAN_B, 0, s>>>(in, n, partial.p);
    k_scan_partials<<<1, 1024, 0, s>>>(partial.p, nb, d_total);
    k_scan_down<<<(unsigned)nb, SCAN_B, 0, s>>>(in, out, n, partial.p);
    HIP_OK(hipGetLastError());
}

uint64_t scan_exclusive_u32(const uint32_t *in, uint32_t *out, size_t n, hipStream_t s) {
    DevBuf<uint32_t> tot(1, s);
    scan_exclusive_u32_async(in, out, n, tot.p, s);
    uint32_t h = 0;
    dgx_read_back(&h, tot.p, sizeof(uint32_t), s);
    return h;
}

namespace {
void run_passes(Key *keys, size_t n, const std::vector<int> &passes, hipStream_t s);

// Pinned host word that the sort kernels set when a look-back wait exceeds its
// bound (it never should: every wait is for a tile that is already running).
uint32_t *g_fault = nullptr;
std::once_flag g_fault_once;
uint32_t *fault_word() {
    std::call_once(g_fault_once, [] {
        void *p = nullptr;
        HIP_OK(hipHostMalloc(&p, 64, hipHostMallocMapped));
        std::memset(p, 0, 64);
        g_fault = (uint32_t *)p;
    });
    return g_fault;
}
}  // namespace

uint32_t *dgx_fault_word() { return fault_word(); }

void sort_fault_check() {
    if (g_fault && __atomic_exchange_n(g_fault, 0u, __ATOMIC_ACQ_REL)) {
        dgx_set_error("a look-back wait (radix sort or single-pass scan) exceeded its bound; that result is invalid");
        throw DgxError();
    }
}

static void check_sort_size(size_t n) {
    if (n > 0xffffffffull - 1024 * SITEMS) {  // 32-bit indices, up to the largest tile past the end
        dgx_set_error("radix_sort_keys: %zu keys exceed the 32-bit index range", n);
        throw DgxError();
    }
}

void radix_sort_keys(Key *keys, size_t n, hipStream_t s, int begin_bit, int end_bit) {
    if (n < 2) return;
    check_sort_size(n);
    if (n <= kBlockSort) {
        sort_block(keys, n, s);
        return;
    }
    std::vector<int> passes;
    for (int p = 0; p < 16; ++p)
        if (!(8 * p + 8 <= begin_bit || 8 * p >= end_bit)) passes.push_back(8 * p);
    run_passes(keys, n, passes, s);
}


namespace {

// Workspace of one sort of rb-bit digits, zeroed by one fill: GH_COPIES x 16 x 256 global
// counters, 16 tile counters, the look-back status words and `extra` words for
// the caller; then the plan.
struct PassSpace {
    int np, nt, rb;
    size_t n, ntiles;
    DevBuf<uint8_t> ws;
    uint32_t *ghist, *ctr, *extra;
    SortPlan *plan;
    uint64_t *status;
    uint32_t pmask = 0;
    uint64_t packed = 0;
    PassSpace(size_t n_, const std::vector<int> &passes, int rb_, size_t nextra, hipStream_t s)
        : np((int)passes.size()), nt(sort_threads(n_, rb_)), rb(rb_), n(n_) {
        ntiles = (n + (size_t)nt * kSortItems - 1) / ((size_t)nt * kSortItems);
        const size_t off_status = (GH_COPIES * 16 * 256 * 4 + 16 * 4 + nextra * 4 + 255) / 256 * 256;
        const size_t off_plan = off_status + (ntiles << rb) * sizeof(uint64_t);
        ws.alloc(off_plan + sizeof(SortPlan), s);
        ghist = (uint32_t *)ws.p;
        ctr = ghist + GH_COPIES * 16 * 256;
        extra = ctr + 16;
        status = (uint64_t *)(ws.p + off_status);
        plan = (SortPlan *)(ws.p + off_plan);
        HIP_OK(hipMemsetAsync(ws.p, 0, off_plan, s));
        for (int j = 0; j < np; ++j) {
            const int slot = rb == 8 ? passes[j] / 8 : j;  // of the counters
            pmask |= 1u << slot;
            packed |= (uint64_t)slot << (4 * j);
        }
    }
};
// The passes over keys kp (temporary kt), counted in w.ghist.  fail, may_skip: as in k_sort_plan.
void launch_passes(PassSpace &w, Key *kp, Key *kt, const std::vector<int> &passes, hipStream_t s,
                   uint32_t *fail = nullptr, bool may_skip = false) {
    const size_t n = w.n;
    const int np = w.np, nt = w.nt;
    SortPlan *plan = w.plan;
    uint64_t *status = w.status;
    uint32_t *ctr = w.ctr;
    if (w.rb == 9) k_sort_plan<9><<<1, 1024, 0, s>>>(w.ghist, (uint32_t)n, w.packed, np, plan, fail, may_skip);
    else k_sort_plan<8><<<1, 1024, 0, s>>>(w.ghist, (uint32_t)n, w.packed, np, plan, fail, may_skip);
    HIP_OK(hipGetLastError());
    uint32_t *fault = fault_word();
    const unsigned grid = (unsigned)w.ntiles;
    for (int j = 0; j < np; ++j) {
        if (w.rb == 9)
            k_onesweep<1024, 9><<<grid, 1024, 0, s>>>(kp, kt, (uint32_t)n, passes[j], j, plan, status, ctr, fault);
        else if (nt == 1024)
            k_onesweep<1024, 8><<<grid, 1024, 0, s>>>(kp, kt, (uint32_t)n, passes[j], j, plan, status, ctr, fault);
        else if (nt == 512)
            k_onesweep<512, 8><<<grid, 512, 0, s>>>(kp, kt, (uint32_t)n, passes[j], j, plan, status, ctr, fault);
        else
            k_onesweep<256, 8><<<grid, 256, 0, s>>>(kp, kt, (uint32_t)n, passes[j], j, plan, status, ctr, fault);
        HIP_OK(hipGetLastError());
    }
}
void launch_hist(PassSpace &w, const Key *keys, hipStream_t s) {
    const unsigned gb = (unsigned)std::min<size_t>(grid_for(w.n, SB * GH_U), 1024);
    k_global_hist<<<gb, SB, 0, s>>>(keys, w.n, w.ghist, w.pmask);
    HIP_OK(hipGetLastError());
}
void run_passes(Key *keys, size_t n, const std::vector<int> &passes, hipStream_t s) {
    if (passes.empty()) return;
    PassSpace w(n, passes, 8, 0, s);
    launch_hist(w, keys, s);
    DevBuf<Key> ktmp(n, s);
    launch_passes(w, keys, ktmp.p, passes, s);
    k_sort_finish<<<(unsigned)std::min<size_t>(grid_for(n, 256), 512), 256, 0, s>>>(keys, ktmp.p, n, w.np, w.plan);
    HIP_OK(hipGetLastError());
}

}  // namespace

namespace {
// Runs of keys that agree above bit 64 + sh put in order.  nlong: a zeroed word.
void order_runs(Key *keys, const Key *from, size_t n, int sh, const uint32_t *skip, uint32_t *nlong, uint32_t *list,
                uint32_t *fail, HugeRuns *huge, hipStream_t s) {
    k_sort_runs<<<grid_for(n, SB), SB, 0, s>>>(keys, from, n, sh, skip, nlong, list);
    const unsigned g = (unsigned)std::min<size_t>(512, std::max<size_t>(64, n >> 14));
    k_sort_long_runs<<<g, 1024, 0, s>>>(keys, n, sh, skip, nlong, list, fail, huge);
    HIP_OK(hipGetLastError());
}
}  // namespace

struct TopSort::Impl {
    size_t n;
    hipStream_t s;
    std::vector<int> passes;
    std::unique_ptr<PassSpace> w;
    DevBuf<Key> tmp;
    DevBuf<uint32_t> list;
};

TopSort::TopSort(Key *keys, size_t n, hipStream_t s) : p_(new Impl()), keys_(keys) {
    check_sort_size(n);
    p_->n = n;
    p_->s = s;
    if (n <= kBlockSort) return;
    uint32_t lg = 0;
    while (lg < 32 && (size_t(1) << lg) < n) ++lg;
    // 18 bits (6 levels) more than n distinct keys need: clouds a few thousand
    // times denser than their mean still leave few runs of equal top bits
    const int np = std::min(8, std::max(4, (int)(lg + 18 + 7) / 8));
    // More than 2^22 keys and up to 2^27 take five digits of 9 bits instead of six of
    // 8 (a key's top bit is 0 and left out).  A pass is bound by its 32 bytes a key:
    // 504 us at 64M keys with 8 bits, 561 with 9, whose runs are shorter; with the
    // counting and balancing, 16 Gaussians of 64M points take 6.51 ms instead of
    // 6.83, 16M points 1.81 instead of 1.89.
    const int np9 = (int)(lg + 18 + 8) / 9;
    if (lg >= 20 && np9 < np && np9 <= 5) {
        for (int j = 0; j < np9; ++j) p_->passes.push_back(127 - 9 * np9 + 9 * j);
        p_->w.reset(new PassSpace(n, p_->passes, 9, 1, s));
    } else {
        for (int j = 0; j < np; ++j) p_->passes.push_back(128 - 8 * np + 8 * j);
        p_->w.reset(new PassSpace(n, p_->passes, 8, 1, s));
    }
    p_->tmp.alloc(n, s);
    p_->list.alloc(n / kRunCap + 1, s);
}
TopSort::~TopSort() {}
int TopSort::top_shift() const { return p_->w ? p_->passes[0] - 64 : 0; }
// An odd number of passes ends in the other buffer, so it starts there.
Key *TopSort::input() const { return p_->w && (p_->w->np & 1) ? p_->tmp.p : keys_; }
TopHist TopSort::hist() const {
    if (!p_->w) return TopHist{nullptr, 0, 0, 0};
    const PassSpace &w = *p_->w;
    return TopHist{w.ghist + (w.rb == 8 ? (p_->passes[0] / 8) * 256 : 0), (uint32_t)w.np,
                   (uint32_t)(p_->passes[0] - 64), (uint32_t)w.rb};
}
void TopSort::sort(bool counted, uint32_t *fail, HugeRuns *huge, bool may_skip) {
    if (p_->n < 2) return;
    if (!p_->w) {
        sort_block(keys_, p_->n, p_->s);
        return;
    }
    PassSpace &w = *p_->w;
    Key *a = input(), *b = a == keys_ ? p_->tmp.p : keys_;
    if (!counted)
        k_top_hist<<<(unsigned)std::min<size_t>(grid_for(p_->n, SB * GH_U), 1024), SB, 0, p_->s>>>(a, p_->n, hist());
    launch_passes(w, a, b, p_->passes, p_->s, fail, may_skip);
    order_runs(keys_, a, p_->n, top_shift(), &w.plan->skip, w.extra, p_->list.p, fail, huge, p_->s);
}

void sort_keys_again(Key *keys, size_t n, hipStream_t s, int begin_bit, uint32_t why, const HugeRuns *huge,
                     int top_shift, uint32_t *fail) {
    if (n < 2) return;
    if (why == kTopHuge && huge) {
        HugeRuns h;
        dgx_read_back(&h, huge, sizeof h, s);
        // some 60 us each, against ten passes over all keys
        if (h.count <= std::min<size_t>(HugeRuns::kMax, std::max<size_t>(4, n >> 19))) {
            for (uint32_t r = 0; r < h.count; ++r)
                radix_sort_keys(keys + h.at[r], h.len[r], s, begin_bit, 64 + top_shift);
            return;
        }
    }
    if (n > kBlockSort && why != kTopAgain) {
        DevBuf<uint32_t> w(2 + n / kRunCap + 1, s);  // long runs, fail, list
        HIP_OK(hipMemsetAsync(w.p, 0, 8, s));
        radix_sort_keys(keys, n, s, 64, 128);
        order_runs(keys, keys, n, 0, nullptr, w.p, w.p + 2, fail ? fail : w.p + 1, nullptr, s);
        if (fail) return;
        uint32_t left = 0;
        dgx_read_back(&left, w.p + 1, 4, s);
        if (!left) return;
    }
    radix_sort_keys(keys, n, s, begin_bit, 128);
}
