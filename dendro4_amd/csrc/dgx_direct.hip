// dgx_direct.hip -- sparse FP64 direct solver of the coarsest multigrid level
// (nested dissection + multifrontal Gauss-Jordan sweeps), see dgx_direct.h.
//
// Reference counterpart: the coarse-grid PCLU of the DAMG V-cycle
// (bin/optionsFBM:57, src/omg/blockDiag.cpp:780-1047 and 1172-1308), a sparse
// LU of the coarsest level's matrix through PETSc.
#include "dgx_direct.h"
#include <cstdio>
#include <string>
#include <chrono>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <functional>
#include <iterator>
#include <limits>
#include <numeric>
#include <thread>

#include "../../include/dendro_mi355x.h"

// ------------------------------------------------------------ host plan ----
namespace {

// Runs body(lo, hi, t) over [0, n) in up to 8 contiguous ranges on host
// threads; each range writes only its own outputs, so the result does not
// depend on the split.
template <typename F>
void parallel_ranges(size_t n, size_t grain, F body) {
    const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
    const unsigned t = (unsigned)std::min<size_t>(std::min(8u, hw), std::max<size_t>(1, n / grain));
    if (t <= 1) {
        body(size_t(0), n, 0u);
        return;
    }
    std::vector<std::thread> th;
    for (unsigned k = 1; k < t; ++k) th.emplace_back(body, n * k / t, n * (k + 1) / t, k);
    body(size_t(0), n / t, 0u);
    for (auto &x : th) x.join();
}

// Geometric nested dissection of the interior-node graph.  A part is split by
// a plane c_a = t: L = nodes with c_a < t, the separator S = nodes with
// c_a >= t that have a neighbour in L, R = the rest; no edge joins L and R.
// Candidate planes lie on the grid lines of the largest power-of-two spacing
// that cuts the part's extent into at least kBins pieces, so they follow the
// octree's own cell faces.  The plane minimises |S| / min(|L|, |R|) over the
// three axes with both sides holding at least 15% of the part, so cuts go
// through coarse regions of an adaptive mesh where they are cheap.  The counts
// come from histograms: #L(t) = #{c < t}, #S(t) = #{m < t} - #{c < t} where m is
// the smallest coordinate over a node and its neighbours in the part.
struct Dissection {
    static constexpr uint32_t kBins = 256;
    // parts at least this large split their two halves over two host threads (a
    // thread costs some 30 us; 6,159 nodes take 0.60 ms, 0.96 on one thread),
    // down to kParDepth levels of the tree (at most 2^kParDepth threads)
    static constexpr size_t kParMin = 1500;
    static constexpr int kParDepth = 3;
    uint32_t ni = 0, leaf = 128;
    const std::vector<uint32_t> &roff, &rcol;  // interior graph (diagonal included)
    const std::vector<uint32_t> &xyz;          // 3 per interior node
    // stamp[v] = id of the part v was last placed in; parts split concurrently
    // are disjoint, and a neighbour in another part never carries this part's
    // id, so relaxed accesses suffice
    std::vector<std::atomic<uint32_t>> stamp;
    // smallest coordinates over a node and its neighbours in its part, kept from
    // part to part: a split changes them only for nodes next to the separator
    // (computing them for every node of every part was most of the dissection:
    // 1.32 ms for 6,159 nodes, 0.96 now)
    std::vector<uint32_t> low;
    std::atomic<uint32_t> next_id{0};

    // A subtree: its fronts in creation order (children before parents), each
    // front's nodes and children (indices into this list), and its roots.
    struct Forest {
        std::vector<std::vector<uint32_t>> S, kids;
        std::vector<uint32_t> roots;
    };

    Dissection(const std::vector<uint32_t> &ro, const std::vector<uint32_t> &rc, const std::vector<uint32_t> &c,
               uint32_t n_int, uint32_t lf)
        : ni(n_int), leaf(lf), roff(ro), rcol(rc), xyz(c), stamp(n_int), low(3 * (size_t)n_int) {
        for (auto &a : stamp) a.store(0, std::memory_order_relaxed);
    }

    static Forest single(std::vector<uint32_t> &&P) {
        Forest f;
        f.S.push_back(std::move(P));
        f.kids.emplace_back();
        f.roots.push_back(0);
        return f;
    }

    // low of v, whose part is cur
    void low3(uint32_t v, uint32_t cur) {
        uint32_t *m = &low[3 * (size_t)v];
        m[0] = xyz[3 * (size_t)v];
        m[1] = xyz[3 * (size_t)v + 1];
        m[2] = xyz[3 * (size_t)v + 2];
        for (uint32_t k = roff[v]; k < roff[v + 1]; ++k) {
            const uint32_t w = rcol[k];
            if (stamp[w].load(std::memory_order_relaxed) != cur) continue;
            const uint32_t *c = &xyz[3 * (size_t)w];
            m[0] = std::min(m[0], c[0]);
            m[1] = std::min(m[1], c[1]);
            m[2] = std::min(m[2], c[2]);
        }
    }

    Forest run_all() {
        std::vector<uint32_t> all(ni);
        std::iota(all.begin(), all.end(), 0u);
        return run(all, all, 0);
    }

    // The part P, of which `changed` are the nodes whose low is out of date.
    Forest run(std::vector<uint32_t> P, const std::vector<uint32_t> &changed, int depth) {
        const size_t np = P.size();
        if (np == 0) return {};
        if (np <= leaf) return single(std::move(P));
        const uint32_t cur = next_id.fetch_add(1, std::memory_order_relaxed) + 1;
        for (uint32_t v : P) stamp[v].store(cur, std::memory_order_relaxed);
        for (uint32_t v : changed) low3(v, cur);
        uint32_t bmin[3] = {~0u, ~0u, ~0u}, bmax[3] = {0, 0, 0};
        for (size_t i = 0; i < np; ++i) {
            for (int a = 0; a < 3; ++a) {
                const uint32_t c = xyz[3 * (size_t)P[i] + a];
                bmin[a] = std::min(bmin[a], c);
                bmax[a] = std::max(bmax[a], c);
            }
        }
        int best_a = -1;
        uint32_t best_t = 0;
        double best_cost = std::numeric_limits<double>::infinity();
        const size_t lo = std::max<size_t>(1, (size_t)(0.15 * (double)np));
        uint32_t hc[kBins + 1], hm[kBins + 1];
        for (int a = 0; a < 3; ++a) {
            if (bmax[a] == bmin[a]) continue;
            int sh = 0;  // grid spacing 2^sh: the extent spans at most kBins cells
            while (((bmax[a] >> sh) - (bmin[a] >> sh)) >= kBins) ++sh;
            const uint32_t base = bmin[a] >> sh;
            std::fill(hc, hc + kBins + 1, 0u);
            std::fill(hm, hm + kBins + 1, 0u);
            for (size_t i = 0; i < np; ++i) {
                ++hc[(xyz[3 * (size_t)P[i] + a] >> sh) - base];
                ++hm[(low[3 * (size_t)P[i] + a] >> sh) - base];
            }
            // plane t_b = (base + b) << sh: #{c < t_b} = sum of hc below b
            size_t nL = 0, nM = 0;
            for (uint32_t b = 1; b <= kBins; ++b) {
                nL += hc[b - 1];
                nM += hm[b - 1];
                if (nL < lo) continue;
                if (np - nL < lo) break;
                const size_t nS = nM - nL, nR = np - nM;
                if (nR < lo) continue;
                const double cost = (double)nS / (double)std::min(nL, nR);
                if (cost < best_cost) {
                    best_cost = cost;
                    best_a = a;
                    best_t = (base + b) << sh;
                }
            }
        }
        if (best_a < 0) return single(std::move(P));  // no admissible plane: one dense front
        std::vector<uint32_t> L, R, Sv;
        for (size_t i = 0; i < np; ++i) {
            const uint32_t v = P[i];
            if (xyz[3 * (size_t)v + best_a] < best_t) L.push_back(v);
            else if (low[3 * (size_t)v + best_a] < best_t) Sv.push_back(v);
            else R.push_back(v);
        }
        std::vector<uint32_t>().swap(P);
        // the nodes of L and R next to S, each once (0 is no part's id)
        std::vector<uint32_t> nextL, nextR;
        for (uint32_t v : Sv) stamp[v].store(0, std::memory_order_relaxed);
        for (uint32_t v : Sv)
            for (uint32_t k = roff[v]; k < roff[v + 1]; ++k) {
                const uint32_t w = rcol[k];
                if (stamp[w].load(std::memory_order_relaxed) != cur) continue;
                stamp[w].store(0, std::memory_order_relaxed);
                (xyz[3 * (size_t)w + best_a] < best_t ? nextL : nextR).push_back(w);
            }
        Forest fl, fr;
        if (depth < kParDepth && L.size() >= kParMin && R.size() >= kParMin) {
            std::thread th([&] { fl = run(std::move(L), nextL, depth + 1); });
            fr = run(std::move(R), nextR, depth + 1);
            th.join();
        } else {
            fl = run(std::move(L), nextL, depth + 1);
            fr = run(std::move(R), nextR, depth + 1);
        }
        // the fronts of L, then those of R (renumbered), then the separator
        Forest out;
        const uint32_t shift = (uint32_t)fl.S.size();
        out.S = std::move(fl.S);
        out.kids = std::move(fl.kids);
        out.roots = std::move(fl.roots);
        for (size_t f = 0; f < fr.S.size(); ++f) {
            for (uint32_t &c : fr.kids[f]) c += shift;
            out.S.push_back(std::move(fr.S[f]));
            out.kids.push_back(std::move(fr.kids[f]));
        }
        for (uint32_t r : fr.roots) out.roots.push_back(r + shift);
        if (Sv.empty()) return out;  // the part was disconnected along the plane
        out.S.push_back(std::move(Sv));
        out.kids.push_back(std::move(out.roots));
        out.roots.assign(1, (uint32_t)(out.S.size() - 1));
        return out;
    }
};

}  // namespace

namespace {

// Place of elimination position p in front F (F.m: not in it); upos holds the
// fronts' positions, ascending behind the s of the separator.
__host__ __device__ inline uint32_t front_place(const MfFront &F, const uint32_t *upos, uint32_t p) {
    if (p - F.ws < F.s) return p - F.ws;
    const uint32_t *u = upos + F.idx;
    uint32_t lo = F.s, hi = F.m;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (u[mid] < p) lo = mid + 1;
        else hi = mid;
    }
    return lo < F.m && u[lo] == p ? lo : F.m;
}

// DGX_SETUP_TIMING=1: the phases of an analysis, one line on stderr.
struct PhaseLog {
    bool on;
    std::chrono::steady_clock::time_point t = std::chrono::steady_clock::now();
    std::string log;
    PhaseLog() {
        static const bool timing = [] {
            const char *e = getenv("DGX_SETUP_TIMING");
            return e && e[0] == '1';
        }();
        on = timing;
    }
    void lap(const char *what) {
        if (!on) return;
        const auto now = std::chrono::steady_clock::now();
        char b[64];
        snprintf(b, sizeof b, " %s %.2f", what, std::chrono::duration<double, std::milli>(now - t).count());
        log += b;
        t = now;
    }
};

}  // namespace

// The plan's fronts, maps and work items from the interior graph (P.n, P.ni and
// P.inode are set).
static void mf_symbolic(MfPlan &P, const std::vector<uint32_t> &roff, const std::vector<uint32_t> &rcol,
                        const std::vector<uint32_t> &cxyz, uint64_t max_entries, uint32_t leaf, uint32_t dense) {
    PhaseLog pl;
    auto lap = [&](const char *what) { pl.lap(what); };
    const uint32_t ni = P.ni;
    // nested dissection; positions in front order (postorder), nodes in list order
    struct {
        std::vector<std::vector<uint32_t>> S, kids;
    } D;
    std::vector<uint32_t> &pos = P.pos, &front_of = P.front_of;
    {
        Dissection nd(roff, rcol, cxyz, ni, ni <= dense ? std::max(ni, 1u) : leaf);
        Dissection::Forest fo = nd.run_all();
        D.S = std::move(fo.S);
        D.kids = std::move(fo.kids);
        pos.assign(ni, 0);
        uint32_t next_pos = 0;
        for (const auto &sep : D.S)
            for (uint32_t v : sep) pos[v] = next_pos++;
    }
    const uint32_t nf = (uint32_t)D.S.size();
    lap("dissection");
    std::vector<uint32_t> sstart(nf), send(nf), at_pos(ni);
    front_of.resize(ni);
    for (uint32_t f = 0; f < nf; ++f) {
        sstart[f] = pos[D.S[f][0]];
        send[f] = sstart[f] + (uint32_t)D.S[f].size();
        for (uint32_t v : D.S[f]) {
            front_of[v] = f;
            at_pos[pos[v]] = v;
        }
    }
    // update sets, as elimination positions (ascending)
    std::vector<std::vector<uint32_t>> U(nf);
    P.height.assign(nf, 0);
    {
        // sorted lists: the union of the children's sets behind S, then what the
        // nodes of S add to it
        std::vector<uint32_t> mark(ni, 0xffffffffu), both, add, tmp;
        for (uint32_t f = 0; f < nf; ++f) {
            both.clear();
            uint32_t h = 0;
            for (uint32_t c : D.kids[f]) {
                const auto from = std::lower_bound(U[c].begin(), U[c].end(), send[f]);
                tmp.clear();
                std::set_union(both.begin(), both.end(), from, U[c].end(), std::back_inserter(tmp));
                both.swap(tmp);
                h = std::max(h, P.height[c] + 1);
            }
            P.height[f] = h;
            for (uint32_t p : both) mark[p] = f;
            add.clear();
            for (uint32_t v : D.S[f])
                for (uint32_t k = roff[v]; k < roff[v + 1]; ++k) {
                    const uint32_t p = pos[rcol[k]];
                    if (p < send[f] || mark[p] == f) continue;
                    mark[p] = f;
                    add.push_back(p);
                }
            std::sort(add.begin(), add.end());
            U[f].resize(both.size() + add.size());
            std::merge(both.begin(), both.end(), add.begin(), add.end(), U[f].begin());
        }
    }
    lap("update-sets");
    // fronts
    P.fronts.resize(nf);
    uint64_t off = 0, upd = 0;
    uint32_t idxo = 0, nl = 0, invo = 0, fmo = 0;
    for (uint32_t f = 0; f < nf; ++f) {
        MfFront &F = P.fronts[f];
        F.s = (uint32_t)D.S[f].size();
        F.m = F.s + (uint32_t)U[f].size();
        if (F.m > kMfMaxFront) {
            dgx_set_error("coarse solver: a front of %u nodes exceeds %u (coarsest level too large)", F.m,
                          kMfMaxFront);
            throw DgxError();
        }
        F.off = off;
        off += (uint64_t)F.m * F.m;
        F.idx = idxo;
        idxo += F.m;
        F.upd = (uint32_t)upd;
        upd += F.m - F.s;
        F.ws = sstart[f];
        F.ch0 = nl;
        F.nch = (uint32_t)D.kids[f].size();
        nl += F.nch;
        for (uint32_t c : D.kids[f]) {
            invo += F.m;
            fmo += P.fronts[c].m - P.fronts[c].s;
        }
        P.max_m = std::max(P.max_m, F.m);
        P.max_s = std::max(P.max_s, F.s);
    }
    if (off > max_entries) {
        dgx_set_error("coarse solver: the frontal matrices need %llu doubles (limit %llu)", (unsigned long long)off,
                      (unsigned long long)max_entries);
        throw DgxError();
    }
    P.front_entries = off;
    P.upd_len = upd;
    P.idx.resize(idxo);
    P.links.resize(nl);
    P.inv.assign(invo, -1);
    P.fmap.resize(fmo);
    // local positions: pm[elimination position] = place in the current front
    std::vector<uint32_t> pm(ni, 0xffffffffu);
    P.upos.resize(idxo);
    invo = 0;
    fmo = 0;
    for (uint32_t f = 0; f < nf; ++f) {
        const MfFront &F = P.fronts[f];
        uint32_t *ix = P.idx.data() + F.idx;
        for (uint32_t p = 0; p < F.s; ++p) {
            ix[p] = P.inode[D.S[f][p]];
            P.upos[F.idx + p] = sstart[f] + p;
            pm[sstart[f] + p] = p;
        }
        for (uint32_t p = 0; p < (uint32_t)U[f].size(); ++p) {
            ix[F.s + p] = P.inode[at_pos[U[f][p]]];
            P.upos[F.idx + F.s + p] = U[f][p];
            pm[U[f][p]] = F.s + p;
        }
        for (uint32_t l = 0; l < F.nch; ++l) {
            const uint32_t c = D.kids[f][l];
            MfLink &L = P.links[F.ch0 + l];
            L.child = c;
            L.inv = invo;
            L.fmap = fmo;
            const std::vector<uint32_t> &uc = U[c];
            for (uint32_t i = 0; i < (uint32_t)uc.size(); ++i) {
                const uint32_t p = pm[uc[i]];
                if (p >= F.m || (p < F.s ? sstart[f] + p : U[f][p - F.s]) != uc[i]) {
                    dgx_set_error("coarse solver: a child update index is missing from its parent front");
                    throw DgxError();
                }
                P.inv[invo + p] = (int32_t)i;
                P.fmap[fmo + i] = p;
            }
            invo += F.m;
            fmo += (uint32_t)uc.size();
        }
    }
    lap("fronts+maps");
    // levels by height, with their work items and scratch
    uint32_t H = 0;
    for (uint32_t f = 0; f < nf; ++f) H = std::max(H, P.height[f] + 1);
    P.lvl_fronts.assign(H, {});
    P.lvl_fwd.assign(H, {});
    P.lvl_bwd.assign(H, {});
    P.lvl_gather.assign(H, {});
    P.lvl_max_m.assign(H, 0);
    P.lvl_max_s.assign(H, 0);
    P.lvl_tc.assign(H, 0);
    for (uint32_t f = 0; f < nf; ++f) {
        const uint32_t h = P.height[f];
        MfFront &F = P.fronts[f];
        F.dinv = (uint32_t)P.lvl_fronts[h].size();
        F.tc = P.lvl_tc[h];
        P.lvl_tc[h] += 4ull * kGJ * F.m;
        P.lvl_fronts[h].push_back(f);
        P.lvl_max_m[h] = std::max(P.lvl_max_m[h], F.m);
        P.lvl_max_s[h] = std::max(P.lvl_max_s[h], F.s);
        const uint32_t u = F.m - F.s;
        for (uint32_t r = 0; u == 0 && r < F.s; r += kGather) P.lvl_fwd[h].push_back({f, r});
        for (uint32_t r = 0; r < u; r += 16) P.lvl_fwd[h].push_back({f, r});
        for (uint32_t r = 0; r < F.s; r += 16) P.lvl_bwd[h].push_back({f, r});
        if (F.nch)
            for (uint32_t r = 0; r < F.m; r += 4) P.lvl_gather[h].push_back({f, r});
    }
    for (uint32_t h = 0; h < H; ++h) {
        P.tc_max = std::max(P.tc_max, P.lvl_tc[h]);
        P.dinv_max = std::max(P.dinv_max, (uint32_t)P.lvl_fronts[h].size());
    }
    if (P.dinv_max > 65535) {  // fronts of a level index grid dimension y of the factorisation
        dgx_set_error("coarse solver: %u fronts in one tree level (limit 65535)", P.dinv_max);
        throw DgxError();
    }
    lap("levels");
    if (pl.on) fprintf(stderr, "coarse analysis: %u interior nodes, %u fronts, ms:%s\n", ni, nf, pl.log.c_str());
}

MfPlan mf_plan(uint32_t n, size_t E, const uint32_t *conn, const uint16_t *meta, const uint8_t *bdy,
               const uint32_t *xyz, uint64_t max_entries, uint32_t leaf, uint32_t dense) {
    MfPlan P;
    P.n = n;
    if (E * 64 > 0xffffffffull) {
        dgx_set_error("coarse solver: %zu elements exceed the 32-bit contribution index", E);
        throw DgxError();
    }
    // interior numbering
    std::vector<int32_t> iid(n, -1);
    for (uint32_t i = 0; i < n; ++i)
        if (!bdy[i]) {
            iid[i] = (int32_t)P.inode.size();
            P.inode.push_back(i);
        }
    const uint32_t ni = (uint32_t)P.inode.size();
    P.ni = ni;
    // interior ids of each element's vertices (original vertex order), and the
    // incidences (interior node, element, vertex) in element order
    std::vector<int32_t> eid(8 * E);
    std::vector<uint32_t> ioff(ni + 1, 0);
    for (size_t e = 0; e < E; ++e)
        for (int j = 0; j < 8; ++j) {
            const int32_t v = iid[conn[(size_t)j * E + e]];
            eid[8 * e + j] = v;
            if (v >= 0) ++ioff[v + 1];
        }
    for (uint32_t i = 0; i < ni; ++i) ioff[i + 1] += ioff[i];
    std::vector<uint32_t> inc(ioff[ni]);  // e * 8 + vertex
    {
        std::vector<uint32_t> fill(ioff.begin(), ioff.end() - 1);
        for (size_t e = 0; e < E; ++e)
            for (uint32_t j = 0; j < 8; ++j) {
                const int32_t v = eid[8 * e + j];
                if (v >= 0) inc[fill[v]++] = (uint32_t)(e * 8 + j);
            }
    }
    // matrix pattern over the interior rows (diagonal included), columns in
    // the order the incident elements first reach them
    std::vector<uint32_t> roff(ni + 1, 0), rcol;
    {
        std::vector<std::vector<uint32_t>> part(8);
        parallel_ranges(ni, 4096, [&](size_t lo, size_t hi, unsigned t) {
            std::vector<uint32_t> mark(ni, 0xffffffffu), &out = part[t];
            out.reserve((hi - lo) * 27);
            for (uint32_t i = (uint32_t)lo; i < hi; ++i) {
                const size_t before = out.size();
                for (uint32_t q = ioff[i]; q < ioff[i + 1]; ++q) {
                    const int32_t *ids = &eid[(inc[q] >> 3) * 8];
                    for (int j = 0; j < 8; ++j) {
                        const int32_t w = ids[j];
                        if (w >= 0 && mark[w] != i) {
                            mark[w] = i;
                            out.push_back((uint32_t)w);
                        }
                    }
                }
                if (out.size() == before) out.push_back(i);  // an interior node of no element keeps its diagonal
                roff[i + 1] = (uint32_t)(out.size() - before);
            }
        });
        for (uint32_t i = 0; i < ni; ++i) roff[i + 1] += roff[i];
        rcol.reserve(roff[ni]);
        for (auto &pv : part) rcol.insert(rcol.end(), pv.begin(), pv.end());
    }
    const uint32_t nnz = roff[ni];
    std::vector<uint32_t> cxyz(3 * (size_t)ni);
    for (uint32_t i = 0; i < ni; ++i)
        for (int a = 0; a < 3; ++a) cxyz[3 * (size_t)i + a] = xyz[3 * (size_t)P.inode[i] + a];
    mf_symbolic(P, roff, rcol, cxyz, max_entries, leaf, dense);
    // places of the matrix entries: the device computes them as it assembles
    // (k_mf_assemble), a caller of the analysis alone gets them listed
    P.a_dst.resize(nnz);
    std::atomic<bool> outside{false};
    parallel_ranges(ni, 4096, [&](size_t lo, size_t hi, unsigned) {
        for (size_t i = lo; i < hi; ++i)
            for (uint32_t k = roff[i]; k < roff[i + 1]; ++k) {
                const uint32_t c = rcol[k], pi = P.pos[i], pj = P.pos[c];
                const MfFront &F = P.fronts[P.front_of[pi <= pj ? i : c]];
                const uint32_t a = front_place(F, P.upos.data(), pi), b = front_place(F, P.upos.data(), pj);
                if (a >= F.m || b >= F.m) outside = true;
                else P.a_dst[k] = F.off + (uint64_t)a * F.m + b;
            }
    });
    if (outside) {
        dgx_set_error("coarse solver: a matrix entry falls outside its front");
        throw DgxError();
    }
    // element-matrix contributions of each entry, in element order: row i's
    // entries come from its incident elements (in element order), each
    // element adding vals[e*64 + k*8 + j] to (ids[j^c], ids[k^c])
    P.a_off.assign(nnz + 1, 0);
    {
        std::vector<std::vector<uint32_t>> part(8);
        parallel_ranges(ni, 4096, [&](size_t lo, size_t hi, unsigned t) {
            std::vector<uint32_t> slot(ni, 0), cnt, start, &out = part[t];
            std::vector<std::pair<uint32_t, uint32_t>> buf;  // (entry in row, contribution)
            out.reserve((size_t)(ioff[hi] - ioff[lo]) * 8);
            for (uint32_t i = (uint32_t)lo; i < hi; ++i) {
                const uint32_t r0 = roff[i], rn = roff[i + 1] - r0;
                for (uint32_t k = r0; k < roff[i + 1]; ++k) slot[rcol[k]] = k - r0;
                cnt.assign(rn + 1, 0);
                buf.clear();
                for (uint32_t q = ioff[i]; q < ioff[i + 1]; ++q) {
                    const uint32_t e = inc[q] >> 3, jj = inc[q] & 7u;
                    const uint32_t c = (meta[e] >> 8) & 7u, j = jj ^ c;  // row i is child-frame vertex j
                    const int32_t *ids = &eid[8 * (size_t)e];
                    for (uint32_t kk = 0; kk < 8; ++kk) {
                        const int32_t col = ids[kk];
                        if (col < 0) continue;
                        const uint32_t k = kk ^ c, a = slot[col];
                        buf.push_back({a, (uint32_t)(e * 64 + k * 8 + j)});
                        ++cnt[a + 1];
                    }
                }
                for (uint32_t a = 0; a < rn; ++a) cnt[a + 1] += cnt[a];
                const size_t base = out.size();
                out.resize(base + buf.size());
                start.assign(cnt.begin(), cnt.end());
                for (const auto &pr : buf) out[base + start[pr.first]++] = pr.second;  // stable: element order
                for (uint32_t a = 0; a < rn; ++a) P.a_off[r0 + a + 1] = cnt[a + 1] - cnt[a];
            }
        });
        for (uint32_t k = 0; k < nnz; ++k) P.a_off[k + 1] += P.a_off[k];
        P.a_src.clear();
        P.a_src.reserve(P.a_off[nnz]);
        for (auto &pv : part) P.a_src.insert(P.a_src.end(), pv.begin(), pv.end());
    }
    return P;
}

// ------------------------------------------------------------- kernels ----
namespace {

constexpr int MB = 256;
constexpr uint32_t kGJT = 64;                       // update tile
typedef double d4 __attribute__((ext_vector_type(4)));

__global__ void k_mf_fill0(double *F, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * MB + threadIdx.x; i < n; i += (uint64_t)gridDim.x * MB) F[i] = 0.0;
}

// ---- the matrix graph of the coarsest level, from its DA
constexpr uint32_t kNoId = 0xffffffffu;
// Elements at a node of a 2:1 balanced octree: in each of the 8 directions the
// leaf at the node and its 7 siblings, whose hanging vertices may refer to it.
constexpr uint32_t kMaxInc = 64, kMaxRow = 8 * kMaxInc;

__global__ void __launch_bounds__(MB) k_cgr_flags(const uint8_t *__restrict__ bdy, uint32_t n, uint32_t *flag) {
    const uint32_t i = blockIdx.x * MB + threadIdx.x;
    if (i <= n) flag[i] = i < n && !bdy[i] ? 1u : 0u;
}
// Interior node ids and coordinates.
__global__ void __launch_bounds__(MB) k_cgr_nodes(const uint8_t *__restrict__ bdy, uint32_t n,
                                                  const uint32_t *__restrict__ iid, const uint32_t *__restrict__ n2l,
                                                  const uint32_t *__restrict__ x, const uint32_t *__restrict__ y,
                                                  const uint32_t *__restrict__ z, uint32_t *inode, uint32_t *xyz) {
    const uint32_t i = blockIdx.x * MB + threadIdx.x;
    if (i >= n || bdy[i]) return;
    const uint32_t v = iid[i], l = n2l[i];
    inode[v] = i;
    xyz[3 * (size_t)v] = x[l];
    xyz[3 * (size_t)v + 1] = y[l];
    xyz[3 * (size_t)v + 2] = z[l];
}
// Interior ids of each element's vertices and each incidence's arrival rank at
// its node.
__global__ void __launch_bounds__(MB) k_cgr_elems(const uint32_t *__restrict__ conn, const uint8_t *__restrict__ bdy,
                                                  const uint32_t *__restrict__ iid, uint32_t ne, uint32_t *eid,
                                                  uint32_t *rank, uint32_t *deg) {
    const uint32_t t = blockIdx.x * MB + threadIdx.x, e = t >> 3, j = t & 7u;
    if (e >= ne) return;
    const uint32_t v = conn[(size_t)j * ne + e], id = bdy[v] ? kNoId : iid[v];
    eid[t] = id;
    if (id != kNoId) rank[t] = atomicAdd(&deg[id], 1u);
}
__global__ void __launch_bounds__(MB) k_cgr_fill(const uint32_t *__restrict__ eid, const uint32_t *__restrict__ rank,
                                                 const uint32_t *__restrict__ ioff, uint32_t n8, uint32_t *inc) {
    const uint32_t t = blockIdx.x * MB + threadIdx.x;
    if (t < n8 && eid[t] != kNoId) inc[ioff[eid[t]] + rank[t]] = t;
}
// One wave per interior row: its incidences put in element order, and its
// columns (the node itself included) in the order those elements first reach
// them, to cand + 8 ioff[i].  64 candidates at a time; one is new if no earlier
// candidate of the 64 and no column found before equals it.
__global__ void __launch_bounds__(MB) k_cgr_rows(const uint32_t *__restrict__ ni, const uint32_t *__restrict__ ioff,
                                                 uint32_t *__restrict__ inc, const uint32_t *__restrict__ eid,
                                                 uint32_t *__restrict__ cand, uint32_t *__restrict__ rlen,
                                                 uint32_t *err) {
    __shared__ uint32_t s_inc[MB / 64][kMaxInc], s_col[MB / 64][kMaxRow];
    const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u, i = blockIdx.x * (MB / 64) + w;
    if (i >= *ni) return;
    const uint32_t q0 = ioff[i], deg = ioff[i + 1] - q0;
    if (deg > kMaxInc) {
        if (lane == 0) atomicOr(err, 1u);
        return;
    }
    uint32_t *out = cand + 8 * (size_t)q0;
    if (deg == 0) {  // a DA's nodes are those that its elements refer to
        if (lane == 0) atomicOr(err, 2u);
        return;
    }
    const uint32_t mine = lane < deg ? inc[q0 + lane] : kNoId;
    uint32_t before = 0;
    for (uint32_t t = 0; t < deg; ++t) before += (uint32_t)__builtin_amdgcn_readlane(mine, t) < mine ? 1u : 0u;
    if (lane < deg) {
        s_inc[w][before] = mine;
        inc[q0 + before] = mine;
    }
    __builtin_amdgcn_wave_barrier();
    uint32_t found = 0;
    for (uint32_t c0 = 0; c0 < 8 * deg; c0 += 64) {
        const uint32_t c = c0 + lane;
        const uint32_t id = c < 8 * deg ? eid[(s_inc[w][c >> 3] & ~7u) + (c & 7u)] : kNoId;
        bool seen = id == kNoId;
        for (uint32_t t = 0; t < found; ++t) seen = seen || s_col[w][t] == id;
        for (uint32_t t = 0; t < 63; ++t) {
            const uint32_t o = (uint32_t)__builtin_amdgcn_readlane(id, t);
            seen = seen || (o == id && t < lane);
        }
        const uint64_t news = __ballot(!seen);
        if (!seen) {
            const uint32_t at = found + (uint32_t)__popcll(news & ((1ull << lane) - 1ull));
            s_col[w][at] = id;
            out[at] = id;
        }
        __builtin_amdgcn_wave_barrier();
        found += (uint32_t)__popcll(news);
    }
    if (lane == 0) rlen[i] = found;
}
__global__ void __launch_bounds__(MB) k_cgr_compact(uint32_t ni, const uint32_t *__restrict__ ioff,
                                                    const uint32_t *__restrict__ cand,
                                                    const uint32_t *__restrict__ roff, uint32_t *rcol) {
    const uint32_t i = blockIdx.x * (MB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (i >= ni) return;
    const uint32_t r0 = roff[i], len = roff[i + 1] - r0;
    for (uint32_t k = lane; k < len; k += 64) rcol[r0 + k] = cand[8 * (size_t)ioff[i] + k];
}

constexpr uint32_t kAsm = 8;
// Assembly, one wave per row i of the matrix and one lane per entry: the sum of
// its element-matrix contributions in element order, stored at its place in the
// front that eliminates the earlier of its two nodes (the places are distinct).
// The host used to list every contribution and place and upload them: 3.7 of the
// 9.6 ms of an analysis of 12,000 nodes.
__global__ void __launch_bounds__(MB) k_mf_assemble(uint32_t ni, const uint32_t *__restrict__ roff,
                                                    const uint32_t *__restrict__ rcol,
                                                    const uint32_t *__restrict__ ioff,
                                                    const uint32_t *__restrict__ inc, const uint32_t *__restrict__ eid,
                                                    const uint16_t *__restrict__ meta,
                                                    const uint32_t *__restrict__ pos,
                                                    const uint32_t *__restrict__ front_of,
                                                    const MfFront *__restrict__ fronts,
                                                    const uint32_t *__restrict__ upos, const double *__restrict__ vals,
                                                    double *F, uint32_t *bad) {
    const uint32_t i = blockIdx.x * (MB / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (i >= ni) return;
    const uint32_t r1 = roff[i + 1], q0 = ioff[i], q1 = ioff[i + 1];
    for (uint32_t k = roff[i] + lane; k < r1; k += 64) {
        const uint32_t col = rcol[k];
        double v = 0.0;
        for (uint32_t q = q0; q < q1; q += kAsm) {  // kAsm elements' loads in flight together
            uint32_t t[kAsm], c[kAsm], hit[kAsm];
            double first[kAsm];
#pragma unroll
            for (uint32_t b = 0; b < kAsm; ++b) t[b] = q + b < q1 ? inc[q + b] : kNoId;
#pragma unroll
            for (uint32_t b = 0; b < kAsm; ++b) {
                hit[b] = c[b] = 0;
                if (t[b] == kNoId) continue;
                c[b] = (meta[t[b] >> 3] >> 8) & 7u;
                const uint32_t *ids = eid + (t[b] & ~7u);
#pragma unroll
                for (uint32_t kk = 0; kk < 8; ++kk) hit[b] |= ids[kk] == col ? 1u << kk : 0u;
            }
            auto at = [&](uint32_t b) {  // child-frame row j of the element's matrix
                const uint32_t k = ((uint32_t)__ffs(hit[b]) - 1u) ^ c[b], j = (t[b] & 7u) ^ c[b];
                return vals[64 * (size_t)(t[b] >> 3) + k * 8 + j];
            };
#pragma unroll
            for (uint32_t b = 0; b < kAsm; ++b) first[b] = hit[b] ? at(b) : 0.0;
#pragma unroll
            for (uint32_t b = 0; b < kAsm; ++b) {
                if (hit[b]) v += first[b];
                for (hit[b] &= hit[b] - 1; hit[b]; hit[b] &= hit[b] - 1) v += at(b);
            }
        }
        const uint32_t pi = pos[i], pj = pos[col];
        const MfFront f = fronts[front_of[pi <= pj ? i : col]];
        const uint32_t a = front_place(f, upos, pi), b = front_place(f, upos, pj);
        if (a < f.m && b < f.m) F[f.off + (uint64_t)a * f.m + b] = v;
        else atomicOr(bad, 2u);
    }
}

// Extend-add: each parent row adds its children's update rows, child by child.
// Four rows per workgroup, one wave per row.
__global__ void __launch_bounds__(MB) k_mf_gather(const MfItem *__restrict__ items, const MfFront *__restrict__ fr,
                                                  const MfLink *__restrict__ links, const int32_t *__restrict__ inv,
                                                  const uint32_t *__restrict__ fmap, double *F) {
    const MfItem it = items[blockIdx.x];
    const MfFront f = fr[it.front];
    const uint32_t p = it.r0 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= f.m) return;
    double *Fr = F + f.off + (uint64_t)p * f.m;
    for (uint32_t l = 0; l < f.nch; ++l) {
        const MfLink L = links[f.ch0 + l];
        const int32_t ip = inv[L.inv + p];
        if (ip < 0) continue;
        const MfFront c = fr[L.child];
        const uint32_t uc = c.m - c.s;
        const double *Ur = F + c.off + (uint64_t)(c.s + ip) * c.m + c.s;
        for (uint32_t q = lane; q < uc; q += 64) Fr[fmap[L.fmap + q]] += Ur[q];
    }
}

// Blocked Gauss-Jordan of the fronts of one tree level, 32 pivots K = [k0,
// k0 + kb) per launch and 64 x 64 tiles of each front.  With D = F[K,K]^-1,
// C = F[:,K] and W = D F[K,:] outside K, D in its columns K:
//   F[i,j] = (j in K ? 0 : F[i,j]) - C[i,:] W[:,j]  for i outside K, F[K,:] = W.
// A launch reads F only in the tile it writes; F[K,:] and C come from two
// scratch panels that the launch before filled while it wrote those rows and
// columns, and D from the workgroup of that launch that holds the next pivot
// block, which inverts it (it is scheduled first).  The panels and D alternate
// between two sets.  Every tile forms its own 64 columns of W.
//
// What bounds it: the serial chain of launches, pivots and divisions, except for
// dense fronts of thousands of rows (FP64 rate).  Both products are FP64 matrix
// instructions (16 x 16 x 4): their operands come from LDS or L2 once per 16
// products.  Three launches per block step (inverse by 1024 threads with two
// barriers per pivot, panels, update with vector FMAs and a scalar loop for the
// columns K) took 14.4 + 7.6 + 25.5 us on the fronts of a 3M-point 4-Gaussian
// octree's coarsest level; one step now takes 16.8 us, and each tree level 9.7 us for
// its first launch.

// x of the lanes 16 g .. 16 g + 15, in every group of 16 lanes
__device__ __forceinline__ double group_bcast(double x, int g) {
    uint32_t w[2] = {(uint32_t)__double_as_longlong(x), (uint32_t)(__double_as_longlong(x) >> 32)};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto a = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);
        const uint32_t y = (g & 1) ? a[1] : a[0];
        const auto b = __builtin_amdgcn_permlane32_swap(y, y, false, false);
        w[h] = (g & 2) ? b[1] : b[0];
    }
    return __longlong_as_double((uint64_t)w[1] << 32 | w[0]);
}
// x of lane R of the lane's group of 16
template <int R>
__device__ __forceinline__ double lane_bcast(double x) {
    const uint64_t v = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, 0x150 + R, 0xf, 0xf, false),
                   hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), 0x150 + R, 0xf, 0xf, false);
    return __longlong_as_double((uint64_t)hi << 32 | lo);
}
// One pivot (row and column R) of the inversion below.
template <int R>
__device__ __forceinline__ void invert_pivot(double X[4], bool &ok) {
    constexpr int G = R & 3, U = R >> 2;
    const uint32_t lj = threadIdx.x & 15, lg = (threadIdx.x >> 4) & 3;
    const double f = group_bcast(X[U], G), piv = lane_bcast<R>(f), inv = 1.0 / piv;
    ok = ok && piv > 0.0 && piv < INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const bool col = u == U && lg == G;
        const double a = lane_bcast<R>(X[u]), b = col ? 1.0 : a, q = b * inv;
        const double t = fma(fma(-q, piv, b), inv, q);  // b / piv: one correction of b * inv
        const double x = (col ? 0.0 : X[u]) - f * t;
        X[u] = lj == R ? t : x;
    }
}
// Inverse of the 16 x 16 matrix held by one wave, by Gauss-Jordan without
// pivoting: X[u] of lane 16 g + j is the entry (j, g + 4 u).  A pivot row is
// broadcast within the groups of 16 lanes, a pivot column across them: no LDS and
// no barrier.  ok becomes false for a pivot that is not positive.
__device__ __forceinline__ void invert16(double X[4], bool &ok) {
    invert_pivot<0>(X, ok);
    invert_pivot<1>(X, ok);
    invert_pivot<2>(X, ok);
    invert_pivot<3>(X, ok);
    invert_pivot<4>(X, ok);
    invert_pivot<5>(X, ok);
    invert_pivot<6>(X, ok);
    invert_pivot<7>(X, ok);
    invert_pivot<8>(X, ok);
    invert_pivot<9>(X, ok);
    invert_pivot<10>(X, ok);
    invert_pivot<11>(X, ok);
    invert_pivot<12>(X, ok);
    invert_pivot<13>(X, ok);
    invert_pivot<14>(X, ok);
    invert_pivot<15>(X, ok);
}
// (A B)^T + c for 16 x 16 blocks in the layout of invert16, b holding B^T: that
// layout is the matrix instructions' first operand, the second operand's
// transpose and the result's transpose.
__device__ __forceinline__ d4 mul16(const double a[4], const double b[4], d4 c) {
#pragma unroll
    for (int k = 0; k < 4; ++k) c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], b[k], c, 0, 0, 0);
    return c;
}
// Inverse of the symmetric 32 x 32 matrix of blocks X[x][y] by its 2 x 2 block
// form: P = A00^-1, H = A10 P, S = A11 - H A01, Q = S^-1; the inverse is
// [P + H^T Q H, -H^T Q; -Q H, Q].  Half the pivots' work of a plain 32 x 32
// Gauss-Jordan: k_mf_gj_first takes 9.7 us with it, 12.3 without.
__device__ __forceinline__ bool invert32(double X[2][2][4]) {
    bool ok = true;
    double P[4], H[4], G[4], Q[4], N[4];  // G = H^T
    const d4 zero = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int u = 0; u < 4; ++u) Q[u] = half ? X[1][1][u] : X[0][0][u];
        invert16(Q, ok);
        if (half) break;
        const d4 h = mul16(Q, X[1][0], zero), g = mul16(X[1][0], Q, zero);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            P[u] = Q[u];
            H[u] = h[u];
            G[u] = g[u];
        }
        const d4 t = mul16(H, X[1][0], zero);
#pragma unroll
        for (int u = 0; u < 4; ++u) X[1][1][u] -= t[u];
    }
    const d4 lo = mul16(G, Q, zero), up = mul16(Q, G, zero);
#pragma unroll
    for (int u = 0; u < 4; ++u) N[u] = up[u];
    const d4 c = mul16(N, G, zero);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        X[0][0][u] = P[u] + c[u];
        X[0][1][u] = -up[u];
        X[1][0][u] = -lo[u];
        X[1][1][u] = Q[u];
    }
    return ok;
}
// The inverse of the kb x kb pivot block in the result layout (v[bi][bj][r] of
// lane 16 g + j: entry (16 bi + g + 4 r, 16 bj + j)), padded with an identity, to
// D (32 x 32).
__device__ __forceinline__ void invert_block(const double v[2][2][4], uint32_t kb, double *D, uint32_t *bad) {
    const uint32_t lj = threadIdx.x & 15, lg = (threadIdx.x >> 4) & 3;
    double X[2][2][4];
#pragma unroll
    for (uint32_t bi = 0; bi < 2; ++bi)
#pragma unroll
        for (uint32_t bj = 0; bj < 2; ++bj)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t i = 16 * bi + lg + 4 * r, j = 16 * bj + lj;
                X[bj][bi][r] = i < kb && j < kb ? v[bi][bj][r] : (i == j ? 1.0 : 0.0);
            }
    if (!invert32(X)) atomicOr(bad, 1u);
#pragma unroll
    for (uint32_t bi = 0; bi < 2; ++bi)
#pragma unroll
        for (uint32_t bj = 0; bj < 2; ++bj)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) D[(16 * bi + lg + 4 * r) * kGJ + 16 * bj + lj] = X[bj][bi][r];
}

// The panels and the inverse of the first pivot block: 64 columns of F[K,:] and
// 64 rows of F[:,K] per workgroup.
__global__ void __launch_bounds__(MB) k_mf_gj_first(const double *__restrict__ F, const MfFront *__restrict__ fr,
                                                    const uint32_t *__restrict__ lvl, double *__restrict__ TC,
                                                    double *__restrict__ dinv, uint32_t *bad) {
    const MfFront f = fr[lvl[blockIdx.y]];
    const uint32_t n = f.m, c0 = blockIdx.x * kGJT;
    if (!f.s || c0 >= n) return;
    const uint32_t kb = min(kGJ, f.s);
    const double *A = F + f.off;
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        const uint32_t lj = threadIdx.x & 15, lg = threadIdx.x >> 4;
        double v[2][2][4];
#pragma unroll
        for (uint32_t bi = 0; bi < 2; ++bi)
#pragma unroll
            for (uint32_t bj = 0; bj < 2; ++bj)
#pragma unroll
                for (uint32_t r = 0; r < 4; ++r) {
                    const uint32_t i = 16 * bi + lg + 4 * r, j = 16 * bj + lj;
                    v[bi][bj][r] = i < kb && j < kb ? A[(size_t)i * n + j] : 0.0;
                }
        invert_block(v, kb, dinv + (size_t)f.dinv * (2 * kGJ * kGJ), bad);
        return;
    }
    // the first workgroup's other waves do its share
    const uint32_t t0 = blockIdx.x == 0 ? threadIdx.x - 64 : threadIdx.x, nt = blockIdx.x == 0 ? MB - 64 : MB;
    double *R = TC + f.tc, *C = R + (size_t)kGJ * n;
    for (uint32_t t = t0; t < kGJT * kGJ; t += nt) {
        const uint32_t q = t / kGJT, j = c0 + t % kGJT, i = c0 + t / kGJ, c = t % kGJ;
        if (q < kb && j < n) R[(size_t)q * n + j] = A[(size_t)q * n + j];
        if (c < kb && i < n) C[(size_t)i * kGJ + c] = A[(size_t)i * n + c];
    }
}

__global__ void __launch_bounds__(MB) k_mf_gj_step(double *__restrict__ F, const MfFront *__restrict__ fr,
                                                   const uint32_t *__restrict__ lvl, uint32_t k0,
                                                   double *__restrict__ TC, double *__restrict__ dinv, uint32_t *bad) {
    const MfFront f = fr[lvl[blockIdx.y]];
    const uint32_t n = f.m, nt = (n + kGJT - 1) / kGJT;
    uint32_t tile = blockIdx.x;
    if (k0 >= f.s || tile >= nt * nt) return;
    const uint32_t kb = min(kGJ, f.s - k0), kn = k0 + kGJ, kbn = kn < f.s ? min(kGJ, f.s - kn) : 0u;
    if (kbn) {  // the tile of the next pivot block first
        const uint32_t d = kn / kGJT * (nt + 1);
        tile = tile == 0 ? d : tile == d ? 0u : tile;
    }
    const uint32_t i0 = tile / nt * kGJT, j0 = tile % nt * kGJT, par = (k0 / kGJ) & 1u;
    double *A = F + f.off, *P = TC + f.tc;
    const double *R = P + (size_t)(par * 2 * kGJ) * n, *C = R + (size_t)kGJ * n;
    double *Rn = P + (size_t)((par ^ 1u) * 2 * kGJ) * n, *Cn = Rn + (size_t)kGJ * n;
    double *Dv = dinv + (size_t)(2 * f.dinv + par) * (kGJ * kGJ), *Dn = dinv + (size_t)(2 * f.dinv + (par ^ 1u)) * (kGJ * kGJ);
    __shared__ double Ws[kGJ][kGJT + 2];
    const uint32_t w = threadIdx.x >> 6, lj = threadIdx.x & 15, lg = (threadIdx.x >> 4) & 3;
    const uint32_t wi = i0 + (w >> 1) * 32, wj = j0 + (w & 1) * 32;  // the wave's 32 x 32
    // k of the matrix instructions: step ks of lane group lg is 8 lg + ks
    const uint32_t c0 = 8 * lg;
    double dv[2][8], rv[8], cv[2][8], a[2][2][4];
    const uint32_t jw = j0 + 16 * w + lj;  // the wave's columns of W
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        rv[k] = c0 + k < kb && jw < n ? R[(size_t)(c0 + k) * n + jw] : 0.0;
        dv[0][k] = Dv[lj * kGJ + c0 + k];
        dv[1][k] = Dv[(16 + lj) * kGJ + c0 + k];
    }
#pragma unroll
    for (uint32_t b = 0; b < 2; ++b)
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t i = wi + 16 * b + lj;
            cv[b][k] = c0 + k < kb && i < n ? C[(size_t)i * kGJ + c0 + k] : 0.0;
        }
#pragma unroll
    for (uint32_t bi = 0; bi < 2; ++bi)
#pragma unroll
        for (uint32_t bj = 0; bj < 2; ++bj)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t i = wi + 16 * bi + lg + 4 * r, j = wj + 16 * bj + lj;
                const bool in = i < n && j < n && !(j >= k0 && j < k0 + kb);
                a[bi][bj][r] = in ? A[(size_t)i * n + j] : 0.0;
            }
    {
        d4 t0 = {0.0, 0.0, 0.0, 0.0}, t1 = t0;
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            t0 = __builtin_amdgcn_mfma_f64_16x16x4f64(dv[0][k], rv[k], t0, 0, 0, 0);
            t1 = __builtin_amdgcn_mfma_f64_16x16x4f64(dv[1][k], rv[k], t1, 0, 0, 0);
        }
        const bool jK = jw >= k0 && jw < k0 + kb;
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t q = lg + 4 * r;
            Ws[q][16 * w + lj] = jK ? Dv[q * kGJ + jw - k0] : t0[r];
            Ws[16 + q][16 * w + lj] = jK ? Dv[(16 + q) * kGJ + jw - k0] : t1[r];
        }
    }
    __syncthreads();
    const uint32_t lw = (w & 1) * 32 + lj;
    d4 acc[2][2] = {};
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        const double b0 = Ws[c0 + k][lw], b1 = Ws[c0 + k][lw + 16];
#pragma unroll
        for (uint32_t b = 0; b < 2; ++b) {
            acc[b][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(cv[b][k], b0, acc[b][0], 0, 0, 0);
            acc[b][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(cv[b][k], b1, acc[b][1], 0, 0, 0);
        }
    }
#pragma unroll
    for (uint32_t bi = 0; bi < 2; ++bi)
#pragma unroll
        for (uint32_t bj = 0; bj < 2; ++bj)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) {
                const uint32_t i = wi + 16 * bi + lg + 4 * r, j = wj + 16 * bj + lj;
                const bool iK = i >= k0 && i < k0 + kb;
                const double v = iK ? Ws[i - k0][j - j0] : a[bi][bj][r] - acc[bi][bj][r];
                a[bi][bj][r] = v;
                if (i >= n || j >= n) continue;
                A[(size_t)i * n + j] = v;
                if (i - kn < kbn) Rn[(size_t)(i - kn) * n + j] = v;  // i < kn: i - kn wraps past kbn
                if (j - kn < kbn) Cn[(size_t)i * kGJ + (j - kn)] = v;
            }
    if (kbn && wi == kn && wj == kn) invert_block(a, kbn, Dn, bad);
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Each wave of a 16-row work item takes 4 consecutive rows and forms their
// products with a vector in LDS, over columns [0, ncol).  A lane keeps 4 rows x 4
// column chunks of loads in flight, so a row costs a few memory round trips
// instead of one per 64 columns; the order of the sums is fixed.  The first round
// is loaded while the vector is still being gathered (load, then dot behind the
// barrier).
struct Rows4 {
    const double *Ar[4];
    bool ok[4];
    uint32_t ncol, lane;
    double a[4][4];
    __device__ __forceinline__ Rows4(const double *A, uint64_t ld, uint32_t rb, uint32_t r_end, uint32_t nc,
                                     uint32_t ln)
        : ncol(nc), lane(ln) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            ok[q] = rb + q < r_end;
            Ar[q] = A + (uint64_t)(ok[q] ? rb + q : 0u) * ld;
        }
    }
    __device__ __forceinline__ void load(uint32_t j0) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) a[q][u] = j0 + 64 * u < ncol && ok[q] ? Ar[q][j0 + 64 * u] : 0.0;
    }
    __device__ __forceinline__ void dot(const double *vl, double acc[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = 0.0;
        for (uint32_t j0 = lane; j0 < ncol; j0 += 64 * 4) {
            if (j0 != lane) load(j0);
            double v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = j0 + 64 * u < ncol ? vl[j0 + 64 * u] : 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[q] = fma(a[q][u], v[u], acc[q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = wave_sum(acc[q]);
    }
};

// The sum of the children's updates at the front's position p, child by child.
__device__ __forceinline__ double child_updates(const MfSolveItem &f, const uint32_t *__restrict__ src,
                                                const double *upd, uint32_t p, double v) {
    for (uint32_t l = 0; l < f.nch; l += 2) {
        const uint32_t *q = src + f.src + (size_t)l * f.m + p;
        const bool two = l + 1 < f.nch;
        const uint32_t s0 = q[0], s1 = two ? q[f.m] : 0u;
        const double u0 = upd[s0], u1 = two ? upd[s1] : 0.0;
        v += u0;
        if (two) v += u1;
    }
    return v;
}

// Forward sweep of one level: w_S = b_S + children's updates (kept in ws for
// the backward sweep), then the update rows upd = w_U + P21 w_S, with
// P21 = -F21 F11^-1 in rows s.. of the front.  16 rows per workgroup.  Bound: the
// chain of dependent loads of a launch (there are two per tree level and V-cycle),
// so an item carries its front's fields and src the update's index itself.  Found
// through item, front, link and child, with the rows loaded behind the barrier, a
// forward launch took 9.4 us and a backward one 8.1 in the V-cycles of a 16M-point
// 4-Gaussian octree; now 7.9 and 7.6.  An item of a front without update rows
// gathers kGather values of w_S.  Workgroups past the items store the boundary
// rows, z = b.
template <typename T>
__global__ void __launch_bounds__(MB) k_mf_fwd(const MfSolveItem *__restrict__ items, uint32_t nitems,
                                               const uint32_t *__restrict__ src, const uint32_t *__restrict__ idx,
                                               const double *__restrict__ F, const T *__restrict__ b, double *ws,
                                               double *upd, const uint8_t *__restrict__ bdy, uint32_t n, T *z) {
    extern __shared__ double wl[];
    if (blockIdx.x >= nitems) {
        const uint32_t i = (blockIdx.x - nitems) * MB + threadIdx.x;
        if (i < n && bdy[i]) z[i] = b[i];
        return;
    }
    const MfSolveItem f = items[blockIdx.x];
    const uint32_t u = f.m - f.s, lane = threadIdx.x & 63;
    if (u == 0) {
        const uint32_t p = f.r0 + threadIdx.x;
        if (p < f.s) ws[f.ws + p] = child_updates(f, src, upd, p, (double)b[idx[f.idx + p]]);
        return;
    }
    const uint32_t rb = f.r0 + (threadIdx.x >> 6) * 4, r1 = min(f.r0 + 16u, u);
    Rows4 rows(F + f.off + (uint64_t)f.s * f.m, f.m, rb, r1, f.s, lane);
    rows.load(lane);
    const bool out = lane < 4 && rb + lane < r1;
    const double wu = out ? child_updates(f, src, upd, f.s + rb + lane, 0.0) : 0.0;
    for (uint32_t p = threadIdx.x; p < f.s; p += MB) {
        const double v = child_updates(f, src, upd, p, (double)b[idx[f.idx + p]]);
        wl[p] = v;
        if (f.r0 == 0) ws[f.ws + p] = v;
    }
    __syncthreads();
    if (rb >= r1) return;
    double acc[4];
    rows.dot(wl, acc);
    if (out) {
        const double a = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
        upd[f.upd + rb + lane] = wu + a;
    }
}

// Backward sweep of one level: x_S = P11 w_S - P12 x_U (rows 0..s-1 of the
// front hold [F11^-1, F11^-1 F12]); x_U are ancestors' nodes, solved already.
template <typename T>
__global__ void __launch_bounds__(MB) k_mf_bwd(const MfSolveItem *__restrict__ items, const uint32_t *__restrict__ idx,
                                               const double *__restrict__ F, const double *__restrict__ ws,
                                               double *x, T *z) {
    extern __shared__ double vl[];
    const MfSolveItem f = items[blockIdx.x];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t rb = f.r0 + (threadIdx.x >> 6) * 4, r1 = min(f.r0 + 16u, f.s);
    Rows4 rows(F + f.off, f.m, rb, r1, f.m, lane);
    rows.load(lane);
    const uint32_t at = lane < 4 && rb + lane < r1 ? idx[f.idx + rb + lane] : 0u;
    for (uint32_t j = threadIdx.x; j < f.m; j += MB) vl[j] = j < f.s ? ws[f.ws + j] : -x[idx[f.idx + j]];
    __syncthreads();
    if (rb >= r1) return;
    double acc[4];
    rows.dot(vl, acc);
    if (lane < 4 && rb + lane < r1) {
        const double a = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
        x[at] = a;
        z[at] = (T)a;
    }
}

// The arrays of a plan, gathered in host memory and uploaded with one copy (one
// copy each took some 40 calls of a few microseconds).
struct PlanPacker {
    struct Part {
        const void *src;
        size_t bytes, at;
        std::function<void(uint8_t *)> set;
    };
    std::vector<Part> parts;
    size_t total = 0;
    template <typename T>
    void add(DevView<T> &d, const std::vector<T> &h) {
        parts.push_back({h.data(), h.size() * sizeof(T), total,
                         [&d](uint8_t *q) { d.p = reinterpret_cast<T *>(q); }});
        total += (h.size() * sizeof(T) + 255) / 256 * 256;
    }
    // host keeps the bytes until the copy is done
    void upload(DevBuf<uint8_t> &dev, std::vector<uint8_t> &host, hipStream_t s) {
        host.resize(total);
        dev.alloc(total, s);
        for (const Part &p : parts) {
            if (p.bytes) std::memcpy(host.data() + p.at, p.src, p.bytes);
            p.set(dev.p + p.at);
        }
        if (total) HIP_OK(hipMemcpyAsync(dev.p, host.data(), total, hipMemcpyHostToDevice, s));
    }
};
template <typename T>
void download(std::vector<T> &h, const T *d, size_t n, hipStream_t s) {
    h.resize(n);
    if (n) HIP_OK(hipMemcpyAsync(h.data(), d, n * sizeof(T), hipMemcpyDeviceToHost, s));
}

}  // namespace

CoarseInputs coarse_graph(const DaDevice &d, hipStream_t s) {
    CoarseInputs in;
    const uint32_t n = in.n = d.n_nodes, ne = (uint32_t)d.n_elem;
    if (d.n_elem * 64 > 0xffffffffull) {
        dgx_set_error("coarse solver: %zu elements exceed the 32-bit contribution index", d.n_elem);
        throw DgxError();
    }
    CoarseGraph &g = in.g;
    DevBuf<uint32_t> flag((size_t)n + 1, s), iid((size_t)n + 1, s), inode(n, s), xyz(3 * (size_t)n, s),
        rank(8 * (size_t)ne, s), cand(64 * (size_t)ne, s);
    // node degrees and row lengths (one more each, for the totals), results
    const size_t n1 = (size_t)n + 1;
    DevBuf<uint32_t> cnt(2 * n1 + 3, s);
    uint32_t *deg = cnt.p, *rlen = deg + n1, *res = rlen + n1;  // res: interior nodes, entries, error
    HIP_OK(hipMemsetAsync(cnt.p, 0, (2 * n1 + 3) * 4, s));
    g.ioff.alloc(n1, s);
    g.roff.alloc(n1, s);
    g.eid.alloc(8 * (size_t)ne, s);
    g.inc.alloc(8 * (size_t)ne, s);
    k_cgr_flags<<<grid_for(n1, MB), MB, 0, s>>>(d.bdy_node.p, n, flag.p);
    scan_exclusive_u32_async(flag.p, iid.p, n1, res, s);
    k_cgr_nodes<<<grid_for(n1, MB), MB, 0, s>>>(d.bdy_node.p, n, iid.p, d.n2l.p, d.x.p, d.y.p, d.z.p, inode.p, xyz.p);
    k_cgr_elems<<<grid_for(8 * (size_t)ne, MB), MB, 0, s>>>(d.conn.p, d.bdy_node.p, iid.p, ne, g.eid.p, rank.p, deg);
    scan_exclusive_u32_async(deg, g.ioff.p, n1, nullptr, s);
    k_cgr_fill<<<grid_for(8 * (size_t)ne, MB), MB, 0, s>>>(g.eid.p, rank.p, g.ioff.p, 8 * ne, g.inc.p);
    k_cgr_rows<<<grid_for(n, MB / 64), MB, 0, s>>>(res, g.ioff.p, g.inc.p, g.eid.p, cand.p, rlen, res + 2);
    scan_exclusive_u32_async(rlen, g.roff.p, n1, res + 1, s);
    HIP_OK(hipGetLastError());
    uint32_t h[3];
    dgx_read_back(h, res, sizeof h, s);
    if (h[2]) {
        if (h[2] & 2u) dgx_set_error("coarse solver: an interior node of no element");
        else dgx_set_error("coarse solver: a node with more than %u elements (octree not 2:1 balanced)", kMaxInc);
        throw DgxError();
    }
    in.ni = h[0];
    g.rcol.alloc(h[1], s);
    if (in.ni)
        k_cgr_compact<<<grid_for(in.ni, MB / 64), MB, 0, s>>>(in.ni, g.ioff.p, cand.p, g.roff.p, g.rcol.p);
    HIP_OK(hipGetLastError());
    download(in.inode, inode.p, in.ni, s);
    download(in.xyz, xyz.p, 3 * (size_t)in.ni, s);
    download(in.roff, g.roff.p, (size_t)in.ni + 1, s);
    download(in.rcol, g.rcol.p, h[1], s);
    HIP_OK(hipStreamSynchronize(s));
    return in;
}

MfPlan coarse_plan(const CoarseInputs &in, uint32_t dense) {
    MfPlan P;
    P.n = in.n;
    P.ni = in.ni;
    P.inode = in.inode;
    // the fronts may take at most 4 GiB of doubles
    mf_symbolic(P, in.roff, in.rcol, in.xyz, (4ull << 30) / 8, 128, dense);
    return P;
}

std::unique_ptr<CoarseSolver> coarse_upload(MfPlan &&plan, CoarseInputs &&in, hipStream_t s) {
    std::unique_ptr<CoarseSolver> cs(new CoarseSolver());
    cs->plan = std::move(plan);
    cs->g = std::move(in.g);
    const MfPlan &P = cs->plan;
    cs->n = in.n;
    cs->ni = P.ni;
    cs->nfronts = (uint32_t)P.fronts.size();
    cs->levels = (uint32_t)P.lvl_fronts.size();
    PlanPacker pk;
    pk.add(cs->fronts, P.fronts);
    pk.add(cs->links, P.links);
    pk.add(cs->inv, P.inv);
    pk.add(cs->fmap, P.fmap);
    pk.add(cs->idx, P.idx);
    pk.add(cs->upos, P.upos);
    pk.add(cs->pos, P.pos);
    pk.add(cs->front_of, P.front_of);
    cs->lvl_fronts.resize(cs->levels);
    cs->lvl_fwd.resize(cs->levels);
    cs->lvl_bwd.resize(cs->levels);
    cs->lvl_gather.resize(cs->levels);
    // the solve sweeps' items with their fronts' fields, and for each position of a
    // parent the places of its children's updates (past the last update: 0)
    std::vector<uint32_t> src(P.inv.size(), (uint32_t)P.upd_len);
    for (const MfFront &F : P.fronts)
        for (uint32_t l = F.ch0; l < F.ch0 + F.nch; ++l)
            for (uint32_t p = 0; p < F.m; ++p) {
                const int32_t ip = P.inv[P.links[l].inv + p];
                if (ip >= 0) src[P.links[l].inv + p] = P.fronts[P.links[l].child].upd + (uint32_t)ip;
            }
    pk.add(cs->src, src);
    auto solve_items = [&](const std::vector<MfItem> &it) {
        std::vector<MfSolveItem> v;
        v.reserve(it.size());
        for (const MfItem &i : it) {
            const MfFront &F = P.fronts[i.front];
            // a front's links follow each other in inv, m entries each
            v.push_back({F.off, F.m, F.s, F.idx, F.upd, F.ws, F.nch ? P.links[F.ch0].inv : 0u, F.nch, i.r0});
        }
        return v;
    };
    std::vector<std::vector<MfSolveItem>> fwd, bwd;
    for (uint32_t h = 0; h < cs->levels; ++h) {
        fwd.push_back(solve_items(P.lvl_fwd[h]));
        bwd.push_back(solve_items(P.lvl_bwd[h]));
        pk.add(cs->lvl_fronts[h], P.lvl_fronts[h]);
        pk.add(cs->lvl_fwd[h], fwd[h]);
        pk.add(cs->lvl_bwd[h], bwd[h]);
        pk.add(cs->lvl_gather[h], P.lvl_gather[h]);
    }
    std::vector<uint8_t> host;
    pk.upload(cs->packed, host, s);
    cs->F.alloc(P.front_entries, s);
    cs->upd.alloc(P.upd_len + 1, s);
    HIP_OK(hipMemsetAsync(cs->upd.p + P.upd_len, 0, sizeof(double), s));
    cs->ws.alloc(P.ni, s);
    cs->x.alloc(in.n, s);
    HIP_OK(hipStreamSynchronize(s));  // the upload reads host memory
    return cs;
}

std::unique_ptr<CoarseSolver> coarse_analyse(const DaDevice &d, hipStream_t s, uint32_t dense) {
    CoarseInputs in = coarse_graph(d, s);
    MfPlan plan = coarse_plan(in, dense);
    return coarse_upload(std::move(plan), std::move(in), s);
}

void coarse_factor(CoarseSolver &cs, const DaDevice &d, double lap_fac, double mass_fac, hipStream_t s) {
    const MfPlan &P = cs.plan;
    DevBuf<uint32_t> bad(1, s);
    HIP_OK(hipMemsetAsync(bad.p, 0, 4, s));
    {
        DevBuf<double> vals((size_t)64 * d.n_elem, s);
        if (d.n_elem) da_element_matrices(d, lap_fac, mass_fac, vals.p, s);
        if (P.front_entries)
            k_mf_fill0<<<(unsigned)std::min<uint64_t>(grid_for(P.front_entries, MB), 8192), MB, 0, s>>>(
                cs.F.p, P.front_entries);
        if (cs.ni)
            k_mf_assemble<<<grid_for(cs.ni, MB / 64), MB, 0, s>>>(cs.ni, cs.g.roff.p, cs.g.rcol.p, cs.g.ioff.p,
                                                                 cs.g.inc.p, cs.g.eid.p, d.meta.p, cs.pos.p,
                                                                 cs.front_of.p, cs.fronts.p, cs.upos.p, vals.p,
                                                                 cs.F.p, bad.p);
        HIP_OK(hipGetLastError());
    }
    DevBuf<double> TC(std::max<uint64_t>(P.tc_max, 1), s), dinv((size_t)std::max(P.dinv_max, 1u) * 2 * kGJ * kGJ, s);
    for (uint32_t h = 0; h < cs.levels; ++h) {
        const uint32_t nf = (uint32_t)P.lvl_fronts[h].size();
        if (!P.lvl_gather[h].empty())
            k_mf_gather<<<(unsigned)P.lvl_gather[h].size(), MB, 0, s>>>(cs.lvl_gather[h].p, cs.fronts.p,
                                                                        cs.links.p, cs.inv.p, cs.fmap.p, cs.F.p);
        const uint32_t mm = P.lvl_max_m[h];
        const uint32_t nt = grid_for(mm, kGJT);
        if (!P.lvl_max_s[h]) continue;
        k_mf_gj_first<<<dim3(nt, nf), MB, 0, s>>>(cs.F.p, cs.fronts.p, cs.lvl_fronts[h].p, TC.p, dinv.p, bad.p);
        for (uint32_t k0 = 0; k0 < P.lvl_max_s[h]; k0 += kGJ)
            k_mf_gj_step<<<dim3(nt * nt, nf), MB, 0, s>>>(cs.F.p, cs.fronts.p, cs.lvl_fronts[h].p, k0, TC.p, dinv.p,
                                                          bad.p);
        HIP_OK(hipGetLastError());
    }
    uint32_t hbad = 0;
    dgx_read_back(&hbad, bad.p, 4, s);
    if (hbad & 2u) {
        dgx_set_error("coarse solver: a matrix entry falls outside its front");
        throw DgxError();
    }
    if (hbad) {
        dgx_set_error("multigrid: coarse matrix is not positive definite (a pivot is not positive)");
        throw DgxError();
    }
}

template <typename T>
void coarse_solve(CoarseSolver &cs, const uint8_t *bdy, const T *b, T *z, hipStream_t s) {
    const MfPlan &P = cs.plan;
    for (uint32_t h = 0; h < std::max(cs.levels, 1u); ++h) {
        const uint32_t items = cs.levels ? (uint32_t)P.lvl_fwd[h].size() : 0u, rest = h ? 0u : grid_for(cs.n, MB);
        if (items + rest)
            k_mf_fwd<T><<<items + rest, MB, cs.levels ? P.lvl_max_s[h] * sizeof(double) : 0, s>>>(
                cs.levels ? cs.lvl_fwd[h].p : nullptr, items, cs.src.p, cs.idx.p, cs.F.p, b, cs.ws.p, cs.upd.p, bdy,
                cs.n, z);
    }
    for (uint32_t h = cs.levels; h-- > 0;)
        k_mf_bwd<T><<<(unsigned)P.lvl_bwd[h].size(), MB, P.lvl_max_m[h] * sizeof(double), s>>>(
            cs.lvl_bwd[h].p, cs.idx.p, cs.F.p, cs.ws.p, cs.x.p, z);
    HIP_OK(hipGetLastError());
}
template void coarse_solve<double>(CoarseSolver &, const uint8_t *, const double *, double *, hipStream_t);
template void coarse_solve<float>(CoarseSolver &, const uint8_t *, const float *, float *, hipStream_t);

// ------------------------------------------------------- C ABI (host plan) ----
struct dgx_direct_plan_s {
    MfPlan plan;
};

extern "C" {

int dgx_direct_plan_host(uint32_t n, uint64_t n_elem, const uint32_t *conn, const uint16_t *meta, const uint8_t *bdy,
                         const uint32_t *xyz, uint32_t leaf, uint32_t dense, dgx_direct_plan *out,
                         dgx_direct_sizes *sz) {
    if (!out || !sz || (n_elem && (!conn || !meta)) || (n && (!bdy || !xyz))) {
        dgx_set_error("direct plan: null argument");
        return -1;
    }
    try {
        std::unique_ptr<dgx_direct_plan_s> h(new dgx_direct_plan_s());
        h->plan = mf_plan(n, n_elem, conn, meta, bdy, xyz, ~0ull, leaf ? leaf : 128, dense);
        const MfPlan &P = h->plan;
        sz->interior = P.ni;
        sz->fronts = P.fronts.size();
        sz->links = P.links.size();
        sz->levels = P.lvl_fronts.size();
        sz->entries = P.front_entries;
        sz->idx_len = P.idx.size();
        sz->inv_len = P.inv.size();
        sz->fmap_len = P.fmap.size();
        sz->a_nnz = P.a_dst.size();
        sz->a_src_len = P.a_src.size();
        sz->upd_len = P.upd_len;
        sz->max_m = P.max_m;
        sz->max_s = P.max_s;
        *out = h.release();
        return 0;
    } catch (DgxError &) {
        return -1;
    } catch (std::exception &e) {
        dgx_set_error("direct plan: %s", e.what());
        return -1;
    }
}

int dgx_direct_plan_export(dgx_direct_plan h, uint64_t *front9, uint64_t *link3, int32_t *inv, uint32_t *fmap,
                           uint32_t *idx, uint32_t *a_off, uint32_t *a_src, uint64_t *a_dst, uint32_t *inode) {
    if (!h) {
        dgx_set_error("direct plan: null handle");
        return -1;
    }
    const MfPlan &P = h->plan;
    if (front9)
        for (size_t f = 0; f < P.fronts.size(); ++f) {
            const MfFront &F = P.fronts[f];
            const uint64_t v[9] = {F.off, F.m, F.s, F.idx, F.upd, F.ws, F.ch0, F.nch, P.height[f]};
            std::memcpy(front9 + 9 * f, v, sizeof(v));
        }
    if (link3)
        for (size_t l = 0; l < P.links.size(); ++l) {
            link3[3 * l] = P.links[l].child;
            link3[3 * l + 1] = P.links[l].inv;
            link3[3 * l + 2] = P.links[l].fmap;
        }
    if (inv) std::copy(P.inv.begin(), P.inv.end(), inv);
    if (fmap) std::copy(P.fmap.begin(), P.fmap.end(), fmap);
    if (idx) std::copy(P.idx.begin(), P.idx.end(), idx);
    if (a_off) std::copy(P.a_off.begin(), P.a_off.end(), a_off);
    if (a_src) std::copy(P.a_src.begin(), P.a_src.end(), a_src);
    if (a_dst) std::copy(P.a_dst.begin(), P.a_dst.end(), a_dst);
    if (inode) std::copy(P.inode.begin(), P.inode.end(), inode);
    return 0;
}

int dgx_direct_plan_free(dgx_direct_plan h) {
    delete h;
    return 0;
}

}  // extern "C"
