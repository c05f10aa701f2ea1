// Numeric multifrontal factorisation on gfx950.
//
// Fronts are processed level by level (height above the leaves), all fronts
// of a level and all frequencies of a batch in the same launches:
//   1. assemble: every entry of a front is written once, as the sum of the
//      children's Schur complements (pulled through child->parent index maps)
//      and of the original matrix entries the front owns (each has one
//      destination, so no atomics);
//   2. partial LU of the first p columns with row pivoting restricted to the
//      p fully summed rows (the front's structure never changes):
//      - fronts with m <= small_max: one workgroup each, which does step 1 too
//        and keeps the front in LDS throughout;
//      - larger fronts: blocked right-looking LU, per panel step a panel
//        kernel (pivot search, scaling, the swaps within the panel), a kernel
//        that replays the swaps on the other columns and solves the U rows,
//        and an MFMA trailing update of the remaining front (which leaves the
//        Schur complement in F22).
// Factors stay in place in the front arena (L11\U11 and L21 in the first p
// columns, U12 in the first p rows); the pivot swaps go to piv[pos0 + j].
#include <algorithm>
#include <utility>

#include "engine.hpp"
#include "mfma.hpp"
#include "prof.hpp"

namespace gfdfd {


// ---------------------------------------------------------------------------
// DevPlan
// ---------------------------------------------------------------------------
// Small fronts (order <= the plan's small_max) are assembled and factored in
// one kernel each, so every small front gets a slot with its own list of
// original entries; the blocked fronts' entries are listed by column.
// Small subtrees: a front belongs when its order is at most small_max and all
// its children belong (leaves included), so a whole subtree can be factored
// by the persistent launch and the level path never waits on it.
// Fronts are in postorder, so each maximal subtree is a contiguous range
// ending at its root.
void DevPlan::build_small(const Plan &pl, std::vector<FrontDev> &fd) {
    const int nfr = (int)pl.fronts.size();
    std::vector<char> in(nfr, 0), small(nfr, 0);
    for (const LevelPlan &L : pl.levels)
        for (int f : L.small) small[f] = 1;
    for (int f = 0; f < nfr; f++) {   // postorder: children first
        const Front &F = pl.fronts[f];
        bool ok = pl.grid && small[f] && F.m <= kSubMaxM && F.nchild <= kAsmMaxChildren;
        for (int c = 0; c < F.nchild && ok; c++) ok = in[pl.children[F.child_off + c]] != 0;
        in[f] = ok;
    }
    std::vector<int> slot(nfr, -1), first, last, lo(nfr);
    int nslot = 0;
    for (int f = 0; f < nfr; f++) {   // lowest front of f's subtree
        const Front &F = pl.fronts[f];
        lo[f] = f;
        for (int c = 0; c < F.nchild; c++) lo[f] = std::min(lo[f], lo[pl.children[F.child_off + c]]);
        if (small[f]) slot[f] = nslot++;
    }
    for (int f = 0; f < nfr; f++)
        if (in[f]) {
            const Front &F = pl.fronts[f];
            sub_mmax = std::max(sub_mmax, F.m);
            for (int k = 0; k < F.p; k++) {
                const double t = F.m - k - 1;
                sub_flops += 4.0 * (2.0 * t * t + t);
            }
            sub_elems += (double)F.m * F.m;
            if (F.parent < 0 || !in[F.parent]) {
                for (int g = lo[f]; g <= f; g++)
                    if (!in[g]) throw std::logic_error("small subtree is not a contiguous postorder range");
                first.push_back(lo[f]);
                last.push_back(f);
            }
        }
    nroots = (int)first.size();
    // original entries: the small fronts' by slot (local offsets), the blocked fronts' by column
    std::vector<std::vector<std::pair<int64_t, int>>> per_slot(nslot);
    std::vector<int> cptr;
    for (int f = 0; f < nfr; f++) {
        if (slot[f] < 0) {
            fd[f].slot = (int)cptr.size();
            cptr.resize(cptr.size() + pl.fronts[f].m + 1, 0);
        } else {
            fd[f].slot = slot[f];
        }
    }
    std::vector<std::vector<std::pair<int64_t, int>>> per_col(cptr.size());
    std::vector<std::pair<int64_t, int>> starts;   // buf_off -> front
    for (int f = 0; f < nfr; f++) starts.push_back({pl.fronts[f].buf_off, f});
    std::sort(starts.begin(), starts.end());
    for (size_t e = 0; e < pl.orig_q.size(); e++) {
        const int64_t d = pl.orig_dst[e];
        auto it = std::upper_bound(starts.begin(), starts.end(), std::make_pair(d, INT32_MAX));
        if (it == starts.begin()) throw std::logic_error("original entry before the first front");
        const int f = std::prev(it)->second;
        const Front &F = pl.fronts[f];
        const int64_t o = d - F.buf_off;
        if (o >= (int64_t)F.m * F.m) throw std::logic_error("original entry outside its front");
        if (slot[f] >= 0) per_slot[slot[f]].push_back({pl.orig_q[e], (int)o});
        else per_col[fd[f].slot + o / F.m].push_back({pl.orig_q[e], (int)o});
    }
    std::vector<int64_t> optr(nslot + 1, 0), oq;
    std::vector<int> ooff;
    for (int k = 0; k < nslot; k++) {
        for (auto &e : per_slot[k]) { oq.push_back(e.first); ooff.push_back(e.second); }
        optr[k + 1] = (int64_t)oq.size();
    }
    std::vector<int64_t> lq;
    std::vector<int> loff;
    for (size_t c = 0; c < cptr.size(); c++) {
        cptr[c] = (int)lq.size();
        for (auto &e : per_col[c]) { lq.push_back(e.first); loff.push_back(e.second); }
    }
    root_first = dev_upload(first);
    root_last = dev_upload(last);
    small_optr = dev_upload(optr);
    small_oq = dev_upload(oq);
    small_ooff = dev_upload(ooff);
    large_cptr = dev_upload(cptr);
    large_oq = dev_upload(lq);
    large_ooff = dev_upload(loff);
    bytes += (2 * first.size() + ooff.size() + cptr.size() + loff.size()) * 4 +
             (optr.size() + oq.size() + lq.size()) * 8;
    for (int l = 0; l < pl.nlevels; l++) {
        const LevelPlan &L = pl.levels[l];
        // the level's small fronts outside the subtrees
        std::vector<FrontDev> sm;
        int smm = 0;
        double el = 0, sfl = 0, sel = 0;
        for (int f : L.small)
            if (!in[f]) {
                const Front &F = pl.fronts[f];
                sm.push_back(fd[f]);
                smm = std::max(smm, F.m);
                sel += 2.0 * F.m * F.m;
                for (int k = 0; k < F.p; k++) {
                    const double t = F.m - k - 1;
                    sfl += 4.0 * (2.0 * t * t + t);
                }
            }
        for (int f : L.large) el += (double)pl.fronts[f].m * pl.fronts[f].m;
        lv_small_rest.push_back(dev_upload(sm));
        n_small_rest.push_back((int)sm.size());
        small_mmax_rest.push_back(smm);
        asm_elems_large.push_back(el);
        small_rest_flops.push_back(sfl);
        small_rest_elems.push_back(sel);
    }
}

DevPlan::DevPlan(std::shared_ptr<const Plan> p) : host(std::move(p)) {
    const Plan &pl = *host;
    std::vector<FrontDev> fd(pl.fronts.size());
    for (size_t f = 0; f < pl.fronts.size(); f++) {
        const Front &F = pl.fronts[f];
        fd[f] = {F.p, F.m, F.pos0, F.nchild, F.child_off, F.level, -1, 0, F.buf_off, F.fv_off, F.idx_off, F.inv_off};
    }
    build_small(pl, fd);
    fronts = dev_upload(fd);
    children = dev_upload(pl.children);
    idx = dev_upload(pl.idx);
    inv = dev_upload(pl.inv);
    perm = dev_upload(pl.perm);
    iperm = dev_upload(pl.iperm);
    colptr = dev_upload(pl.colptr);
    rowind = dev_upload(pl.rowind);
    bytes += fd.size() * sizeof(FrontDev) + (pl.children.size() + pl.idx.size() + pl.inv.size() +
                                            2 * pl.perm.size() + pl.colptr.size() + pl.rowind.size()) * 4;
    // gather sources of every front row before pivoting, at the front's work rows:
    // [X position or -1, W row of a child's contribution or -1, a second one or -1]
    {
        std::vector<int> g((size_t)pl.fv_rows * 3, -1);
        for (const Front &F : pl.fronts)
            for (int i = 0; i < F.m; i++) {
                int *r = &g[(size_t)(F.fv_off + i) * 3];
                if (i < F.p) r[0] = F.pos0 + i;
                int k = 1;
                for (int c = 0; c < F.nchild; c++) {
                    const Front &C = pl.fronts[pl.children[F.child_off + c]];
                    const int a = pl.inv[C.inv_off + i];
                    if (a < 0) continue;
                    if (k == 3) throw std::logic_error("front row with more than two child contributions");
                    r[k++] = (int)(C.fv_off + C.p + a);
                }
            }
        gsrc_id = dev_upload(g);
        bytes += g.size() * 4;
    }
    // CSR-of-M -> CSC map, valid when the pattern is symmetric (grid plans)
    if (pl.grid) {
        std::vector<int64_t> t(pl.nnz);
        std::vector<int> fill(pl.n, 0);
        for (int c = 0; c < pl.n; c++)
            for (int q = pl.colptr[c]; q < pl.colptr[c + 1]; q++) {
                int r = pl.rowind[q];
                // row r of M: its entries in column order are the rows of CSC column r (symmetric pattern)
                t[pl.colptr[r] + fill[r]++] = q;
            }
        tq = dev_upload(t);
        bytes += t.size() * 8;
    }
    for (const LevelPlan &L : pl.levels) {
        std::vector<int> all(L.small);
        all.insert(all.end(), L.large.begin(), L.large.end());
        std::vector<FrontDev> lf;
        int haskids = 0;
        for (int f : all) {
            lf.push_back(fd[f]);
            haskids |= pl.fronts[f].nchild > 0;
        }
        lv_children.push_back(haskids);
        lv_fr.push_back(dev_upload(lf));
        lv_all.push_back(dev_upload(all));
        n_small.push_back((int)L.small.size());
        n_large.push_back((int)L.large.size());
        n_all.push_back((int)all.size());
        mmax_all.push_back(std::max(L.small_mmax, L.large_mmax));
        int pm = 0;
        for (int f : all) pm = std::max(pm, pl.fronts[f].p);
        pmax_all.push_back(pm);
    }
    // tile lists of every blocked step
    std::vector<TileDev> tl;
    std::vector<Tile> tmp;
    steps.resize(pl.levels.size());
    for (size_t l = 0; l < pl.levels.size(); l++) {
        const LevelPlan &L = pl.levels[l];
        for (int k0 = 0; k0 < L.large_pmax; k0 += pl.nb) {
            step_tiles(pl, L, k0, kTile, tmp);
            steps[l].push_back({(int64_t)tl.size(), (int)tmp.size()});
            for (const Tile &t : tmp) tl.push_back({t.front, t.ti, t.tj});
        }
    }
    // the two-panel schedule: per 64-column block b0 of a level, the thin update
    // (rows from b0 + 32, the second panel's columns: fronts with p > b0 + 32)
    // and the depth-min(64, p - b0) trailing update
    if (pl.nb != 32) throw std::logic_error("the blocked path assumes 32-column panels");
    deep_steps.resize(pl.levels.size());
    for (size_t l = 0; l < pl.levels.size(); l++) {
        const LevelPlan &L = pl.levels[l];
        for (int b0 = 0; b0 < L.large_pmax; b0 += 64) {
            DeepStep d;
            d.thin_off = (int64_t)tl.size();
            for (int li = 0; li < (int)L.large.size(); li++) {
                const Front &F = pl.fronts[L.large[li]];
                if (F.p <= b0 + 32) continue;
                const int kb2 = std::min(32, F.p - b0 - 32), t = F.m - b0 - 32;
                for (int ti = 0; ti < (t + kTile - 1) / kTile; ti++) tl.push_back({li, ti, 0});
                d.thin_flops += 8.0 * t * kb2 * 32;
                d.thin_elems += 2.0 * t * kb2 + t * 32.0 + 32.0 * kb2;
                d.trsm_thin_flops += 8.0 * 0.5 * 32 * 32 * kb2;
            }
            d.thin_cnt = (int)(tl.size() - d.thin_off);
            d.deep_off = (int64_t)tl.size();
            for (int li = 0; li < (int)L.large.size(); li++) {
                const Front &F = pl.fronts[L.large[li]];
                if (F.p <= b0) continue;
                const int kd = std::min(64, F.p - b0), t = F.m - b0 - kd;
                for (int j = b0; j < b0 + kd; j++) {
                    const int pe = j < b0 + 32 ? std::min(b0 + 32, b0 + kd) : b0 + kd;   // the panel's end
                    (j < b0 + 32 ? d.panel1_flops : d.panel2_flops) +=
                        8.0 * (F.m - j - 1) * (pe - j - 1) + 6.0 * (F.m - j - 1);
                }
                if (t <= 0) continue;
                const int nt = (t + kTile - 1) / kTile;
                for (int tj = 0; tj < nt; tj++)
                    for (int ti = 0; ti < nt; ti++) tl.push_back({li, ti, tj});
                d.deep_flops += 8.0 * t * t * kd;
                d.deep_elems += 2.0 * t * kd + 2.0 * t * t;
                d.trsm_deep_flops += 8.0 * 0.5 * kd * kd * t;
            }
            d.deep_cnt = (int)(tl.size() - d.deep_off);
            deep_steps[l].push_back(d);
        }
    }
    tiles = dev_upload(tl);
    bytes += tl.size() * sizeof(TileDev);
    for (const Front &F : pl.fronts) max_children = std::max(max_children, F.nchild);
    // single-block levels: every front of the level has at most one pivot block
    // and is stored in the one-product solve format (see k_diag_inv)
    for (size_t l = 0; l < pl.levels.size(); l++)
        single.push_back(pmax_all[l] <= 32 && mmax_all[l] <= kSingleMmax && max_children <= 2 ? 1 : 0);
    lv_single = dev_upload(single);
    // inverse squares for the levels of fewer than kVecSplitFronts multi-block
    // fronts whose pivot blocks fit the inversion kernel's LDS
    {
        std::vector<int> lst;
        std::vector<int64_t> loff;
        vinv.assign(pl.levels.size(), 0);
        vinv_off.assign(pl.levels.size(), nullptr);
        for (size_t l = 0; l < pl.levels.size(); l++) {
            if (single[l] || n_all[l] >= kVecSplitFronts || pmax_all[l] > kVinvPmax || n_all[l] == 0) continue;
            vinv[l] = 1;
            const LevelPlan &L = pl.levels[l];
            std::vector<int> all(L.small);
            all.insert(all.end(), L.large.begin(), L.large.end());
            std::vector<int64_t> off;
            for (int f : all) {
                const int p = pl.fronts[f].p, c = pl.fronts[f].m - p;
                off.push_back(vinv_elems);
                lst.push_back(f);
                loff.push_back(vinv_elems);
                // the square, then L21 inv(L11) (c x p) and inv(U11) U12 (p x c)
                vinv_elems += (int64_t)p * p + 2 * (int64_t)p * c;
                vinv_pmax = std::max(vinv_pmax, p);
                vinv_rect_tiles = std::max(vinv_rect_tiles, 2 * ((p + 63) / 64) * ((c + 63) / 64));
            }
            vinv_off[l] = dev_upload(off);
        }
        vinv_n = (int)lst.size();
        vinv_list = dev_upload(lst);
        vinv_list_off = dev_upload(loff);
        bytes += lst.size() * 12;
    }
    counts.resize(pl.levels.size());
    for (size_t l = 0; l < pl.levels.size(); l++) {
        const LevelPlan &L = pl.levels[l];
        LevelCounts &c = counts[l];
        auto each = [&](const std::vector<int> &v, auto fn) { for (int f : v) fn(pl.fronts[f]); };
        auto tri = [&](const Front &F) {
            double p = F.p, m = F.m;
            c.tri_elems += 0.5 * p * p + p * (m - p);
            c.sum_m += m;
            c.asm_elems += m * m;
        };
        each(L.small, tri);
        each(L.large, tri);
        each(L.small, [&](const Front &F) {
            for (int k = 0; k < F.p; k++) {
                double t = F.m - k - 1;
                c.small_flops += 4.0 * (2.0 * t * t + t);
            }
            c.small_elems += 2.0 * F.m * F.m;
        });
        each(L.small, [&](const Front &F) { c.contrib_elems += (double)F.p * (F.m - F.p); c.sum_p += F.p; });
        each(L.large, [&](const Front &F) { c.contrib_elems += (double)F.p * (F.m - F.p); c.sum_p += F.p; });
        int lpmax = 0;
        for (int f : L.small) lpmax = std::max(lpmax, pl.fronts[f].p);
        for (int f : L.large) lpmax = std::max(lpmax, pl.fronts[f].p);
        for (int b0 = 0; b0 < lpmax; b0 += 32) {
            double fe = 0, be = 0;
            auto blk = [&](const Front &F) {
                if (F.p <= b0) return;
                const double kb = std::min(32, F.p - b0);
                fe += 0.5 * kb * kb + kb * (F.m - b0 - kb);
                be += 0.5 * kb * kb + kb * b0;
                diag_elems += kb * kb;
            };
            each(L.small, blk);
            each(L.large, blk);
            c.fwd_blk_elems.push_back(fe);
            c.bwd_blk_elems.push_back(be);
        }
        for (int k0 = 0; k0 < L.large_pmax; k0 += pl.nb) {
            double gf = 0, ge = 0, pf = 0, tf = 0;
            each(L.large, [&](const Front &F) {
                if (F.p <= k0) return;
                double kb = std::min(pl.nb, F.p - k0), t = F.m - k0 - kb;
                gf += 8.0 * t * t * kb;
                ge += 2.0 * t * kb + 2.0 * t * t;
                for (int j = k0; j < k0 + kb; j++) pf += 8.0 * (F.m - j - 1) * (k0 + kb - j - 1) + 6.0 * (F.m - j - 1);
                tf += 8.0 * 0.5 * kb * kb * t;
            });
            c.gemm_flops.push_back(gf);
            c.gemm_elems.push_back(ge);
            c.panel_flops.push_back(pf);
            c.trsm_flops.push_back(tf);
        }
    }
}

DevPlan::~DevPlan() {
    dev_free(fronts); dev_free(children); dev_free(idx); dev_free(inv); dev_free(perm); dev_free(iperm);
    dev_free(colptr); dev_free(rowind); dev_free(tq); dev_free(tiles);
    dev_free(lv_single);
    dev_free(gsrc_id);
    for (auto p : vinv_off) dev_free(p);
    dev_free(vinv_list);
    dev_free(vinv_list_off);
    dev_free(root_first); dev_free(root_last); dev_free(small_optr); dev_free(small_oq);
    dev_free(small_ooff); dev_free(large_cptr); dev_free(large_oq); dev_free(large_ooff);
    for (auto p : lv_small_rest) dev_free(p);
    for (auto p : lv_fr) dev_free(p);
    for (auto p : lv_all) dev_free(p);
}

template <typename T>
Factors<T>::~Factors() {
    if (graph) (void)hipGraphExecDestroy(graph);
    dev_free(arena);
    dev_free(piv);
    dev_free(rowperm);
    dev_free(sing);
    dev_free(gsrc);
    dev_free(sched);
    dev_free(vinv);
    if (own_vals) dev_free(vals);
}
template struct Factors<double>;
template struct Factors<float>;

// 1+2: assembly of the blocked fronts
// ---------------------------------------------------------------------------
// A workgroup writes a block of whole columns of one front, every entry once,
// as the sum of the children's Schur complements, then adds the columns'
// original entries (each destination is unique, and only this workgroup
// touches these columns: a barrier separates the two, where a scatter launch of
// its own cost 5 us a level).  With up to two children (the grid plans' fronts)
// their values are loaded unconditionally (an entry a child does not cover
// reads the child's block origin and is dropped), four entries at a time, so
// eight loads are in flight before the first add.  grid (fronts, column blocks, nfreq)
template <typename T>
__global__ void __launch_bounds__(256) k_front_assemble(cx<T> *__restrict__ arena, int64_t fstride,
                                                        const FrontDev *__restrict__ lvF,
                                                        const FrontDev *__restrict__ fronts,
                                                        const int *__restrict__ children, const int *__restrict__ inv,
                                                        const int *__restrict__ cptr, const int64_t *__restrict__ oq,
                                                        const int *__restrict__ ooff,
                                                        const cx<double> *__restrict__ vals, int64_t vstride,
                                                        int ncols) {
    extern __shared__ int cmap[];   // [nchild][m]: child row of each front row, or -1
    __shared__ int64_t cbase[kAsmMaxChildren];
    __shared__ int cstride[kAsmMaxChildren];
    const FrontDev F = lvF[blockIdx.x];
    const int m = F.m, nc = F.nchild, c0 = blockIdx.y * ncols, c1 = min(m, c0 + ncols);
    if (c0 >= m) return;
    cx<T> *A = arena + blockIdx.z * fstride;
    cx<T> *G = A + F.buf_off;
    const int tid = threadIdx.x;
    const int o0 = cptr[F.slot + c0], o1 = cptr[F.slot + c1];
    // the children's row maps and block origins, staged once: each entry below
    // then waits on one value load only
    if (tid < nc) {
        const FrontDev C = fronts[children[F.child_off + tid]];
        cbase[tid] = C.buf_off + C.p + (int64_t)C.p * C.m;   // contribution block origin
        cstride[tid] = C.m;
    }
    for (int c = 0; c < nc; c++) {
        const int io = fronts[children[F.child_off + c]].inv_off;
        for (int r = tid; r < m; r += 256) cmap[c * m + r] = inv[io + r];
    }
    __syncthreads();
    const int64_t beg = (int64_t)c0 * m, end = (int64_t)c1 * m;
    if (nc <= 2 && end < (int64_t(1) << 31)) {
        constexpr int U = 4;
        const int tot = (int)end;
        for (int e0 = (int)beg + tid; e0 < tot; e0 += U * 256) {
            cx<T> w[U][2];
            bool ok[U][2];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = e0 + u * 256;
                const int ec = e < tot ? e : (int)beg;
                const int s = ec / m, r = ec - s * m;
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int a = c < nc ? cmap[c * m + r] : -1, b = c < nc ? cmap[c * m + s] : -1;
                    ok[u][c] = a >= 0 && b >= 0;
                    w[u][c] = A[c < nc ? cbase[c] + (ok[u][c] ? a + (int64_t)b * cstride[c] : 0) : F.buf_off];
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = e0 + u * 256;
                if (e >= tot) break;
                cx<T> v = {T(0), T(0)};
                if (ok[u][0]) v = w[u][0];
                if (ok[u][1]) v = cadd(v, w[u][1]);
                G[e] = v;
            }
        }
    } else {
        for (int64_t e = beg + tid; e < end; e += 256) {
            const int s = (int)(e / m), r = (int)(e - (int64_t)s * m);
            cx<T> v = {T(0), T(0)};
            for (int c = 0; c < nc; c++) {
                const int a = cmap[c * m + r], b = cmap[c * m + s];
                if (a >= 0 && b >= 0) v = cadd(v, A[cbase[c] + a + (int64_t)b * cstride[c]]);
            }
            G[e] = v;
        }
    }
    __syncthreads();
    const cx<double> *V = vals + blockIdx.z * vstride;
    for (int e = o0 + tid; e < o1; e += 256) {
        const cx<double> v = V[oq[e]];
        cx<T> &d = G[ooff[e]];
        d.x += (T)v.x;
        d.y += (T)v.y;
    }
}

// ---------------------------------------------------------------------------
// pivot search helper: max cabs1 with the smallest row on ties
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void better(T &best, int &bi, T ob, int oi) {
    if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
}

template <typename T>
__device__ int block_argmax(T best, int bi, T *sb, int *si) {
    // wave reduction then across waves through LDS
    for (int off = 32; off > 0; off >>= 1) {
        T ob = __shfl_xor(best, off);
        int oi = __shfl_xor(bi, off);
        better(best, bi, ob, oi);
    }
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) { sb[w] = best; si[w] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < nw; k++) better(sb[0], si[0], sb[k], si[k]);
    }
    __syncthreads();
    return si[0];
}

// ---------------------------------------------------------------------------
// 3a: small fronts, one workgroup, front in LDS
// ---------------------------------------------------------------------------
// fn(0), fn(1), .. fn(N - 1) with constant indices, so that arrays indexed by
// them stay in registers (a loop whose guard is monotone in its index can be
// rolled again after unrolling, which puts them in scratch)
template <typename Fn, int... I>
__device__ __forceinline__ void static_for_seq(Fn &&fn, std::integer_sequence<int, I...>) {
    (fn(std::integral_constant<int, I>{}), ...);
}
template <int N, typename Fn>
__device__ __forceinline__ void static_for(Fn &&fn) {
    static_for_seq(fn, std::make_integer_sequence<int, N>{});
}
// acc += a*b.  The panel kernels sum an entry's terms from zero and subtract the
// sum once: subtracted one by one every term rounds at the size of the entry,
// which the terms are far below (with the panels' eliminations done so, FP32
// factors' solutions 1.2 to 1.3 times further off: 201x101, 3.8e-6 against
// 2.9e-6, the geometric mean of 12 matrices).
template <typename T>
__device__ __forceinline__ void cmadd_to(T &sx, T &sy, cx<T> a, cx<T> b) {
    sx = fma(-a.y, b.y, fma(a.x, b.x, sx));
    sy = fma(a.y, b.x, fma(a.x, b.y, sy));
}
// c - a*b where a sum cannot be kept, for each step needs the entry: in FP64 the
// product first, so that only the subtraction rounds at the size of c (61x41,
// error 2.26e-15 against 2.37e-15, at no cost); in FP32 fused.  That is 1.68e-6 at
// 61x41, 3 % above the LDS panels (1.62e-6), and 2.9e-6 at 201x101, 4 % below
// them; with the product apart 1.53e-6 and 2.8e-6, the contribution rows 0.4 % of
// a factorisation of 1601x401 slower, and the refinement's second step contracts
// so well that the test of a step expected wrongly finds none on its inputs.
template <typename T>
__device__ __forceinline__ cx<T> cmsub_step(cx<T> c, cx<T> a, cx<T> b) {
    if constexpr (sizeof(T) == 8) return csub(c, cmul_f(a, b));
    else return cmsub_f(c, a, b);
}
// wave-wide maximum and minimum by DPP (row shifts, then row broadcasts): six
// register steps where xor-shuffles take six LDS-crossbar round trips
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(dpp_i<CTRL, ROWS>(__float_as_int(v)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)dpp_i<CTRL, ROWS>((int)(unsigned)b);
    const unsigned hi = (unsigned)dpp_i<CTRL, ROWS>((int)(unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float readlane_t(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double readlane_t(double d, int l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(d);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ cx<T> readlane_t(cx<T> v, int l) {
    return {readlane_t(v.x, l), readlane_t(v.y, l)};
}
// (neither argument is ever a NaN; fmax would quiet each of them first)
__device__ __forceinline__ float max_raw(float a, float b) { return fmax(a, b); }
__device__ __forceinline__ double max_raw(double a, double b) {
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
    v = max_raw(v, dpp_f<0x111, 0xF>(v));   // row_shr 1, 2, 4, 8
    v = max_raw(v, dpp_f<0x112, 0xF>(v));
    v = max_raw(v, dpp_f<0x114, 0xF>(v));
    v = max_raw(v, dpp_f<0x118, 0xF>(v));
    v = max_raw(v, dpp_f<0x142, 0xA>(v));   // row_bcast 15 into rows 1 and 3
    v = max_raw(v, dpp_f<0x143, 0xC>(v));   // row_bcast 31 into rows 2 and 3
    return readlane_t(v, 63);
}
// holds a value's computation where it is called: the reciprocals then run
// beside the pivot search instead of being sunk below it
template <typename T>
__device__ __forceinline__ void pin(cx<T> v) {
    asm volatile("" ::"v"(v.x), "v"(v.y));
}
__device__ __forceinline__ int wave_min(int v) {
    v = min(v, dpp_i<0x111, 0xF>(v));
    v = min(v, dpp_i<0x112, 0xF>(v));
    v = min(v, dpp_i<0x114, 0xF>(v));
    v = min(v, dpp_i<0x118, 0xF>(v));
    v = min(v, dpp_i<0x142, 0xA>(v));
    v = min(v, dpp_i<0x143, 0xC>(v));
    return __builtin_amdgcn_readlane(v, 63);
}

// Partial LU of an m x m front held column-major in LDS (p pivots, row
// pivoting within the p fully-summed rows); rp[i] is the row that ends at position i.
// All 256 threads of the workgroup call it.  Blocked by kLuNb pivots, three
// barriers per panel:
//   - wave 0 factors the panel's kLuNb columns with its rows in registers (lane
//     l holds rows l and, for NR = 2, l + 64).  Rows do not move: each lane
//     carries the position its row has reached, so a swap is two label
//     changes.  The pivot is found by a DPP maximum and a ballot (ties by the
//     lowest position), its row reaches the wave by readlane, and every lane's
//     reciprocal of its own candidate runs beside the search, so the two
//     divisions are off the chain;
//   - the workgroup reads each other column's panel rows and displaced rows
//     through the panel's permutation, forms the U12 rows by forward
//     substitution in registers and writes both back;
//   - one trailing update A22 -= L21 U12 of depth kLuNb with 2 x 2 output tiles
//     per thread.
// Complex products use the explicit fused multiply-adds (cmul_f, cmsub_f): the
// persistent subtree kernel and the level path inline this function and must
// round alike.
constexpr int kLuNb = 8;
struct LuPerm {
    int top[kLuNb];             // row (before the panel) that ends at each panel position
    int q[kLuNb], r[kLuNb];     // positions below the panel that change, and the rows they take
    int nd;
};
template <typename T, int NR>
__device__ __forceinline__ void small_lu_lds(cx<T> *S, int m, int p, int *rp, int *__restrict__ sing, LuPerm *pm) {
    const int tid = threadIdx.x, bs = 256, lane = tid & 63;
    int row[NR];   // wave 0: the row (before all swaps) at the lane's position
#pragma unroll
    for (int k = 0; k < NR; k++) row[k] = lane + 64 * k;
    for (int jb = 0; jb < p; jb += kLuNb) {
        const int je = min(p, jb + kLuNb), nb = je - jb;   // panel columns [jb, je)
        if (tid < 64) {
            cx<T> a[NR][kLuNb];
            int pos[NR];   // position of the lane's row
#pragma unroll
            for (int k = 0; k < NR; k++) {
                const int r = lane + 64 * k;
                pos[k] = r;
#pragma unroll
                for (int c = 0; c < kLuNb; c++)
                    a[k][c] = r < m && c < nb ? S[r + (jb + c) * m] : cx<T>{T(0), T(0)};
            }
            bool zero = false;
#pragma unroll
            for (int jj = 0; jj < kLuNb; jj++) if (jj < nb) {
                const int j = jb + jj;
                // the lane's candidate: rows at positions [j, p); a NaN counts as -1
                T best = T(-2);
                int bp = m;
                cx<T> ca = a[0][jj];
#pragma unroll
                for (int k = 0; k < NR; k++)
                    if (pos[k] >= j && pos[k] < p) {
                        const T v = cabs1(a[k][jj]), w = v >= T(0) ? v : T(-1);
                        if (w > best || (w == best && pos[k] < bp)) {
                            best = w;
                            bp = pos[k];
                            ca = a[k][jj];
                        }
                    }
                const cx<T> rc = crecip(ca);
                const T mx = wave_max(best);
                pin(rc);
                const unsigned long long tie = __ballot(best == mx);
                int L = __ffsll((unsigned long long)tie) - 1;
                if (tie & (tie - 1)) {
                    const int lowest = wave_min(best == mx ? bp : m);
                    L = __ffsll((unsigned long long)__ballot(best == mx && bp == lowest)) - 1;
                }
                const int pr = __builtin_amdgcn_readlane(bp, L);
                zero |= mx == T(0);
                const cx<T> d = readlane_t(rc, L);
                cx<T> u[kLuNb];
#pragma unroll
                for (int c = jj + 1; c < kLuNb; c++) {
                    if constexpr (NR == 1) {
                        u[c] = readlane_t(a[0][c], L);
                    } else {
                        const bool k1 = pos[1] == bp;   // which of the lane's rows is its candidate
                        const cx<T> w = {k1 ? a[1][c].x : a[0][c].x, k1 ? a[1][c].y : a[0][c].y};
                        u[c] = readlane_t(w, L);
                    }
                }
#pragma unroll
                for (int k = 0; k < NR; k++) {
                    pos[k] = pos[k] == pr ? j : pos[k] == j ? pr : pos[k];
                    if (pos[k] > j) {
                        const cx<T> l = cmul_f(a[k][jj], d);
                        a[k][jj] = l;
#pragma unroll
                        for (int c = jj + 1; c < kLuNb; c++) a[k][c] = cmsub_f(a[k][c], l, u[c]);
                    }
                }
            }
            if (zero && lane == 0) atomicOr(sing, 1);
            int base = 0;
#pragma unroll
            for (int k = 0; k < NR; k++) {
                const int r = lane + 64 * k;
                const bool in = r >= jb && r < m;
                if (in) {
#pragma unroll
                    for (int c = 0; c < kLuNb; c++)
                        if (c < nb) S[pos[k] + (jb + c) * m] = a[k][c];
                    if (pos[k] < je) pm->top[pos[k] - jb] = r;
                    rp[pos[k]] = row[k];
                }
                const bool moved = in && pos[k] >= je && pos[k] != r;
                const unsigned long long mv = __ballot(moved);
                if (moved) {
                    const int at = base + __popcll(mv & ((1ull << lane) - 1));
                    pm->q[at] = pos[k];
                    pm->r[at] = r;
                }
                base += __popcll(mv);
            }
            if (lane == 0) pm->nd = base;
            // (one wave: its LDS operations complete in order)
#pragma unroll
            for (int k = 0; k < NR; k++)
                if (lane + 64 * k >= jb && lane + 64 * k < p) row[k] = rp[lane + 64 * k];
        }
        __syncthreads();
        // the other columns: rows of the panel and the rows it displaced, through
        // the permutation; beyond the panel the U12 rows by forward substitution
        {
            const int nd = pm->nd;
            for (int c = tid; c < m; c += bs) {
                if (c >= jb && c < je) continue;
                cx<T> *col = S + c * m;
                cx<T> u[kLuNb];
#pragma unroll
                for (int i = 0; i < kLuNb; i++) u[i] = col[i < nb ? pm->top[i] : jb];
                if (nd > 0) {
                    T wr[kLuNb], wi[kLuNb];
                    static_for<kLuNb>([&](auto k) {
                        const cx<T> w = col[k < nd ? pm->r[k] : jb];
                        wr[k] = w.x;
                        wi[k] = w.y;
                    });
                    static_for<kLuNb>([&](auto k) {
                        if (k < nd) col[pm->q[k]] = {wr[k], wi[k]};
                    });
                }
                if (c >= je)
                    static_for<kLuNb>([&](auto i) {
                        if (i < nb)
                            static_for<i>([&](auto t) { u[i] = cmsub_f(u[i], S[jb + i + (jb + t) * m], u[t]); });
                    });
                static_for<kLuNb>([&](auto i) {
                    if (i < nb) col[jb + i] = u[i];
                });
            }
        }
        __syncthreads();
        if (je >= m) break;
        // trailing update of rows and columns [je, m): 2 x 2 tiles, the tile's
        // rows fastest across threads
        const int q = m - je, qt = (q + 1) >> 1;
        for (int tt = tid; tt < qt * qt; tt += bs) {
            const int r0 = je + 2 * (tt % qt), c0 = je + 2 * (tt / qt);
            const bool r1 = r0 + 1 < m, c1 = c0 + 1 < m;
            cx<T> a00 = S[r0 + c0 * m], a10 = r1 ? S[r0 + 1 + c0 * m] : cx<T>{T(0), T(0)};
            cx<T> a01 = c1 ? S[r0 + (c0 + 1) * m] : cx<T>{T(0), T(0)};
            cx<T> a11 = (r1 && c1) ? S[r0 + 1 + (c0 + 1) * m] : cx<T>{T(0), T(0)};
#pragma unroll 2
            for (int t = jb; t < je; t++) {
                const cx<T> l0 = S[r0 + t * m], l1 = r1 ? S[r0 + 1 + t * m] : cx<T>{T(0), T(0)};
                const cx<T> u0 = S[t + c0 * m], u1 = c1 ? S[t + (c0 + 1) * m] : cx<T>{T(0), T(0)};
                a00 = cmsub_f(a00, l0, u0);
                a10 = cmsub_f(a10, l1, u0);
                a01 = cmsub_f(a01, l0, u1);
                a11 = cmsub_f(a11, l1, u1);
            }
            S[r0 + c0 * m] = a00;
            if (r1) S[r0 + 1 + c0 * m] = a10;
            if (c1) S[r0 + (c0 + 1) * m] = a01;
            if (r1 && c1) S[r0 + 1 + (c0 + 1) * m] = a11;
        }
        __syncthreads();
    }
}

// what a small front's assembly and LU read of the plan and write beside the arena
struct SmallDev {
    const FrontDev *fronts;
    const int *children, *inv;
    const int64_t *optr, *oq;
    const int *ooff;
    const cx<double> *vals;
    int64_t vstride;
    int *rowperm;
    int n;
    int *sing;
};
struct SmallShared {
    LuPerm pm;
    int rp[96];   // row (before all swaps) at each position
    int64_t cbase[kAsmMaxChildren];
    int cstride[kAsmMaxChildren];
};
// LDS of a small front: the front, then its children's row maps
template <typename T>
constexpr size_t small_front_lds(int mmax, int max_children) {
    return sizeof(cx<T>) * (size_t)mmax * mmax + sizeof(int) * (size_t)mmax * max_children;
}
constexpr size_t kSmallLdsMax = 160 * 1024 - 1024, kSubLdsMax = 68 * 1024;

// One small front of one frequency, by 256 threads: pull-assembly in LDS from
// the children's contribution blocks, the original entries added, the partial
// LU, the front written to the arena -- one pass over the front in memory,
// where separate assembly, scatter and LU launches wrote it, updated it, read
// it and wrote it again.  A wave assembles whole columns (lane = row), so the
// row's child entry is found once per lane and the column's once per wave, and
// four columns' loads per child are in flight before the first add; an entry
// no child covers reads the child's block origin and is dropped.  Bound by the
// LU's chain of panels at four workgroups per CU (LDS).  1601x401, four
// frequencies: small fronts 4.7 ms in FP64 and 2.3 in FP32, the factorisation
// 38.6 to 34.6 ms and 24.4 to 22.1.
template <typename T, int NR>
__device__ __forceinline__ void small_front(cx<T> *__restrict__ A, const SmallDev &d, const FrontDev &F, int fq,
                                            cx<T> *S, SmallShared &sh) {
    const int m = F.m, mm = m * m, nc = F.nchild, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int *cmap = reinterpret_cast<int *>(S + mm);   // [nchild][m]: child row of each front row, or -1
    const int64_t o0 = d.optr[F.slot], o1 = d.optr[F.slot + 1];
    if (nc > 0) {
        if (tid < nc) {
            const FrontDev C = d.fronts[d.children[F.child_off + tid]];
            sh.cbase[tid] = C.buf_off + C.p + (int64_t)C.p * C.m;   // contribution block origin
            sh.cstride[tid] = C.m;
        }
        for (int c = 0; c < nc; c++) {
            const int io = d.fronts[d.children[F.child_off + c]].inv_off;
            for (int r = tid; r < m; r += 256) cmap[c * m + r] = d.inv[io + r];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const int r = lane + 64 * k;
            if (r >= m) break;
            constexpr int U = 4;
            for (int s0 = wave * U; s0 < m; s0 += 4 * U) {
                cx<T> v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = {T(0), T(0)};
                for (int c = 0; c < nc; c++) {
                    const int a = cmap[c * m + r], st = sh.cstride[c];
                    const cx<T> *B = A + sh.cbase[c];
                    cx<T> w[U];
                    bool ok[U];
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        const int b = s0 + u < m ? cmap[c * m + s0 + u] : -1;
                        ok[u] = a >= 0 && b >= 0;
                        w[u] = B[ok[u] ? a + b * st : 0];
                    }
#pragma unroll
                    for (int u = 0; u < U; u++)
                        if (ok[u]) v[u] = cadd(v[u], w[u]);
                }
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (s0 + u < m) S[r + (s0 + u) * m] = v[u];
            }
        }
    } else {
        for (int e = tid; e < mm; e += 256) S[e] = {T(0), T(0)};
    }
    __syncthreads();
    const cx<double> *V = d.vals + (int64_t)fq * d.vstride;
    for (int64_t e = o0 + tid; e < o1; e += 256) {
        const cx<double> v = V[d.oq[e]];
        cx<T> &t = S[d.ooff[e]];
        t.x += (T)v.x;
        t.y += (T)v.y;
    }
    __syncthreads();
    small_lu_lds<T, NR>(S, m, F.p, sh.rp, d.sing + fq, &sh.pm);
    for (int r = tid; r < F.p; r += 256) d.rowperm[(int64_t)fq * d.n + F.pos0 + r] = sh.rp[r];
    cx<T> *G = A + F.buf_off;
    for (int e = tid; e < mm; e += 256) G[e] = S[e];
}

// grid (the level's small fronts, nfreq)
template <typename T, int NR>
__global__ void __launch_bounds__(256) k_small_front(cx<T> *__restrict__ arena, int64_t fstride, SmallDev d,
                                                     const FrontDev *__restrict__ lvF) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ SmallShared sh;
    const int fq = blockIdx.y;
    const FrontDev F = lvF[blockIdx.x];
    small_front<T, NR>(arena + fq * fstride, d, F, fq, reinterpret_cast<cx<T> *>(smem_raw), sh);
}

// ---------------------------------------------------------------------------
// 3a': the small subtrees in one persistent launch.  A task is one maximal
// small subtree (fronts first..last, children before parents) for one
// frequency; workgroups take tasks from a global counter until none is left.
// A workgroup factors its subtree's fronts in order: each front is assembled
// in LDS from its children's contribution blocks -- written by this same
// workgroup earlier in the task, so a workgroup barrier is all the
// synchronisation there is -- and its original entries, factored there and
// written to the arena.  No workgroup ever waits for another.  Same
// arithmetic, in the same order, as k_small_front.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_subtree_factor(cx<T> *arena, int64_t fstride, SmallDev d,
                                                        const int *__restrict__ root_first,
                                                        const int *__restrict__ root_last, int nroots, int nf,
                                                        int *__restrict__ counter) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ SmallShared sh;
    __shared__ int task;
    const int tid = threadIdx.x, ntask = nroots * nf;
    for (;;) {
        if (tid == 0) task = atomicAdd(counter, 1);
        __syncthreads();
        const int t = task;
        if (t >= ntask) return;
        const int r = t / nf, fq = t - r * nf;
        const int f0 = root_first[r], f1 = root_last[r];
        for (int f = f0; f <= f1; f++) {
            const FrontDev F = d.fronts[f];
            small_front<T, 1>(arena + (int64_t)fq * fstride, d, F, fq, reinterpret_cast<cx<T> *>(smem_raw), sh);
            __syncthreads();   // the parent, later in this loop, reads this block
        }
    }
}

// ---------------------------------------------------------------------------
// 3b: blocked path for large fronts
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) k_panel(cx<T> *__restrict__ arena, int64_t fstride,
                                               const FrontDev *__restrict__ lvF, int *__restrict__ rowperm, int n,
                                               int k0, int nb, int *__restrict__ sing) {
    __shared__ T sb[4];
    __shared__ int si[4];
    const FrontDev F = lvF[blockIdx.x];
    if (F.p <= k0) return;
    const int fq = blockIdx.y;
    int *rp = rowperm + (int64_t)fq * n + F.pos0;
    if (k0 == 0) {
        for (int r = threadIdx.x; r < F.p; r += blockDim.x) rp[r] = r;
        __syncthreads();
    }
    cx<T> *G = arena + fq * fstride + F.buf_off;
    const int m = F.m, p = F.p, kb = min(nb, p - k0), tid = threadIdx.x, bs = blockDim.x;
    for (int j = k0; j < k0 + kb; j++) {
        T best = T(-1);
        int bi = j;
        for (int r = j + tid; r < p; r += bs) better(best, bi, cabs1(G[r + (int64_t)j * m]), r);
        const int pr = block_argmax(best, bi, sb, si);
        if (tid == 0) {
            const int a = rp[j];
            rp[j] = rp[pr];
            rp[pr] = a;
            if (sb[0] == T(0)) atomicOr(sing + fq, 1);
        }
        if (pr != j)
            for (int c = tid; c < m; c += bs) {
                cx<T> t = G[j + (int64_t)c * m];
                G[j + (int64_t)c * m] = G[pr + (int64_t)c * m];
                G[pr + (int64_t)c * m] = t;
            }
        __syncthreads();
        const cx<T> d = crecip(G[j + (int64_t)j * m]);
        for (int r = j + 1 + tid; r < m; r += bs) G[r + (int64_t)j * m] = cmul(G[r + (int64_t)j * m], d);
        __syncthreads();
        const int rows = m - j - 1, ncol = k0 + kb - j - 1;
        for (int e = tid; e < rows * ncol; e += bs) {
            int c = j + 1 + e / rows, r = j + 1 + e % rows;
            G[r + (int64_t)c * m] = cmsub(G[r + (int64_t)c * m], G[r + (int64_t)j * m], G[j + (int64_t)c * m]);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// 3c: blocked path, panel held in registers.  The pivot candidates of a
// 32-column panel are the front's remaining fully-summed rows [k0, p), one row
// per thread, all its panel columns in that thread's registers.  Rows do not
// move while the panel is factored: each thread carries the position its row
// has reached.  The panel goes eight columns at a time.  Per column every wave
// finds its best candidate (DPP maximum and a ballot) and that lane publishes
// value, position, reciprocal and its entries of the eight columns in the
// wave's slot; one barrier later every thread picks the winning wave and updates
// its own eight entries from that slot (slots alternate, so a step has one
// barrier).  After eight columns the pivot rows' other entries are solved in LDS
// (one lane per column) and every remaining row takes one rank-8 update, which
// keeps those columns off the chain of pivot steps; then the row is rotated
// by eight registers, so the code stays short enough for the instruction
// cache.  k_panel_finish applies the panel's permutation to the front's other
// columns.  Bound by the 32-step chain: a panel in LDS with three barriers per
// column took 48 us (270x145, one FP64 frequency, event-timed), this 27; the 69
// panels of 1601x401, four frequencies, 8.5 ms (those above 318 rows in global
// memory) and 2.9.
// ---------------------------------------------------------------------------
template <typename T>
struct PanelSlot {
    T best;
    int pos;
    cx<T> rc;
    cx<T> row[8];
};
template <typename T, int NW>
__global__ void __launch_bounds__(64 * NW) k_panel_reg(cx<T> *__restrict__ arena, int64_t fstride,
                                                       const FrontDev *__restrict__ lvF, int *__restrict__ piv,
                                                       int *__restrict__ rowperm, int n, int k0, int nb,
                                                       int *__restrict__ sing) {
    __shared__ PanelSlot<T> slot[2][NW];
    __shared__ cx<T> Lb[8][8], Ub[8][24];   // the block's pivot rows: multipliers, entries of the later columns
    const FrontDev F = lvF[blockIdx.x];
    if (F.p <= k0) return;
    const int fq = blockIdx.y;
    cx<T> *G = arena + fq * fstride + F.buf_off;
    const int m = F.m, p = F.p, kb = min(nb, p - k0), np = p - k0;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool in = tid < np;
    // (rows past the panel and columns past kb read a valid entry and become zero)
    T ar[32], ai[32];
    static_for<32>([&](auto c) {
        const cx<T> v = G[(k0 + (in ? tid : 0)) + (int64_t)(k0 + (c < kb ? c : 0)) * m];
        ar[c] = in && c < kb ? v.x : T(0);
        ai[c] = in && c < kb ? v.y : T(0);
    });
    int *rp = rowperm + (int64_t)fq * n + F.pos0 + k0;
    const int row = in ? (k0 == 0 ? tid : rp[tid]) : 0;   // (before all swaps) at the thread's position
    int pos = tid;
    bool zero = false;
    const int n8 = (kb + 7) >> 3;
#pragma unroll 1
    for (int b = 0; b < 4; b++) {
        static_for<8>([&](auto jj) {
            const int j = 8 * b + jj;
            if (j < kb) {
                // the thread's candidate (a NaN counts as -1, rows done or outside as -2)
                const T v = fabs(ar[jj]) + fabs(ai[jj]);
                const T best = in && pos >= j ? (v >= T(0) ? v : T(-1)) : T(-2);
                const cx<T> rc = crecip(cx<T>{ar[jj], ai[jj]});
                const T mx = wave_max(best);
                pin(rc);
                const unsigned long long tie = __ballot(best == mx);
                int L = __ffsll((unsigned long long)tie) - 1;
                if (tie & (tie - 1)) {
                    const int lowest = wave_min(best == mx ? pos : 64 * NW);
                    L = __ffsll((unsigned long long)__ballot(best == mx && pos == lowest)) - 1;
                }
                PanelSlot<T> *sl = slot[jj & 1];
                if (lane == L) {
                    PanelSlot<T> &s = sl[wave];
                    s.best = best;
                    s.pos = pos;
                    s.rc = rc;
                    static_for<8>([&](auto c) {
                        if (c > jj) s.row[c] = {ar[c], ai[c]};
                    });
                }
                __syncthreads();
                T wb = sl[0].best;
                int pr = sl[0].pos, ww = 0;
                static_for<NW>([&](auto w) {
                    if (w > 0) {
                        const T ob = sl[w].best;
                        const int op = sl[w].pos;
                        if (ob > wb || (ob == wb && op < pr)) {
                            wb = ob;
                            pr = op;
                            ww = w;
                        }
                    }
                });
                const PanelSlot<T> &s = sl[ww];
                if (tid == 0) piv[(int64_t)fq * n + F.pos0 + k0 + j] = k0 + pr;
                zero |= wb == T(0);
                pos = pos == pr ? j : pos == j ? pr : pos;
                if (in && pos > j) {
                    const cx<T> l = cmul_f(cx<T>{ar[jj], ai[jj]}, s.rc);
                    ar[jj] = l.x;
                    ai[jj] = l.y;
                    static_for<8>([&](auto c) {
                        if (c > jj) {
                            const cx<T> a = cmsub_step(cx<T>{ar[c], ai[c]}, l, s.row[c]);
                            ar[c] = a.x;
                            ai[c] = a.y;
                        }
                    });
                }
            }
        });
        if (b + 1 < n8) {
            // (a block before the last is full: its eight pivots are the positions 8b .. 8b + 7)
            const int t0 = pos - 8 * b;
            const bool piv_row = in && t0 >= 0 && t0 < 8;
            if (piv_row) {
                static_for<8>([&](auto c) { Lb[t0][c] = {ar[c], ai[c]}; });
                static_for<3>([&](auto g) {
                    if (b + g + 1 < n8) static_for<8>([&](auto c) {
                        Ub[t0][8 * g + c] = {ar[8 * g + 8 + c], ai[8 * g + 8 + c]};
                    });
                });
            }
            __syncthreads();
            if (tid < 8 * (n8 - b - 1)) {
                T ur[8], ui[8];
                static_for<8>([&](auto t) {
                    ur[t] = Ub[t][tid].x;
                    ui[t] = Ub[t][tid].y;
                });
                T sr[8], si[8];
                static_for<8>([&](auto t) { sr[t] = si[t] = T(0); });
                if constexpr (NW == 16) __builtin_amdgcn_sched_barrier(0);   // (128 registers a thread there)
                static_for<8>([&](auto s) {
                    ur[s] -= sr[s];
                    ui[s] -= si[s];
                    static_for<7 - s>([&](auto d) {
                        constexpr int t = s + 1 + d;
                        cmadd_to(sr[t], si[t], Lb[t][s], cx<T>{ur[s], ui[s]});
                    });
                    if constexpr (NW == 16) __builtin_amdgcn_sched_barrier(0);
                });
                static_for<8>([&](auto t) { Ub[t][tid] = {ur[t], ui[t]}; });
            }
            __syncthreads();
            static_for<3>([&](auto g) {
                if (b + g + 1 < n8) {
                    if (piv_row)
                        static_for<8>([&](auto c) {
                            ar[8 * g + 8 + c] = Ub[t0][8 * g + c].x;
                            ai[8 * g + 8 + c] = Ub[t0][8 * g + c].y;
                        });
                    else if (in && t0 >= 8)
                        static_for<8>([&](auto cc) {
                            constexpr int c = 8 * g + 8 + cc;
                            T sr = T(0), si = T(0);
                            static_for<8>([&](auto t) { cmadd_to(sr, si, cx<T>{ar[t], ai[t]}, Ub[t][8 * g + cc]); });
                            ar[c] -= sr;
                            ai[c] -= si;
                        });
                }
            });
        }
        // the next eight columns to the front; after four rotations the order is the first one
        T tr[8], ti[8];
        static_for<8>([&](auto c) {
            tr[c] = ar[c];
            ti[c] = ai[c];
        });
        static_for<24>([&](auto c) {
            ar[c] = ar[c + 8];
            ai[c] = ai[c + 8];
        });
        static_for<8>([&](auto c) {
            ar[c + 24] = tr[c];
            ai[c + 24] = ti[c];
        });
    }
    if (zero && tid == 0) atomicOr(sing + fq, 1);
    if (in) rp[pos] = row;   // (every thread read its row before the first barrier)
    if (in)
        static_for<32>([&](auto c) {
            if (c < kb) G[(k0 + pos) + (int64_t)(k0 + c) * m] = {ar[c], ai[c]};
        });
}
// most candidate rows of a panel in registers: one per thread, 512 threads in
// FP64 (128 registers a row, two waves per SIMD) and 1024 in FP32
template <typename T>
constexpr int kPanelRows = sizeof(T) == 8 ? 512 : 1024;

// After a panel's LU: grid (column or row chunks of 64, fronts, nfreq), one
// wave per chunk.  Chunk x < ccols: 64 columns outside the panel, one per lane
// -- the panel's row permutation and, with TRSM, the U12 rows of the columns
// beyond it by forward substitution, the column's 32 rows in registers.  The
// permutation follows from the swap sequence: lane t tracks where row k0 + t
// (t < 32), or the row that step t - 32 pulled in, ends.  A row outside the
// panel only ever receives one of the panel's first rows, so those are moved
// once every lane holds its sources.  The other chunks: 64 contribution rows,
// x U_kk = a.  Replaces 32 dependent swaps in memory and a triangular
// solve with a shuffle reduction per row in a launch of its own: 345 + 325 us
// against 343 per factorisation of 270x145 (FP64, 22 panels; 386 with the U12 rows'
// terms subtracted one by one).  Bound by the dependent rows at two waves per SIMD
// in FP64 and four in FP32 (registers).
template <typename T, bool TRSM>
__global__ void __launch_bounds__(64) k_panel_finish(cx<T> *__restrict__ arena, int64_t fstride,
                                                     const FrontDev *__restrict__ lvF, const int *__restrict__ piv,
                                                     int n, int k0, int nb, int ccols) {
    __shared__ cx<T> U[32][33];
    __shared__ int src[32], dq[32], dr[32];
    const FrontDev F = lvF[blockIdx.y];
    if (F.p <= k0) return;
    const int fq = blockIdx.z;
    cx<T> *G = arena + fq * fstride + F.buf_off;
    const int m = F.m, p = F.p, kb = min(nb, p - k0), tid = threadIdx.x;
    const bool cols = (int)blockIdx.x < ccols;
    if (cols && (int)blockIdx.x * 64 >= m - kb) return;
    if (!cols && p + ((int)blockIdx.x - ccols) * 64 >= m) return;
    // a contribution row's panel entries (columns past kb read column k0 and are
    // not used), then the panel's block, 16 entries per thread, all in flight
    // before the first is used
    T xr[32], xi[32];
    const int i = p + ((int)blockIdx.x - ccols) * 64 + tid;
    if (!cols)
        static_for<32>([&](auto t) {
            const cx<T> v = G[(i < m ? i : p) + (int64_t)(k0 + (t < kb ? t : 0)) * m];
            xr[t] = v.x;
            xi[t] = v.y;
        });
    if (TRSM || !cols) {
        T ur[16], ui[16];
        static_for<16>([&](auto u) {
            const int e = tid + 64 * u, r = e & 31, c = e >> 5;
            const cx<T> v = G[(k0 + (r < kb ? r : 0)) + (int64_t)(k0 + (c < kb ? c : 0)) * m];
            ur[u] = v.x;
            ui[u] = v.y;
        });
        static_for<16>([&](auto u) {
            const int e = tid + 64 * u, r = e & 31, c = e >> 5;
            U[r][c] = {ur[u], ui[u]};
        });
    }
    if (cols) {
        // columns c outside [k0, k0+kb)
        const int pv = (tid & 31) < kb ? piv[(int64_t)fq * n + F.pos0 + k0 + (tid & 31)] : -1;
        const int row = tid < 32 ? (tid < kb ? k0 + tid : -1) : pv;
        int pos = row;
        bool live = tid < 32 ? tid < kb : pv >= k0 + kb;
        for (int j = 0; j < kb; j++) {
            const int s = __builtin_amdgcn_readlane(pv, j), a = k0 + j;
            if (tid - 32 > j && s == row) live = false;   // pulled in before: tracked by that lane
            pos = pos == a ? s : pos == s ? a : pos;
        }
        if (live && pos < k0 + kb) src[pos - k0] = row;
        const bool out = live && pos >= k0 + kb && pos != row;
        const unsigned long long outs = __ballot(out);
        if (out) {
            const int at = __popcll(outs & ((1ull << tid) - 1));
            dq[at] = pos;
            dr[at] = row;
        }
        const int nd = __popcll(outs);
        const bool moved = __ballot(live && pos != row) != 0;
        __syncthreads();
        int c = blockIdx.x * 64 + tid;
        const bool beyond = c >= k0;
        if (beyond) c += kb;
        if (c >= m || (!moved && !(TRSM && beyond))) return;
        cx<T> *col = G + (int64_t)c * m;
        static_for<32>([&](auto t) {
            const cx<T> v = col[t < kb ? src[t] : k0];
            xr[t] = v.x;
            xi[t] = v.y;
        });
        for (int k = 0; k < nd; k += 8) {
            T wr[8], wi[8];
            static_for<8>([&](auto u) {
                const cx<T> v = col[k + u < nd ? dr[k + u] : k0];
                wr[u] = v.x;
                wi[u] = v.y;
            });
            static_for<8>([&](auto u) {
                if (k + u < nd) col[dq[k + u]] = {wr[u], wi[u]};
            });
        }
        if (TRSM && beyond)
            // eight rows at a time: the terms of the rows above them, then their own
            static_for<4>([&](auto b) {
                T sr[8], si[8];
                static_for<8>([&](auto i) { sr[i] = si[i] = T(0); });
                static_for<8 * b>([&](auto t) {
                    static_for<8>([&](auto i) { cmadd_to(sr[i], si[i], U[8 * b + i][t], cx<T>{xr[t], xi[t]}); });
                    // (keeps the scheduler from hoisting the whole block's LDS reads into registers)
                    if constexpr (sizeof(T) == 8 ? t % 2 == 1 : t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                });
                static_for<8>([&](auto i) {
                    constexpr int t = 8 * b + i;
                    xr[t] -= sr[i];
                    xi[t] -= si[i];
                    static_for<7 - i>([&](auto d) {
                        constexpr int q = i + 1 + d;
                        cmadd_to(sr[q], si[q], U[8 * b + q][t], cx<T>{xr[t], xi[t]});
                    });
                });
                __builtin_amdgcn_sched_barrier(0);
            });
        static_for<32>([&](auto t) {
            if (t < kb) col[k0 + t] = {xr[t], xi[t]};
        });
        return;
    }
    // contribution rows: x U_kk = a, U_kk from the factored panel
    __syncthreads();
    const cx<T> rc = crecip(U[tid & 31][tid & 31]);   // lane t: the reciprocal of pivot t
    static_for<32>([&](auto t) {
        if (t < kb) {
            const cx<T> x = cmul_f(cx<T>{xr[t], xi[t]}, readlane_t(rc, t));
            xr[t] = x.x;
            xi[t] = x.y;
            static_for<31 - t>([&](auto d) {
                constexpr int s = t + 1 + d;
                const cx<T> v = cmsub_step(cx<T>{xr[s], xi[s]}, x, U[t][s]);
                xr[s] = v.x;
                xi[s] = v.y;
            });
        }
        if constexpr (sizeof(T) == 8 || t % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    });
    if (i < m)
        static_for<32>([&](auto t) {
            if (t < kb) G[i + (int64_t)(k0 + t) * m] = {xr[t], xi[t]};
        });
}

// U12 rows of the pivot block: rows [k0, k0+kb) of the columns beyond it,
// solved with the unit lower triangle L[k0:k0+kb, k0:k0+kb].  KB = 32: one
// panel, kb = min(32, p - k0), XW = 64 columns per workgroup; KB = 64: two
// panels at once, kb = min(64, p - k0), 32 columns per workgroup, triangle and
// columns in dynamic LDS.  ccap > 0 ends the columns at min(k0 + ccap, p) (the
// second panel's columns only), else at m.  grid (column chunks, fronts, nfreq)
template <typename T, int KB>
__global__ void __launch_bounds__(256) k_trsm_u(cx<T> *__restrict__ arena, int64_t fstride,
                                               const FrontDev *__restrict__ lvF, int k0, int ccap) {
    constexpr int XW = KB == 32 ? 64 : 32, LPC = 256 / XW;   // columns per workgroup, lanes per column
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T>(*Ls)[KB + 1] = reinterpret_cast<cx<T>(*)[KB + 1]>(smem_raw);
    cx<T>(*Xs)[XW + 1] = reinterpret_cast<cx<T>(*)[XW + 1]>(smem_raw + sizeof(cx<T>) * KB * (KB + 1));
    const FrontDev F = lvF[blockIdx.y];
    if (F.p <= k0) return;
    const int m = F.m, kb = min(KB, F.p - k0), cend = ccap > 0 ? min(k0 + ccap, F.p) : m;
    const int c0 = k0 + kb + blockIdx.x * XW;
    if (c0 >= cend) return;
    cx<T> *G = arena + blockIdx.z * fstride + F.buf_off;
    const int tid = threadIdx.x;
    // unrolled so that a batch of loads is in flight at once
#pragma unroll 4
    for (int e = tid; e < kb * kb; e += 256) {
        int i = e % kb, t = e / kb;
        Ls[i][t] = G[(k0 + i) + (int64_t)(k0 + t) * m];
    }
    // (unconditional: columns past the end read column c0 and are zeroed when stored)
    {
        constexpr int PER = KB * XW / 256;
        cx<T> v[PER];
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int e = tid + 256 * u, i = e % KB, c = e / KB, col = c0 + c;
            v[u] = G[(k0 + (i < kb ? i : 0)) + (int64_t)(col < cend ? col : c0) * m];
        }
#pragma unroll
        for (int u = 0; u < PER; u++) {
            const int e = tid + 256 * u, i = e % KB, c = e / KB, col = c0 + c;
            if (i < kb) Xs[i][c] = col < cend ? v[u] : cx<T>{T(0), T(0)};
        }
    }
    __syncthreads();
    {
        // LPC adjacent lanes (one wave) per column: each sums every LPC-th term
        // of row i's dot product, xor-shuffles add them, lane 0 of the group
        // stores the entry the next rows read
        const int c = tid / LPC, part = tid % LPC;
        for (int i = 1; i < kb; i++) {
            cx<T> acc = {T(0), T(0)};
            for (int t = part; t < i; t += LPC) acc = cmsub(acc, Ls[i][t], Xs[t][c]);
#pragma unroll
            for (int o = 1; o < LPC; o <<= 1) {
                acc.x += __shfl_xor(acc.x, o);
                acc.y += __shfl_xor(acc.y, o);
            }
            if (part == 0) Xs[i][c] = cadd(Xs[i][c], acc);
        }
    }
    __syncthreads();
    for (int e = tid; e < kb * XW; e += 256) {
        int i = e % kb, c = e / kb, col = c0 + c;
        if (col < cend) G[(k0 + i) + (int64_t)col * m] = Xs[i][c];
    }
}
template <typename T, int KB>
constexpr size_t trsm_lds() {
    return sizeof(cx<T>) * KB * (KB + 1) + sizeof(cx<T>) * KB * ((KB == 32 ? 64 : 32) + 1);
}

// ---------------------------------------------------------------------------
// trailing update C -= A*B on MFMA, four real products per complex product,
// 64x64 tiles.  The product's depth is the front's next min(depth, p - k0)
// pivot columns (depth 32: one panel; 64: two panels), taken KB at a time
// through the same LDS with the next chunk's loads in flight during a chunk's
// products, so C is read and written once per `depth` pivots.  The product is
// summed from zero and subtracted from C once: accumulated onto C every step
// rounds at the size of C, which the terms are far below (FP32 factors'
// solutions 1.2 to 1.5 times further off: 201x101, 3.8e-6 against 5.5e-6, the
// geometric mean of 12 matrices).  C is loaded under the last chunk's products,
// when the prefetch registers are free.  The operands are staged as complex
// entries, A by columns and B by its rows, each with the lanes that write it
// along the contiguous direction (staging B by columns put 32 lanes on one bank).
// The updated block starts at row and column k0 + that depth; ccap > 0 ends
// its columns at min(k0 + ccap, p) (the thin update of the second panel's
// columns), else at m.  Bound by each tile's load-stage-product chain at three
// workgroups per CU.  Its share of a factorisation of 1601x401, four frequencies:
// 9.35 ms in FP64 (31 TF/s) and 5.35 in FP32, 9.21 and 5.21 with C in the
// accumulators.  Chunks of 32 columns in FP32: 17.4 ms a factorisation against 17.2.
// Each XCD takes one contiguous range of the tiles (of all frequencies), whose
// operands it reads into its own L2 once: 403x207, two frequencies 555 -> 530 us
// FP64, 421 -> 395 FP32; 1601x401, four, 9.27 -> 9.21 ms and 6.55 -> 6.40.
// 4 waves in 2x2, each wave 32x32 = 2x2 blocks of 16x16.
// MFMA 16x16x4 operand layout: A lane l -> (row l%16, k l/16), B lane l ->
// (k l/16, col l%16).  Accumulator register v of lane l holds column l%16 and
// row 4*(l/16)+v for f32, but row 4*v+l/16 for f64.
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_gemm_update(cx<T> *__restrict__ arena, int64_t fstride, const FrontDev *__restrict__ lvF,
              const TileDev *__restrict__ tiles, int k0, int depth, int ccap) {
    constexpr int KB = 16, PER = KB * 64 / 256;
    __shared__ cx<T> As[KB][64], Bs[64][KB + 1];
    const int item = xcd_range_item(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int freq = item / gridDim.x;
    const TileDev tl = tiles[item - freq * gridDim.x];
    const FrontDev F = lvF[tl.front];
    const int m = F.m, kd = min(depth, F.p - k0);
    const int base = k0 + kd, cend = ccap > 0 ? min(k0 + ccap, F.p) : m;
    const int r0 = base + tl.ti * 64, c0 = base + tl.tj * 64;
    cx<T> *G = arena + freq * fstride + F.buf_off;
    const int tid = threadIdx.x;
    const int lane = tid & 63, w = tid >> 6, wr = (w >> 1) * 32, wc = (w & 1) * 32;
    const int lr = lane & 15, lk = lane >> 4;
    // addresses: a uniform base per operand and 32-bit byte offsets within 64 columns of it
    const char *Ga = reinterpret_cast<const char *>(G + (int64_t)k0 * m + r0);   // column k of A at k m
    char *Gc = reinterpret_cast<char *>(G + (int64_t)c0 * m);                    // column j of B and C at j m
    auto at = [](const char *base, int e) {
        return *reinterpret_cast<const cx<T> *>(base + (unsigned)e * (unsigned)sizeof(cx<T>));
    };
    // a chunk's operands, loaded unconditionally (entries outside read the
    // operand's first and are zeroed when staged) so that they stay in flight
    T ax[PER], ay[PER], bx[PER], by[PER];
    auto load_chunk = [&](int kc) {
        const int kb = min(KB, kd - kc);
        static_for<PER>([&](auto u) {
            const int e = tid + 256 * u, i = e & 63, k = e >> 6;
            const cx<T> v = at(Ga, k < kb && r0 + i < m ? i + (kc + k) * m : 0);
            ax[u] = v.x;
            ay[u] = v.y;
        });
        static_for<PER>([&](auto u) {
            const int e = tid + 256 * u, k = e % KB, j = e / KB;
            const cx<T> v = at(Gc, k < kb && c0 + j < cend ? (k0 + kc + k) + j * m : 0);
            bx[u] = v.x;
            by[u] = v.y;
        });
    };
    auto stage_chunk = [&](int kc) {
        const int kb = min(KB, kd - kc);
        static_for<PER>([&](auto u) {
            const int e = tid + 256 * u, i = e & 63, ka = e >> 6, kb2 = e % KB, j = e / KB;
            const bool ina = ka < kb && r0 + i < m, inb = kb2 < kb && c0 + j < cend;
            As[ka][i] = {ina ? ax[u] : T(0), ina ? ay[u] : T(0)};
            Bs[j][kb2] = {inb ? bx[u] : T(0), inb ? by[u] : T(0)};
        });
    };
    typename mfma_t<T>::acc cr[2][2], ci[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            cr[a][b] = typename mfma_t<T>::acc{0, 0, 0, 0};
            ci[a][b] = cr[a][b];
        }
    auto products = [&](int kc) {
        const int kend = (min(KB, kd - kc) + 3) & ~3;
#pragma unroll 1
        for (int kk = 0; kk < kend; kk += 4) {
            const int k = kk + lk;
            cx<T> av[2], bv[2];
#pragma unroll
            for (int a = 0; a < 2; a++) av[a] = As[k][wr + a * 16 + lr];
#pragma unroll
            for (int b = 0; b < 2; b++) bv[b] = Bs[wc + b * 16 + lr][k];
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int a = 0; a < 2; a++) cmma<T>(av[a].x, av[a].y, bv[b].x, bv[b].y, cr[a][b], ci[a][b]);
        }
    };
    load_chunk(0);
    int kc = 0;
    for (; kc + KB < kd; kc += KB) {
        stage_chunk(kc);
        __syncthreads();
        load_chunk(kc + KB);   // in flight during this chunk's products
        products(kc);
        __syncthreads();   // every wave is done with this chunk
    }
    stage_chunk(kc);
    __syncthreads();
    // the tile of C, in flight during the last chunk's products
    T gx[2][2][4], gy[2][2][4];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = r0 + wr + a * 16 + mfma_t<T>::row(lk, v), j = wc + b * 16 + lr;
                const cx<T> c = at(Gc, row < m && c0 + j < cend ? row + j * m : 0);
                gx[a][b][v] = c.x;
                gy[a][b][v] = c.y;
            }
    products(kc);
    int ms = m;
    asm("" : "+s"(ms));   // (the stores' offsets computed anew rather than kept through the products)
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int row = r0 + wr + a * 16 + mfma_t<T>::row(lk, v), j = wc + b * 16 + lr;
                if (row < ms && c0 + j < cend)
                    *reinterpret_cast<cx<T> *>(Gc + (unsigned)(row + j * ms) * (unsigned)sizeof(cx<T>)) = {
                        gx[a][b][v] - cr[a][b][v], gy[a][b][v] - ci[a][b][v]};
            }
}

// zero-pivot flags cleared by a kernel rather than a memset node, so the
// factorisation can be captured into a graph and replayed
__global__ void k_clear_flags(int *__restrict__ flags, int count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) flags[i] = 0;
}

// ---------------------------------------------------------------------------
// gather sources after pivoting, per frequency: row i of a front takes the
// sources of its row rowperm(i) (pivot rows) or i (contribution rows), so a
// forward sweep reads one table entry per row.  grid (row chunks, nfreq)
// ---------------------------------------------------------------------------
__global__ void k_gsrc(const FrontDev *__restrict__ fronts, int nfronts, const int *__restrict__ rowperm, int n,
                       const int *__restrict__ gsrc_id, int64_t fv_rows, int *__restrict__ gsrc) {
    const int f = blockIdx.x;
    if (f >= nfronts) return;
    const FrontDev F = fronts[f];
    const int *rp = rowperm + (int64_t)blockIdx.y * n + F.pos0;
    int *out = gsrc + ((int64_t)blockIdx.y * fv_rows + F.fv_off) * 3;
    const int *in = gsrc_id + F.fv_off * 3;
    for (int i = threadIdx.x; i < F.m; i += blockDim.x) {
        const int s = i < F.p ? rp[i] : i;
        out[3 * i] = in[3 * s];
        out[3 * i + 1] = in[3 * s + 1];
        out[3 * i + 2] = in[3 * s + 2];
    }
}

// ---------------------------------------------------------------------------
// solve format: every 32x32 diagonal block of a front's pivot block is
// replaced in place by its inverses -- strictly lower part: inverse of the
// unit lower block of L11, upper part with diagonal: inverse of the upper
// block of U11 -- so that the substitutions apply each diagonal block as one
// small dense product on the matrix cores instead of a 32-step dependent
// chain.  Fronts of single-block levels (p <= 32) go one step further: L21 is
// replaced by L21 inv(L11) and U12 by inv(U11) U12, which turns each of their
// forward and backward substitutions -- for M as for M^T -- into one product
// with no dependent phase:  [y; w2 - L21 y] = [inv(L11); L21 inv(L11)] w1  and
// x1 = [inv(U11), -inv(U11) U12] [y1; x2].  Computed in FP64 for both factor
// precisions (the block is staged in the factor precision, exact in FP64).
// One workgroup per front, grid (fronts, nfreq); every global load of the
// front is issued a phase ahead of its use (the next block, or the rows below,
// while a block is inverted; the columns beyond, during the rows' products).
// Bound by each workgroup's serial path: three per compute unit (registers
// held to that, LDS allows no more) take 2.7 ms at 1601x401, four FP64
// frequencies, where two took 3.6.
// ---------------------------------------------------------------------------
// every lane takes the value that lane q of its group of four holds (DPP quad permute)
__device__ __forceinline__ int quad_bcast_i(int v, int q) {
    switch (q) {
    case 0: return __builtin_amdgcn_mov_dpp(v, 0x00, 0xF, 0xF, false);
    case 1: return __builtin_amdgcn_mov_dpp(v, 0x55, 0xF, 0xF, false);
    case 2: return __builtin_amdgcn_mov_dpp(v, 0xAA, 0xF, 0xF, false);
    default: return __builtin_amdgcn_mov_dpp(v, 0xFF, 0xF, 0xF, false);
    }
}
__device__ __forceinline__ double quad_bcast(double d, int q) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(d);
    const unsigned lo = (unsigned)quad_bcast_i((int)(unsigned)b, q);
    const unsigned hi = (unsigned)quad_bcast_i((int)(unsigned)(b >> 32), q);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ cx<double> quad_bcast(cx<double> v, int q) {
    return {quad_bcast(v.x, q), quad_bcast(v.y, q)};
}
__device__ __forceinline__ double readlane_d(double d, int l) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(d);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <typename T>
__device__ __forceinline__ cx<double> c64(cx<T> v) {
    return {(double)v.x, (double)v.y};
}
// c + a b with every fused multiply-add written out
__device__ __forceinline__ cx<double> cmac_f(cx<double> c, cx<double> a, cx<double> b) {
    return {fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y))};
}

// Inverses of the NB x NB block D (NB = 8, 16, 24 or 32, the identity beyond the
// block's order): the unit lower inverse into LI and the upper inverse into UI,
// each complete with its zeros (LI with its unit diagonal).  Waves 0-1 build
// LI, waves 2-3 UI at the same time; four lanes per column j, lane part holding
// rows 4k + part in registers.  Right-looking: at step t the lane holding row
// t hands x_t to its group of four (DPP), and every lane updates its rows below
// t (above t for UI) -- no LDS round trip and no barrier inside the chain.
template <typename T, int NB>
__device__ __forceinline__ void tri_inverses(const cx<T> (*D)[33], cx<double> (*LI)[33], cx<double> (*UI)[33],
                                             int tid) {
    constexpr int NK = NB / 4;
    const int j = (tid & 127) >> 2, part = tid & 3;
    cx<double> acc[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) acc[k] = {4 * k + part == j ? 1.0 : 0.0, 0.0};
    // column t of the block for the lane's rows, read a step ahead; the
    // scheduling barrier per step keeps the unrolled chain from hoisting every
    // LDS read at once
    cx<T> an[NK];
    if (tid < 128) {
        // column j of inv(L): x_t final once rows < t are applied; rows i > t -= L[i][t] x_t
#pragma unroll
        for (int k = 0; k < NK; k++) an[k] = D[4 * k + part][0];
#pragma unroll
        for (int t = 0; t < NB - 1; t++) {
            const int q = t & 3, kt = t >> 2;
            cx<T> ac[NK];
#pragma unroll
            for (int k = kt; k < NK; k++) ac[k] = an[k];
            if (t + 1 < NB - 1)
#pragma unroll
                for (int k = (t + 1) >> 2; k < NK; k++) an[k] = D[4 * k + part][t + 1];
            const cx<double> x = quad_bcast(acc[kt], q);
#pragma unroll
            for (int k = kt; k < NK; k++) {
                cx<double> a = c64(ac[k]);
                if (k == kt && part <= q) a = {0.0, 0.0};
                acc[k] = cmsub_f(acc[k], a, x);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (j < NB)
#pragma unroll
            for (int k = 0; k < NK; k++) LI[4 * k + part][j] = acc[k];
    } else {
        // column j of inv(U): x_t = acc_t / U[t][t] once rows > t are applied; rows i < t -= U[i][t] x_t
        // lane l holds 1 / U[l % 32][l % 32]; step t reads lane t's (readlane)
        const int dl = tid & 31;
        const cx<double> rl = crecip(c64(D[dl][dl]));
#pragma unroll
        for (int k = 0; k < NK; k++) an[k] = D[4 * k + part][NB - 1];
#pragma unroll
        for (int t = NB - 1; t >= 0; t--) {
            const int q = t & 3, kt = t >> 2;
            cx<T> ac[NK];
#pragma unroll
            for (int k = 0; k <= kt; k++) ac[k] = an[k];
            if (t > 0)
#pragma unroll
                for (int k = 0; k <= (t - 1) >> 2; k++) an[k] = D[4 * k + part][t - 1];
            const cx<double> x = quad_bcast(cmul(acc[kt], cx<double>{readlane_d(rl.x, t), readlane_d(rl.y, t)}), q);
            if (part == q) acc[kt] = x;
#pragma unroll
            for (int k = 0; k <= kt; k++) {
                cx<double> a = c64(ac[k]);
                if (k == kt && part >= q) a = {0.0, 0.0};
                acc[k] = cmsub_f(acc[k], a, x);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (j < NB)
#pragma unroll
            for (int k = 0; k < NK; k++) UI[4 * k + part][j] = acc[k];
    }
}

// L21 <- L21 inv(L11) on a chunk of 32 rows staged as V[i][s] (zero beyond the
// front), on the matrix cores: wave w computes one 16 x 16 tile of the
// transposed product (rows t: columns of L21, columns i: its rows), so each
// accumulator register stores 16 consecutive rows of one column of G.  K runs
// from the tile's first column (inv(L11) is zero above its diagonal).
template <typename T>
__device__ __forceinline__ void l21_mfma(const cx<T> (*V)[33], const cx<double> (*LI)[33], cx<T> *G, int m, int p,
                                         int r0, int wave, int lane) {
    const int ntt = (p + 15) >> 4, lr = lane & 15, lk = lane >> 4;
    if (wave >= 2 * ntt) return;
    const int t0 = (wave % ntt) * 16, i0 = (wave / ntt) * 16;
    if (r0 + i0 >= m) return;
    d4v cr = {0.0, 0.0, 0.0, 0.0}, ci = cr;
    const int kend = (p + 3) & ~3;
    for (int k0 = t0; k0 < kend; k0 += 4) {
        const cx<double> a = LI[k0 + lk][t0 + lr];       // A[t][s] = inv(L11)[s][t]
        const cx<double> b = c64(V[i0 + lr][k0 + lk]);   // B[s][i] = L21[i][s]
        cmma<double>(a.x, a.y, b.x, b.y, cr, ci);
    }
    const int i = i0 + lr;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int t = t0 + mfma_t<double>::row(lk, v);
        if (t < p && r0 + i < m) G[r0 + i + (int64_t)t * m] = {(T)cr[v], (T)ci[v]};
    }
}

// U12 <- inv(U11) U12 on a chunk of 32 columns staged as V[c][s]: wave w
// computes one 16 x 16 tile of the transposed product (rows c: columns of U12,
// columns i: its rows); K runs from the tile's first row (inv(U11) is zero
// below its diagonal).
template <typename T>
__device__ __forceinline__ void u12_mfma(const cx<T> (*V)[33], const cx<double> (*UI)[33], cx<T> *G, int m, int p,
                                         int c0, int wave, int lane) {
    const int nit = (p + 15) >> 4, lr = lane & 15, lk = lane >> 4;
    if (wave >= 2 * nit) return;
    const int i0 = (wave % nit) * 16, cc0 = (wave / nit) * 16;
    if (c0 + cc0 >= m) return;
    d4v cr = {0.0, 0.0, 0.0, 0.0}, ci = cr;
    const int kend = (p + 3) & ~3;
    for (int k0 = i0; k0 < kend; k0 += 4) {
        const cx<double> a = c64(V[cc0 + lr][k0 + lk]);   // A[c][s] = U12[s][c]
        const cx<double> b = UI[i0 + lr][k0 + lk];        // B[s][i] = inv(U11)[i][s]
        cmma<double>(a.x, a.y, b.x, b.y, cr, ci);
    }
    const int i = i0 + lr;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int c = c0 + cc0 + mfma_t<double>::row(lk, v);
        if (i < p && c < m) G[i + (int64_t)c * m] = {(T)cr[v], (T)ci[v]};
    }
}

template <typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
k_diag_inv(cx<T> *__restrict__ arena, int64_t fstride, const FrontDev *__restrict__ fronts,
           const int *__restrict__ lv_single) {
    __shared__ cx<T> D[32][33];   // the block being inverted, then the rectangles' chunks
    __shared__ cx<double> LI[32][33], UI[32][33];
    const FrontDev F = fronts[blockIdx.x];
    cx<T> *G = arena + blockIdx.y * fstride + F.buf_off;
    const int m = F.m, p = F.p, tid = threadIdx.x;
    if (p == 0) return;
    const bool single = lv_single[F.level] && p <= 32;
    // chunk loads: four entries per thread, entry e = tid + 256u at (e % 32,
    // e / 32) of a 32 x 32 tile; out-of-range entries read G[0] and are
    // replaced when staged (unconditional loads stay in flight together)
    cx<T> rb[4], rl[4], ru[4];
    auto load_block = [&](int b0) {
        const int kb = min(32, p - b0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, i = e & 31, t = e >> 5;
            rb[u] = G[i < kb && t < kb ? b0 + i + (int64_t)(b0 + t) * m : 0];
        }
    };
    auto load_l21 = [&](int r0) {   // rows r0 + i, columns s < p
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, i = e & 31, s = e >> 5;
            rl[u] = G[r0 + i < m && s < p ? r0 + i + (int64_t)s * m : 0];
        }
    };
    auto load_u12 = [&](int c0) {   // rows s < p, columns c0 + c
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, s = e & 31, c = e >> 5;
            ru[u] = G[s < p && c0 + c < m ? s + (int64_t)(c0 + c) * m : 0];
        }
    };
    load_block(0);
    if (single && p < m) load_l21(p);
    for (int b0 = 0; b0 < p; b0 += 32) {
        const int kb = min(32, p - b0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, i = e & 31, t = e >> 5;
            D[i][t] = i < kb && t < kb ? rb[u] : cx<T>{i == t ? T(1) : T(0), T(0)};
        }
        __syncthreads();
        if (b0 + 32 < p) load_block(b0 + 32);
        // the block's order rounded up to 8 (the padding is the identity)
        if (kb <= 8) tri_inverses<T, 8>(D, LI, UI, tid);
        else if (kb <= 16) tri_inverses<T, 16>(D, LI, UI, tid);
        else if (kb <= 24) tri_inverses<T, 24>(D, LI, UI, tid);
        else tri_inverses<T, 32>(D, LI, UI, tid);
        __syncthreads();
        for (int e = tid; e < kb * kb; e += 256) {
            const int i = e % kb, t = e / kb;
            const cx<double> v = i > t ? LI[i][t] : UI[i][t];
            G[b0 + i + (int64_t)(b0 + t) * m] = {(T)v.x, (T)v.y};
        }
    }
    if (!single) return;
    const int wave = tid >> 6, lane = tid & 63;
    if (p < m) load_u12(p);   // in flight during the L21 products
    for (int r0 = p; r0 < m; r0 += 32) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, i = e & 31, s = e >> 5;
            D[i][s] = r0 + i < m && s < p ? rl[u] : cx<T>{T(0), T(0)};
        }
        __syncthreads();
        if (r0 + 32 < m) load_l21(r0 + 32);
        l21_mfma<T>(D, LI, G, m, p, r0, wave, lane);
        __syncthreads();
    }
    for (int c0 = p; c0 < m; c0 += 32) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u, s = e & 31, c = e >> 5;
            D[c][s] = s < p && c0 + c < m ? ru[u] : cx<T>{T(0), T(0)};
        }
        __syncthreads();
        if (c0 + 32 < m) load_u12(c0 + 32);
        u12_mfma<T>(D, UI, G, m, p, c0, wave, lane);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// driver
// ---------------------------------------------------------------------------
namespace {
size_t g_panel_lds_cap = 0;   // 0: none
// The default: the small fronts level by level, and (g_deep_min_m < 0) two panels
// per step only where the trailing update is bound by its passes over memory.
// The persistent subtree launch is a serial chain of fronts per workgroup:
// 61x41, one FP64 frequency, 0.91 ms per factorisation against 0.52 level by
// level; 1601x401, four frequencies, 43.0 against 42.3.  Two panels per step
// trade a pass over the trailing block for three more launches and a 64-row
// triangular solve.  Two panels on every level / one / by the rule, ms: FP64
// 270x145 1.67 / 1.32 / 1.31, 1601x401 with four frequencies 28.5 / 25.1 / 25.1,
// 2001x2001 143.5 / 144.2 / 144.2, 3001x3001 407 / 423 / 423; FP32 1601x401 with
// four 17.8 / 17.3 / 17.1, with eight 31.2 / 31.4 / 30.5, 801x801 with four 20.2 /
// 20.0 / 19.7, 2401x801 with four 62.1 / 66.3 / 62.4, 2001x2001 72.9 / 75.7 / 71.9.
// FP32 gains from fronts of order 384 once the level's tiles fill the device
// several times over; FP64 only on grids of millions of points.
int g_persistent = 0;    // small subtrees in one persistent launch
int g_deep_min_m = -1;   // blocked levels with a front of order >= this take the two-panel schedule
constexpr int kDeepFp32M = 384, kDeepFp32Tiles = 6 * 256;
template <typename T>
bool deep_level(const LevelPlan &L, const DevPlan::DeepStep &first, int nf) {
    if (g_deep_min_m >= 0) return L.large_mmax >= g_deep_min_m;
    return sizeof(T) == 4 && L.large_mmax >= kDeepFp32M && (int64_t)first.deep_cnt * nf >= kDeepFp32Tiles;
}
}
void set_factor_tuning(int panel_lds_cap, int persistent, int deep_min_m) {
    g_panel_lds_cap = panel_lds_cap > 0 ? (size_t)panel_lds_cap : 0;
    g_persistent = persistent != 0;
    g_deep_min_m = deep_min_m;
}

template <typename T>
void factor_numeric(const DevPlan &dp, Factors<T> &F, const cx<double> *vals, int64_t vstride, hipStream_t st) {
    const Plan &pl = *dp.host;
    const int nf = F.nfreq;
    F.vinv_ready = false;   // the single-vector path's inverse squares follow the new factors
    hipLaunchKernelGGL(k_clear_flags, dim3((nf + 63) / 64), dim3(64), 0, st, F.sing, nf);
    static bool attr_set = false;
    if (!attr_set) {
        // fronts of up to 90x90 complex doubles live in LDS (gfx950: 160 KB per CU)
        for (const void *k : {reinterpret_cast<const void *>(&k_small_front<double, 1>),
                              reinterpret_cast<const void *>(&k_small_front<double, 2>),
                              reinterpret_cast<const void *>(&k_small_front<float, 1>),
                              reinterpret_cast<const void *>(&k_small_front<float, 2>)})
            GFDFD_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLdsMax));
        GFDFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_subtree_factor<double>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSubLdsMax));
        GFDFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_subtree_factor<float>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSubLdsMax));
        GFDFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_trsm_u<double, 64>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)trsm_lds<double, 64>()));
        GFDFD_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_trsm_u<float, 64>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)trsm_lds<float, 64>()));
        attr_set = true;
    }
    const bool sub = g_persistent && dp.nroots > 0 && F.sched;
    const SmallDev sd{dp.fronts, dp.children, dp.inv, dp.small_optr, dp.small_oq, dp.small_ooff,
                      vals,      vstride,     F.rowperm, pl.n,     F.sing};
    if (dp.max_children > kAsmMaxChildren) throw std::logic_error("front assembly: too many children");
    if (sub) {
        const int ntask = dp.nroots * nf;
        const size_t lds = small_front_lds<T>(dp.sub_mmax, dp.max_children);
        if (lds > kSubLdsMax) throw std::logic_error("subtree front exceeds its LDS");
        hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(64), 0, st, F.sched, 1);
        ProfScope ps(K_SUBTREE, st, dp.sub_flops * nf, 3.0 * dp.sub_elems * sizeof(cx<T>) * nf);
        // every workgroup takes tasks until none is left; a few per CU keep the CUs busy
        const int grid = std::min(ntask, 256 * 8);
        hipLaunchKernelGGL(k_subtree_factor<T>, dim3(grid), dim3(256), lds, st, F.arena, F.fstride, sd, dp.root_first,
                           dp.root_last, dp.nroots, nf, F.sched);
    }
    for (int l = 0; l < pl.nlevels; l++) {
        const LevelPlan &L = pl.levels[l];
        const DevPlan::LevelCounts &cnt = dp.counts[l];
        const double es = sizeof(cx<T>) * (double)nf;
        // the small fronts: every one of the level, or those outside the subtrees
        const int n_small = sub ? dp.n_small_rest[l] : dp.n_small[l];
        if (n_small > 0) {
            const int smm = sub ? dp.small_mmax_rest[l] : L.small_mmax;
            const size_t lds = small_front_lds<T>(smm, dp.max_children);
            if (lds > kSmallLdsMax) throw std::logic_error("small front exceeds LDS");
            ProfScope ps(K_SMALL_LU, st, (sub ? dp.small_rest_flops[l] : cnt.small_flops) * nf,
                         (sub ? dp.small_rest_elems[l] : cnt.small_elems) * es);
            const FrontDev *list = sub ? dp.lv_small_rest[l] : dp.lv_fr[l];
            if (smm <= 64)
                hipLaunchKernelGGL((k_small_front<T, 1>), dim3(n_small, nf), dim3(256), lds, st, F.arena, F.fstride,
                                   sd, list);
            else
                hipLaunchKernelGGL((k_small_front<T, 2>), dim3(n_small, nf), dim3(256), lds, st, F.arena, F.fstride,
                                   sd, list);
        }
        const FrontDev *lvL = dp.lv_fr[l] + dp.n_small[l];   // the level's blocked fronts
        if (dp.n_large[l] > 0) {
            ProfScope ps(K_FRONT_ASSEMBLE, st, 0.0, dp.asm_elems_large[l] * es);
            // about 16 entries per thread, in whole columns
            const int ncols = std::max(1, 4096 / L.large_mmax);
            const size_t lds = sizeof(int) * (size_t)dp.max_children * L.large_mmax;
            if (lds > 64 * 1024) throw std::logic_error("front assembly: too large a front for the row maps");
            hipLaunchKernelGGL(k_front_assemble<T>, dim3(dp.n_large[l], (L.large_mmax + ncols - 1) / ncols, nf),
                               dim3(256), lds, st, F.arena, F.fstride, lvL, dp.fronts, dp.children, dp.inv,
                               dp.large_cptr, dp.large_oq, dp.large_ooff, vals, vstride, ncols);
        }
        if (dp.n_large[l] > 0) {
            const size_t lds32 = trsm_lds<T, 32>(), lds64 = trsm_lds<T, 64>();
            // one 32-column panel of every blocked front of the level: its LU (in
            // registers, or in global memory when the candidate rows are too many
            // or exceed the caller's cap), the row permutation on the other columns
            // with the contribution rows and, with trsm, the U12 rows
            auto panel = [&](int k0, double flops, bool trsm, double trsm_flops) {
                const int rows = L.large_pmax - k0;
                const size_t plds = (size_t)rows * pl.nb * sizeof(cx<T>);
                const int ccols = (L.large_mmax + 63) / 64;   // m - kb columns of any front fit
                const int crows = (L.large_mmax + 63) / 64;
                if (rows <= kPanelRows<T> && (!g_panel_lds_cap || plds <= g_panel_lds_cap)) {
                    {
                        ProfScope ps(K_PANEL, st, flops * nf, 0.0);
                        const dim3 g(dp.n_large[l], nf);
#define PANEL(NW)                                                                                                   \
    hipLaunchKernelGGL((k_panel_reg<T, NW>), g, dim3(64 * NW), 0, st, F.arena, F.fstride, lvL, F.piv, F.rowperm,     \
                       pl.n, k0, pl.nb, F.sing)
                        if (rows <= 64) PANEL(1);
                        else if (rows <= 128) PANEL(2);
                        else if (rows <= 256) PANEL(4);
                        else if (rows <= 512) PANEL(8);
                        else if constexpr (sizeof(T) == 4) PANEL(16);
#undef PANEL
                    }
                    ProfScope ps(K_PANEL_APPLY, st, trsm ? trsm_flops * nf : 0.0, 0.0);
                    if (trsm)
                        hipLaunchKernelGGL((k_panel_finish<T, true>), dim3(ccols + crows, dp.n_large[l], nf), dim3(64),
                                           0, st, F.arena, F.fstride, lvL, F.piv, pl.n, k0,
                                           pl.nb, ccols);
                    else
                        hipLaunchKernelGGL((k_panel_finish<T, false>), dim3(ccols + crows, dp.n_large[l], nf),
                                           dim3(64), 0, st, F.arena, F.fstride, lvL, F.piv, pl.n,
                                           k0, pl.nb, ccols);
                } else {
                    {
                        ProfScope ps(K_PANEL, st, flops * nf, 0.0);
                        hipLaunchKernelGGL(k_panel<T>, dim3(dp.n_large[l], nf), dim3(256), 0, st, F.arena, F.fstride,
                                           lvL, F.rowperm, pl.n, k0, pl.nb, F.sing);
                    }
                    if (trsm) {
                        ProfScope ps(K_TRSM, st, trsm_flops * nf, 0.0);
                        hipLaunchKernelGGL((k_trsm_u<T, 32>), dim3(ccols, dp.n_large[l], nf), dim3(256), lds32, st,
                                           F.arena, F.fstride, lvL, k0, 0);
                    }
                }
            };
            auto gemm = [&](int64_t off, int cnt, int k0, int depth, int ccap, double flops, double elems) {
                if (cnt <= 0) return;
                ProfScope ps(K_GEMM, st, flops * nf, elems * es);
                hipLaunchKernelGGL(k_gemm_update<T>, dim3(cnt, nf), dim3(256), 0, st, F.arena, F.fstride, lvL,
                                   dp.tiles + off, k0, depth, ccap);
            };
            if (deep_level<T>(L, dp.deep_steps[l][0], nf)) {
                // two panels per block: panel 1; its U rows and update on panel 2's
                // columns only; panel 2; the U rows of both panels (one 64-row
                // solve) and one depth-64 trailing update, so the trailing block
                // is read and written once per 64 pivots.  Panel 2's row swaps
                // reach the not yet updated columns and panel 1's L columns alike,
                // which keeps the deferred update consistent.
                int bi = 0;
                for (int b0 = 0; b0 < L.large_pmax; b0 += 64, bi++) {
                    const auto &d = dp.deep_steps[l][bi];
                    panel(b0, d.panel1_flops, false, 0.0);
                    if (d.thin_cnt > 0) {
                        {
                            ProfScope ps(K_TRSM, st, d.trsm_thin_flops * nf, 0.0);
                            hipLaunchKernelGGL((k_trsm_u<T, 32>), dim3(1, dp.n_large[l], nf), dim3(256),
                                               lds32, st, F.arena, F.fstride, lvL,
                                               b0, 64);
                        }
                        gemm(d.thin_off, d.thin_cnt, b0, 32, 64, d.thin_flops, d.thin_elems);
                        panel(b0 + 32, d.panel2_flops, false, 0.0);
                    }
                    {
                        ProfScope ps(K_TRSM, st, d.trsm_deep_flops * nf, 0.0);
                        const int colchunks = (L.large_mmax - b0 + 31) / 32;
                        hipLaunchKernelGGL((k_trsm_u<T, 64>), dim3(colchunks, dp.n_large[l], nf), dim3(256),
                                           lds64, st, F.arena, F.fstride, lvL, b0,
                                           0);
                    }
                    gemm(d.deep_off, d.deep_cnt, b0, 64, 0, d.deep_flops, d.deep_elems);
                }
            } else {
                int si = 0;
                for (int k0 = 0; k0 < L.large_pmax; k0 += pl.nb, si++) {
                    panel(k0, cnt.panel_flops[si], true, cnt.trsm_flops[si]);
                    const auto &sp = dp.steps[l][si];
                    gemm(sp.first, sp.second, k0, 32, 0, cnt.gemm_flops[si], cnt.gemm_elems[si]);
                }
            }
        }
    }
    const int nfr = (int)pl.fronts.size();
    hipLaunchKernelGGL(k_gsrc, dim3(nfr, nf), dim3(64), 0, st, dp.fronts, nfr, F.rowperm, pl.n, dp.gsrc_id, pl.fv_rows,
                       F.gsrc);
    {
        ProfScope ps(K_DIAG_INV, st, 0.0, 2.0 * dp.diag_elems * sizeof(cx<T>) * nf);
        hipLaunchKernelGGL(k_diag_inv<T>, dim3(nfr, nf), dim3(256), 0, st, F.arena, F.fstride, dp.fronts,
                           dp.lv_single);
    }
    GFDFD_HIP(hipGetLastError());
}

template void factor_numeric<double>(const DevPlan &, Factors<double> &, const cx<double> *, int64_t, hipStream_t);
template void factor_numeric<float>(const DevPlan &, Factors<float> &, const cx<double> *, int64_t, hipStream_t);

}  // namespace gfdfd
