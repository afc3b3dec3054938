// Row order, permuted pattern and level sets of the ILU(0) preconditioner (see ilu_plan.h).
//
// Order within a sub-problem: the rows of group 0 (all rows, or Taylor-Hood velocities),
// then those of group 1 (Taylor-Hood pressures), which keeps ILU(0) pivots non-zero for
// the zero pressure-pressure block. Within a group either the natural order, or a
// multicolour order: a greedy colouring of the group's rows (in natural order, each row
// takes the smallest colour none of its already coloured neighbours in the group has),
// rows sorted by (colour, index). Rows of one colour of one group are independent, so the
// triangular solves have at most as many levels as there are colours. Levels: a row's
// lower level is one more than the largest level of the columns left of its diagonal,
// its upper level likewise from the right.
#include "ilu_plan.h"

#include <algorithm>
#include <climits>
#include <thread>
#include <utility>

namespace pyhip {

int ilu_plan_host(int64_t n, const int32_t *rs, const int32_t *col, const std::vector<int64_t> &sub_off,
                  const std::vector<char> &is_p, int order, int auto_levels, IluHostPlan &out, std::string &err) {
    out = IluHostPlan();
    const int nsub = (int)sub_off.size() - 1;
    const int64_t nnz = rs[n];
    if ((int64_t)is_p.size() != n || nsub < 0) {
        err = "ILU(0) plan: inconsistent arguments";
        return -1;
    }
    std::vector<int32_t> perm(n), iperm(n);
    // multicolour order for the sub-problems with mc[s] (colours are computed for all
    // rows; the neighbours of a row are in its own sub-problem)
    auto make_perm = [&](const std::vector<char> &mc) {
        std::vector<int32_t> color(n, 0);
        bool any = false;
        for (char c : mc) any = any || c;
        if (any) {
            std::vector<int32_t> mark;   // mark[c] == row: colour c taken by a neighbour
            for (int64_t i = 0; i < n; i++) {
                for (int32_t k = rs[i]; k < rs[i + 1]; k++) {
                    const int32_t c = col[k];
                    if (c < i && is_p[c] == is_p[i]) {
                        if ((size_t)color[c] >= mark.size()) mark.resize(color[c] + 1, -1);
                        mark[color[c]] = (int32_t)i;
                    }
                }
                int32_t c = 0;
                while ((size_t)c < mark.size() && mark[c] == i) c++;
                color[i] = c;
            }
        }
        int64_t w = 0;
        std::vector<int32_t> rows;
        for (int s = 0; s < nsub; s++)
            for (char g = 0; g < 2; g++) {
                rows.clear();
                for (int64_t i = sub_off[s]; i < sub_off[s + 1]; i++)
                    if (is_p[i] == g) rows.push_back((int32_t)i);
                if (mc[s])
                    std::stable_sort(rows.begin(), rows.end(),
                                     [&](int32_t x, int32_t y) { return color[x] < color[y]; });
                for (int32_t r : rows) perm[w++] = r;
            }
        for (int64_t i = 0; i < n; i++) iperm[perm[i]] = (int32_t)i;
    };
    std::vector<int32_t> prs(n + 1, 0), pcol(nnz), psrc(nnz), pdiag(n, -1), lev(n, 0);
    auto make_pattern = [&]() -> int {
        std::vector<std::pair<int32_t, int32_t>> tmp;
        for (int64_t i = 0; i < n; i++) {
            const int32_t o = perm[i];
            tmp.clear();
            for (int32_t k = rs[o]; k < rs[o + 1]; k++) tmp.push_back({iperm[col[k]], k});
            std::sort(tmp.begin(), tmp.end());
            prs[i + 1] = prs[i] + (int32_t)tmp.size();
            pdiag[i] = -1;
            for (size_t t = 0; t < tmp.size(); t++) {
                pcol[prs[i] + t] = tmp[t].first;
                psrc[prs[i] + t] = tmp[t].second;
                if (tmp[t].first == i) pdiag[i] = prs[i] + (int32_t)t;
            }
            if (pdiag[i] < 0) {
                err = "ILU(0): a row has no structural diagonal entry";
                return -1;
            }
        }
        return 0;
    };
    // lower levels (depends on smaller columns)
    auto lower_levels = [&]() {
        int32_t nl = 0;
        for (int64_t i = 0; i < n; i++) {
            int32_t l = 0;
            for (int32_t k = prs[i]; k < pdiag[i]; k++) l = std::max(l, lev[pcol[k]] + 1);
            lev[i] = l;
            nl = std::max(nl, l + 1);
        }
        return nl;
    };
    int rc0;
    std::vector<char> mc(nsub, order == 2 ? 1 : 0);
    make_perm(mc);
    if ((rc0 = make_pattern())) return rc0;
    int32_t nlo = lower_levels();
    if (order == 0 && nlo > auto_levels) {
        // per sub-problem, so that its order does not depend on the batch
        bool any = false;
        for (int s = 0; s < nsub; s++) {
            int32_t nl = 0;
            for (int64_t i = sub_off[s]; i < sub_off[s + 1]; i++) nl = std::max(nl, lev[i] + 1);
            mc[s] = nl > auto_levels;
            any = any || mc[s];
        }
        if (any) {
            make_perm(mc);
            if ((rc0 = make_pattern())) return rc0;
            nlo = lower_levels();
        }
    }
    auto bucket = [&](int32_t nl, std::vector<int32_t> &rows, std::vector<int64_t> &ptr) {
        ptr.assign(nl + 1, 0);
        for (int64_t i = 0; i < n; i++) ptr[lev[i] + 1]++;
        for (int32_t l = 0; l < nl; l++) ptr[l + 1] += ptr[l];
        rows.resize(n);
        std::vector<int64_t> f(ptr.begin(), ptr.end() - 1);
        for (int64_t i = 0; i < n; i++) rows[f[lev[i]]++] = (int32_t)i;
    };
    bucket(nlo, out.lo_rows, out.lo_ptr);
    // upper levels (depends on larger columns), computed in decreasing row order
    int32_t nup = 0;
    for (int64_t i = n - 1; i >= 0; i--) {
        int32_t l = 0;
        for (int32_t k = pdiag[i] + 1; k < prs[i + 1]; k++) l = std::max(l, lev[pcol[k]] + 1);
        lev[i] = l;
        nup = std::max(nup, l + 1);
    }
    bucket(nup, out.up_rows, out.up_ptr);
    bool mc_any = false;
    for (char c : mc) mc_any = mc_any || c;
    out.perm = std::move(perm);
    out.prs = std::move(prs);
    out.pcol = std::move(pcol);
    out.psrc = std::move(psrc);
    out.pdiag = std::move(pdiag);
    out.multicolor = mc_any;
    return 0;
}

// Stable sort of rows [b, e) by decreasing key(row) >= 0; tmp, cnt: scratch
template <typename K>
static void sort_decreasing(int32_t *b, int32_t *e, K key, std::vector<int32_t> &tmp, std::vector<int32_t> &cnt) {
    const int64_t n = e - b;
    if (std::is_sorted(b, e, [&](int32_t x, int32_t y) { return key(x) > key(y); })) return;
    int32_t top = 0;
    for (int32_t *r = b; r < e; r++) top = std::max(top, key(*r));
    if (n < 16 || top > 4 * n) {   // few rows, or more counters than rows
        std::stable_sort(b, e, [&](int32_t x, int32_t y) { return key(x) > key(y); });
        return;
    }
    cnt.assign(top + 2, 0);
    for (int32_t *r = b; r < e; r++) cnt[top - key(*r) + 1]++;
    for (int32_t k = 0; k <= top; k++) cnt[k + 1] += cnt[k];
    tmp.assign(b, e);
    for (int32_t r : tmp) b[cnt[top - key(r)]++] = r;
}

template <typename F>
static void parallel_subs(int n, F &&fn) {
    unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    if (n < 64) nt = 1;
    const int per = (n + (int)nt - 1) / (int)nt;
    std::vector<std::thread> th;
    for (int b = 0; b < n; b += per) {
        const int e = std::min(n, b + per);
        if (nt == 1) fn(b, e);
        else th.emplace_back([&fn, b, e]() { fn(b, e); });
    }
    for (auto &x : th) x.join();
}

// One side (lower or upper) of the sliced plan for the handled sub-problems: level lists
// from the merged level lists `rows` / `ptr` of the whole batch.
static int sliced_side(const IluHostPlan &H, const std::vector<int32_t> &rows, const std::vector<int64_t> &ptr,
                       bool lower, const std::vector<int32_t> &slot_of, const IluSlicedPlan &P, const std::vector<int32_t> &row_sub, IluSlicedSide &S,
                       std::vector<int32_t> &big, std::vector<int64_t> &big_ptr, std::string &err) {
    const int nh = (int)P.subs.size(), nl = (int)ptr.size() - 1;
    auto len = [&](int32_t r) { return lower ? H.pdiag[r] - H.prs[r] : H.prs[r + 1] - H.pdiag[r] - 1; };
    // rows of each handled sub-problem in level order, and each one's level
    std::vector<int64_t> start(nh + 1, 0);
    for (int t = 0; t < nh; t++) start[t + 1] = start[t] + P.rows[t];
    std::vector<int64_t> pos(start.begin(), start.end() - 1);
    std::vector<int32_t> level(start[nh]);
    S.order.resize(start[nh]);
    big_ptr.assign(1, 0);
    for (int l = 0; l < nl; l++) {
        for (int64_t w = ptr[l]; w < ptr[l + 1]; w++) {
            const int32_t r = rows[w], t = slot_of[row_sub[r]];
            if (t < 0) {
                big.push_back(r);
                continue;
            }
            level[pos[t]] = l;
            S.order[pos[t]++] = r;
        }
        if ((int64_t)big.size() > big_ptr.back()) big_ptr.push_back((int64_t)big.size());
    }
    // the slices of sub-problem t, whose levels are sorted: f(wave, level, lanes, first row, rows, chunks)
    auto cut = [&](int t, auto f) {
        for (int64_t a = start[t]; a < start[t + 1];) {
            int64_t e = a;
            while (e < start[t + 1] && level[e] == level[a]) e++;
            const int64_t R = e - a;
            const int32_t longest = len(S.order[a]);
            // lanes that still leave the level at most one slice per wave
            int fill = P.tiny[t] ? 4 : 1;
            while (!P.tiny[t] && fill < 16 && 2 * fill * R <= kIluSliceLanes * kIluSliceWaves && fill < longest) fill *= 2;
            int k = 0;
            for (int64_t b = a; b < e; k++) {
                int lanes = fill;
                const int32_t n = len(S.order[b]);
                while (lanes < 16 && (n + lanes - 1) / lanes > kIluChunk) lanes *= 2;
                const int m = (int)std::min<int64_t>(kIluSliceLanes / lanes, e - b);
                const int steps = (n + lanes - 1) / lanes;
                f(k % kIluSliceWaves, (int)level[a], lanes, b, m, std::max(1, (steps + kIluChunk - 1) / kIluChunk));
                b += m;
            }
            a = e;
        }
    };
    S.nlev.resize(nh);
    std::vector<int64_t> c0((size_t)nh * kIluSliceWaves + 1, 0);
    parallel_subs(nh, [&](int t0, int t1) {
        std::vector<int32_t> tmp, cnt;
        for (int t = t0; t < t1; t++) {
            int32_t *o = S.order.data();
            for (int64_t a = start[t], e; a < start[t + 1]; a = e) {
                for (e = a; e < start[t + 1] && level[e] == level[a];) e++;
                sort_decreasing(o + a, o + e, len, tmp, cnt);
            }
            S.nlev[t] = start[t + 1] > start[t] ? level[start[t + 1] - 1] + 1 : 0;
            int64_t *c = c0.data() + (size_t)t * kIluSliceWaves + 1;
            cut(t, [&](int w, int, int, int64_t, int, int nch) { c[w] += nch; });
            for (int w = 0; w < kIluSliceWaves; w++) c[w] = (c[w] + kIluDepth - 1) / kIluDepth * kIluDepth;
        }
    });
    for (size_t w = 1; w < c0.size(); w++) c0[w] += c0[w - 1];
    if (c0.back() > INT32_MAX || start[nh] > INT32_MAX) {
        err = "ILU(0) sliced plan: too many chunks";
        return -1;
    }
    S.chunk0.assign(c0.begin(), c0.end());
    S.chunk.resize(c0.back());
    parallel_subs(nh, [&](int t0, int t1) {
        for (int t = t0; t < t1; t++) {
            const int64_t *c = c0.data() + (size_t)t * kIluSliceWaves;
            int64_t at[kIluSliceWaves];
            uint16_t last[kIluSliceWaves] = {0};
            std::copy(c, c + kIluSliceWaves, at);
            cut(t, [&](int w, int lev, int lanes, int64_t b, int m, int nch) {
                const uint16_t base = (uint16_t)(lev | __builtin_ctz(lanes) << 12);
                for (int q = 0; q < nch; q++)
                    S.chunk[at[w]++] = IluChunk{(int32_t)b, q * kIluChunk, t,
                                                (uint16_t)(base | (q + 1 < nch ? 1 << 15 : 0)), (uint16_t)m};
                last[w] = (uint16_t)lev;
            });
            // padding stays on the wave's last level
            for (int w = 0; w < kIluSliceWaves; w++)
                while (at[w] < c[w + 1]) S.chunk[at[w]++] = IluChunk{0, 0, t, last[w], 0};
        }
    });
    return 0;
}

void ilu_sliced_expand(const IluHostPlan &H, const IluSlicedPlan &P, bool lower, std::vector<uint16_t> &idx,
                       std::vector<int32_t> &src) {
    const IluSlicedSide &S = lower ? P.lo : P.up;
    idx.resize(S.chunk.size() * kIluChunkIdx);
    src.assign(S.chunk.size() * kIluChunkVal, -1);
    for (size_t c = 0; c < S.chunk.size(); c++) {
        const IluChunk &C = S.chunk[c];
        const int32_t r0 = P.row0[C.slot];
        for (int lane = 0; lane < kIluSliceLanes; lane++) {
            const IluLane L = ilu_chunk_lane(C, lane, S.order.data(), H.prs.data(), H.pdiag.data(), lower);
            uint16_t *ix = idx.data() + c * kIluChunkIdx + lane * 8;
            for (int j = 0; j < kIluChunk; j++) {
                const bool in = L.e(j) < L.len;
                ix[j] = (uint16_t)(in ? H.pcol[L.k0 + L.e(j)] - r0 : P.rows[C.slot]);
                if (in) src[c * kIluChunkVal + (j / 2) * 2 * kIluSliceLanes + 2 * lane + j % 2] = L.k0 + L.e(j);
            }
            ix[kIluChunk] = L.row >= 0 ? (uint16_t)(L.row - r0) : kIluNoRow;
            ix[kIluChunk + 1] = C.mark;
        }
    }
}

int ilu_sliced_host(const IluHostPlan &H, const std::vector<int64_t> &sub_off, int cap, IluSlicedPlan &out,
                    std::string &err) {
    out = IluSlicedPlan();
    const int nsub = (int)sub_off.size() - 1;
    const int64_t n = (int64_t)H.perm.size();
    if (cap >= (int)kIluNoRow) {
        err = "ILU(0) sliced plan: more rows than 16-bit indices";
        return -1;
    }
    // levels of each sub-problem on each side: the merged lists' levels that hold its rows
    std::vector<int32_t> row_sub(n), levels[2];
    for (int s = 0; s < nsub; s++)
        for (int64_t r = sub_off[s]; r < sub_off[s + 1]; r++) row_sub[r] = s;
    for (int u = 0; u < 2; u++) {
        const auto &rows = u ? H.up_rows : H.lo_rows;
        const auto &ptr = u ? H.up_ptr : H.lo_ptr;
        levels[u].assign(nsub, 0);
        for (size_t l = 0; l + 1 < ptr.size(); l++)
            for (int64_t w = ptr[l]; w < ptr[l + 1]; w++) levels[u][row_sub[rows[w]]] = (int32_t)l + 1;
    }
    std::vector<int32_t> order;
    std::vector<char> tiny(nsub, 0);
    int64_t ntiny = 0;
    for (int s = 0; s < nsub; s++) {
        const int64_t m = sub_off[s + 1] - sub_off[s];
        const int64_t entries = (int64_t)H.prs[sub_off[s + 1]] - H.prs[sub_off[s]] - m;
        if (m <= 0 || m > cap || levels[0][s] > kIluMaxLevels || levels[1][s] > kIluMaxLevels ||
            entries > kIluEntriesPerLevel * (levels[0][s] + levels[1][s]))
            continue;
        order.push_back(s);
        tiny[s] = m <= kIluTinyRows;
        for (int64_t r = sub_off[s]; r < sub_off[s + 1] && tiny[s]; r++)
            tiny[s] = H.pdiag[r] - H.prs[r] <= 4 * kIluChunk && H.prs[r + 1] - H.pdiag[r] - 1 <= 4 * kIluChunk;
        ntiny += tiny[s];
    }
    if (ntiny >= kIluTinyCount)
        order.erase(std::remove_if(order.begin(), order.end(), [&](int32_t s) { return tiny[s] != 0; }), order.end());
    // longest first: the last workgroups to start are the shortest
    std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
        return sub_off[a + 1] - sub_off[a] > sub_off[b + 1] - sub_off[b];
    });
    std::vector<int32_t> slot_of(nsub, -1);
    for (size_t t = 0; t < order.size(); t++) {
        const int s = order[t];
        slot_of[s] = (int32_t)t;
        out.subs.push_back(s);
        out.row0.push_back((int32_t)sub_off[s]);
        out.rows.push_back((int32_t)(sub_off[s + 1] - sub_off[s]));
        out.tiny.push_back(tiny[s]);
        out.max_rows = std::max(out.max_rows, out.rows.back());
    }
    if (out.subs.empty()) {
        out.lo.chunk0 = out.up.chunk0 = {0};
        out.big_lo = H.lo_rows;
        out.big_up = H.up_rows;
        out.big_lo_ptr = H.lo_ptr;
        out.big_up_ptr = H.up_ptr;
        return 0;
    }
    int rc = sliced_side(H, H.lo_rows, H.lo_ptr, true, slot_of, out, row_sub, out.lo, out.big_lo,
                         out.big_lo_ptr, err);
    if (!rc)
        rc = sliced_side(H, H.up_rows, H.up_ptr, false, slot_of, out, row_sub, out.up, out.big_up,
                         out.big_up_ptr, err);
    return rc;
}

void ilu_level_host(const IluHostPlan &H, std::vector<int32_t> rows, const std::vector<int64_t> &ptr, bool lower,
                    IluLevelSide &out) {
    out = IluLevelSide();
    auto steps_of = [&](int32_t r) {
        const int32_t n = lower ? H.pdiag[r] - H.prs[r] : H.prs[r + 1] - H.pdiag[r] - 1;
        return (n + 7) / 8;
    };
    out.order = std::move(rows);
    std::vector<int32_t> tmp, cnt;
    for (size_t l = 0; l + 1 < ptr.size(); l++) {
        int32_t *R = out.order.data() + ptr[l];
        sort_decreasing(R, out.order.data() + ptr[l + 1], steps_of, tmp, cnt);
        IluLevel L;
        L.rows = (int32_t)(ptr[l + 1] - ptr[l]);
        L.row0 = (int32_t)ptr[l];
        // narrow levels: more lanes per row, for more loads in flight
        L.lanes = L.rows <= 16384 ? 8 : L.rows <= 65536 ? 4 : 2;
        for (int32_t b = 0; b < L.rows;) {
            const int g = L.nseg++, steps = steps_of(R[b]);
            int32_t e = b;
            // the last segment takes every row that is left
            while (e < L.rows && (g == kIluSegments - 1 || steps_of(R[e]) == steps)) e++;
            L.seg_row[g] = b;
            L.seg_row[g + 1] = e;
            L.steps[g] = steps;
            L.off[g] = out.entries;
            out.entries += (int64_t)(e - b) * 8 * steps;
            b = e;
        }
        out.lev.push_back(L);
    }
}

void ilu_level_expand(const IluHostPlan &H, const IluLevelSide &S, bool lower, std::vector<int32_t> &row,
                      std::vector<int32_t> &col, std::vector<int32_t> &src, std::vector<int32_t> &rsrc) {
    row.resize(S.order.size());
    rsrc.resize(S.order.size());
    col.resize(S.entries);
    src.resize(S.entries);
    for (const IluLevel &L : S.lev)
        for (int32_t i = 0; i < L.rows; i++) {
            const int32_t r = S.order[L.row0 + i], k0 = lower ? H.prs[r] : H.pdiag[r] + 1,
                          n = (lower ? H.pdiag[r] : H.prs[r + 1]) - k0;
            row[L.row0 + i] = ilu_level_row(r, H.prs.data(), H.pdiag.data(), H.perm.data(), lower);
            rsrc[L.row0 + i] = H.pdiag[r];
            for (int st = 0; st < 8; st++)
                ilu_level_stripe(L, i, st, [&](int64_t at, int k) {
                    col[at] = ilu_level_col(r, k0, n, k, H.pcol.data(), H.perm.data());
                    src[at] = k < n ? k0 + k : -1;
                });
        }
}

}  // namespace pyhip
