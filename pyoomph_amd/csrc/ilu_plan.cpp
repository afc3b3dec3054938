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

// One side (lower or upper) of the sliced plan for the handled sub-problems: level lists
// from the merged level lists `rows` / `ptr` of the whole batch.
static int sliced_side(const IluHostPlan &H, const std::vector<int32_t> &rows, const std::vector<int64_t> &ptr,
                       bool lower, const std::vector<int32_t> &slot_of, const IluSlicedPlan &P, const std::vector<int32_t> &row_sub, IluSlicedSide &S,
                       std::vector<int32_t> &big, std::vector<int64_t> &big_ptr, std::string &err) {
    const int nh = (int)P.subs.size(), nl = (int)ptr.size() - 1;
    // per handled sub-problem: (level, rows) lists in level order
    std::vector<std::vector<std::pair<int32_t, std::vector<int32_t>>>> lists(nh);
    big_ptr.assign(1, 0);
    for (int l = 0; l < nl; l++) {
        for (int64_t w = ptr[l]; w < ptr[l + 1]; w++) {
            const int32_t r = rows[w], t = slot_of[row_sub[r]];
            if (t < 0) {
                big.push_back(r);
                continue;
            }
            if (lists[t].empty() || lists[t].back().first != l) lists[t].push_back({l, {}});
            lists[t].back().second.push_back(r);
        }
        if ((int64_t)big.size() > big_ptr.back()) big_ptr.push_back((int64_t)big.size());
    }
    auto len = [&](int32_t r) { return lower ? H.pdiag[r] - H.prs[r] : H.prs[r + 1] - H.pdiag[r] - 1; };
    S.chunk0.assign(1, 0);
    struct Slice {
        int level, lanes;
        size_t b, n;
        const std::vector<int32_t> *rows;
    };
    for (int t = 0; t < nh; t++) {
        const int32_t r0 = P.row0[t], dummy = P.rows[t];
        std::vector<std::vector<Slice>> waves(kIluSliceWaves);
        for (size_t l = 0; l < lists[t].size(); l++) {
            auto &R = lists[t][l].second;
            std::stable_sort(R.begin(), R.end(), [&](int32_t a, int32_t b) { return len(a) > len(b); });
            // lanes that still leave the level at most one slice per wave
            int fill = 1;
            while (fill < 16 && 2 * fill * (int64_t)R.size() <= kIluSliceLanes * kIluSliceWaves && fill < len(R[0]))
                fill *= 2;
            int k = 0;
            for (size_t b = 0; b < R.size(); k++) {
                int lanes = fill;
                while (lanes < 16 && (len(R[b]) + lanes - 1) / lanes > kIluChunk) lanes *= 2;
                const size_t m = std::min<size_t>(kIluSliceLanes / lanes, R.size() - b);
                waves[k % kIluSliceWaves].push_back({(int)l, lanes, b, m, &R});
                b += m;
            }
        }
        S.nlev.push_back((int32_t)lists[t].size());
        for (const auto &tasks : waves) {
            const size_t first = S.chunk0.back();
            uint16_t mark = 0;
            // appends an empty chunk
            auto chunk = [&]() -> size_t {
                const size_t c = S.idx.size() / kIluChunkIdx;
                S.idx.resize((c + 1) * kIluChunkIdx, (uint16_t)dummy);
                S.src.resize((c + 1) * kIluChunkVal, -1);
                for (int lane = 0; lane < kIluSliceLanes; lane++) {
                    S.idx[c * kIluChunkIdx + lane * 8 + kIluChunk] = kIluNoRow;
                    S.idx[c * kIluChunkIdx + lane * 8 + kIluChunk + 1] = mark;
                }
                return c;
            };
            for (const Slice &sl : tasks) {
                const std::vector<int32_t> &R = *sl.rows;
                const int lanes = sl.lanes, w = (len(R[sl.b]) + lanes - 1) / lanes;
                const int nch = std::max(1, (w + kIluChunk - 1) / kIluChunk);
                const uint16_t base = (uint16_t)(sl.level | __builtin_ctz(lanes) << 12);
                size_t c0 = 0;
                for (int c = 0; c < nch; c++) {
                    mark = (uint16_t)(base | (c + 1 < nch ? 1 << 15 : 0));
                    const size_t at = chunk();
                    if (c == 0) c0 = at;
                    for (int lane = 0; lane < kIluSliceLanes; lane++)
                        if ((size_t)(lane / lanes) < sl.n)
                            S.idx[at * kIluChunkIdx + lane * 8 + kIluChunk] =
                                (uint16_t)(R[sl.b + lane / lanes] - r0);
                }
                for (size_t q = 0; q < sl.n; q++) {
                    const int32_t r = R[sl.b + q], k0 = lower ? H.prs[r] : H.pdiag[r] + 1;
                    for (int e = 0; e < len(r); e++) {
                        const int step = e / lanes, j = step % kIluChunk;
                        const size_t lane = q * lanes + e % lanes, c = c0 + step / kIluChunk;
                        S.idx[c * kIluChunkIdx + lane * 8 + j] = (uint16_t)(H.pcol[k0 + e] - r0);
                        S.src[c * kIluChunkVal + (j / 2) * 2 * kIluSliceLanes + 2 * lane + j % 2] = k0 + e;
                    }
                }
            }
            mark &= 0xfff;   // padding stays on the wave's last level
            while ((S.idx.size() / kIluChunkIdx - first) % kIluDepth) chunk();
            if (S.src.size() >= (size_t)INT32_MAX) {
                err = "ILU(0) sliced plan: too many entries";
                return -1;
            }
            S.chunk0.push_back((int32_t)(S.idx.size() / kIluChunkIdx));
        }
    }
    return 0;
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
    for (int s = 0; s < nsub; s++) {
        const int64_t m = sub_off[s + 1] - sub_off[s];
        const int64_t entries = (int64_t)H.prs[sub_off[s + 1]] - H.prs[sub_off[s]] - m;
        if (m > 0 && m <= cap && levels[0][s] <= kIluMaxLevels && levels[1][s] <= kIluMaxLevels &&
            entries <= kIluEntriesPerLevel * (levels[0][s] + levels[1][s]))
            order.push_back(s);
    }
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
        out.max_rows = std::max(out.max_rows, out.rows.back());
    }
    int rc = sliced_side(H, H.lo_rows, H.lo_ptr, true, slot_of, out, row_sub, out.lo, out.big_lo,
                         out.big_lo_ptr, err);
    if (!rc)
        rc = sliced_side(H, H.up_rows, H.up_ptr, false, slot_of, out, row_sub, out.up, out.big_up,
                         out.big_up_ptr, err);
    return rc;
}

int ilu_level_host(const IluHostPlan &H, const std::vector<int32_t> &big_rows, const std::vector<int64_t> &big_ptr,
                   bool lower, IluLevelSide &out, std::string &err) {
    out = IluLevelSide();
    auto len = [&](int32_t r) { return lower ? H.pdiag[r] - H.prs[r] : H.prs[r + 1] - H.pdiag[r] - 1; };
    std::vector<int32_t> R;
    for (size_t l = 0; l + 1 < big_ptr.size(); l++) {
        R.assign(big_rows.begin() + big_ptr[l], big_rows.begin() + big_ptr[l + 1]);
        auto steps_of = [&](int32_t r) { return (len(r) + 7) / 8; };
        std::stable_sort(R.begin(), R.end(), [&](int32_t a, int32_t b) { return steps_of(a) > steps_of(b); });
        IluLevel L;
        L.rows = (int32_t)R.size();
        L.row0 = (int32_t)out.row.size();
        // narrow levels: more lanes per row, for more loads in flight
        L.lanes = L.rows <= 16384 ? 8 : L.rows <= 65536 ? 4 : 2;
        const int ns = 8 / L.lanes;
        for (int32_t b = 0; b < L.rows;) {
            const int g = L.nseg++, steps = steps_of(R[b]);
            int32_t e = b;
            // the last segment takes every row that is left
            while (e < L.rows && (g == kIluSegments - 1 || steps_of(R[e]) == steps)) e++;
            L.seg_row[g] = b;
            L.seg_row[g + 1] = e;
            L.steps[g] = steps;
            L.off[g] = (int64_t)out.col.size();
            const int64_t S = (int64_t)(e - b) * L.lanes;
            out.col.resize(out.col.size() + S * ns * steps);
            out.src.resize(out.col.size(), -1);
            for (int32_t q = b; q < e; q++) {
                const int32_t r = R[q], k0 = lower ? H.prs[r] : H.pdiag[r] + 1, n = len(r);
                const int32_t pad = n ? H.perm[H.pcol[k0]] : H.perm[r];
                for (int k = 0; k < 8 * steps; k++) {
                    const int st = k % 8, u = st % L.lanes, j = st / L.lanes;
                    const int64_t at = L.off[g] + ((int64_t)(k / 8) * ns + j) * S + (int64_t)(q - b) * L.lanes + u;
                    out.col[at] = k < n ? H.perm[H.pcol[k0 + k]] : pad;
                    out.src[at] = k < n ? k0 + k : -1;
                }
            }
            b = e;
        }
        for (const int32_t r : R) {
            const bool last = lower && H.prs[r + 1] - H.pdiag[r] == 1;
            out.row.push_back(last ? (H.perm[r] | kIluLast) : H.perm[r]);
            out.rsrc.push_back(H.pdiag[r]);
        }
        out.lev.push_back(L);
    }
    if (out.col.size() >= (size_t)INT64_C(1) << 40) {
        err = "ILU(0) level plan: too many entries";
        return -1;
    }
    return 0;
}

}  // namespace pyhip
