// Host entry points to the ILU(0) plan builder for tests on the CPU (no device work):
// they expose the row order, the permuted pattern and the level sets.
#include <cstring>
#include <string>

#include "ilu_plan.h"

using namespace pyhip;

namespace {
thread_local std::string g_ilu_err;
}

extern "C" {

const char *pyhip_ilu_plan_error(void) { return g_ilu_err.c_str(); }

// is_p may be null (one group per sub-problem); order as ilu_plan_host
void *pyhip_ilu_plan_new(int64_t n, const int32_t *rs, const int32_t *col, int nsub, const int64_t *sub_off,
                         const int8_t *is_p, int order, int auto_levels) {
    if (n < 0 || !rs || !col || nsub < 1 || !sub_off || sub_off[0] != 0 || sub_off[nsub] != n || order < 0 ||
        order > 2) {
        g_ilu_err = "invalid arguments";
        return nullptr;
    }
    std::vector<int64_t> off(sub_off, sub_off + nsub + 1);
    std::vector<char> g(n, 0);
    if (is_p)
        for (int64_t i = 0; i < n; i++) g[i] = is_p[i] ? 1 : 0;
    IluHostPlan *P = new IluHostPlan();
    if (ilu_plan_host(n, rs, col, off, g, order, auto_levels, *P, g_ilu_err)) {
        delete P;
        return nullptr;
    }
    return P;
}

// sizes[0..3] = lower levels, upper levels, nnz, multicolour flag
int pyhip_ilu_plan_sizes(const void *h, int64_t *sizes) {
    const IluHostPlan *P = (const IluHostPlan *)h;
    if (!P || !sizes) return -1;
    sizes[0] = (int64_t)P->lo_ptr.size() - 1;
    sizes[1] = (int64_t)P->up_ptr.size() - 1;
    sizes[2] = (int64_t)P->pcol.size();
    sizes[3] = P->multicolor ? 1 : 0;
    return 0;
}

int pyhip_ilu_plan_copy(const void *h, int32_t *perm, int32_t *prs, int32_t *pcol, int32_t *psrc, int32_t *pdiag,
                        int32_t *lo_rows, int64_t *lo_ptr, int32_t *up_rows, int64_t *up_ptr) {
    const IluHostPlan *P = (const IluHostPlan *)h;
    if (!P) return -1;
    auto cp = [](auto *dst, const auto &v) {
        if (dst && !v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
    };
    cp(perm, P->perm);
    cp(prs, P->prs);
    cp(pcol, P->pcol);
    cp(psrc, P->psrc);
    cp(pdiag, P->pdiag);
    cp(lo_rows, P->lo_rows);
    cp(lo_ptr, P->lo_ptr);
    cp(up_rows, P->up_rows);
    cp(up_ptr, P->up_ptr);
    return 0;
}

// The sliced plan of a plan (ilu_sliced_host with `cap`), side 0 lower / 1 upper. sizes:
// [0] handled sub-problems, [1] chunks, [2] rows of the other sub-problems, [3] their
// levels. Null arrays are not written.
int pyhip_ilu_sliced_copy(const void *h, int nsub, const int64_t *sub_off, int cap, int side, int64_t *sizes,
                          int32_t *subs, int32_t *nlev, int32_t *chunk0, uint16_t *idx, int32_t *src, int32_t *big,
                          int64_t *big_ptr) {
    const IluHostPlan *P = (const IluHostPlan *)h;
    if (!P || !sizes || !sub_off || nsub < 1) return -1;
    IluSlicedPlan Q;
    if (ilu_sliced_host(*P, std::vector<int64_t>(sub_off, sub_off + nsub + 1), cap, Q, g_ilu_err)) return -1;
    const IluSlicedSide &S = side ? Q.up : Q.lo;
    std::vector<uint16_t> x;
    std::vector<int32_t> sr;
    if (idx || src) ilu_sliced_expand(*P, Q, side == 0, x, sr);
    const auto &bg = side ? Q.big_up : Q.big_lo;
    const auto &bp = side ? Q.big_up_ptr : Q.big_lo_ptr;
    sizes[0] = (int64_t)Q.subs.size();
    sizes[1] = (int64_t)S.chunk.size();
    sizes[2] = (int64_t)bg.size();
    sizes[3] = (int64_t)bp.size() - 1;
    auto cp = [](auto *dst, const auto &v) {
        if (dst && !v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
    };
    cp(subs, Q.subs);
    cp(nlev, S.nlev);
    cp(chunk0, S.chunk0);
    cp(idx, x);
    cp(src, sr);
    cp(big, bg);
    cp(big_ptr, bp);
    return 0;
}

// The level-by-level layout of one side (0 lower, 1 upper) of the sub-problems above `cap`
// rows (ilu_level_host). sizes: [0] levels, [1] rows, [2] entries; levels [nlev][4 + 9 + 8 + 8]:
// rows, row0, lanes, nseg, seg_row, steps, off. Null arrays are not written.
int pyhip_ilu_level_copy(const void *h, int nsub, const int64_t *sub_off, int cap, int side, int64_t *sizes,
                         int64_t *levels, int32_t *row, int32_t *col, int32_t *src, int32_t *rsrc) {
    const IluHostPlan *P = (const IluHostPlan *)h;
    if (!P || !sizes || !sub_off || nsub < 1) return -1;
    IluSlicedPlan Q;
    IluLevelSide S;
    if (ilu_sliced_host(*P, std::vector<int64_t>(sub_off, sub_off + nsub + 1), cap, Q, g_ilu_err)) return -1;
    ilu_level_host(*P, side ? Q.big_up : Q.big_lo, side ? Q.big_up_ptr : Q.big_lo_ptr, side == 0, S);
    std::vector<int32_t> r, c, sr, rsr;
    if (row || col || src || rsrc) ilu_level_expand(*P, S, side == 0, r, c, sr, rsr);
    sizes[0] = (int64_t)S.lev.size();
    sizes[1] = (int64_t)S.order.size();
    sizes[2] = S.entries;
    if (levels)
        for (const IluLevel &L : S.lev) {
            for (int64_t v : {(int64_t)L.rows, (int64_t)L.row0, (int64_t)L.lanes, (int64_t)L.nseg}) *levels++ = v;
            for (int32_t v : L.seg_row) *levels++ = v;
            for (int32_t v : L.steps) *levels++ = v;
            for (int64_t v : L.off) *levels++ = v;
        }
    auto cp = [](auto *dst, const auto &v) {
        if (dst && !v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
    };
    cp(row, r);
    cp(col, c);
    cp(src, sr);
    cp(rsrc, rsr);
    return 0;
}

void pyhip_ilu_plan_free(void *h) { delete (IluHostPlan *)h; }

}  // extern "C"
