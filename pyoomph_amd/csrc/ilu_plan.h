// Row order, permuted pattern and level sets of the ILU(0) preconditioner (host, once per
// pattern; see ilu_plan.cpp). No reference counterpart: pyoomph solves with SuperLU
// (pyoomph/solvers/scipy.py:47-104); this preconditioner serves the batched GMRES/CG.
#pragma once
#include <cstdint>
#include <string>
#include <vector>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define PYHIP_HD __host__ __device__
#else
#define PYHIP_HD
#endif

namespace pyhip {

struct IluHostPlan {
    std::vector<int32_t> perm;               // [n] new -> old
    std::vector<int32_t> prs, pcol, psrc;    // permuted column-sorted pattern, source entry
    std::vector<int32_t> pdiag;              // [n] diagonal position
    std::vector<int32_t> lo_rows, up_rows;   // rows grouped by lower / upper solve level
    std::vector<int64_t> lo_ptr, up_ptr;     // level boundaries
    bool multicolor = false;                 // some sub-problem takes the multicolour order
};

// order: 0 auto (multicolour for each sub-problem whose natural order has more than
// auto_levels lower-solve levels), 1 natural, 2 multicolour. is_p[i] = 1 puts row i in
// the second group of its sub-problem (Taylor-Hood pressures). Returns 0 or -1 (err).
int ilu_plan_host(int64_t n, const int32_t *rs, const int32_t *col, const std::vector<int64_t> &sub_off,
                  const std::vector<char> &is_p, int order, int auto_levels, IluHostPlan &out, std::string &err);

// Sliced copy of the triangular factors for the sub-problems of at most `cap` rows, whose
// solves run in one workgroup of kIluSliceWaves waves each (ilu_sliced.h). Every level of a
// sub-problem's lower and upper solve is cut into slices of 64 lanes, `lanes` lanes per row (a
// power of two): rows sorted by decreasing length within the level, wide enough that a
// narrow level spreads over all waves and a row takes at most kIluChunk steps where 16 lanes
// allow it. Lane = row-in-slice * lanes + u takes the row's entries u, u + lanes, ...: one
// step each. A slice is stored in chunks of kIluChunk steps (one, unless a row has more than
// 16 * kIluChunk entries), every lane's part of a chunk contiguous for 16-byte loads:
//   idx [chunk][lane][8]      local columns of the steps, the lane's local row (kIluNoRow:
//                             none), the chunk's mark
//   val [chunk][3][lane][2]   factor entries, two steps at a time
// Mark: level | log2(lanes) << 12 | 1 << 15 where the slice goes on in the next chunk.
// Slice k of a level belongs to wave k mod kIluSliceWaves; a wave's chunks follow each other
// in level order, padded with empty ones to a multiple of kIluDepth, so that a wave reads one
// stream. Columns and rows are local to the sub-problem (16 bits); steps past a row's end
// point at the local row `rows` (one past the last), where the solve keeps a zero.
// The host cuts the levels (IluChunk: 16 bytes a chunk); the chunks' columns and the place of
// their factor entries are written out where they are used, by kernels (ilu_sliced.h) or for
// tests (ilu_sliced_expand): written out by the host and copied, the padded arrays took up to ten
// times the rest of a first solve (4096 P1 meshes of 8 x 8: 17 ms without them, 173 with).
constexpr int kIluSliceLanes = 64;
constexpr int kIluSliceWaves = 16;
constexpr int kIluChunk = 6;
constexpr int kIluDepth = 3;                // chunks a wave loads ahead
constexpr int kIluChunkIdx = kIluSliceLanes * 8, kIluChunkVal = kIluSliceLanes * kIluChunk;
constexpr uint16_t kIluNoRow = 0xffff;
constexpr int kIluMaxLevels = 4096;
struct IluChunk {
    int32_t at;        // its rows: [at, at + n) of the side's row list
    int32_t first;     // their first step in this chunk
    int32_t slot;      // handled sub-problem
    uint16_t mark, n;  // n 0: padding
};
struct IluSlicedSide {
    std::vector<int32_t> nlev;               // [handled] levels of each sub-problem
    std::vector<int32_t> chunk0;             // [handled * waves + 1] first chunk of each wave
    std::vector<int32_t> order;              // permuted rows by (sub-problem, level, decreasing length)
    std::vector<IluChunk> chunk;
};
struct IluSlicedPlan {
    std::vector<int32_t> subs, row0, rows;   // handled sub-problems (longest first), first permuted row, row count
    IluSlicedSide lo, up;
    std::vector<int32_t> big_lo, big_up;     // rows of the other sub-problems by level (as lo_rows / up_rows)
    std::vector<int64_t> big_lo_ptr, big_up_ptr;
    int max_rows = 0;                        // largest handled sub-problem
    std::vector<char> tiny;                  // [handled] four lanes a row, see ilu_sliced_host
};

// Lane `lane` of a chunk: its permuted row (-1: none), the row's entries on this side
// [k0, k0 + len) of the permuted pattern and the lane's entry of step j, e(j) (< len: taken)
struct IluLane {
    int32_t row, k0, len, lanes, e0;
    PYHIP_HD int32_t e(int j) const { return e0 + j * lanes; }
};
PYHIP_HD inline IluLane ilu_chunk_lane(const IluChunk &C, int lane, const int32_t *order, const int32_t *prs,
                                       const int32_t *pdiag, bool lower) {
    const int sh = (C.mark >> 12) & 7;
    IluLane L = {-1, 0, 0, 1 << sh, 0};
    if ((lane >> sh) >= C.n) return L;
    L.row = order[C.at + (lane >> sh)];
    L.k0 = lower ? prs[L.row] : pdiag[L.row] + 1;
    L.len = (lower ? pdiag[L.row] : prs[L.row + 1]) - L.k0;
    L.e0 = C.first * L.lanes + (lane & (L.lanes - 1));
    return L;
}

// The sliced plan of H (ilu_plan_host); cap < 65535. A sub-problem is handled if it has at
// most cap rows and kIluMaxLevels levels on each side, and at most kIluEntriesPerLevel
// triangle entries per level (both sides; but see tiny ones): one CU takes about 0.28 us per 1000 entries
// (P2 Poisson 41^2, 67 k entries in 7 + 7 levels: 22 us; 64^2, 166 k in 7 + 7: 47 us;
// Taylor-Hood 26^2, 223 k in 23 + 23: 58 us), a launch per level about 3 us (42, 42 and
// 150 us). Decided per sub-problem, so that its solve is the same alone and in any batch.
// Tiny sub-problems, of at most kIluTinyRows rows with at most 4 kIluChunk entries a side,
// always take four lanes a row: a lane's two running sums are then two of the level kernels'
// stripes, combined by the same tree, so that the level launches give the same bits and may serve
// them. They do for kIluTinyCount of them or more, since a workgroup takes its own
// chain of levels, 512 at a time on the 256 CUs, where a launch takes a level of all of them: Newton
// solves of 2048 / 4096 with 49 rows 6.6 / 12.6 ms by workgroups, 6.5 / 8.1 by launches; with 121
// rows 10.3 / 19.4 and 11.2 / 16.1; with 225 rows (P2) 21.8 / 41.6 and 30.5 / 38.2.
// Returns 0 or -1 (err).
constexpr int64_t kIluEntriesPerLevel = 10000;
constexpr int kIluTinyRows = 256;
constexpr int kIluTinyCount = 3072;
int ilu_sliced_host(const IluHostPlan &H, const std::vector<int64_t> &sub_off, int cap, IluSlicedPlan &out,
                    std::string &err);
// idx and, as indices in the permuted pattern (-1: none), val of a side
void ilu_sliced_expand(const IluHostPlan &H, const IluSlicedPlan &P, bool lower, std::vector<uint16_t> &idx,
                       std::vector<int32_t> &src);

// Level-by-level solves of the other sub-problems, a launch per level, in the problem's own
// row numbering. A level's rows are sorted by decreasing entry count and cut into segments of
// equal step counts (a step: 8 entries of a row); `lanes` lanes take a row. Entry e of a row
// belongs to stripe e mod 8, lane u of the row to the stripes u, u + lanes, ...: stored
// [step][stripe / lanes][row in segment * lanes + u], so that a thread's entries come from
// addresses it computes from the segment's numbers alone, without row pointers. Padding
// repeats the row's first column with factor entry 0.
constexpr int kIluSegments = 8;
struct IluLevel {
    int32_t rows = 0, row0 = 0, lanes = 1, nseg = 0;
    int32_t seg_row[kIluSegments + 1] = {0};   // first row of each segment within the level
    int32_t steps[kIluSegments] = {0};
    int64_t off[kIluSegments] = {0};           // first entry of each segment
};
constexpr int32_t kIluLast = INT32_MIN;        // row mark (sign bit): no upper entries
// Place of entry k (0 .. 8 steps - 1) of the level's row i, in segment g
PYHIP_HD inline int64_t ilu_level_place(const IluLevel &L, int g, int32_t i, int k) {
    const int ns = 8 / L.lanes, st = k % 8;
    const int64_t S = (int64_t)(L.seg_row[g + 1] - L.seg_row[g]) * L.lanes;
    return L.off[g] + ((int64_t)(k / 8) * ns + st / L.lanes) * S + (int64_t)(i - L.seg_row[g]) * L.lanes + st % L.lanes;
}
struct IluLevelSide {
    std::vector<IluLevel> lev;
    std::vector<int32_t> order;              // permuted rows by (level, decreasing steps)
    int64_t entries = 0;
};
// rows / ptr: the permuted rows of the other sub-problems by level (IluSlicedPlan)
void ilu_level_host(const IluHostPlan &H, std::vector<int32_t> rows, const std::vector<int64_t> &ptr, bool lower,
                    IluLevelSide &out);
// Written out, by kernels (ilu_levels.h) or for tests: problem rows (lower: | kIluLast where
// it applies), problem columns, permuted-pattern index of each entry (-1: padding) and of each
// row's pivot
void ilu_level_expand(const IluHostPlan &H, const IluLevelSide &S, bool lower, std::vector<int32_t> &row,
                      std::vector<int32_t> &col, std::vector<int32_t> &src, std::vector<int32_t> &rsrc);
// f(place, k) for the entries st, st + 8, ... of the level's row i, with its row's entries on
// this side [k0, k0 + n) of the permuted pattern: k < n the row's k-th, else padding
template <typename F>
PYHIP_HD inline void ilu_level_stripe(const IluLevel &L, int32_t i, int st, F f) {
    int g = 0;
    while (i >= L.seg_row[g + 1]) g++;
    for (int k = st; k < 8 * L.steps[g]; k += 8) f(ilu_level_place(L, g, i, k), k);
}
PYHIP_HD inline int32_t ilu_level_col(int32_t r, int32_t k0, int32_t n, int k, const int32_t *pcol, const int32_t *perm) {
    return perm[k < n ? pcol[k0 + k] : n ? pcol[k0] : r];
}
PYHIP_HD inline int32_t ilu_level_row(int32_t r, const int32_t *prs, const int32_t *pdiag, const int32_t *perm, bool lower) {
    return lower && prs[r + 1] - pdiag[r] == 1 ? (perm[r] | kIluLast) : perm[r];
}

}  // namespace pyhip
