"""ILU(0) row order and level schedule (host code, no GPU): the permuted pattern is the
symmetric permutation of the matrix pattern, every level of the triangular solves holds
rows that do not depend on each other, the multicolour order keeps same-coloured rows of
a group apart, and each sub-problem's order is the one it has alone in the batch."""
import ctypes

import numpy as np
import pytest
import scipy.sparse as sp

from pyoomph_amd import _lib
from tests.oracle_bridge import oracle_problem

AUTO, NATURAL, MULTICOLOR = 0, 1, 2


def _lib_ilu():
    L = _lib.load()
    L.pyhip_ilu_plan_new.restype = ctypes.c_void_p
    L.pyhip_ilu_plan_new.argtypes = [ctypes.c_int64, _lib.c_i32p, _lib.c_i32p, ctypes.c_int, _lib.c_i64p,
                                     ctypes.POINTER(ctypes.c_int8), ctypes.c_int, ctypes.c_int]
    L.pyhip_ilu_plan_sizes.argtypes = [ctypes.c_void_p, _lib.c_i64p]
    L.pyhip_ilu_plan_copy.argtypes = [ctypes.c_void_p] + [_lib.c_i32p] * 6 + [_lib.c_i64p, _lib.c_i32p, _lib.c_i64p]
    L.pyhip_ilu_plan_free.argtypes = [ctypes.c_void_p]
    L.pyhip_ilu_plan_error.restype = ctypes.c_char_p
    return L


def _plan(rs, col, sub_off, is_p=None, order=AUTO, auto_levels=64):
    L = _lib_ilu()
    rs = np.ascontiguousarray(rs, np.int32)
    col = np.ascontiguousarray(col, np.int32)
    so = np.ascontiguousarray(sub_off, np.int64)
    n = len(rs) - 1
    g = None if is_p is None else np.ascontiguousarray(is_p, np.int8)
    h = L.pyhip_ilu_plan_new(n, rs.ctypes.data_as(_lib.c_i32p), col.ctypes.data_as(_lib.c_i32p), len(so) - 1,
                             so.ctypes.data_as(_lib.c_i64p),
                             None if g is None else g.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)), order,
                             auto_levels)
    if not h:
        raise RuntimeError(L.pyhip_ilu_plan_error().decode())
    sz = np.zeros(4, np.int64)
    assert L.pyhip_ilu_plan_sizes(h, sz.ctypes.data_as(_lib.c_i64p)) == 0
    nlo, nup, nnz, mc = (int(v) for v in sz)
    out = dict(perm=np.zeros(n, np.int32), prs=np.zeros(n + 1, np.int32), pcol=np.zeros(nnz, np.int32),
               psrc=np.zeros(nnz, np.int32), pdiag=np.zeros(n, np.int32), lo_rows=np.zeros(n, np.int32),
               lo_ptr=np.zeros(nlo + 1, np.int64), up_rows=np.zeros(n, np.int32), up_ptr=np.zeros(nup + 1, np.int64))
    ptr = [v.ctypes.data_as(_lib.c_i64p if v.dtype == np.int64 else _lib.c_i32p) for v in out.values()]
    assert L.pyhip_ilu_plan_copy(h, *ptr) == 0
    L.pyhip_ilu_plan_free(h)
    out["multicolor"] = bool(mc)
    return out


def _batch(parts):
    """block-diagonal column-sorted structural pattern of several oracle problems, with
    the group of each row (1: Taylor-Hood pressure)"""
    mats, off, grp = [], [0], []
    for op in parts:
        G = op.geqn
        ns = G.shape[1]
        r = np.repeat(G, ns, axis=1).ravel()
        c = np.tile(G, (1, ns)).ravel()
        m = (r >= 0) & (c >= 0)
        mats.append(sp.csr_matrix((np.ones(m.sum()), (r[m], c[m])), shape=(op.ndof, op.ndof)))
        off.append(off[-1] + op.ndof)
        g = np.zeros(op.ndof, np.int8)
        if op.nvalue == 3:
            p = op.eqn[:, 2]
            g[p[p >= 0]] = 1
        grp.append(g)
    A = sp.block_diag(mats).tocsr()
    A.sum_duplicates()
    A.sort_indices()
    return A, np.array(off), np.concatenate(grp)


def _check_plan(A, off, grp, P):
    n = A.shape[0]
    rs, col = A.indptr, A.indices
    perm = P["perm"]
    assert np.array_equal(np.sort(perm), np.arange(n))
    iperm = np.empty(n, np.int64)
    iperm[perm] = np.arange(n)
    # each sub-problem keeps its own block of positions; group 0 rows come first
    for s in range(len(off) - 1):
        blk = perm[off[s]:off[s + 1]]
        assert blk.min() == off[s] and blk.max() == off[s + 1] - 1
        g = grp[blk]
        assert np.all(np.diff(g.astype(int)) >= 0)
    # permuted pattern = pattern of Pi A Pi^T, column-sorted, psrc points to the entry
    B = A[perm][:, perm].tocsr()
    B.sort_indices()
    assert np.array_equal(P["prs"], B.indptr) and np.array_equal(P["pcol"], B.indices)
    rows_new = np.repeat(np.arange(n), np.diff(P["prs"]))
    rows_old = np.repeat(np.arange(n), np.diff(rs))
    assert np.array_equal(rows_old[P["psrc"]], perm[rows_new])
    assert np.array_equal(col[P["psrc"]], perm[P["pcol"]])
    assert np.array_equal(P["pcol"][P["pdiag"]], np.arange(n))
    # level sets: every row in exactly one level; a row's lower (upper) neighbours sit in
    # earlier levels, so the rows of one level do not depend on each other
    for rows, ptr, side in ((P["lo_rows"], P["lo_ptr"], -1), (P["up_rows"], P["up_ptr"], 1)):
        assert ptr[0] == 0 and ptr[-1] == n and np.all(np.diff(ptr) > 0)
        assert np.array_equal(np.sort(rows), np.arange(n))
        lev = np.empty(n, np.int64)
        lev[rows] = np.repeat(np.arange(len(ptr) - 1), np.diff(ptr))
        pc = P["pcol"]
        dep = (pc < rows_new) if side < 0 else (pc > rows_new)
        assert np.all(lev[pc[dep]] < lev[rows_new[dep]])
        # each level is as early as it can be (one more than its deepest dependency)
        deepest = np.full(n, -1, np.int64)
        np.maximum.at(deepest, rows_new[dep], lev[pc[dep]])
        assert np.array_equal(lev, deepest + 1)
    return iperm


def test_natural_order_is_the_identity_and_levels_follow_the_mesh():
    parts = [oracle_problem("bratu", N=9, space="C2", lam=1.0), oracle_problem("poisson", N=2)]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, order=NATURAL)
    assert np.array_equal(P["perm"], np.arange(A.shape[0])) and not P["multicolor"]
    _check_plan(A, off, grp, P)


@pytest.mark.parametrize("order", [NATURAL, MULTICOLOR])
def test_taylor_hood_pressures_follow_velocities(order):
    parts = [oracle_problem("ns", N=6), oracle_problem("bratu", N=5, space="C1", lam=1.0), oracle_problem("ns", N=4)]
    A, off, grp = _batch(parts)
    assert grp.sum() > 0
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=order)
    _check_plan(A, off, grp, P)


def test_multicolour_order_separates_neighbours():
    parts = [oracle_problem("bratu", N=16, space="C2", lam=1.0), oracle_problem("ns", N=6),
             oracle_problem("rd", N=4, f=np.zeros(729))]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=MULTICOLOR)
    assert P["multicolor"]
    _check_plan(A, off, grp, P)
    # rows of one colour are a run of consecutive positions with no coupling between them;
    # the colour classes are the lower-solve levels restricted to one group
    n = A.shape[0]
    lev = np.empty(n, np.int64)
    lev[P["lo_rows"]] = np.repeat(np.arange(len(P["lo_ptr"]) - 1), np.diff(P["lo_ptr"]))
    rows_new = np.repeat(np.arange(n), np.diff(P["prs"]))
    pc = P["pcol"]
    g_new = grp[P["perm"]]
    same = (g_new[rows_new] == g_new[pc]) & (pc != rows_new)
    assert np.all(lev[rows_new[same]] != lev[pc[same]])
    # greedy colouring needs at most (largest group degree + 1) colours per group, so the
    # lower solve of the batch has at most that many levels per group
    deg = np.bincount(rows_new[same], minlength=n).max()
    assert len(P["lo_ptr"]) - 1 <= 2 * (deg + 1)
    Pn = _plan(A.indptr, A.indices, off, is_p=grp, order=NATURAL)
    assert len(P["lo_ptr"]) < len(Pn["lo_ptr"])


def _restrict(P, off, s):
    """the plan of sub-problem s, in its own numbering"""
    r0, r1 = off[s], off[s + 1]
    perm = P["perm"][r0:r1] - r0
    prs = P["prs"][r0:r1 + 1] - P["prs"][r0]
    pcol = P["pcol"][P["prs"][r0]:P["prs"][r1]] - r0
    return perm, prs, pcol


def test_each_sub_problem_keeps_its_own_order_in_a_batch():
    """auto order: a sub-problem switches to multicolour by its own level count, so its
    order is the same alone and in any batch"""
    parts = [oracle_problem("bratu", N=24, space="C2", lam=1.0), oracle_problem("bratu", N=3, space="C2", lam=1.0),
             oracle_problem("ns", N=8), oracle_problem("poisson", N=1)]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=AUTO, auto_levels=20)
    _check_plan(A, off, grp, P)
    switched = []
    for s in range(len(parts)):
        B = A[off[s]:off[s + 1], off[s]:off[s + 1]].tocsr()
        B.sort_indices()
        g = grp[off[s]:off[s + 1]]
        alone = _plan(B.indptr, B.indices, [0, B.shape[0]], is_p=g, order=AUTO, auto_levels=20)
        perm, prs, pcol = _restrict(P, off, s)
        assert np.array_equal(perm, alone["perm"])
        assert np.array_equal(prs, alone["prs"]) and np.array_equal(pcol, alone["pcol"])
        switched.append(alone["multicolor"])
    # the large sub-problems switch, the small ones keep the natural order
    assert switched[0] and not switched[1] and not switched[3]
    assert P["multicolor"]


def test_missing_diagonal_is_an_error():
    A = sp.csr_matrix(np.array([[1.0, 1.0, 0.0], [1.0, 0.0, 1.0], [0.0, 1.0, 1.0]]))
    A.eliminate_zeros()
    with pytest.raises(RuntimeError, match="diagonal"):
        _plan(A.indptr, A.indices, [0, 3], order=NATURAL)


def test_level_schedule_solves_like_a_sequential_sweep():
    """a triangular solve done level by level (all rows of a level at once, from values
    of earlier levels) equals the row-by-row forward and backward substitution"""
    parts = [oracle_problem("ns", N=5), oracle_problem("bratu", N=7, space="C2", lam=1.0)]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=MULTICOLOR)
    n = A.shape[0]
    rng = np.random.default_rng(3)
    B = A[P["perm"]][:, P["perm"]].tocsr()
    B.sort_indices()
    B.data = rng.uniform(0.1, 1.0, B.nnz)
    B.setdiag(B.diagonal() + 10.0)
    b = rng.standard_normal(n)
    Lo = sp.tril(B, -1).tocsr()
    y = np.zeros(n)
    for l in range(len(P["lo_ptr"]) - 1):
        rows = P["lo_rows"][P["lo_ptr"][l]:P["lo_ptr"][l + 1]]
        y[rows] = b[rows] - Lo[rows] @ y
    ys = np.zeros(n)
    for i in range(n):
        ys[i] = b[i] - (Lo[i] @ ys)[0]
    assert np.allclose(y, ys, rtol=1e-13, atol=1e-13)
    x = np.zeros(n)
    d = B.diagonal()
    Us = sp.triu(B, 1).tocsr()
    for l in range(len(P["up_ptr"]) - 1):
        rows = P["up_rows"][P["up_ptr"][l]:P["up_ptr"][l + 1]]
        x[rows] = (y[rows] - Us[rows] @ x) / d[rows]
    xs = np.zeros(n)
    for i in range(n - 1, -1, -1):
        xs[i] = (y[i] - (Us[i] @ xs)[0]) / d[i]
    assert np.allclose(x, xs, rtol=1e-13, atol=1e-13)


def _sliced(P_args, off, cap, side):
    """Copy of one side (0 lower, 1 upper) of the sliced plan (ilu_sliced_host)."""
    L = _lib_ilu()
    A, grp, order = P_args
    rs, col = np.ascontiguousarray(A.indptr, np.int32), np.ascontiguousarray(A.indices, np.int32)
    so, g = np.ascontiguousarray(off, np.int64), np.ascontiguousarray(grp, np.int8)
    h = L.pyhip_ilu_plan_new(len(rs) - 1, rs.ctypes.data_as(_lib.c_i32p), col.ctypes.data_as(_lib.c_i32p), len(so) - 1,
                             so.ctypes.data_as(_lib.c_i64p), g.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)), order, 64)
    assert h
    vp = ctypes.c_void_p
    f = L.pyhip_ilu_sliced_copy
    f.argtypes = [vp, ctypes.c_int, _lib.c_i64p, ctypes.c_int, ctypes.c_int, _lib.c_i64p] + [vp] * 7
    sz = np.zeros(4, np.int64)
    head = [h, len(so) - 1, so.ctypes.data_as(_lib.c_i64p), cap, side, sz.ctypes.data_as(_lib.c_i64p)]
    assert f(*head, *[None] * 7) == 0
    ns, nc, nb, nbl = (int(v) for v in sz)
    out = dict(subs=np.zeros(ns, np.int32), nlev=np.zeros(ns, np.int32), chunk0=np.zeros(16 * ns + 1, np.int32),
               idx=np.zeros((nc, 64, 8), np.uint16), src=np.zeros((nc, 3, 64, 2), np.int32), big=np.zeros(nb, np.int32),
               big_ptr=np.zeros(nbl + 1, np.int64))
    assert f(*head, *[v.ctypes.data for v in out.values()]) == 0
    L.pyhip_ilu_plan_free(h)
    return out


@pytest.mark.parametrize("cap", [0, 60, 1000])
@pytest.mark.parametrize("order", [AUTO, NATURAL, MULTICOLOR])
def test_sliced_solve_emulated_equals_the_triangular_solves(order, cap):
    """The slices, walked as the one-workgroup solve walks them, give the triangular solves
    of the permuted factor; sub-problems above the cap stay in the level lists."""
    import scipy.sparse.linalg as sl
    parts = [oracle_problem("ns", N=6), oracle_problem("bratu", N=9, space="C1", lam=1.0), oracle_problem("poisson", N=2),
             oracle_problem("poisson", N=11)]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=order)
    n = A.shape[0]
    rng = np.random.default_rng(1)
    lu = rng.uniform(-0.05, 0.05, len(P["pcol"]))
    lu[P["pdiag"]] = rng.uniform(1.0, 2.0, n)
    b = rng.standard_normal(n)
    F = sp.csr_matrix((lu, P["pcol"], P["prs"]), shape=(n, n))
    D = sp.diags(lu[P["pdiag"]])
    want = {0: sl.spsolve_triangular((sp.tril(F, -1) + sp.eye(n)).tocsr(), b, lower=True),
            1: sl.spsolve_triangular((sp.triu(F, 1) + D).tocsr(), b, lower=False)}
    small = [s for s in range(len(parts)) if off[s + 1] - off[s] <= cap]
    for side in (0, 1):
        S = _sliced((A, grp, order), off, cap, side)
        assert sorted(S["subs"]) == small
        # rows of the other sub-problems, every one in a level of its own side
        rest = np.concatenate([np.arange(off[s], off[s + 1]) for s in range(len(parts)) if s not in small] or [[]])
        assert np.array_equal(np.sort(S["big"]), rest) and S["big_ptr"][-1] == len(rest)
        for t, s in enumerate(S["subs"]):
            r0, m = off[s], off[s + 1] - off[s]
            x = np.append(b[r0:r0 + m], 0.0)
            seen = np.zeros(m, int)
            for lv in range(S["nlev"][t]):
                new = {}
                for wave in range(16 * t, 16 * t + 16):
                    lo, hi = S["chunk0"][wave:wave + 2]
                    assert (hi - lo) % 3 == 0
                    marks = S["idx"][lo:hi, :, 7].astype(int)
                    assert np.all(marks == marks[:, :1]) and np.all(np.diff(marks[:, 0] & 0xfff) >= 0)
                    acc = np.zeros(64)
                    for ch in range(lo, hi):
                        mark = int(S["idx"][ch, 0, 7])
                        if mark & 0xfff != lv:
                            continue
                        lanes = 1 << ((mark >> 12) & 7)
                        c = S["idx"][ch, :, :6].astype(int).T            # [step][lane]
                        q = S["src"][ch].transpose(0, 2, 1).reshape(6, 64)
                        assert lanes <= 16 and np.all(c <= m) and np.all((q < 0) == (c == m))
                        acc += (np.where(q >= 0, lu[q], 0.0) * x[c]).sum(0)
                        if mark >> 15:
                            continue
                        lane, acc, row = acc, np.zeros(64), S["idx"][ch, :, 6]
                        for g in range(0, 64, lanes):
                            if row[g] == 0xffff:
                                continue
                            assert np.all(row[g:g + lanes] == row[g])
                            r = int(row[g])
                            v = x[r] - lane[g:g + lanes].sum()
                            new[r] = v / lu[P["pdiag"][r0 + r]] if side else v
                            seen[r] += 1
                for r, v in new.items():   # rows of one level do not read each other
                    x[r] = v
            assert np.all(seen == 1)
            assert np.allclose(x[:m], want[side][r0:r0 + m], rtol=1e-12, atol=1e-13)


@pytest.mark.parametrize("cap", [0, 60])
@pytest.mark.parametrize("order", [AUTO, NATURAL, MULTICOLOR])
def test_level_solve_emulated_equals_the_triangular_solves(order, cap):
    """The level layout of the sub-problems above the cap, walked as the level kernels walk it
    (first lower level with the second, rows without upper entries finished by the lower
    solve), gives z = (L U)^-1 v in the problem's own numbering."""
    import scipy.sparse.linalg as sl
    parts = [oracle_problem("ns", N=6), oracle_problem("bratu", N=9, space="C1", lam=1.0), oracle_problem("poisson", N=11)]
    A, off, grp = _batch(parts)
    P = _plan(A.indptr, A.indices, off, is_p=grp, order=order)
    n = A.shape[0]
    rng = np.random.default_rng(2)
    lu = rng.uniform(-0.05, 0.05, len(P["pcol"]))
    lu[P["pdiag"]] = rng.uniform(1.0, 2.0, n)
    v = rng.standard_normal(n)
    F = sp.csr_matrix((lu, P["pcol"], P["prs"]), shape=(n, n))
    D = sp.diags(lu[P["pdiag"]])
    want = np.empty(n)
    w = sl.spsolve_triangular((sp.tril(F, -1) + sp.eye(n)).tocsr(), v[P["perm"]], lower=True)
    want[P["perm"]] = sl.spsolve_triangular((sp.triu(F, 1) + D).tocsr(), w, lower=False)
    big = np.concatenate([np.arange(off[s], off[s + 1]) for s in range(len(parts)) if off[s + 1] - off[s] > cap])

    L = _lib_ilu()
    rs, col = np.ascontiguousarray(A.indptr, np.int32), np.ascontiguousarray(A.indices, np.int32)
    so, g = np.ascontiguousarray(off, np.int64), np.ascontiguousarray(grp, np.int8)
    h = L.pyhip_ilu_plan_new(n, rs.ctypes.data_as(_lib.c_i32p), col.ctypes.data_as(_lib.c_i32p), len(so) - 1,
                             so.ctypes.data_as(_lib.c_i64p), g.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)), order, 64)
    f = L.pyhip_ilu_level_copy
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, _lib.c_i64p, ctypes.c_int, ctypes.c_int, _lib.c_i64p] + \
        [ctypes.c_void_p] * 5
    sides = []
    for side in (0, 1):
        sz = np.zeros(3, np.int64)
        head = [h, len(so) - 1, so.ctypes.data_as(_lib.c_i64p), cap, side, sz.ctypes.data_as(_lib.c_i64p)]
        assert f(*head, *[None] * 5) == 0
        a = (np.zeros((sz[0], 29), np.int64), np.zeros(sz[1], np.int32), np.zeros(sz[2], np.int32),
             np.zeros(sz[2], np.int32), np.zeros(sz[1], np.int32))
        assert f(*head, *[q.ctypes.data for q in a]) == 0
        sides.append(a)
    L.pyhip_ilu_plan_free(h)

    def row_sums(lv, col, src, x):
        rows, _, lanes, nseg = (int(q) for q in lv[:4])
        seg, steps, offs = lv[4:13], lv[13:21], lv[21:29]
        out, ns = np.zeros(rows), 8 // lanes
        for k in range(nseg):
            S = int(seg[k + 1] - seg[k]) * lanes
            m = S * ns * int(steps[k])
            c, q = col[offs[k]:offs[k] + m], src[offs[k]:offs[k] + m]
            e = (np.where(q >= 0, lu[q], 0.0) * x[c]).reshape(-1, seg[k + 1] - seg[k], lanes)
            out[seg[k]:seg[k + 1]] = e.sum(axis=(0, 2))
        assert seg[0] == 0 and seg[nseg] == rows
        return out

    y, z = np.full(n, np.nan), np.full(n, np.nan)
    levels, row, col, src, rsrc = sides[0]
    for k, lv in enumerate(levels):
        r = row[lv[1]:lv[1] + lv[0]]
        i, last = r & 0x7fffffff, r < 0
        # the second level reads v itself: its columns all lie in the first
        s = row_sums(lv, col, src, v if k <= 1 else y)
        y[i] = v[i] - s
        z[i[last]] = y[i[last]] / lu[rsrc[lv[1]:lv[1] + lv[0]][last]]
    levels, row, col, src, rsrc = sides[1]
    assert np.all(np.isfinite(z[row[:levels[0][0]]]))   # the first upper level is already done
    for lv in levels[1:]:
        r = row[lv[1]:lv[1] + lv[0]]
        z[r] = (y[r] - row_sums(lv, col, src, z)) / lu[rsrc[lv[1]:lv[1] + lv[0]]]
    assert np.allclose(z[big], want[big], rtol=1e-12, atol=1e-13)
    assert np.all(np.isnan(np.delete(z, big)))


def test_sliced_plan_of_many_small_problems_costs_about_as_much_as_their_row_order():
    """The layout is written out where it is used; the plan itself only cuts the levels. With
    the padded arrays written by the host it took 28 times the row order here, now 0.5."""
    import time
    A, off, grp = _batch([oracle_problem("bratu", N=8, space="C1", lam=1.0)])
    n, count = A.shape[0], 2048   # fewer than take the level lists
    rs = np.concatenate([A.indptr[:-1] + i * A.nnz for i in range(count)] + [[A.nnz * count]]).astype(np.int32)
    col = np.concatenate([A.indices + i * n for i in range(count)]).astype(np.int32)
    so, g = np.arange(count + 1, dtype=np.int64) * n, np.tile(grp, count).astype(np.int8)
    L, vp = _lib_ilu(), ctypes.c_void_p
    f = L.pyhip_ilu_sliced_copy
    f.argtypes = [vp, ctypes.c_int, _lib.c_i64p, ctypes.c_int, ctypes.c_int, _lib.c_i64p] + [vp] * 7
    order, sliced = [], []
    for _ in range(3):
        t = time.perf_counter()
        h = L.pyhip_ilu_plan_new(n * count, rs.ctypes.data_as(_lib.c_i32p), col.ctypes.data_as(_lib.c_i32p), count,
                                 so.ctypes.data_as(_lib.c_i64p), g.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)), AUTO, 64)
        order.append(time.perf_counter() - t)
        sz = np.zeros(4, np.int64)
        t = time.perf_counter()
        assert f(h, count, so.ctypes.data_as(_lib.c_i64p), 20000, 0, sz.ctypes.data_as(_lib.c_i64p), *[None] * 7) == 0
        sliced.append(time.perf_counter() - t)
        L.pyhip_ilu_plan_free(h)
        assert sz[0] == count
    assert min(sliced) <= 6 * min(order)


def test_level_plan_of_a_long_band_costs_less_than_its_row_order():
    """The level lists of a matrix that no workgroup takes (120000 rows, half bandwidth 2: a
    plugin factorises such a matrix anew every time): 0.04 of the row order, 0.7 when the
    padded columns were written by the host."""
    import time
    n = 120000
    A = sp.diags([np.ones(n - abs(k)) for k in range(-2, 3)], range(-2, 3), shape=(n, n)).tocsr()
    A.sort_indices()
    rs, col = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    so, g = np.array([0, n], np.int64), np.zeros(n, np.int8)
    L, vp = _lib_ilu(), ctypes.c_void_p
    f = L.pyhip_ilu_level_copy
    f.argtypes = [vp, ctypes.c_int, _lib.c_i64p, ctypes.c_int, ctypes.c_int, _lib.c_i64p] + [vp] * 5
    order, level = [], []
    for _ in range(3):
        t = time.perf_counter()
        h = L.pyhip_ilu_plan_new(n, rs.ctypes.data_as(_lib.c_i32p), col.ctypes.data_as(_lib.c_i32p), 1,
                                 so.ctypes.data_as(_lib.c_i64p), g.ctypes.data_as(ctypes.POINTER(ctypes.c_int8)), AUTO, 64)
        order.append(time.perf_counter() - t)
        sz = np.zeros(3, np.int64)
        t = time.perf_counter()
        assert f(h, 1, so.ctypes.data_as(_lib.c_i64p), 20000, 0, sz.ctypes.data_as(_lib.c_i64p), *[None] * 5) == 0
        level.append(time.perf_counter() - t)
        L.pyhip_ilu_plan_free(h)
        assert sz[1] == n
    assert min(level) <= 0.35 * min(order)


@pytest.mark.parametrize("kind,kw,tiny", [("bratu", dict(N=4, space="C1", lam=1.0), True),
                                          ("poisson", dict(N=4), True), ("ns", dict(N=2), False)])
def test_many_tiny_problems_take_the_level_lists(kind, kw, tiny):
    """3072 sub-problems of at most 256 short rows share the level launches, 3071 take a
    workgroup each, and so do rows of more than 24 entries a side; every slice of a tiny one
    has four lanes a row (the sums of the level kernels)."""
    A, off, grp = _batch([oracle_problem(kind, **kw)])
    n = A.shape[0]
    for count in (3071, 3072):
        B = sp.csr_matrix((np.ones(A.nnz * count), np.tile(A.indices, count) + np.repeat(np.arange(count) * n, A.nnz),
                           np.concatenate([A.indptr[:-1] + i * A.nnz for i in range(count)] + [[A.nnz * count]])),
                          shape=(n * count, n * count))
        S = _sliced((B, np.tile(grp, count), AUTO), np.arange(count + 1) * n, 20000, 0)
        assert len(S["subs"]) == (0 if tiny and count == 3072 else count)
        assert len(S["big"]) == n * (count - len(S["subs"]))
        if tiny and len(S["subs"]):
            rows = S["idx"][:, :, 6] != 0xffff
            assert set((S["idx"][rows.any(1), 0, 7] >> 12) & 7) == {2}


@pytest.mark.parametrize("n,band", [(130, 129), (260, 259), (700, 120)])
@pytest.mark.parametrize("order", [NATURAL, MULTICOLOR])
def test_slices_over_several_chunks(order, n, band):
    """Rows of more than 96 entries a side (16 lanes, 6 steps): their slices go on over two and
    three chunks, every entry taken once, by the lane of its row, the same row in each chunk, with
    the go-on mark on all but the last."""
    offs = [k for k in range(-band, band + 1)]
    A = sp.diags([np.ones(n - abs(k)) for k in offs], offs, shape=(n, n)).tocsr()
    A.sort_indices()
    off, grp = np.array([0, n]), np.zeros(n, np.int8)
    P = _plan(A.indptr, A.indices, off, order=order)
    for side in (0, 1):
        S = _sliced((A, grp, order), off, 1000, side)
        k0, k1 = (P["prs"][:-1], P["pdiag"]) if side == 0 else (P["pdiag"] + 1, P["prs"][1:])
        taken, longest = [], 0
        for w in range(16):
            rows, length = None, 0
            for ch in range(*S["chunk0"][w:w + 2]):
                q = S["src"][ch].transpose(0, 2, 1).reshape(6, 64)
                row, mark = S["idx"][ch, :, 6], int(S["idx"][ch, 0, 7])
                assert rows is None or np.array_equal(rows, row)
                r = np.broadcast_to(row.astype(int), q.shape)[q >= 0]
                assert np.all((q[q >= 0] >= k0[r]) & (q[q >= 0] < k1[r]))
                assert np.array_equal(S["idx"][ch, :, :6].T[q >= 0], P["pcol"][q[q >= 0]])
                taken.append(q[q >= 0])
                length += 1
                longest = max(longest, length)
                rows, length = (row, length) if mark >> 15 else (None, 0)
            assert rows is None
        assert np.array_equal(np.sort(np.concatenate(taken)),
                              np.concatenate([np.arange(a, b) for a, b in zip(k0, k1)]))
        assert longest == -(-int((k1 - k0).max()) // 96)
