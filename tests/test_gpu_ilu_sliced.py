"""One-workgroup ILU(0) solves (ilu_sliced.h): sub-problems on both sides of the rule that
hands them a workgroup, alone and mixed in one batch, and in the solver plugin."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sl

pytestmark = pytest.mark.gpu


def _solve(parts, precision="f64"):
    from pyoomph_amd.problem import Problem
    P = Problem(parts)
    P.preconditioner = "ilu0"
    if precision == "f32":
        P.linear_precision = "f32"
    st = P.solve()
    x = P.get_current_dofs()
    assert all(s["converged"] and s["linear_failures"] == 0 for s in st)
    return [P.sub_dofs(i, x) for i in range(len(parts))]


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_batch_of_handled_and_level_scheduled_problems_equals_each_alone(gpu, precision):
    from pyoomph_amd import workloads as wl
    # 64^2 P2: more entries than a workgroup takes; the others: one workgroup each, natural
    # order up to N = 17 P2, multicolour above; 2^2 P1: a single unknown
    parts = [wl.bratu(17, "C2", 1.5), wl.bratu(64, "C2", 1.0), wl.bratu(2, "C1", 2.0), wl.bratu(33, "C1", 0.7),
             wl.bratu(23, "C2", 2.5)]
    together = _solve(parts, precision)
    for mp, x in zip(parts, together):
        assert np.array_equal(x, _solve([mp], precision)[0])


@pytest.mark.parametrize("n,band", [(1, 1), (63, 3), (65, 64), (1500, 40), (20001, 2)])
def test_plugin_solves_matrices_at_the_edges_of_the_rule(gpu, n, band):
    """One row; rows of a slice and of a level that do not fill it; dense rows, many lanes
    each; one row more than a workgroup's LDS holds."""
    from pyoomph_amd.plugins import HIPKrylovSerial
    rng = np.random.default_rng(n)
    offs = [k for k in range(-band, band + 1) if abs(k) < n]
    A = sp.diags([rng.uniform(-1, 1, n - abs(k)) for k in offs], offs, shape=(n, n)).tolil()
    A.setdiag(2.0 * band + 2.0)
    A = A.tocsr()
    b = rng.standard_normal(n)
    x = b.copy()
    S = HIPKrylovSerial(None)
    S.solve_serial(1, n, A.nnz, 1, A.data, A.indices, A.indptr, None, n, 1)
    S.solve_serial(2, n, A.nnz, 1, None, None, None, x, n, 1)
    want = sl.spsolve(A.tocsc(), b)
    assert np.linalg.norm(x - want) <= 1e-9 * np.linalg.norm(want)


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_large_problem_solves_again_after_a_small_one(gpu, precision):
    """The LDS limit of the kernel is one of the function, whatever problem was set up last:
    9801 rows (78 KB in FP64), then 49, both alive, then the large one without a new set-up."""
    import torch
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem

    def solve(P):
        with torch.cuda.stream(P._stream):
            P.dofs.zero_()
        assert all(s["converged"] and s["linear_failures"] == 0 for s in P.solve())
        return P.get_current_dofs()

    large, small = (Problem([wl.bratu(N, "C1", 1.0)]) for N in (100, 8))
    for P in (large, small):
        P.preconditioner, P.linear_precision = "ilu0", precision
    x = solve(large)
    solve(small)
    assert np.array_equal(x, solve(large))


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("N,space", [(2, "C1"), (4, "C2"), (8, "C1")])
def test_tiny_problems_have_the_same_bits_in_workgroups_and_level_launches(gpu, N, space, precision):
    """3072 tiny sub-problems share the level launches; a few of them take a workgroup each."""
    from pyoomph_amd import workloads as wl
    few = [wl.bratu(N, space, 0.5 + 0.7 * i) for i in range(4)]
    # a larger one beside them keeps its workgroup
    want = _solve(few, precision)
    got = _solve(few * 768 + [wl.bratu(20, "C2", 1.0)], precision)
    for i in (0, 1, 2, 3, 1536, 3071):
        assert np.array_equal(got[i], want[i % 4])
    assert np.array_equal(got[-1], _solve([wl.bratu(20, "C2", 1.0)], precision)[0])


@pytest.mark.parametrize("n", [65, 96, 97, 130, 200, 256, 257, 300])
def test_dense_matrices_are_factorised_exactly(gpu, n):
    """ILU(0) of a full matrix is its LU in any order: rows of more than 64 lower and upper
    entries, of exactly kIluRow = 256 entries (in LDS) and more (in memory), and slices that go
    on over two and three chunks (more than 96 entries a side). One iteration then leaves the
    rounding of an elimination, n 2^-52 times a growth of at most 2 on a diagonally dominant
    matrix, far below the 1e-10 at which a solve with wrong factors would stop."""
    from pyoomph_amd.plugins import HIPKrylovSerial
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n))
    A[np.arange(n), np.arange(n)] = np.abs(A).sum(1) + 1.0
    A = sp.csr_matrix(A)
    b = rng.standard_normal(n)
    x = b.copy()
    S = HIPKrylovSerial(None)
    S.solve_serial(1, n, A.nnz, 1, A.data, A.indices, A.indptr, None, n, 1)
    S.solve_serial(2, n, A.nnz, 1, None, None, None, x, n, 1)
    assert np.linalg.norm(A @ x - b) <= 8 * n * 2.0**-52 * np.linalg.norm(b)
