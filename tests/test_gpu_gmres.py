"""GMRES orthogonalisation kernels (gmres_kernels.h) at the edges of their chunks: systems
around 256, 512 and 1024 rows per block, odd row counts, and one whose reductions take a
launch of their own; batches whose sub-problems use different chunk lengths."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as sl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 255, 257, 32768, 32769, 131073, 700001])
def test_plugin_gmres_solves_nonsymmetric_systems(gpu, n):
    from pyoomph_amd.plugins import HIPKrylovSerial
    rng = np.random.default_rng(n)
    # a convection-dominated chain with random far couplings: a dozen ILU(0)-GMRES iterations
    far = max(1, n // 3)
    A = (sp.diags([np.full(n, 4.0), rng.uniform(-2.5, -0.5, n - 1), rng.uniform(0.0, 1.0, n - 1)], [0, -1, 1])
         + sp.diags([rng.uniform(-0.8, 0.8, n - far)], [far], shape=(n, n))).tocsr()
    A.sum_duplicates()
    A.sort_indices()
    b = rng.standard_normal(n)
    x = b.copy()
    S = HIPKrylovSerial(None)
    S.solve_serial(1, n, A.nnz, 1, A.data, A.indices, A.indptr, None, n, 1)
    S.solve_serial(2, n, A.nnz, 1, None, None, None, x, n, 1)
    # the solver's stop is a relative residual of 1e-10 (1 % slack in its final check)
    assert np.linalg.norm(A @ x - b) <= 1.02e-10 * np.linalg.norm(b)
    if n < 1000:
        want = sl.spsolve(A.tocsc(), b)
        assert np.linalg.norm(x - want) <= 1e-8 * np.linalg.norm(want)


@pytest.mark.parametrize("opts", [dict(preconditioner="amg"), dict(preconditioner="ilu0"),
                                  dict(preconditioner="amg", linear_precision="f32"),
                                  dict(preconditioner="jacobi", gmres_restart=200)])
def test_gmres_batch_with_different_chunk_lengths_equals_alone(gpu, opts):
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem

    def solve(parts):
        P = Problem(parts)
        P.krylov = "gmres"
        for k, v in opts.items():
            setattr(P, k, v)
        P.gmres_max_iters = 20000
        st = P.solve()
        assert all(s["converged"] for s in st)
        x = P.get_current_dofs()
        return [P.sub_dofs(i, x) for i in range(len(parts))]

    parts = [wl.bratu(9, "C1", 1.0), wl.bratu(100, "C2", 1.0), wl.bratu(40, "C2", 2.0)]
    if opts["preconditioner"] == "jacobi":
        parts = [wl.bratu(9, "C1", 1.0), wl.bratu(30, "C2", 2.0)]
    for mp, x in zip(parts, solve(parts)):
        assert np.array_equal(x, solve([mp])[0])


def test_sums_by_blocks_and_by_launches_have_the_same_bits(gpu):
    """3481 rows (14 chunks: every block adds up the partials), alone and beside 297025 rows (291
    chunks: launches add them from 29 vectors on), with more than 29 iterations."""
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem

    def solve(parts):
        P = Problem(parts)
        P.krylov, P.preconditioner, P.gmres_restart, P.gmres_max_iters = "gmres", "ilu0", 60, 20000
        st = P.solve()
        assert all(s["converged"] for s in st) and st[0]["linear_iters"] > 2 * 29
        return P.sub_dofs(0, P.get_current_dofs())

    small = wl.bratu(60, "C1", 1.5)
    assert np.array_equal(solve([small]), solve([small, wl.bratu(546, "C1", 1.0)]))
