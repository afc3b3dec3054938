"""Preconditioned CG vector kernels (cg_kernels.h) at the edges of their chunks: sub-problems
below and above 256, 32768 and 131072 rows, one whose sums take a launch of their own, and a
batch whose sub-problems stop at different iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _solve(parts, precision="f64", precond="amg"):
    from pyoomph_amd.problem import Problem
    P = Problem(parts)
    P.krylov, P.preconditioner, P.linear_precision = "cg", precond, precision
    st = P.solve()
    assert all(s["converged"] and s["linear_failures"] == 0 for s in st)
    x = P.get_current_dofs()
    return [P.sub_dofs(i, x) for i in range(len(parts))], P


@pytest.mark.parametrize("precision,precond", [("f64", "amg"), ("f32", "amg"), ("f64", "ilu0")])
def test_batch_of_different_chunk_lengths_equals_alone(gpu, precision, precond):
    from pyoomph_amd import workloads as wl
    sizes = [(2, "C1"), (16, "C1"), (17, "C1"), (91, "C2"), (46, "C2")]
    if precond == "amg":
        sizes.append((182, "C2"))   # 131769 rows: 1024-row chunks
    parts = [wl.bratu(N, sp, 0.7 + 0.3 * i) for i, (N, sp) in enumerate(sizes)]
    together, _ = _solve(parts, precision, precond)
    for mp, x in zip(parts, together):
        assert np.array_equal(x, _solve([mp], precision, precond)[0][0])


def test_sums_of_a_long_vector(gpu):
    """813^2 rows: 646 chunks, summed by a launch of their own. The residual of the solution
    is below the Newton tolerance."""
    from pyoomph_amd import workloads as wl
    (x,), P = _solve([wl.bratu(814, "C1", 1.0)])
    assert P.ndof == 813 * 813
    assert np.max(np.abs(P.get_residuals())) < 1e-8 and np.isfinite(x).all()
