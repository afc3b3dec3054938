"""The V-cycle's coarse levels in one workgroup per sub-problem against the same levels in
launches of their own: a small sub-problem runs the whole cycle in its workgroup when it is
alone, and only the last levels beside a large one; the bits have to be the same. The row products of the set-up take other lane counts
alone than in the batch (by the mean row length), with the same sums. Sizes: below
the coarsest level's 48 rows, just above, one pass of 256 rows and the next, several levels,
and sub-problems of one batch that end on different levels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["bratu", "rd", "ns"])
def test_tail_gives_the_bits_of_the_launches(gpu, kind, precision):
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem
    if kind == "ns" and precision == "f32":
        pytest.skip("the block preconditioner runs FP64 solves")
    small = {"bratu": lambda: [wl.bratu(N, sp, 1.5) for N, sp in
                               ((3, "C2"), (4, "C2"), (9, "C1"), (8, "C2"), (9, "C2"), (33, "C1"), (25, "C2"))],
             "rd": lambda: [wl.reaction_diffusion_cube(N) for N in (2, 3, 5)],
             "ns": lambda: [wl.lid_driven_cavity(N, 50.0) for N in (3, 9)]}[kind]()
    large = {"bratu": lambda: wl.bratu(96, "C2", 1.5), "rd": lambda: wl.reaction_diffusion_cube(11),
             "ns": lambda: wl.lid_driven_cavity(40, 50.0)}[kind]()

    def solve(parts):
        P = Problem(parts)
        if kind == "ns":
            P.preconditioner, P.newton_solver_tolerance = "block", 1e-9
        else:
            P.krylov, P.preconditioner = "cg", "amg"
        P.linear_precision = precision
        assert all(s["converged"] for s in P.solve())
        return P, P.get_current_dofs()

    B, xb = solve(small + [large])
    for i, part in enumerate(small):
        _, xa = solve([part])
        assert np.array_equal(xa, B.sub_dofs(i, xb)), i
