"""spmv variants with one row per lane group (spmv.h): the same bits as 8 lanes over 256-row
blocks, on every matrix of a solve (finest, coarse, transfer), in FP64 and FP32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["bratu_small", "bratu", "rd", "ns"])
def test_one_row_variants_keep_bits(gpu, monkeypatch, kind, precision):
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem
    if kind == "ns" and precision == "f32":
        pytest.skip("the block preconditioner runs FP64 solves")
    parts = {"bratu_small": lambda: [wl.bratu(3, "C1", 1.0), wl.bratu(2, "C2", 2.0)],
             "bratu": lambda: [wl.bratu(33, "C2", 2.0), wl.bratu(40, "C1", 1.0)],
             "rd": lambda: [wl.reaction_diffusion_cube(7)], "ns": lambda: [wl.lid_driven_cavity(9)]}[kind]()
    xs = []
    for v in ("8", "9", "10", "11", None):   # None: the rule
        if v is None:
            monkeypatch.delenv("PYHIP_SPMV_LPR", raising=False)
        else:
            monkeypatch.setenv("PYHIP_SPMV_LPR", v)
        P = Problem(parts)
        if kind == "ns":
            P.preconditioner, P.newton_solver_tolerance = "block", 1e-10
        else:
            P.krylov, P.preconditioner = "cg", "amg"
        P.linear_precision = precision
        st = P.solve()
        assert all(s["converged"] for s in st)
        xs.append(P.get_current_dofs())
    for x in xs[1:]:
        assert np.array_equal(x, xs[0])
