"""Element kernels and the gather at the edges of their workgroups: one element, a last
workgroup that is nearly empty, exactly full ones and the next size (128 triangles; 32768, 65536
and 81920 triangles, where FP64 changes the kernel; 7 and 28 bricks, 128 (element, node)
pairs of Taylor-Hood elements, 512 matrix entries), steady and with the time derivative.

Bar: FP64 bitwise against the oracle (1e-12 where the exponential enters, as in the parity
tests). FP32 against FP64, relative to the largest entry: (27 + 16 N) 2^-24. A sum of at most
27 points gives 27 * 2^-24; the rounded coordinates (2^-25 in the unit square) enter the
tangents with shape derivatives whose absolute sum is at most 8, over tangents of length 1 / N,
8 N * 2^-25 = 4 N * 2^-24, and the entry holds four factors of the metric (two gradients and
the weight, of degree two)."""
import numpy as np
import pytest

from oracle import timestepping as ots
from tests.test_gpu_parity import build, rel

pytestmark = pytest.mark.gpu

SIZES = ([("bratu", dict(N=N, space=sp, lam=2.0)) for sp in ("C1", "C2") for N in (2, 8, 9, 17)] +
         [("bratu", dict(N=N, space=sp, lam=2.0)) for sp, N in (("C1", 181), ("C1", 182), ("C2", 127), ("C2", 128),
                                                                ("C2", 182))] +
         [("poisson", dict(N=N)) for N in (2, 8, 9, 181, 182, 203)] +
         [("rd", dict(N=N)) for N in (1, 2, 3, 4)] +
         [("ns", dict(N=N)) for N in (2, 4, 15)])


@pytest.mark.parametrize("transient", [False, True])
@pytest.mark.parametrize("kind,kw", SIZES)
def test_assembly_at_workgroup_edges(gpu, kind, kw, transient):
    import torch
    P, op = build(kind, kw)
    if not P.ndof:
        pytest.skip("no free value")
    rng = np.random.default_rng(kw["N"])
    x, h1, h2 = (rng.uniform(-0.4, 0.4, P.ndof) for _ in range(3))
    P.set_current_dofs(x)
    tw = ots.bdf2_weights(0.05, 0.08)
    if transient:
        P.set_time_state(tw, *(torch.tensor(h, dtype=torch.float64, device=P.device) for h in (h1, h2)))
        op.set_time(tw, h1, h2)
    r, rs, col, val = op.get_jacobian(x)
    R, J = P.assemble_jacobian()
    only = P.get_residuals()
    r32, v32 = P.assemble_device("f32")
    _, v64 = P.assemble_device("f64")
    assert np.array_equal(J.indptr, rs) and np.array_equal(J.indices, col)
    assert rel(J.data, val) <= 1e-12 and rel(R, r) <= 1e-12
    if kind != "bratu":
        assert np.array_equal(J.data, val)
    if kind not in ("bratu", "poisson"):
        assert np.array_equal(R, r)
    assert np.array_equal(only, R)
    scale = float(v64.abs().max())
    tol = (27 + 16 * kw["N"]) * 2.0**-24
    assert float((v32.double() - v64).abs().max()) <= tol * scale
    assert np.max(np.abs(r32.cpu().numpy() - R)) <= tol * max(scale, np.max(np.abs(R)))


@pytest.mark.parametrize("kind,kw", [("bratu", dict(N=N, space=sp, lam=float(N * N))) for sp, N in
                                     (("C1", 181), ("C1", 182), ("C2", 127), ("C2", 128), ("C2", 182))] +
                         [("poisson", dict(N=N)) for N in (127, 182, 203)])
def test_fp32_sources_on_many_elements(gpu, kind, kw):
    """The FP32 bar above is relative to the stiffness, beside which a source of order h^2 does not
    count on a fine mesh. Here lambda = N^2 makes the Bratu terms as large as the stiffness, and
    the residual without dofs is the source alone, held to the same bar relative to its own
    largest entry."""
    import torch
    P, op = build(kind, kw)
    tol = (27 + 16 * kw["N"]) * 2.0**-24

    def assemble():
        out = [P.assemble_device(p) for p in ("f32", "f64")]
        torch.cuda.synchronize()
        return out

    rng = np.random.default_rng(kw["N"])
    if kind == "bratu":
        P.set_current_dofs(rng.uniform(-0.4, 0.4, P.ndof))
        (r32, v32), (r64, v64) = assemble()
        assert float((v32.double() - v64).abs().max()) <= tol * float(v64.abs().max())
        assert float((r32 - r64).abs().max()) <= tol * max(float(v64.abs().max()), float(r64.abs().max()))
    P.set_current_dofs(np.zeros(P.ndof))
    (r32, _), (r64, _) = assemble()
    assert float(r64.abs().max()) > 0 and float((r32 - r64).abs().max()) <= tol * float(r64.abs().max())


@pytest.mark.parametrize("transient", [False, True])
@pytest.mark.parametrize("cubes", [(1,), (1, 1), (1, 1, 1), (1,) * 7, (2,), (2, 1), (13,), (13, 5), (14,)])
def test_brick_kernels_meet_at_their_rule(gpu, cubes, transient):
    """1, 2, 3, 7, 8, 9, 2197, 2322 and 2744 bricks, on both sides of the sizes where the FP64
    residual and the FP64 matrix change the kernel: the residual alone, the residual beside the
    matrix and each cube's residual alone in a problem are the same bits."""
    import torch
    from pyoomph_amd import workloads as wl
    from pyoomph_amd.problem import Problem
    tw = ots.bdf2_weights(0.05, 0.08)

    def assemble(parts, x, h1, h2):
        P = Problem(parts)
        P.set_current_dofs(x)
        if transient:
            P.set_time_state(tw, *(torch.tensor(h, dtype=torch.float64, device=P.device) for h in (h1, h2)))
        res, vals = P.assemble_device("f64")
        torch.cuda.synchronize()
        return P, P.get_residuals(), res.cpu().numpy(), vals.cpu().numpy()

    parts = [wl.reaction_diffusion_cube(N, seed=i) for i, N in enumerate(cubes)]
    rng = np.random.default_rng(len(cubes))
    v = [rng.uniform(-0.4, 0.4, sum((2 * N - 1) ** 3 for N in cubes)) for _ in range(3)]
    P, only, res, vals = assemble(parts, *v)
    assert np.array_equal(only, res) and np.isfinite(vals).all()
    d = e = 0
    for N, part in zip(cubes, parts):
        n = (2 * N - 1) ** 3
        _, o1, r1, v1 = assemble([part], *(x[d:d + n] for x in v))
        assert np.array_equal(o1, only[d:d + n]) and np.array_equal(r1, res[d:d + n])
        assert np.array_equal(v1, vals[e:e + v1.size])
        d, e = d + n, e + v1.size
