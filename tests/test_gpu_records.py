"""A scattered numbering, whose arrays are plain records, against the numbering
of the generator, whose arrays are interleaved: the same mesh, state and
directions, so every result is the same sum in another order.

Both round at the size of what they sum; the fields carry noise in every
component, so no result is small against its terms, and 1e-11 of the largest value
of each component is some thousand roundings."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from aerof_dev_amd import FlowParams, LowMachPrec, ViscousParams, init_state
from aerof_dev_amd import mesh as M

pytestmark = pytest.mark.gpu
LM = LowMachPrec(min_mach=0.02, slope=1.5, cutoff=0.9, shock_reducer=0.3, irey=1e-4)
FLOWS = {
    "euler": dict(mach=0.5),
    "euler first order": dict(mach=0.5, second_order=False),
    "low Mach": dict(mach=0.1, low_mach=LM),
    "viscous": dict(mach=0.4, p_inf=1.0 / (1.4 * 0.16), viscous=ViscousParams(reynolds=50.0, viscous_cst=1.0)),
}


@pytest.fixture(scope="module")
def meshes():
    """A viscous channel of 17,576 nodes (275 slices, the last of 40 nodes) and the
    same with its nodes shuffled, and the map old -> new."""
    m = M.kuhn_box(25, 25, 25, jitter=0.15, seed=3, face_codes=M.VISCOUS_CHANNEL)
    renum = np.random.default_rng(5).permutation(m.num_nodes).astype(np.int32)
    s = M.renumber(m, renum)
    for x, scattered in ((m, False), (s, True)):
        e = M.edges(x).astype(np.int64)
        a, b = np.concatenate([e[:, 0], e[:, 1]]), np.concatenate([e[:, 1], e[:, 0]])
        lines = np.unique((a // 64) * x.num_nodes + b // 8).size / a.size
        assert (lines > 0.25) == scattered
    return m, s, renum


def _pair(gpu, meshes, flow):
    """Per mesh: operator, and a function that puts a host field into its order."""
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    m, s, renum = meshes
    p = FlowParams(alpha=0.05, **FLOWS[flow])
    old = np.empty_like(renum)
    old[renum] = np.arange(renum.size)
    both = []
    for mesh, order in ((m, np.arange(renum.size)), (s, old)):
        both.append((SpaceOperator(mesh, p), lambda f, order=order: torch.from_numpy(f[order].copy()).to(gpu)))
    U = init_state(p, m.X, "noise", 0.02, seed=5)
    # in the velocity too: where a difference is zero, the limiter's derivative hangs
    # on the rounding of the slope beside it
    du = 0.02 * p.mach * np.random.default_rng(8).standard_normal((U.shape[0], 3))
    U[:, 4] += (U[:, 1:4] * du).sum(1) + 0.5 * U[:, 0] * (du ** 2).sum(1)
    U[:, 1:4] += U[:, :1] * du
    return p, both, U, renum


def _same(a, b, renum, what):
    a, b = a.cpu().numpy(), b.cpu().numpy()[renum]
    a, b = (x.reshape(x.shape[0], -1) for x in (a, b))
    err = np.abs(a - b).max(0) / np.abs(a).max(0)
    print(f"[records] {what}: {err.max():.1e}", flush=True)
    assert np.all(np.isfinite(a)) and np.all(err <= 1e-12), what


@pytest.mark.parametrize("flow", list(FLOWS))
def test_residual_and_implicit(gpu, meshes, flow):
    import torch
    from aerof_dev_amd.operators import GmresSolver, MatVecProdFD, MatVecProdH1
    p, both, U, renum = _pair(gpu, meshes, flow)
    rng = np.random.default_rng(6)
    v = rng.standard_normal(U.shape)
    res = []
    for op, put in both:
        Ud, out = put(U), {}
        R, V = torch.empty_like(Ud), torch.empty_like(Ud)
        assert op.compute_residual(Ud, R) == 0
        out["residual"] = R
        op.conservative_to_primitive(Ud, V)
        g = [torch.empty_like(Ud) for _ in range(3)]
        op.compute_gradients(V, *g)
        out["gradients"] = torch.cat(g, 1)
        h1, dt = MatVecProdH1(op), torch.empty(op.num_nodes, dtype=torch.float64, device=gpu)
        h1.timestep(Ud, 20.0, dt)
        out["time step"] = dt
        y, x = torch.empty_like(Ud), torch.empty_like(Ud)
        h1.evaluate(Ud, dt, 0)
        h1.apply(put(v), y)
        h1.prec_apply(put(v), x)
        out["H1 product"], out["block Jacobi"] = y, x
        z = torch.empty_like(Ud)
        its, _ = GmresSolver(op, 30, 1e-13, 300).solve(put(v), z)
        assert its < 300
        h1.apply(z, (w := torch.empty_like(Ud)))
        assert float(torch.linalg.norm(w - put(v))) <= 1e-11 * float(torch.linalg.norm(put(v)))
        if not p.viscous:
            fd, q = MatVecProdFD(op, 2), torch.empty_like(Ud)
            assert fd.evaluate(Ud, dt) == 0 and fd.apply(put(v * np.abs(U)), q) == 0
            fd.release()
        # the other ways to the same residual give the same bits
        Q = torch.empty_like(Ud)
        from aerof_dev_amd._abi import check, lib
        assert check(lib().aerofx_residual_noalloc(op._h, C.c_void_p(Ud.data_ptr()), C.c_void_p(Q.data_ptr()), 0),
                     "residual_noalloc") == 0
        assert torch.equal(Q, R)
        op.set_residual_kernels("staged")
        assert op.compute_residual(Ud, Q) == 0 and torch.equal(Q, R)
        res.append(out)
    for k in res[0]:
        _same(res[0][k], res[1][k], renum, f"{flow} {k}")
    for op, _ in both:
        op.close()


@pytest.mark.parametrize("flow", [f for f in FLOWS if f != "low Mach"])
def test_derivatives(gpu, meshes, flow):
    import torch
    from aerof_dev_amd.operators import MatVecProdH2
    p, both, U, renum = _pair(gpu, meshes, flow)
    rng = np.random.default_rng(7)
    dU, lam, dX = rng.standard_normal(U.shape) * np.abs(U), rng.standard_normal(U.shape), \
        rng.standard_normal((U.shape[0], 3)) * 1e-2
    res = []
    for op, put in both:
        Ud, out = put(U), {}
        new = lambda w=5: torch.empty((U.shape[0], w), dtype=torch.float64, device=gpu)  # noqa: E731
        for name, a, b in (("dR/dU", dU, None), ("dR/dX", None, dX)):
            d = new()
            assert op.compute_derivative_of_residual(Ud, d, None if a is None else put(a),
                                                     None if b is None else put(b)) == 0
            out[name] = d
        gu, gx, gu2 = new(), new(3), new()
        op.compute_transpose_derivative_of_residual(Ud, put(lam), gu, gx)
        op.compute_transpose_derivative_of_residual(Ud, put(lam), gu2)
        out["dR/dU^T"], out["dR/dX^T"], out["dR/dU^T alone"] = gu, gx, gu2
        h2, y = MatVecProdH2(op), new()
        assert h2.evaluate(Ud) == 0 and h2.apply(put(dU), y) == 0
        h2.release()
        out["exact product"] = y
        jU, jX = new(), new(3)
        out["J"] = torch.tensor([op.wall_force(Ud, (0.3, 0.1, 1.0), jU, jX)] * U.shape[0], dtype=torch.float64)
        wall = jU.abs().sum(1) > 0
        assert 0 < int(wall.sum()) < U.shape[0]
        out["dJ/dU"], out["dJ/dX"] = jU, jX
        res.append(out)
    for k in res[0]:
        _same(res[0][k], res[1][k], renum, f"{flow} {k}")
    for op, _ in both:
        op.close()


@pytest.mark.parametrize("flow", ["euler", "viscous"])
def test_newton(gpu, meshes, flow):
    """Eight steps of each numbering: the Krylov solves stop at their tolerance
    (1e-2), not at the same vector, so the histories agree to that, and the first
    residual to rounding."""
    from aerof_dev_amd.operators import steady_solve
    p, both, U, renum = _pair(gpu, meshes, flow)
    h = [steady_solve(op, put(U), precision=0, max_steps=8)["history"] for op, put in both]
    for op, _ in both:
        op.close()
    assert len(h[0]) == len(h[1]) == 9
    assert abs(h[0][0] - h[1][0]) <= 1e-12 * h[0][0]
    assert np.max(np.abs(h[0] - h[1]) / h[0]) <= 3e-2


def test_failsafe(gpu, meshes):
    """Tags and residual of the scattered numbering against the oracle's (the tags
    go by the edges' direction, so the numberings tag different nodes)."""
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    m = meshes[1]
    p = FlowParams(mach=0.5)
    N = m.num_nodes
    U = init_state(p, m.X, "noise", 0.01, seed=8)
    bad = U.copy()
    bad[[N // 2, N - 1], 4] = -2.0
    om = O.OracleMesh(m, p)
    tags = np.zeros((3, N), dtype=np.int32)
    op = SpaceOperator(m, p)
    op.set_failsafe(2)
    R = torch.empty((N, 5), dtype=torch.float64, device=gpu)
    for state in (bad, U):
        Rr, ierr, _ = om.residual_fs(state, 2, tags)
        assert op.compute_residual(torch.from_numpy(state).to(gpu), R) == ierr
        np.testing.assert_array_equal(np.stack(op.failsafe_nodes()), tags)
    assert ierr == 0 and tags[2].any()
    assert np.abs(R.cpu().numpy() - Rr).max() <= 1e-12 * np.abs(Rr).max()
    op.close()
