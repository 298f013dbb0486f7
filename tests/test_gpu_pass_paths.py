"""Paths of the passes that regularly numbered boxes and channels do not take.

The gradient pass holds the different neighbours of 64 consecutive nodes in LDS:
512 in the first batch of loads, the rest in a loop, up to 1024 (beyond, or with a
row of more than 64 neighbours, it gathers per entry); it reads 16 neighbours'
places at a time.  The meshes here lie on both sides of each limit.  From 6144
slices of 64 nodes on the flux pass takes whole rows, unless one is too long; of a
shuffled numbering the arrays are plain records.  The residual is held
against the oracle to 1e-12 of each sum's magnitude, as on any mesh."""
import os
import sys

import numpy as np
import pytest

import oracle as O
from aerof_dev_amd import FlowParams, LowMachPrec, init_state
from aerof_dev_amd import mesh as M
sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_edge_cases import _cone  # noqa: E402

pytestmark = pytest.mark.gpu
LM = LowMachPrec(min_mach=0.02, slope=1.5, cutoff=0.9, shock_reducer=0.3, irey=1e-4)


def _shuffled(m, seed, run=1):
    """The nodes, or runs of consecutive ones, in random order."""
    N = m.num_nodes
    order = np.random.default_rng(seed).permutation((N + run - 1) // run)
    old = (order[:, None] * run + np.arange(run)).ravel()
    renum = np.empty(N, dtype=np.int32)
    renum[old[old < N]] = np.arange(N, dtype=np.int32)
    return M.renumber(m, renum)


def _split(m, which):
    """The tets `which`, each divided into four around its centroid."""
    tets = np.asarray(m.tets)
    X, new = [np.asarray(m.X)], [np.delete(tets, which, axis=0)]
    for k, t in enumerate(which):
        c = m.num_nodes + k
        X.append(m.X[tets[t]].mean(axis=0, keepdims=True))
        for v in range(4):
            q = tets[t].copy()
            q[v] = c
            new.append(q[None, :])
    return M.Mesh(np.vstack(X), np.vstack(new).astype(np.int32), m.faces, m.codes)


def _neighbours(m):
    nb = [[] for _ in range(m.num_nodes)]
    for a, b in M.edges(m):
        nb[a].append(b)
        nb[b].append(a)
    return nb


def _halo_of(target, m):
    """The mesh with 64 scattered nodes numbered first that have exactly `target`
    different neighbours."""
    nb = [set(x) for x in _neighbours(m)]
    first, seen, rest = [], set(), list(np.random.default_rng(2).permutation(m.num_nodes))
    for left in range(64, 0, -1):  # what is missing, spread over the nodes left
        miss = target - len(seen)
        gain = [len(nb[n] - seen) for n in rest]
        k = min((q for q, g in enumerate(gain) if g <= miss), key=lambda q: abs(gain[q] - miss / left))
        seen |= nb[rest[k]]
        first.append(rest.pop(k))
    assert len(seen) == target
    renum = np.empty(m.num_nodes, dtype=np.int32)
    renum[np.array(first + sorted(rest))] = np.arange(m.num_nodes, dtype=np.int32)
    return M.renumber(m, renum)


def _divided():
    """Every tet divided: the corners have up to 38 neighbours, the centroids 4."""
    m = M.kuhn_box(7, 6, 6, jitter=0.15, seed=3)
    return _split(m, np.arange(m.num_tets))


MESHES = {  # name: (mesh, most neighbours of a slice, most of a node)
    "shuffled": (lambda: _shuffled(M.kuhn_box(36, 36, 36, jitter=0.15, seed=3), 1), (513, 1024), (14, 14)),
    "shuffled by eights": (lambda: _shuffled(M.kuhn_box(36, 36, 36, jitter=0.15, seed=3), 1, 8), (513, 1024), (14, 14)),
    "512 in a slice": (lambda: _halo_of(512, M.kuhn_box(11, 11, 12, jitter=0.15, seed=3)), (512, 512), (14, 14)),
    "513 in a slice": (lambda: _halo_of(513, M.kuhn_box(11, 11, 12, jitter=0.15, seed=3)), (513, 513), (14, 14)),
    "1024 in a slice": (lambda: _halo_of(1024, _divided()), (1024, 1024), (30, 64)),
    "1025 in a slice": (lambda: _halo_of(1025, _divided()), (1025, 1025), (30, 64)),
    "16 neighbours": (lambda: _cone(15), (17, 17), (16, 16)),
    "17 neighbours": (lambda: _cone(16), (18, 18), (17, 17)),
    "33 neighbours": (lambda: _cone(32), (34, 34), (33, 33)),
    "64 neighbours": (lambda: _cone(63), (64, 65), (64, 64)),
    "65 neighbours": (lambda: _cone(64), (64, 66), (65, 65)),
    "63 nodes": (lambda: M.kuhn_box(6, 2, 2, jitter=0.15, seed=3), (1, 63), (4, 14)),
    "64 nodes": (lambda: M.kuhn_box(3, 3, 3, jitter=0.15, seed=3), (1, 64), (4, 14)),
    "65 nodes": (lambda: _split(M.kuhn_box(3, 3, 3, jitter=0.15, seed=3), [17]), (1, 65), (4, 15)),
}


def _mesh(name):
    make, halo, degree = MESHES[name]
    m = make()
    nb = _neighbours(m)
    most = max(len(set().union(*nb[s:s + 64])) for s in range(0, m.num_nodes, 64))
    deg = max(map(len, nb))
    print(f"[paths] {name}: {m.num_nodes} nodes, {most} in a slice, {deg} of a node", flush=True)
    assert halo[0] <= most <= halo[1] and degree[0] <= deg <= degree[1]
    if name.endswith("nodes"):
        assert m.num_nodes == int(name.split()[0])
    # records from 256 slices on where the entries name more lines of eight nodes
    # than a quarter of their number: the shuffled mesh alone
    lines = sum(len({n // 8 for row in nb[s:s + 64] for n in row}) for s in range(0, m.num_nodes, 64))
    records = m.num_nodes > 255 * 64 and lines > 0.25 * sum(map(len, nb))
    assert records == (name == "shuffled")
    return m


def _check_residual(gpu, m, p, U):
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    ref = O.OracleMesh(m, p).residual(U, want_abs=True)
    assert ref["ierr"] == 0
    op = SpaceOperator(m, p)
    R = torch.full((m.num_nodes, 5), float("nan"), dtype=torch.float64, device=gpu)
    assert op.compute_residual(torch.from_numpy(U).to(gpu), R) == 0
    assert np.max(np.abs(R.cpu().numpy() - ref["R"]) / np.maximum(ref["Rabs"], 1e-300)) <= 1e-12
    op.close()


@pytest.mark.parametrize("second_order", [True, False])
@pytest.mark.parametrize("name", list(MESHES))
def test_residual(gpu, name, second_order):
    m = _mesh(name)
    p = FlowParams(mach=0.5, alpha=0.05, yaw=0.03, second_order=second_order)
    _check_residual(gpu, m, p, init_state(p, m.X, "noise", 0.005, seed=12))


FLOWS = {"supersonic": dict(mach=2.2), "stiffened": dict(mach=0.5, pstiff=2.0),
         "supersonic stiffened": dict(mach=3.0, pstiff=0.3)}


def _flow(flow, second_order):
    """Mesh, parameters and state; the stiffened gas between slip walls alone (the
    farfield flux is the perfect gas's), with the energy of its pressure."""
    kw = FLOWS[flow]
    walls = dict(face_codes=(M.AEROFX_BC_SLIP_WALL,) * 6) if "pstiff" in kw else {}
    m = M.kuhn_box(7, 6, 5, jitter=0.15, seed=3, **walls)
    p = FlowParams(alpha=0.3, yaw=0.2, second_order=second_order, **kw)
    U = init_state(FlowParams(alpha=0.3, yaw=0.2, mach=p.mach), m.X, "noise", 0.02, seed=13)
    U[:, 4] += p.gamma * p.pstiff / (p.gamma - 1.0)
    return m, p, U


@pytest.mark.parametrize("second_order", [True, False])
@pytest.mark.parametrize("flow", list(FLOWS))
def test_residual_of_flows(gpu, flow, second_order):
    _check_residual(gpu, *_flow(flow, second_order))


# ---------------------------------------------------------------------------
# the derivatives over the same paths: <lam, dR> and the transposed products,
# bounded as in test_gpu_passes.py
# ---------------------------------------------------------------------------
def _check_duality(gpu, m, p, U):
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    U = torch.from_numpy(U).to(gpu)
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(gpu)  # noqa: E731
    N = m.num_nodes
    h = float(np.median(np.linalg.norm(m.X[m.tets[:, 0]] - m.X[m.tets[:, 1]], axis=1)))
    lam, dU, dX = rnd(N, 5), rnd(N, 5) * U.abs().mean(0), rnd(N, 3) * 0.1 * h
    op = SpaceOperator(m, p)
    du, dx = torch.empty_like(U), torch.empty_like(U)
    assert op.compute_derivative_of_residual(U, du, dU, None) == 0
    assert op.compute_derivative_of_residual(U, dx, None, dX) == 0
    gu, gx = torch.empty_like(U), torch.empty_like(dX)
    op.compute_transpose_derivative_of_residual(U, lam, gu, gx)
    for fwd, rev in ((lam * du, gu * dU), (lam * dx, gx * dX)):
        S = float(fwd.abs().sum() + rev.abs().sum())
        assert abs(float(fwd.sum() - rev.sum())) <= 1e-12 * S
    op.close()


@pytest.mark.parametrize("name", ["shuffled", "shuffled by eights", "513 in a slice", "1025 in a slice", "33 neighbours", "65 nodes"])
def test_duality(gpu, name):
    m = _mesh(name)
    p = FlowParams(mach=0.5, alpha=0.05, yaw=0.03)
    _check_duality(gpu, m, p, init_state(p, m.X, "noise", 0.005, seed=12))


@pytest.mark.parametrize("second_order", [True, False])
@pytest.mark.parametrize("flow", list(FLOWS))
def test_duality_of_flows(gpu, flow, second_order):
    _check_duality(gpu, *_flow(flow, second_order))


# ---------------------------------------------------------------------------
# whole rows per wave: 74^3 nodes, 6332 slices, the last of 24 nodes
# ---------------------------------------------------------------------------
@pytest.fixture(scope="module")
def large():
    m = M.kuhn_box(73, 73, 73, jitter=0.15, seed=3)
    assert m.num_nodes % 64 and (m.num_nodes + 63) // 64 >= 6144
    return m


@pytest.mark.parametrize("second_order", [True, False])
@pytest.mark.parametrize("low_mach", [None, LM])
def test_residual_by_rows(gpu, large, low_mach, second_order):
    p = FlowParams(mach=0.05 if low_mach else 0.5, alpha=0.05, second_order=second_order, low_mach=low_mach)
    _check_residual(gpu, large, p, init_state(p, large.X, "noise", 0.01, seed=12))


def test_failsafe_by_rows(gpu, large):
    """Tags and count of a state with two nodes of negative pressure, one of them
    the last, then the residual with their neighbours first order."""
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    m, p = large, FlowParams(mach=0.5)
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


# ---------------------------------------------------------------------------
# a node of more neighbours than one lane should take beside a large mesh: the
# edge passes go by entries (a limit of 32 below 12288 slices)
# ---------------------------------------------------------------------------
def _beside(m, other):
    n = m.num_nodes
    return M.Mesh(np.vstack([m.X, other.X + 5.0]), np.vstack([m.tets, other.tets + n]).astype(np.int32),
                  np.vstack([m.faces, other.faces + n]).astype(np.int32),
                  np.concatenate([m.codes, other.codes]).astype(np.int32))


@pytest.mark.parametrize("k", [31, 32])
def test_residual_of_hub_beside_large_mesh(gpu, large, k):
    m = _beside(large, _cone(k))
    p = FlowParams(mach=0.5, alpha=0.05)
    _check_residual(gpu, m, p, init_state(p, m.X, "noise", 0.005, seed=12))


@pytest.mark.parametrize("k", [31, 32])
def test_duality_of_hub_beside_large_mesh(gpu, k):
    m = _beside(M.kuhn_box(45, 45, 46, jitter=0.15, seed=3), _cone(k))
    p = FlowParams(mach=0.5, alpha=0.05)
    _check_duality(gpu, m, p, init_state(p, m.X, "noise", 0.005, seed=12))
