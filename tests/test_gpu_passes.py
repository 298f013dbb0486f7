"""The derivative passes at the sizes where their split changes: 64-node slices
(one node short, exact, two over), meshes on both sides of the adjoint's rules for
whole rows and streams (1536 and 3072 slices; at first order the adjoint goes by
entries on all of them), and rows too long for the tables in LDS (a cone with
two 301-neighbour hubs: the gradient pass gathers per entry, the viscous
Jacobian runs its kernel per entry).  Both directions read the same tables,
normals and gradients: test_gpu_pass_paths.py holds the residual, which reads
them too, against the oracle at such sizes.

Tangent and adjoint are the exact derivative of one residual, so <lam, dR> and
the transposed products differ by rounding alone: each side is a sum of
products of which the largest partial sums are bounded by S = sum |lam dR|
(and its mirror), over a chain of a few hundred operations per term: 1e-12 S
is some ten times the rounding of such a chain (a few hundred times 1.1e-16,
averaging down over the sum) and any wrong edge, slot or lane is far above it.
"""
import os
import sys

import numpy as np
import pytest

import oracle as O
from aerof_dev_amd import FlowParams, init_state
from aerof_dev_amd import mesh as M
sys.path.insert(0, os.path.dirname(__file__))
from test_gpu_high_degree import _mesh as _cone_mesh  # noqa: E402
from test_gpu_viscous import ns_params  # noqa: E402

pytestmark = pytest.mark.gpu

MESHES = {
    "63": lambda: M.kuhn_box(6, 2, 2, jitter=0.15, seed=3),
    "64": lambda: M.kuhn_box(3, 3, 3, jitter=0.15, seed=3),
    "66": lambda: M.kuhn_box(10, 2, 1, jitter=0.15, seed=3),
    "cone": _cone_mesh,
    "1521 slices": lambda: M.kuhn_box(45, 45, 45, jitter=0.15, seed=3),
    "1554 slices": lambda: M.kuhn_box(45, 45, 46, jitter=0.15, seed=3),
    "3102 slices": lambda: M.kuhn_box(57, 57, 58, jitter=0.15, seed=3),
}


@pytest.mark.parametrize("second_order", [True, False])
@pytest.mark.parametrize("name", list(MESHES))
def test_tangent_adjoint_duality_at_edges(gpu, name, second_order):
    import torch
    from aerof_dev_amd.operators import SpaceOperator
    m = MESHES[name]()
    p = FlowParams(mach=0.5, alpha=0.05, yaw=0.03, second_order=second_order)
    U = torch.from_numpy(init_state(p, m.X, "noise", 0.01, seed=12)).to(gpu)
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(gpu)
    N = m.num_nodes
    h = float(np.median(np.linalg.norm(m.X[m.tets[:, 0]] - m.X[m.tets[:, 1]], axis=1)))
    lam, dU, dX = rnd(N, 5), rnd(N, 5) * U.abs().mean(0), rnd(N, 3) * 0.1 * h
    op = SpaceOperator(m, p)
    du, dx = torch.empty_like(U), torch.empty_like(U)
    assert op.compute_derivative_of_residual(U, du, dU, None) == 0
    assert op.compute_derivative_of_residual(U, dx, None, dX) == 0
    gu, gx, gu2 = torch.empty_like(U), torch.empty_like(dX), torch.empty_like(U)
    op.compute_transpose_derivative_of_residual(U, lam, gu, gx)
    op.compute_transpose_derivative_of_residual(U, lam, gu2)
    for fwd, rev in ((lam * du, gu * dU), (lam * dx, gx * dX), (lam * du, gu2 * dU)):
        S = float(fwd.abs().sum() + rev.abs().sum())
        assert abs(float(fwd.sum() - rev.sum())) <= 1e-12 * S
    op.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_viscous_jacobian_of_hubs(gpu, precision):
    import torch
    from aerof_dev_amd.operators import MatVecProdH1, SpaceOperator
    m = _cone_mesh()
    p = ns_params(0.3, 40.0)
    U = init_state(p, m.X, "noise", 0.01, seed=13)
    om = O.OracleMesh(m, p)
    V = om.residual(U)["V"]
    dt = om.timestep(V, 20.0)
    Dr, Ar = om.apply_bcs_jacobian(U, *om.jacobian(V, dt))
    op = SpaceOperator(m, p)
    h1 = MatVecProdH1(op)
    h1.evaluate(torch.from_numpy(U).to(gpu), torch.from_numpy(dt).to(gpu), precision)
    D, A = h1.blocks()
    tol = 1e-12 if precision == 0 else 1e-6
    assert np.max(np.abs(D - Dr) / np.abs(Dr).max(axis=(1, 2))[:, None, None]) <= tol
    assert np.max(np.abs(A - Ar) / (np.abs(Ar).max(axis=(2, 3))[:, :, None, None] + 1e-300)) <= tol
    op.close()
