"""Solves at the sizes where the small-problem kernels change: blocks of the preconditioner
of 64 unknowns (registers) and of 63 and 65 (LDS), last blocks of every kind, one-workgroup
Arnoldi steps up to their limits, against the dense solution or the other precision."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as T
from wavebem_amd import mesh as M
from wavebem_amd.bem import BEMProblem, Config

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_available")]


def _solve(m, bc, **cfg):
    phi, dphi = bc * m.surface_nodes, bc * m.other_nodes
    with BEMProblem(m, Config(**cfg)) as p:
        p.compute_constraints(bc)
        p.assemble_system()
        st = p.solve_system(phi, dphi, bc)
    return np.where(m.other_nodes > 0, phi, dphi), st


# 54 (one short block), 294 = 4 * 64 + 38, 384 = 6 * 64 dofs
@pytest.mark.parametrize("n", [2, 6, 7])
@pytest.mark.parametrize("precision", ["fp64", "fp32_ir"])
def test_block_inverse_and_small_arnoldi(n, precision):
    m = M.box_mesh(n=n, hi=(1.0, 0.8, 0.6), dirichlet_top=True)
    bc = np.random.default_rng(n).standard_normal(m.n_dofs)
    ptr, idx = M.double_nodes_csr(m.support_points)
    # coincident dofs carry one value, as boundary data does
    bc = bc[[idx[a] for a in ptr[:-1]]]
    H, G = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx)
    cons = O.compute_constraints(ptr, idx, m.surface_nodes, bc)
    x0 = T.dense_solution(H, G, m.surface_nodes, m.other_nodes, cons, bc)
    its = {}
    for block in (64, 63, 65):
        x, st = _solve(m, bc, precision=precision, precond_block=block, precond_coarse=0,
                       solver_tolerance=1e-12)
        assert np.abs(x - x0).max() < 1e-8 * np.abs(x0).max()
        its[block] = st["iterations"]
    # a wrong inverse still converges, in many more steps; blocks one wider or narrower
    # change the count by a few
    assert its[64] <= max(its[63], its[65]) + 6


# 3,750 and 4,056 dofs: within the limit of a one-workgroup step, the basis outgrowing it
# during the solve; 4,374: above
@pytest.mark.parametrize("n", [24, 25, 26])
def test_small_arnoldi_limits(n):
    m = M.box_mesh(n=n, hi=(1.0, 0.8, 0.6), dirichlet_top=True)
    X = m.support_points
    bc = np.where(m.surface_nodes > 0, np.cos(3 * X[:, 0]) * X[:, 1], 0.2 * X[:, 0])
    a, sa = _solve(m, bc, precision="fp64")
    b, sb = _solve(m, bc, precision="fp32_ir")
    assert sa["true_rel_residual"] < 1e-9 and sb["true_rel_residual"] < 1e-9
    assert np.abs(a - b).max() < 1e-8 * np.abs(a).max()


# constraint lines written by the product's launch: none, and 52 and 112 of them (less than a
# wavefront, a part of a block)
@pytest.mark.parametrize("n, lines", [(4, False), (4, True), (9, True)])
@pytest.mark.parametrize("precision", ["fp64", "fp32_ir"])
def test_product_writes_constraint_lines(n, lines, precision):
    m = M.box_mesh(n=n, hi=(1.0, 0.8, 0.6), dirichlet_top=True)
    ptr, idx = M.double_nodes_csr(m.support_points)
    H, G = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx)
    rng = np.random.default_rng(n)
    bc = rng.standard_normal(m.n_dofs)[[idx[a] for a in ptr[:-1]]]
    src = rng.standard_normal(m.n_dofs)
    with BEMProblem(m, Config(precision=precision)) as p:
        if lines:
            p.compute_constraints(bc)
        else:
            p.set_constraints([], [0], [], [], [])
        p.assemble_system()
        dst = p.constrained_vmult(src)
    if lines:
        cons = O.compute_constraints(ptr, idx, m.surface_nodes, bc)
        A, _ = T.explicit_system(H, G, m.surface_nodes, m.other_nodes, cons, bc)
        want = A @ src
    else:
        want = O.vmult(G, H, O.compute_alpha(H), m.surface_nodes, m.other_nodes, src)
    # FP64: sums of n products; FP32-IR: entries to 2^-33
    tol = 1e-12 if precision == "fp64" else 1e-9
    assert np.abs(dst - want).max() < tol * np.abs(want).max()
