"""The strip kernel of the regular-cell assembly over every rule order and over lines of
every kind: full (8 dofs), short, two shared short ones (9 = 5 + 4), fewer rows than one
block, rounds with idle wavefronts.  G, H and alpha against the oracle's assembly."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as T
from tests.test_strip_plan import replay
from wavebem_amd import mesh as M
from wavebem_amd.bem import BEMProblem, Config, host_strip_plan

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_available")]


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-10), ("fp32_ir", 1e-9)])
@pytest.mark.parametrize("q", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("n", [2, 7, 8, 12])
def test_strip_rules(n, q, precision, bar):
    m = M.box_mesh(n=n, hi=(1.0, 0.8, 0.6), dirichlet_top=True)
    ptr, idx = M.double_nodes_csr(m.support_points)
    H0, G0 = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx, q_order=q)
    with BEMProblem(m, Config(precision=precision, quadrature_order=q),
                    double_nodes=(ptr, idx)) as p:
        p.assemble_system()
        G, H = p.matrices()
        alpha = p.compute_alpha()
    # sums of q^2 products per entry, in FP64 (stored as 2^-33 relative in FP32-IR)
    assert T.row_scaled_err(G, G0) < bar
    assert T.row_scaled_err(H, H0) < bar
    # one rounding of every entry of the row at most
    a0 = -H0.sum(axis=1)
    assert np.abs(alpha - a0).max() < bar * np.abs(H0).sum(axis=1).max()


def holed_mesh(kind):
    """One structured patch whose grid has missing cells: lines with gaps inside, lines of a
    strip that are empty, so that a round's four lines hold any number of columns."""
    na, npos = 23, 29  # cells
    keep = np.ones((na, npos), bool)
    if kind == "ring":
        keep[4:19, 5:24] = False
    elif kind == "dots":  # 2 x 2 cells each, whose middle dof goes
        for a in range(1, na - 2, 3):
            for b in range(1 + a % 2, npos - 2, 4):
                keep[a:a + 2, b:b + 2] = False
    else:  # stairs
        keep = np.arange(npos)[None, :] <= np.arange(na)[:, None] * 1.3 + 1
        keep &= np.arange(npos)[None, :] >= np.arange(na)[:, None] * 1.3 - 12
    u, v = np.meshgrid(np.linspace(0, 1, npos + 1), np.linspace(0, 0.8, na + 1))
    X = np.stack([u, v, 0.3 * u * v + 0.1 * u * u], -1).reshape(-1, 3)
    d = np.arange(X.shape[0]).reshape(na + 1, npos + 1)
    cells = np.stack([d[:-1, :-1], d[:-1, 1:], d[1:, :-1], d[1:, 1:]], -1)[keep]
    used, cells = np.unique(cells, return_inverse=True)
    cells = cells.reshape(-1, 4).astype(np.int32)
    n, nc = len(used), len(cells)
    surf = (np.arange(n) % 2).astype(float)
    return M.SurfaceMesh(X[used], cells, np.ones(nc, np.int8), np.zeros(nc, np.int32), surf,
                         1.0 - surf, np.zeros(n, np.int32))


@pytest.mark.parametrize("precision,bar", [("fp64", 1e-10), ("fp32_ir", 1e-9)])
@pytest.mark.parametrize("kind", ["ring", "dots", "stairs"])
def test_strips_with_holes(kind, precision, bar):
    m = holed_mesh(kind)
    plan = host_strip_plan(m)
    lines = [bin(x).count("1") for x in plan["gaps"][:, 2]]
    assert plan["strip_dofs"] == m.n_dofs and len(set(lines)) > 2
    replay(m, plan)
    ptr, idx = M.double_nodes_csr(m.support_points)
    H0, G0 = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx)
    with BEMProblem(m, Config(precision=precision), double_nodes=(ptr, idx)) as p:
        p.assemble_system()
        G, H = p.matrices()
        alpha = p.compute_alpha()
    assert T.row_scaled_err(G, G0) < bar
    assert T.row_scaled_err(H, H0) < bar
    a0 = -H0.sum(axis=1)
    assert np.abs(alpha - a0).max() < bar * np.abs(H0).sum(axis=1).max()
