"""Several right-hand sides where the batched products' panels end unevenly: columns that
end inside a 64-column panel and a 4-column group, exactly at a panel's end, panels that mix
both operators' columns; one, an odd number and the largest batch of vectors.  Against the
dense solution of every column's own constrained system."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as T
from wavebem_amd import mesh as M
from wavebem_amd.bem import BEMProblem, Config

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("gpu_available")]


def _mesh(name):
    if name == "box":  # 384 = 6 * 64 dofs
        return M.box_mesh(n=7, hi=(1.0, 0.8, 0.6), dirichlet_top=True)
    # 341 and 1,083 dofs: 21 and 59 columns in the last panel
    return M.wigley_tank(**dict(zip(("nh", "nt", "nu", "nd", "ny", "nzd"), name)))


@pytest.mark.parametrize("name", [(6, 2, 3, 4, 4, 2), "box", (12, 4, 6, 8, 8, 3)])
@pytest.mark.parametrize("k", [1, 3, 16])
def test_batched_hi_lo_product(name, k):
    m = _mesh(name)
    ptr, idx = M.double_nodes_csr(m.support_points)
    first = [idx[a] for a in ptr[:-1]]  # coincident dofs carry one value
    bcs = np.random.default_rng(k).standard_normal((k, m.n_dofs)).take(first, axis=1)
    phi, dphi = bcs * m.surface_nodes, bcs * m.other_nodes
    with BEMProblem(m, Config(precision="fp32_ir", solver_tolerance=1e-11)) as p:
        p.compute_constraints(bcs[0])
        p.assemble_system()
        st = p.solve_system_multi(phi, dphi, bcs)
    assert st["true_rel_residual"] < 1e-9
    H, G = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx)
    for v in range(k):
        cons = O.compute_constraints(ptr, idx, m.surface_nodes, bcs[v])
        x0 = T.dense_solution(H, G, m.surface_nodes, m.other_nodes, cons, bcs[v])
        x = np.where(m.other_nodes > 0, phi[v], dphi[v])
        assert np.abs(x - x0).max() < 1e-8 * np.abs(x0).max()


@pytest.mark.parametrize("tmp_vectors", [3, 6, 9])
@pytest.mark.parametrize("precision", ["fp64", "fp32_ir"])
def test_batched_restarts(tmp_vectors, precision):
    """Cycles of 1, 4 and 7 steps with the next step queued before a column is read: right-hand
    sides of several sizes, so that instances end in different steps and cycles and one (zero)
    never starts; the step queued for a cycle that has ended must leave no trace."""
    m = _mesh((12, 4, 6, 8, 8, 3))
    ptr, idx = M.double_nodes_csr(m.support_points)
    first = [idx[a] for a in ptr[:-1]]
    scale = np.array([1.0, 1e-5, 0.0, 1e-9, 1.0])
    bcs = np.random.default_rng(7).standard_normal((5, m.n_dofs)).take(first, axis=1)
    bcs *= scale[:, None]
    phi, dphi = bcs * m.surface_nodes, bcs * m.other_nodes
    with BEMProblem(m, Config(precision=precision, solver_tolerance=1e-11,
                              gmres_max_tmp_vectors=tmp_vectors, solver_max_steps=20000)) as p:
        p.compute_constraints(bcs[0])
        p.assemble_system()
        st = p.solve_system_multi(phi, dphi, bcs)
    assert st["iterations"] > 2 * (tmp_vectors - 2)
    H, G = O.assemble(m.support_points, m.cell_dofs, m.cell_orient, ptr, idx)
    for v in range(5):
        cons = O.compute_constraints(ptr, idx, m.surface_nodes, bcs[v])
        x0 = T.dense_solution(H, G, m.surface_nodes, m.other_nodes, cons, bcs[v])
        x = np.where(m.other_nodes > 0, phi[v], dphi[v])
        # every instance stops at the same absolute residual, 1e-11
        assert np.abs(x - x0).max() < 1e-8 * np.abs(x0).max() + 1e-9
