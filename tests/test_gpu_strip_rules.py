"""The strip kernel of the regular-cell assembly over every rule order and over lines of
every kind: full (8 dofs), short, two shared short ones (9 = 5 + 4), fewer rows than one
block, rounds with idle wavefronts.  G, H and alpha against the oracle's assembly."""
import numpy as np
import pytest

import oracle as O
from tests import helpers as T
from wavebem_amd import mesh as M
from wavebem_amd.bem import BEMProblem, Config

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
