"""The CG scalars worked out inside the vector updates (instances of few row
blocks) against the separate finisher: a small instance solved alone takes
the first, in a batch with one of more than 512 blocks the second."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("solver,nrhs", [(0, 1), (1, 1), (1, 2)])
def test_small_instance_alone_and_beside_a_large_one(pkg, orc, solver, nrhs, precision):
    small, large = pkg.grids.cartesian(9, 8, 7), pkg.grids.cartesian(56, 56, 56)
    perm = pkg.fields.perm_c1(small.num_cells, 40)
    bt, bv = cases.xdrop_bc(small)
    G, icp = pkg.grids.concat([small, large])
    # the large instance starts converged: no pressure drop and no sources
    BT, _ = cases.xdrop_bc(G)
    BV = np.zeros((nrhs, G.num_half_faces))
    for k in range(nrhs):
        BV[k, :bv.shape[0]] = (1 + k) * bv
    K = np.concatenate([perm, pkg.fields.perm_c1(large.num_cells, 41)])
    s = pkg.HybridSolver(0)
    s.init(G, K, (0, 0, 0), BT, None, inst_cellpos=icp)
    tm, rm = cases.unit_fluid(G.num_cells)
    kw = dict(residual_tolerance=1e-12, precision=precision, linsolver_type=solver, element_operator=False)
    src = np.zeros((nrhs, G.num_cells)) if nrhs > 1 else np.zeros(G.num_cells)
    s.solve(tm, rm, src, BT, BV if nrhs > 1 else BV[0], **kw)
    v = np.atleast_2d(s.getSolution()[2])[:, :bv.shape[0]]
    ref = orc.solve(small, perm, tm[:small.num_cells], rm[:small.num_cells], np.zeros(small.num_cells), bt, bv, tol=1e-14)
    alone = pkg.HybridSolver(0)
    alone.init(small, perm, (0, 0, 0), bt, None)
    alone.solve(tm[:small.num_cells], rm[:small.num_cells], np.zeros(small.num_cells), bt, bv, **kw)
    # solves to 1e-12 of a system with a condition number below 1e4
    assert cases.rel_err(alone.getSolution()[2], ref.outflux) < 1e-8
    for k in range(nrhs):
        assert cases.rel_err(v[k], (1 + k) * ref.outflux) < 1e-8
