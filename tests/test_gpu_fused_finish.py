"""The CG scalars worked out inside the vector updates (instances of few row
blocks) against the separate finisher: a small instance solved alone takes
the first, in a batch with one of more than 1024 blocks the second."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("solver,nrhs", [(0, 1), (1, 1), (1, 2)])
def test_small_instance_alone_and_beside_a_large_one(pkg, orc, solver, nrhs, precision):
    small, large = pkg.grids.cartesian(9, 8, 7), pkg.grids.cartesian(72, 72, 72)
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


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("n", [55, 56, 69])
def test_more_partials_than_one_round_of_loads(pkg, solver, precision, n):
    """Around 512 and just below 1024 partials of the assembled operator (rows of 1024
    faces), each summed eight loads at a time; a uniform medium has the closed form
    v = k dp / L."""
    g = pkg.grids.cartesian(n, n, n)
    nc = g.num_cells
    bt, bv = cases.xdrop_bc(g, 1.0, 0.0)
    s = pkg.HybridSolver(0)
    s.init(g, pkg.fields.diag_perm(np.ones(nc), np.ones(nc), np.ones(nc)), (0, 0, 0), bt, None)
    tm, rm = cases.unit_fluid(nc)
    s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12, precision=precision, linsolver_type=solver)
    exact = np.zeros(g.num_half_faces)
    exact[g.side == 1], exact[g.side == 0] = 1.0 / n, -1.0 / n
    v = np.asarray(s.getSolution()[2]).reshape(-1)
    # solves to 1e-12 of a system with a condition number of about n^2 < 5e3
    assert np.max(np.abs(v - exact)[(g.side == 0) | (g.side == 1)]) < 1e-8


@pytest.mark.parametrize("solver", [0, 1])
@pytest.mark.parametrize("element_operator,n", [(0, 70), (0, 71), (2, 63), (2, 64), (2, 65)])
def test_both_sides_of_the_limit_in_mixed_precision(pkg, element_operator, n, solver):
    """Just below and above 1024 partials of each operator: one per 1024 face rows
    (1020 and 1064), or one per 256 cells of a colour (978, 1024 and 1074)."""
    g = pkg.grids.cartesian(n, n, n)
    nc = g.num_cells
    bt, bv = cases.xdrop_bc(g, 1.0, 0.0)
    s = pkg.HybridSolver(0)
    s.init(g, pkg.fields.diag_perm(np.ones(nc), np.ones(nc), np.ones(nc)), (0, 0, 0), bt, None)
    tm, rm = cases.unit_fluid(nc)
    s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12, precision="mixed", linsolver_type=solver,
            element_operator=element_operator)
    assert s.report.element_operator == (1 if element_operator else 0)
    exact = np.zeros(g.num_half_faces)
    exact[g.side == 1], exact[g.side == 0] = 1.0 / n, -1.0 / n
    v = np.asarray(s.getSolution()[2]).reshape(-1)
    # solves to 1e-12 of a system with a condition number of about n^2 < 6e3
    assert np.max(np.abs(v - exact)[(g.side == 0) | (g.side == 1)]) < 1e-8
