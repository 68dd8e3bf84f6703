"""The averaging transfer between the faces and the first coarse level against the
oracle: Dirichlet rows left out of the cycle also where the solver type starts
from zero, several sweeps, periodic pairs, and blocks one cell thick."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kw", [dict(linsolver_type=0, precond=1), dict(smooth_steps=2),
                                dict(linsolver_type=0, precond=1, element_operator=2)])
@pytest.mark.parametrize("dims", [(2, 2, 2), (7, 1, 5), (13, 10, 6)])
def test_dirichlet_rows_and_sweeps(pkg, orc, dims, kw, precision):
    g = pkg.grids.cartesian(*dims, 1.0, 1.0, 0.5)
    nc = g.num_cells
    perm = pkg.fields.perm_c1(nc, 8)
    bt, bv = cases.xdrop_bc(g, 3.0, 1.0)
    tm, rm = cases.unit_fluid(nc)
    s = pkg.HybridSolver(0)
    s.init(g, perm, (0, 0, 0), bt, None)
    s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12, precision=precision, **kw)
    p, _, v = s.getSolution()
    ref = orc.solve(g, perm, tm, rm, np.zeros(nc), bt, bv, tol=1e-14)
    # solves to 1e-12 of systems with condition numbers below 1e4
    assert cases.rel_err(p, ref.cell_pressure) < 1e-8
    assert cases.rel_err(v, ref.outflux) < 1e-8


@pytest.mark.parametrize("dims", [(4, 4, 4), (9, 6, 5)])
def test_periodic_pairs(pkg, orc, dims):
    g = pkg.grids.cartesian(*dims)
    nc = g.num_cells
    perm = pkg.fields.perm_c1(nc, 9)
    bt, bv, partner = cases.periodic_bc(g)
    tm, rm = cases.unit_fluid(nc)
    s = pkg.HybridSolver(0)
    s.init(g, perm, (0, 0, 0), bt, partner)
    s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12)
    ref = orc.solve(g, perm, tm, rm, np.zeros(nc), bt, bv, partner=partner, tol=1e-14)
    assert cases.rel_err(s.getSolution()[2], ref.outflux) < 1e-8


def test_smoother_weights_of_a_batch(pkg, orc):
    """Every level's weight of two unlike instances in one handle is the smaller
    of theirs alone (the largest eigenvalue of a block-diagonal operator)."""
    gs = [pkg.grids.cartesian(12, 9, 7), pkg.grids.cartesian(10, 10, 10, 1.0, 1.0, 0.4)]
    perms = [pkg.fields.perm_c1(g.num_cells, 30 + t) for t, g in enumerate(gs)]
    G, icp = pkg.grids.concat(gs)
    bt, bv = cases.xdrop_bc(G)
    s = pkg.HybridSolver(0)
    s.init(G, np.concatenate(perms), (0, 0, 0), bt, None, inst_cellpos=icp)
    tm, rm = cases.unit_fluid(G.num_cells)
    s.solve(tm, rm, np.zeros(G.num_cells), bt, bv, residual_tolerance=1e-8)
    w = s.report.as_dict()["smoother_weights"][0]
    alone = []
    for g, perm in zip(gs, perms):
        b, v = cases.xdrop_bc(g)
        q = pkg.HybridSolver(0)
        q.init(g, perm, (0, 0, 0), b, None)
        tm, rm = cases.unit_fluid(g.num_cells)
        q.solve(tm, rm, np.zeros(g.num_cells), b, v, residual_tolerance=1e-8)
        alone.append(q.report.as_dict()["smoother_weights"][0])
    # 12 Lanczos steps come within a few percent of the eigenvalue from below
    assert 0.97 * min(alone) <= w <= 1.05 * min(alone), (w, alone)


@pytest.mark.parametrize("dims", [(2, 2, 2), (7, 1, 5), (13, 10, 6)])
@pytest.mark.parametrize("element_operator", [0, 2])
def test_post_sweep_written_with_known_weights(pkg, orc, dims, element_operator):
    """Mixed precision: the first solve of a permeability fills the post-smoothing
    operator after the weights' estimate, later ones together with A P."""
    g = pkg.grids.cartesian(*dims, 1.0, 1.0, 0.5)
    nc = g.num_cells
    perm = pkg.fields.perm_c1(nc, 12)
    bt, bv = cases.xdrop_bc(g, 3.0, 1.0)
    tm, rm = cases.unit_fluid(nc)
    ref = orc.solve(g, perm, tm, rm, np.zeros(nc), bt, bv, tol=1e-14)
    s = pkg.HybridSolver(0)
    s.init(g, perm, (0, 0, 0), bt, None)
    its = []
    for _ in range(3):
        s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12, precision="mixed",
                element_operator=element_operator)
        its.append(s.report.iterations)
        # solves to 1e-12 of systems with condition numbers below 1e4
        assert cases.rel_err(s.getSolution()[2], ref.outflux) < 1e-8
    # the same preconditioner up to the order of FP32 sums
    assert max(its) - min(its) <= 2


@pytest.mark.parametrize("precision,element_operator", [("fp64", 0), ("mixed", 0), ("mixed", 2)])
@pytest.mark.parametrize("precond", [0, 1])
@pytest.mark.parametrize("smooth_steps", [1, 2])
@pytest.mark.parametrize("solver", [0, 1])
def test_reduction_is_relative_to_the_solver_types_start(pkg, solver, smooth_steps, precond, precision,
                                                         element_operator):
    """Solver type 0 starts from zero, the others from the Dirichlet values, with
    either preconditioner: the residual that the tolerance is relative to."""
    import scipy.sparse as sp
    g = pkg.grids.cartesian(13, 10, 6, 1.0, 1.0, 0.5)
    nc = g.num_cells
    bt, bv = cases.xdrop_bc(g, 30.0, 29.0)
    tm, rm = cases.unit_fluid(nc)
    s = pkg.HybridSolver(0)
    s.init(g, pkg.fields.perm_c1(nc, 8), (0, 0, 0), bt, None)
    s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-5, precision=precision, precond=precond,
            linsolver_type=solver, smooth_steps=smooth_steps, element_operator=element_operator)
    x = np.asarray(s.getSolution()[1])
    ptr, col, val, b = s.system()
    A = sp.csr_matrix((val, col, ptr), shape=(b.shape[0],) * 2)
    x0 = np.zeros_like(b)
    if solver:
        # Dirichlet rows are the ones with a single nonzero entry
        off = np.asarray(abs(A - sp.diags(A.diagonal())).sum(axis=1)).reshape(-1)
        x0 = np.where(off == 0, b / A.diagonal(), 0.0)
    r, r0 = np.linalg.norm(b - A @ x), np.linalg.norm(b - A @ x0)
    assert s.report.reduction <= 1e-5
    # the report's own FP64 residual of the same x, up to the rounding of A x (1e-16 of |b|)
    assert abs(s.report.reduction - r / r0) < 1e-4 * s.report.reduction + 1e-12
