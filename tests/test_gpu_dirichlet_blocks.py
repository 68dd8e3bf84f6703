"""Multigrid aggregates all of whose faces are Dirichlet faces (a one-cell instance
in a batch, a cell cut off inside a larger instance): their coarse rows are zero,
and neither they nor the other instances may suffer from that."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu

MODES = [("fp64", 0), ("mixed", 0), ("mixed", 2)]


@pytest.mark.parametrize("precision,element_operator", MODES)
@pytest.mark.parametrize("smooth_steps", [1, 2])
@pytest.mark.parametrize("cells", [(1, 1, 1)])
def test_small_instance_beside_a_larger_one(pkg, orc, cells, smooth_steps, precision, element_operator):
    small, large = pkg.grids.cartesian(*cells), pkg.grids.cartesian(12, 10, 8)
    bts, bvs = np.zeros(small.num_half_faces, np.int32), np.zeros(small.num_half_faces)
    outer = np.asarray(small.nb) < 0
    bts[outer] = cases.DIR
    bvs[outer] = 1.0 + np.arange(outer.sum())
    btl, bvl = cases.xdrop_bc(large)
    Ks = pkg.fields.perm_c1(small.num_cells, 3)
    Kl = pkg.fields.perm_c1(large.num_cells, 4)
    G, icp = pkg.grids.concat([small, large])
    bt, bv = np.concatenate([bts, btl]), np.concatenate([bvs, bvl])
    s = pkg.HybridSolver(0)
    s.init(G, np.concatenate([Ks, Kl]), (0, 0, 0), bt, None, inst_cellpos=icp)
    tm, rm = cases.unit_fluid(G.num_cells)
    kw = dict(residual_tolerance=1e-12, precision=precision, smooth_steps=smooth_steps,
              element_operator=element_operator, linsolver_maxit=200)
    for _ in range(2):   # the second solve of a handle takes the weights and lists it keeps
        s.solve(tm, rm, np.zeros(G.num_cells), bt, bv, **kw)
        p, _, v = s.getSolution()
        alone = pkg.HybridSolver(0)
        alone.init(large, Kl, (0, 0, 0), btl, None)
        alone.solve(*cases.unit_fluid(large.num_cells), np.zeros(large.num_cells), btl, bvl, **kw)
        w, wa = s.report.as_dict()["smoother_weights"], alone.report.as_dict()["smoother_weights"]
        nl = alone.report.levels - 1
        # 12 Lanczos steps of the same operator (the other instance adds rows whose
        # eigenvalues are not the largest) come within a few percent of one value
        assert np.allclose(w[:nl], wa[:nl], rtol=0.05), (w, wa)
        assert abs(s.report.iterations - alone.report.iterations) <= 2
        nc = 0
        for g, K, b, x in ((small, Ks, bts, bvs), (large, Kl, btl, bvl)):
            n, h = g.num_cells, g.num_half_faces
            ref = orc.solve(g, K, np.ones(n), np.zeros(n), np.zeros(n), b, x, tol=1e-14)
            # solves to 1e-12 of systems with condition numbers below 1e4
            assert cases.rel_err(p[nc:nc + n], ref.cell_pressure) < 1e-8
            assert cases.rel_err(v[6 * nc:6 * nc + h], ref.outflux) < 1e-8
            nc += n


def _cut_off(g, cells):
    """Makes every face of the cells a boundary face (also of their neighbours)."""
    nb, twin, hc = np.array(g.nb), g.twin(), g.hf_cell()
    for h in np.flatnonzero(np.isin(hc, cells) & (nb >= 0)):
        nb[h] = nb[twin[h]] = -1
    g.nb = nb.astype(np.int32)
    return np.isin(hc, cells)


@pytest.mark.parametrize("precision,element_operator", MODES)
@pytest.mark.parametrize("linsolver_type", [0, 1])
@pytest.mark.parametrize("block", [1, 2])
def test_cells_cut_off_inside_an_instance(pkg, orc, block, linsolver_type, precision, element_operator):
    """block 1: the last cell of a 9x9x9 box, alone in its aggregate; 2: the eight
    cells of an inner aggregate, each cut off from the others too."""
    g = pkg.grids.cartesian(9, 9, 9) if block == 1 else pkg.grids.cartesian(8, 8, 8)
    nc = g.num_cells
    if block == 1:
        off = [nc - 1]
    else:
        off = [i + 8 * (j + 8 * k) for i in (2, 3) for j in (4, 5) for k in (2, 3)]
    at = _cut_off(g, off)
    K = pkg.fields.perm_c1(nc, 6)
    bt, bv = cases.xdrop_bc(g)
    bt[at], bv[at] = cases.DIR, np.linspace(0.2, 0.8, at.sum())
    tm, rm = cases.unit_fluid(nc)
    ref = orc.solve(g, K, tm, rm, np.zeros(nc), bt, bv, tol=1e-14)
    s = pkg.HybridSolver(0)
    s.init(g, K, (0, 0, 0), bt, None)
    for _ in range(2):
        s.solve(tm, rm, np.zeros(nc), bt, bv, residual_tolerance=1e-12, precision=precision, precond=1,
                linsolver_type=linsolver_type, element_operator=element_operator, linsolver_maxit=200)
        p, _, v = s.getSolution()
        # solves to 1e-12 of a system with a condition number below 1e4
        assert cases.rel_err(p, ref.cell_pressure) < 1e-8
        assert cases.rel_err(v, ref.outflux) < 1e-8
