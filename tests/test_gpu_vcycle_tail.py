"""The one-workgroup tail of the V-cycle against the oracle: tails that hold
only the coarsest level, a smoothed transfer, every level of small instances,
and instances of uneven size in one launch; a tail asked for beyond what fits
starts at the finest level that does."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("tail", [0, 64, 200, 100000])
@pytest.mark.parametrize("sizes", [[(4, 4, 4)], [(9, 8, 7), (3, 2, 5), (17, 12, 9)], [(40, 33, 21)]])
def test_tail_levels(pkg, orc, sizes, tail, precision):
    gs = [pkg.grids.cartesian(*d) for d in sizes]
    G, icp = pkg.grids.concat(gs)
    perms = [pkg.fields.perm_c1(g.num_cells, 20 + t) for t, g in enumerate(gs)]
    bcs = [cases.xdrop_bc(g) for g in gs]
    tm, rm = cases.unit_fluid(G.num_cells)
    bt = np.concatenate([b[0] for b in bcs])
    bv = np.concatenate([b[1] for b in bcs])
    src = np.zeros((3, G.num_cells))
    src[1, 0], src[1, -1] = 1e-13, -1e-13
    bvs = np.stack([bv, bv, 2.0 * bv])
    s = pkg.HybridSolver(0)
    s.init(G, np.concatenate(perms), (0, 0, 0), bt, None, inst_cellpos=icp)
    s.solve(tm, rm, src, bt, bvs, residual_tolerance=1e-12, precision=precision, tail_rows=tail, autotune=False)
    p, _, v = s.getSolution()
    for k in range(3):
        for t, g in enumerate(gs):
            c = slice(icp[t], icp[t + 1])
            h = slice(6 * icp[t], 6 * icp[t + 1])
            ref = orc.solve(g, perms[t], tm[c], rm[c], src[k, c], bt[h], bvs[k, h], tol=1e-14)
            # solves to 1e-12 of systems with condition numbers below 1e4
            assert cases.rel_err(p[k, c], ref.cell_pressure) < 1e-8
            assert cases.rel_err(v[k, h], ref.outflux) < 1e-8
