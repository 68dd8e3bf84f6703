"""Mixed precision on systems that the iteration solves exactly in a few steps, so
that its FP32 residual ends in rounding while the true one does not: boxes of a
few cells with every outer face a Dirichlet face, alone and in a batch."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("element_operator", [0, 2])
@pytest.mark.parametrize("linsolver_type,smooth_steps", [(0, 1), (1, 1), (1, 2)])
@pytest.mark.parametrize("dims", [(1, 1, 1), (1, 1, 2), (2, 1, 1), (1, 1, 3), (2, 2, 1), (1, 3, 2)])
def test_all_outer_faces_dirichlet(pkg, orc, dims, linsolver_type, smooth_steps, element_operator):
    g = pkg.grids.cartesian(*dims)
    large = pkg.grids.cartesian(9, 8, 7)
    for seed in (3, 4, 5):
        K = pkg.fields.perm_c1(g.num_cells, seed)
        bt, bv = np.zeros(g.num_half_faces, np.int32), np.zeros(g.num_half_faces)
        outer = np.asarray(g.nb) < 0
        bt[outer] = cases.DIR
        bv[outer] = 1.0 + np.arange(outer.sum())
        tm, rm = cases.unit_fluid(g.num_cells)
        ref = orc.solve(g, K, tm, rm, np.zeros(g.num_cells), bt, bv, tol=1e-14)
        G, icp = pkg.grids.concat([g, large])
        btl, bvl = cases.xdrop_bc(large)
        KG = np.concatenate([K, pkg.fields.perm_c1(large.num_cells, seed)])
        for grid, k, b, v, part in ((g, K, bt, bv, None),
                                    (G, KG, np.concatenate([bt, btl]), np.concatenate([bv, bvl]), icp)):
            s = pkg.HybridSolver(0)
            s.init(grid, k, (0, 0, 0), b, None, inst_cellpos=part)
            tm, rm = cases.unit_fluid(grid.num_cells)
            s.solve(tm, rm, np.zeros(grid.num_cells), b, v, residual_tolerance=1e-12, precision="mixed",
                    linsolver_type=linsolver_type, smooth_steps=smooth_steps, element_operator=element_operator,
                    linsolver_maxit=400)
            p, _, q = s.getSolution()
            # solves to 1e-12 of systems with condition numbers below 1e4
            assert cases.rel_err(p[:g.num_cells], ref.cell_pressure) < 1e-8
            assert cases.rel_err(q[:g.num_half_faces], ref.outflux) < 1e-8
