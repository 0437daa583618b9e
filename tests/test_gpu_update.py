"""k_update (r -= alpha q, two cells a turn): an odd number of cells, fewer
cells than a block has threads, and more than its blocks take in one turn.

The residual that the CG iteration carries along (its history) must be the
oracle's residual of the iterate it stops at.  Both are sums of the same
products in FP64, apart by rounding: a few hundred operations an iteration on
values up to the first residual, 1e-13 of it, taken as 1e-9 of a residual
that is still above 1e-4 of it; a lost cell would show as 1 / sqrt(n) or more.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(7, 9, 5), (31, 33, 35), (64, 64, 64), (83, 81, 79), (104, 102, 100)])
def test_carried_residual_is_the_iterates(pps, orc, shape, method):
    print("carried residual", shape, method, flush=True)
    g = pps.Grid.make(*shape)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 10.0, 1.5, seed=4)
    um, vm, wm = pps.pressure_masks(g)
    A = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    og = orc.OrcGrid.make(*shape)
    Ah = A.cpu().numpy()
    with pps.Solver(g, method=method) as s:
        for its in (1, 3):
            p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
            s.solve(A, p, 1e-300, 1.2, its)
            carried = s.history()[-1]
            r = orc.residual_field(og, Ah, np.ascontiguousarray(p.cpu().numpy()))
            true = float(np.sqrt((r ** 2).mean()))
            print(f"   {its}: carried {carried:.12e} true {true:.12e}", flush=True)
            assert abs(carried - true) <= 1e-9 * true
