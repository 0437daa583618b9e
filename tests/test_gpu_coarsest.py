"""The dense inverse of the coarsest level (k_bottom_build_reg up to 64
cells, k_bottom_build_lds to 90, k_bottom_build beyond), on grids small
enough that the finest level is the coarsest: one refinement step from zero
is then x = Minv b, the mean taken off, and must equal numpy's pseudo-
inverse solution of the same system."""
import numpy as np
import pytest

from helpers import sparse_matrix

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# sizes around the register form's limits: one cell row, a row count that is
# no multiple of 4, full 64 cells, periodic wraps of size 1 and 2, then the
# LDS form (75 and 90 cells) and the global one (91 cells)
CASES = [
    ((3, 1, 1), (0,) * 6), ((3, 3, 3), (0,) * 6), ((7, 3, 3), (0,) * 6), ((4, 4, 4), (0,) * 6),
    ((4, 4, 4), (1,) * 6), ((2, 8, 4), (1, 0, 0, 1, 0, 0)), ((5, 5, 3), (1, 0, 0, 1, 0, 0)),
    ((5, 6, 3), (1, 0, 0, 1, 0, 0)), ((7, 13, 1), (1, 0, 0, 1, 0, 0)),
]


@pytest.mark.parametrize("shape,bc", CASES)
@pytest.mark.parametrize("method,tol", [("fp64", 1e-11), ("mixed", 1e-4)])
def test_coarsest_level_is_solved_exactly(pps, orc, shape, bc, method, tol):
    print("coarsest level", shape, bc, method, flush=True)
    g = pps.Grid.make(*shape, bdry_cond=bc)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.3)], 1.0, 10.0, 1.5, seed=2)
    um, vm, wm = pps.pressure_masks(g)
    A = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    with pps.Solver(g, method=method, outer=pps.OUTER_REFINE) as s:
        p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
        s.solve(A, p, 1e-300, 1.2, 1)
    og = orc.OrcGrid.make(*shape, bc=bc)
    Ah = np.ascontiguousarray(A.cpu().numpy())
    x = np.linalg.pinv(sparse_matrix(og, Ah).toarray(), rcond=1e-11) @ Ah[7].ravel()
    got = g.interior(p).cpu().numpy().ravel()
    # condition numbers of these systems stay below 1e4: 1e-16 (FP64) and
    # 6e-8 (FP32 inverse and right-hand side) times that, with a margin
    err = np.abs((got - got.mean()) - (x - x.mean())).max() / np.abs(x - x.mean()).max()
    print(f"   err {err:.2e}", flush=True)
    assert err <= tol
