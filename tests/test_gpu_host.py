"""Host arrays through the pinned pieces (stage_copy): the solve must be the
device entry's bit for bit, ghost cells included, on both sides of the size
below which the runtime copies, with remainders of a chunk, with p below that
size and above it, a second time on the same pieces, and from pinned arrays.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("shape", [(24, 20, 28), (48, 48, 48), (52, 50, 54), (100, 102, 98), (128, 128, 128)])
def test_host_solve_is_the_device_solve(pps, shape, pinned):
    print("host arrays", shape, pinned, flush=True)
    g = pps.Grid.make(*shape)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 10.0, 1.5, seed=4)
    um, vm, wm = pps.pressure_masks(g)
    A = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    tol = 1e-8 * float(torch.sqrt((A[7] ** 2).mean()))
    p0 = torch.rand(g.shape_p, dtype=torch.float64, generator=torch.Generator().manual_seed(3))
    Ah = A.cpu().pin_memory() if pinned else A.cpu()
    with pps.Solver(g, method="fp64") as s:
        p = p0.cuda()
        s.solve(A, p, tol, 1.2, 50)
        want = p.cpu().numpy()
        for turn in range(2):
            ph = (p0.clone().pin_memory() if pinned else p0.clone()).numpy()
            s.new_solver_mg(Ah.numpy(), ph, tol, 1.2, 50, 2)
            assert np.array_equal(ph, want), (turn, float(np.abs(ph - want).max()))


@pytest.mark.parametrize("flag", [1, 2])
def test_host_free_solve_is_the_device_solve(pps, flag):
    """Three or four arrays in one copy, the mask's cells half the size of the
    others'."""
    shape = (52, 50, 54)
    print("host free solver", shape, flag, flush=True)
    g = pps.Grid.make(*shape)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 10.0, 1.5, seed=4)
    A = pps.setup_poisson(g, u, v, w, *pps.pressure_masks(g), rho, 1.0)
    rng = np.random.default_rng(7)
    mask = rng.choice([0, 1, 2, 3], size=g.shape_p, p=[0.4, 0.25, 0.25, 0.1]).astype(np.int32)
    gas = rng.standard_normal(g.shape_p) if flag == 1 else None
    p0 = rng.standard_normal(g.shape_p)
    Ah = A.cpu().numpy()
    with pps.Solver(g, method="sor") as s:
        p = torch.from_numpy(p0).cuda()
        it, t2 = s.free_solve(A, p, torch.from_numpy(mask).cuda(), torch.from_numpy(gas).cuda() if flag == 1 else None,
                              flag, 0.0, 1.2, 5)
        want = p.cpu().numpy()
        for turn in range(2):
            ph = p0.copy()
            hit, ierr, ht2 = s.free_solver(Ah, ph, mask, gas, flag, 0.0, 1.2, 5)
            assert (hit, ierr, ht2) == (it, 0, t2), turn
            assert np.array_equal(ph, want), (turn, float(np.abs(ph - want).max()))


def test_host_poi_solve_is_the_device_solve(pps):
    shape = (52, 50, 54)
    print("host poi_solve", shape, flush=True)
    g = pps.Grid.make(*shape)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 10.0, 1.5, seed=4)
    A = pps.setup_poisson(g, u, v, w, *pps.pressure_masks(g), rho, 1.0)
    pps.remove_rhs_mean(g, A)
    p0 = np.random.default_rng(7).standard_normal(g.shape_p)
    with pps.Solver(g, method="fp64") as s:
        p = torch.from_numpy(p0).cuda()
        it = s.poi_solve_device(A, p, 1e-8)
        want = p.cpu().numpy()
        for turn in range(2):
            ph = p0.copy()
            assert s.poi_solve(A.cpu().numpy(), ph, 1e-8) == it
            assert np.array_equal(ph, want), (turn, float(np.abs(ph - want).max()))
