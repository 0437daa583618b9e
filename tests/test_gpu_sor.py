"""RB-SOR iterations queued ahead of their stopping test (NewSolver_std,
newsolver.f90:78-174, and FreeSolver, freesurface.f90:700-855) against the
oracle: p, the iteration count and the history are those of the iteration that
the reference ends at, whatever ends it.  The sweeps keep the reference's
arithmetic (bounds on p as in the tests of whole solves); the norms differ by
the order of their sums.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WALLS, PX = (0,) * 6, (1, 0, 0, 1, 0, 0)


def _system(pps, orc, shape, bc):
    g = pps.Grid.make(*shape, bdry_cond=bc)
    og = orc.OrcGrid.make(*shape, bc=bc)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.6, 0.25)], 1.0, 100.0, 1.5, seed=3)
    um, vm, wm = pps.pressure_masks(g)
    At = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, At)
    return g, og, At, np.ascontiguousarray(At.cpu().numpy())


def _same(og, p, want, bound):
    p, want = og.interior(p.cpu().numpy()), og.interior(want)
    err = np.abs(p - want).max() / np.abs(want).max()
    print(f"   max rel diff {err:.1e}", flush=True)
    assert err <= bound


@pytest.mark.parametrize("norm", [1, 2])
@pytest.mark.parametrize("shape,bc", [((64, 40, 24), WALLS), ((130, 9, 33), WALLS), ((32, 36, 70), PX)])
@pytest.mark.parametrize("last", [1, 2, 7])
def test_new_solver_std_stops_where_the_oracle_does(pps, orc, shape, bc, last, norm):
    print("sor stop", shape, bc, last, norm, flush=True)
    g, og, At, A = _system(pps, orc, shape, bc)
    want = np.zeros(og.shape_p)
    rc, it, t2, hist = orc.newsolver_std(og, A, want, 0.0, 1.2, last, norm)
    assert rc == 0 and it == last + 1 and (last == 1 or t2 < hist[:-1].min())
    # the limit ends it, or a tolerance that this iteration is the first to meet
    for tol, limit in ((0.0, last), (t2 * 1.0000001, last + 1), (t2 * 1.0000001, last + 9)):
        with pps.Solver(g, method="sor") as s:
            p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
            git, gt2 = s.solve(At, p, tol, 1.2, limit, norm)
            ghist = np.array(s.history())
        assert git == (last + 1 if tol == 0.0 else last)
        assert gt2 == pytest.approx(t2, rel=1e-9)
        assert ghist.shape == hist.shape and np.allclose(ghist, hist, rtol=1e-9, atol=0)
        _same(og, p, want, 1e-12)


@pytest.mark.parametrize("shape,bc", [((64, 40, 24), WALLS), ((32, 36, 70), PX)])
def test_new_solver_std_diverges_where_the_oracle_does(pps, orc, shape, bc):
    """beta > 2: the sum passes 1e16 and ends the call, p being that iteration's."""
    print("sor divergence", shape, bc, flush=True)
    g, og, At, A = _system(pps, orc, shape, bc)
    want = np.zeros(og.shape_p)
    rc, it, t2, _ = orc.newsolver_std(og, A, want, 0.0, 2.5, 200, 2)
    assert rc != 0 and 1 < it < 200 and np.isfinite(t2)
    with pps.Solver(g, method="sor") as s:
        p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
        with pytest.raises(pps.PPSError) as e:
            s.solve(At, p, 0.0, 2.5, 200, 2)
        assert e.value.code == pps.ERR_DIVERGED
        assert len(s.history()) == it - 1
    _same(og, p, want, 1e-9)


def test_free_solver_without_iterations(pps, orc):
    """A limit below 1 runs none: it = 1 (a loop of no trips, as the oracle's),
    and the handle's later calls see their own totals."""
    g, og, At, A = _system(pps, orc, (32, 24, 20), WALLS)
    m = torch.zeros(g.shape_p, dtype=torch.int32, device="cuda")
    m[10, 12, 14] = 1
    pgas = torch.ones(g.shape_p, dtype=torch.float64, device="cuda")

    def call(s, limit):
        p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
        it, t2 = s.free_solve(At, p, m, pgas, 1, 0.0, 1.2, limit)
        return it, t2, list(s.history()), p

    with pps.Solver(g, method="sor") as s:
        first = call(s, 5)
        assert first[0] == 6 and len(first[2]) == 5
        for limit in (0, -1, -3):
            print("free solver limit", limit, flush=True)
            want = np.zeros(og.shape_p)
            rc, it, t2, _ = orc.free_solver(og, A, want, m.cpu().numpy(), pgas.cpu().numpy(), 1, 0.0, 1.2, limit)
            none = call(s, limit)
            assert rc == 0 and none[:3] == (it, t2, [])
            assert np.array_equal(og.interior(none[3].cpu().numpy()), og.interior(want))
            again = call(s, 5)
            assert again[:3] == first[:3] and torch.equal(again[3], first[3])
