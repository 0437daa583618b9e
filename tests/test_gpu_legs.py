"""The V-cycle's fused smoothing legs (k_leg_pre / k_leg_post on small levels,
k_march on large ones) and coarse end (k_tail) against the kernels they replace.

One refinement step from zero is x = V(b): the default cycle must equal, to
rounding, the cycle that runs colour by colour (SMOOTH_COLOUR_PASSES: k_rb,
k_resid_restrict(_g), k_prolong_add(_g) and k_bottom_solve) on the same
hierarchy.  Shapes at the edges of the tail's thread and pair counts, odd
and short axes, semi-coarsened boxes, periodic axes, and a non-singular
operator (stored diagonals).  The bounds are rounding of the precision times
the few hundred operations of a cycle, as the sweeps' own tests take them.
"""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

WALLS, PX, PALL = (0,) * 6, (1, 0, 0, 1, 0, 0), (1,) * 6
TOL = {"fp64": 1e-12, "mixed": 2e-5}


def _cycle(pps, g, A, method, **opt):
    with pps.Solver(g, method=method, outer=pps.OUTER_REFINE, **opt) as s:
        p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
        s.solve(A, p, 1e-300, 1.2, 1)
    return g.interior(p).clone()


def _compare(pps, shape, bc, method, shift=0.0, lengths=(1.0, 1.0, 1.0)):
    print("cycle vs colour passes", shape, bc, method, shift, lengths, flush=True)
    g = pps.Grid.make(*shape, bdry_cond=bc, lengths=lengths)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2), (0.8, 0.3, 0.6, 0.12)], 1.0, 100.0, 1.5, seed=4)
    um, vm, wm = pps.pressure_masks(g)
    A = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    if shift:
        A[6] *= 1.0 + shift
    x = _cycle(pps, g, A, method)
    ref = _cycle(pps, g, A, method, smoother=pps.SMOOTH_COLOUR_PASSES, tail_cells=-1)
    err = float((x - ref).abs().max() / ref.abs().max())
    print(f"   err {err:.2e}", flush=True)
    assert err <= TOL[method]


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,bc,lengths", [
    ((32, 32, 32), WALLS, (1.0, 1.0, 1.0)),    # two pairs a thread
    ((28, 14, 12), PX, (1.0, 1.0, 1.0)),       # 7 wide below: a periodic axis odd, the coarsest
    ((17, 16, 16), WALLS, (1.0, 1.0, 1.0)),    # missing second cells
    ((9, 30, 15), WALLS, (1.0, 1.0, 1.0)),
    ((3, 50, 41), WALLS, (0.06, 1.0, 0.8)),    # one pair a row and a half
    ((40, 20, 24), PALL, (1.0, 1.0, 1.0)),
    ((32, 32, 16), WALLS, (1.0, 1.0, 4.0)),    # z kept for two levels
    ((48, 12, 40), PX, (1.0, 1.0, 1.0)),
])
def test_coarse_end_matches_colour_passes(pps, shape, bc, lengths, method):
    _compare(pps, shape, bc, method, lengths=lengths)


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(32, 32, 32), (17, 22, 27)])
def test_coarse_end_with_stored_diagonals(pps, shape, method):
    _compare(pps, shape, WALLS, method, shift=0.02)


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,bc,lengths", [
    ((40, 40, 40), WALLS, (1.0, 1.0, 1.0)),    # a finest level of whole tiles
    ((41, 35, 37), WALLS, (1.0, 1.0, 1.0)),    # remainders in every direction
    ((64, 23, 50), PX, (1.0, 1.0, 1.0)),
    ((48, 48, 32), PALL, (1.0, 1.0, 1.0)),
    ((2, 96, 48), WALLS, (0.02, 1.0, 0.5)),    # one pair a row
    ((64, 64, 17), WALLS, (1.0, 1.0, 1.5)),    # x, y halved, z kept
    ((64, 64, 64), WALLS, (1.0, 1.0, 1.0)),    # 24-plane regions in FP32
])
def test_legs_match_colour_passes(pps, shape, bc, lengths, method):
    _compare(pps, shape, bc, method, lengths=lengths)


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,bc,lengths", [
    ((72, 72, 72), WALLS, (1.0, 1.0, 1.0)),    # whole tiles
    ((73, 67, 71), WALLS, (1.0, 1.0, 1.0)),    # odd rows (4-byte loads), remainders of one tile row
    ((76, 50, 98), WALLS, (1.0, 1.0, 1.0)),    # a last tile of two columns
    ((64, 81, 70), PX, (1.0, 1.0, 1.0)),
    ((66, 70, 76), WALLS, (1.0, 1.0, 1.0)),    # even rows, no multiple of 16 bytes in FP32
    ((96, 64, 64), PALL, (1.0, 1.0, 1.0)),
    ((40, 96, 96), WALLS, (2.0, 1.0, 1.0)),    # x kept
    ((80, 77, 60), WALLS, (1.0, 1.0, 2.0)),    # z kept, y odd
    ((96, 24, 96), PALL, (1.0, 0.25, 1.0)),    # one tile of rows, wrapped onto itself (FP64)
    ((128, 150, 16), PX, (1.0, 1.0, 0.1)),     # short columns
])
def test_marching_legs_match_colour_passes(pps, shape, bc, lengths, method):
    _compare(pps, shape, bc, method, lengths=lengths)


@pytest.mark.parametrize("method", ["fp64", "mixed"])
def test_legs_with_stored_diagonals(pps, method):
    _compare(pps, (45, 40, 33), WALLS, method, shift=0.02)


def test_repeated_solves_swap_buffers(pps):
    """An odd number of cycles leaves the finest level's two iterate buffers
    swapped; a second solve on the handle must not see them as one."""
    g = pps.Grid.make(40, 44, 36)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 100.0, 1.5, seed=4)
    um, vm, wm = pps.pressure_masks(g)
    A = pps.setup_poisson(g, u, v, w, um, vm, wm, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    brms = float(torch.sqrt((A[7] ** 2).mean()))
    with pps.Solver(g, method="fp64") as s:
        for its in (1, 2, 3):
            p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
            s.solve(A, p, 1e-300, 1.2, its)
            p.zero_()
            it, _ = s.solve(A, p, 1e-10 * brms, 1.2, 60, allow_maxit=False)
            print(f"after {its} cycles: {it} iterations", flush=True)
            assert it <= 15


@pytest.mark.parametrize("closed", [0.0, 1e-44])
@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,bc", [
    ((72, 72, 72), WALLS),    # 16-byte loads in both precisions
    ((66, 70, 76), WALLS),    # 16-byte loads in FP64, 4-byte ones in FP32
    ((73, 67, 71), WALLS),    # 4-byte loads, missing second cells
    ((64, 81, 70), PX),       # walls in y and z only
])
def test_marching_legs_with_cells_open_to_one_side(pps, shape, bc, method, closed):
    """Dead ends of one cell (faces closed by the masks, or all but closed: their
    couplings are FP32 denormals) at the walls and beside them.  A marching leg
    holds cells beyond a wall; whatever it takes as their rows, they must not
    reach the cells inside through couplings of zero."""
    print("dead ends", shape, bc, method, closed, flush=True)
    g = pps.Grid.make(*shape, bdry_cond=bc)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2), (0.8, 0.3, 0.6, 0.12)], 1.0, 100.0, 1.5, seed=4)
    masks = pps.pressure_masks(g)
    nx, ny, nz = shape
    ends = [((11, ny - 1, 9), (1, -1)), ((30, 0, 21), (1, 1)), ((37, 40, nz - 1), (2, -1)), ((20, 33, 0), (2, 1))]
    if not bc[0]:   # at the x walls; those of 16 bytes before the high one
        ends += [((nx - q, 9 + 8 * q, 13 + 6 * q), (0, -1)) for q in (1, 2, 3, 4)]
        ends += [((0, 25, 31), (0, 1)), ((nx - 1, ny - 1, 44), (1, -1)), ((nx - 1, ny - 1, 50), (0, -1))]
    for cell, way in ends:
        for a in range(3):
            for side in (-1, 1):
                c = list(cell)
                c[a] += min(side, 0)
                if (a, side) != way and 0 <= c[a] < shape[a] - 1:   # a wall's faces are closed
                    masks[a][g.ng + c[2], g.ng + c[1], g.ng + c[0]] = closed
    A = pps.setup_poisson(g, u, v, w, *masks, rho, 1.0)
    pps.remove_rhs_mean(g, A)
    for cell, way in ends:
        open_ = A[:6, cell[2], cell[1], cell[0]] > 1e-30
        assert open_.nonzero().flatten().tolist() == [2 * way[0] + (way[1] > 0)]
    x = _cycle(pps, g, A, method)
    ref = _cycle(pps, g, A, method, smoother=pps.SMOOTH_COLOUR_PASSES, tail_cells=-1)
    assert bool(torch.isfinite(ref).all())
    err = float((x - ref).abs().max() / ref.abs().max())
    print(f"   err {err:.2e}", flush=True)
    assert err <= TOL[method]


@pytest.mark.parametrize("closed", [1e-40, 1e-44])
@pytest.mark.parametrize("shape", [(48, 48, 48), (72, 72, 72), (73, 67, 71)])
def test_mixed_solve_with_denormal_couplings(pps, shape, closed):
    """A block whose faces are all but closed: in FP32 its diagonals are
    denormals, whose reciprocals overflow.  The mixed solve must converge as the
    FP64 one does (two iterations allowed for the precision)."""
    print("denormal block", shape, closed, flush=True)
    g = pps.Grid.make(*shape)
    rho, u, v, w = pps.synth_fields(g, [(0.4, 0.5, 0.5, 0.2)], 1.0, 100.0, 1.5, seed=4)
    masks = list(pps.pressure_masks(g))
    block = torch.zeros(g.shape_p, dtype=torch.bool, device="cuda")
    lo, hi = g.ng + shape[0] // 4, g.ng + shape[0] // 2
    block[lo:hi, lo:hi, lo:hi] = True
    for a in range(3):
        faces = (block | torch.roll(block, -1, 2 - a)) & (masks[a] > 0)
        masks[a][faces] = closed
        (u, v, w)[a][faces] = 0.0
    A = pps.setup_poisson(g, u, v, w, *masks, rho, 1.0)
    inside = g.interior(block)
    A[7][inside] = 0.0
    A[7][~inside] -= A[7].sum() / (~inside).sum()
    tol = 1e-10 * float((A[7] ** 2).mean().sqrt())
    its = {}
    for method in ("fp64", "mixed"):
        with pps.Solver(g, method=method) as s:
            p = torch.zeros(g.shape_p, dtype=torch.float64, device="cuda")
            its[method] = s.solve(A, p, tol, 1.2, 60, allow_maxit=False)[0]
    print("   iterations", its, flush=True)
    assert its["mixed"] <= its["fp64"] + 2
