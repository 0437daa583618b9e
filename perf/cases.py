"""What the solver is timed on: calls of its public entry points over the
range of sizes, boundary conditions, precisions and directions that users
of the library run, on synthetic droplet fields.

Kinds of a case (`kind`):
  step   one time step's projection from the velocity, mask and density
         fields (Solver.solve_fields with project=True): returns p, u, v, w
  solve  the pressure solve of an assembled 8-slot system on the device
         (Solver.solve): returns p
  grad   forward and backward of PressureSolve: returns p, dJ/dc, dJ/db
  host   the drop-in NewSolverMG call on host arrays (Solver.new_solver_mg):
         returns p
  free   FreeSolver's masked red-black SOR with gas cells, a fixed number
         of iterations (Solver.free_solve): returns p

Sizes nx, ny, nz; per_x 1: periodic in x (walls elsewhere); method: mixed
or fp64 (the free solver has one form); ratio: density of the droplets (1
outside); drops of radius rmin .. rmax in a unit box; rtol: relative
residual of the solve.

The pressure of a closed box is defined up to a constant, which the caller
fixes: it takes the mean off where the directions are FP32 (the FP64 forms
keep a zero mean, the free solver's gas cells fix it by themselves).
"""
import math
import random

import torch

import __graft_entry__

DEV = "cuda"
NG = 2            # ghost layers of padded arrays
FREE_ITERS = 50   # FreeSolver iterations of a pass (the call's default limit)


def _case(name, kind, n, method="mixed", per_x=0, ratio=1000.0, ndrop=1, rmin=0.25, rmax=0.25, rtol=1e-10):
    nx, ny, nz = (n, n, n) if isinstance(n, int) else n
    c = dict(kind=kind, nx=nx, ny=ny, nz=nz, per_x=per_x, method=method, ratio=ratio, ndrop=ndrop, rmin=rmin,
             rmax=rmax, rtol=rtol)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest time step in use (tests, laptop-sized runs): latency and launches
        _case("step32", "step", 32),
        # a plain FP64 solve of the 64^3 unit cube, density ratio 10
        _case("solve64_fp64", "solve", 64, method="fp64", ratio=10.0),
        # an odd, ragged box: sizes the reference's multigrid refuses
        _case("ragged49x64x40_fp64", "solve", (49, 64, 40), method="fp64", ndrop=2, rmin=0.12, rmax=0.2),
        # a time step on a size that is no power of two
        _case("step100", "step", 100, ndrop=8, rmin=0.06, rmax=0.12),
        # the 128^3 single-sphere solve, density ratio 1000
        _case("solve128", "solve", 128),
        # the Fortran caller's drop-in on host arrays, with the default method
        _case("host128_fp64", "host", 128, method="fp64"),
        # the adjoint gradient at 128^3, at PressureSolve's default tolerance
        _case("grad128", "grad", 128, rtol=1e-12),
        # free-surface flow: the masked SOR iteration around gas bubbles
        _case("free128", "free", 128, method="sor", ndrop=8, rmin=0.06, rmax=0.12),
        # the 256^3 64-droplet benchmark solve, periodic in x, both forms
        _case("solve256", "solve", 256, per_x=1, ndrop=64, rmin=0.03, rmax=0.08),
        _case("solve256_fp64", "solve", 256, method="fp64", per_x=1, ndrop=64, rmin=0.03, rmax=0.08),
        # the time step of that box, from the fields
        _case("step256", "step", 256, per_x=1, ndrop=64, rmin=0.03, rmax=0.08),
        # the largest: forward and backward at 512^3, 512 droplets
        _case("grad512", "grad", 512, ndrop=512, rmin=0.01, rmax=0.04),
    ]


def draw(rng):
    kind = rng.choice(["step", "step", "solve", "solve", "grad", "grad", "host", "free"])
    top = 160 if kind in ("host", "free") else 384
    n = math.exp(rng.uniform(math.log(24), math.log(top)))
    nx, ny, nz = (max(20, round(n * rng.uniform(0.65, 1.0))) for _ in range(3))
    per_x = rng.random() < 0.4
    if per_x:   # a periodic axis is coarsened only while it is even
        nx = 2 ** round(math.log2(n))
        nx = min(max(nx, 32), 256)
    elif rng.random() < 0.5:
        nx, ny, nz = (8 * max(3, round(m / 8)) for m in (nx, ny, nz))
    method = {"free": "sor", "host": "fp64"}.get(kind) or rng.choice(["mixed", "mixed", "fp64"])
    ndrop = rng.choice([1, 2, 8, 64])
    rmax = 0.3 / ndrop ** (1 / 3)
    return _case(None, kind, (nx, ny, nz), method, int(per_x), rng.choice([10.0, 100.0, 1000.0]), ndrop, 0.5 * rmax,
                 rmax, 1e-12 if kind == "grad" else 1e-10)


# ---------------------------------------------------------------------------
# inputs, in plain torch: the density of a droplet field with a 1.5-cell
# interface and face velocities uniform in (-1, 1), closed at the walls
# ---------------------------------------------------------------------------
def _pad(f, per_x, walls):
    """Padded copy: x ghosts wrapped when periodic, otherwise (and in y, z)
    the nearest interior value or 0 (walls = "copy" / "zero")."""
    p = torch.zeros([m + 2 * NG for m in f.shape], dtype=f.dtype, device=f.device)
    p[NG:-NG, NG:-NG, NG:-NG] = f
    for g in range(NG):
        if per_x:
            p[:, :, g] = p[:, :, g + f.shape[2]]
            p[:, :, -1 - g] = p[:, :, -1 - g - f.shape[2]]
        elif walls == "copy":
            p[:, :, g] = p[:, :, NG]
            p[:, :, -1 - g] = p[:, :, -1 - NG]
    if walls == "copy":
        for g in range(NG):
            p[:, g], p[:, -1 - g] = p[:, NG], p[:, -1 - NG]
        for g in range(NG):
            p[g], p[-1 - g] = p[NG], p[-1 - NG]
    return p


def _density(case, seed):
    n = (case["nz"], case["ny"], case["nx"])
    h = [1.0 / m for m in n]
    wh = 1.5 * min(h)
    c = torch.zeros(n, dtype=torch.float64, device=DEV)
    r = random.Random(seed)
    for _ in range(case["ndrop"]):
        at = [r.uniform(0.35, 0.65) if case["ndrop"] == 1 else r.random() for _ in range(3)]
        R = r.uniform(case["rmin"], case["rmax"])
        reach = R + 15.0 * wh
        idx, d2 = [], 0.0
        for a in range(3):
            lo, hi = math.floor((at[a] - reach) / h[a]), math.ceil((at[a] + reach) / h[a])
            if a == 2 and case["per_x"]:
                lo, hi = (lo, hi) if hi - lo <= n[a] else (0, n[a])
            else:
                lo, hi = max(lo, 0), min(hi, n[a])
            i = torch.arange(lo, hi, device=DEV)
            d = (i.double() + 0.5) * h[a] - at[a]
            if a == 2 and case["per_x"]:
                d = d - torch.round(d)
            shape = [1, 1, 1]
            shape[a] = -1
            d2 = d2 + (d * d).view(shape)
            idx.append(i % n[a])
        drop = 0.5 * (1.0 - torch.tanh((d2.sqrt() - R) / wh))
        box = c[idx[0][0]:idx[0][-1] + 1, idx[1][0]:idx[1][-1] + 1]
        box.index_add_(2, idx[2], drop)
    return 1.0 + (case["ratio"] - 1.0) * c.clamp(max=1.0)


def _fields(case, seed):
    """Interior rho and face velocities (+x, +y, +z face of every cell)."""
    rho = _density(case, seed)
    gen = torch.Generator(DEV).manual_seed(seed)
    vel = [torch.rand(rho.shape, dtype=torch.float64, device=DEV, generator=gen).mul_(2).sub_(1) for _ in range(3)]
    if not case["per_x"]:
        vel[0][:, :, -1] = 0.0
    vel[1][:, -1] = 0.0
    vel[2][-1] = 0.0
    return rho, vel


def _rhs(case, vel):
    """-div u, mean removed."""
    n = (case["nx"], case["ny"], case["nz"])
    b = torch.zeros_like(vel[0])
    for a in range(3):
        b -= (vel[a] - torch.roll(vel[a], 1, 2 - a)) * n[a]
    return b - b.mean()


def _faces(case, rho):
    """2 / (rho_c + rho_nb) on the +x, +y, +z faces, 0 on walls."""
    c = torch.stack([2.0 / (rho + torch.roll(rho, -1, 2 - a)) for a in range(3)])
    if not case["per_x"]:
        c[0, :, :, -1] = 0.0
    c[1, :, -1] = 0.0
    c[2, -1] = 0.0
    return c


def _target(case, seed):
    """A smooth field: 8 sine modes of random amplitude, wavenumbers 1 .. 4."""
    r = random.Random(seed + 1)
    ax = [(torch.arange(m, dtype=torch.float64, device=DEV) + 0.5) / m for m in (case["nz"], case["ny"], case["nx"])]
    t = torch.zeros([len(a) for a in ax], dtype=torch.float64, device=DEV)
    for _ in range(8):
        k = [2 * math.pi * r.randint(1, 4) for _ in range(3)]
        amp, ph = r.uniform(-1, 1), r.uniform(0, 2 * math.pi)
        t += amp * torch.sin(k[0] * ax[0].view(-1, 1, 1) + k[1] * ax[1].view(1, -1, 1) + k[2] * ax[2] + ph)
    return t


def _gas(rho):
    return rho > rho.mean()


# ---------------------------------------------------------------------------
# what a user's program holds before the call, and the call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    pps = __graft_entry__.load_package()
    px = case["per_x"]
    grid = pps.Grid.make(case["nx"], case["ny"], case["nz"], ng=NG, bdry_cond=(px, 0, 0, px, 0, 0))
    rho, vel = _fields(case, seed)
    b = _rhs(case, vel)
    tol = case["rtol"] * float(torch.sqrt((b * b).mean()))
    s = dict(kind=case["kind"], pps=pps, solver=pps.Solver(grid, method=case["method"]), tol=tol,
             mixed=case["method"] == "mixed")
    if case["kind"] == "grad":
        s["c"] = _faces(case, rho).requires_grad_(True)
        s["b"] = b.requires_grad_(True)
        s["w"] = pps.face_weights(grid)
        s["target"] = _target(case, seed)
        s["rtol"] = case["rtol"]
        return s
    del b
    f = dict(zip(("u", "v", "w"), (_pad(v, px, "zero") for v in vel)), rho=_pad(rho, px, "copy"))
    f["um"], f["vm"], f["wm"] = pps.pressure_masks(grid)
    s["p"] = torch.zeros(grid.shape_p, dtype=torch.float64, device=DEV)
    if case["kind"] == "step":
        s["fields"] = f
        return s
    s["A"] = pps.setup_poisson(grid, f["u"], f["v"], f["w"], f["um"], f["vm"], f["wm"], f["rho"])
    pps.remove_rhs_mean(grid, s["A"])
    if case["kind"] == "host":
        s["A"], s["p"] = s["A"].cpu().numpy(), s["p"].cpu().numpy()
    if case["kind"] == "free":
        s["mask"] = _pad(_gas(rho).to(torch.int32), px, "copy")
        s["gas"] = torch.zeros_like(s["p"])
    return s


def _mean_free(s, p):
    return p - p.mean() if s["mixed"] else p


def run(s):
    kind, solver = s["kind"], s["solver"]
    if kind == "grad":
        p = s["pps"].PressureSolve.apply(s["c"], _mean_free(s, s["b"]), solver, s["w"], s["rtol"], 200)
        p = _mean_free(s, p)
        dc, db = torch.autograd.grad(p, (s["c"], s["b"]), p.detach() - s["target"])
        return dict(p=p.detach(), dc=dc, db=db)
    p = s["p"]
    inner = solver.grid.interior(p)
    if kind == "host":
        p.fill(0.0)
        solver.new_solver_mg(s["A"], p, s["tol"], maxit=100)
        return p
    p.zero_()
    if kind == "free":
        solver.free_solve(s["A"], p, s["mask"], s["gas"], 1, 0.0, 1.2, FREE_ITERS)
        return p
    if kind == "solve":
        solver.solve(s["A"], p, s["tol"], maxit=100)
        return _mean_free(s, inner)
    _, _, u, v, w = solver.solve_fields(s["fields"], p, s["tol"], maxit=100, project=True)
    return dict(p=_mean_free(s, inner), u=u, v=v, w=w)


def work(case):
    """Each input read and each output written once, and the operations of
    one application of the operator (a solve has to do more of both)."""
    n = case["nx"] * case["ny"] * case["nz"]
    per_cell = {"step": 7 + 4, "solve": 8 + 1, "host": 8 + 1, "grad": (3 + 1 + 1) + (1 + 3 + 1), "free": 8 + 0.5 + 1}
    return {"bytes": 8.0 * per_cell[case["kind"]] * n, "flops": (2 if case["kind"] == "grad" else 1) * 13.0 * n}


# ---------------------------------------------------------------------------
# the same values from plain torch in FP64
# ---------------------------------------------------------------------------
def _apply(op, x):
    y = torch.zeros_like(x)
    for a, c in enumerate(op):
        f = c * (x - torch.roll(x, -1, 2 - a))
        y += f
        y -= torch.roll(f, 1, 2 - a)
    return y


def _diag(op):
    d = torch.zeros_like(op[0])
    for a, c in enumerate(op):
        d += c + torch.roll(c, 1, 2 - a)
    return d


class _Multigrid:
    """Symmetric V-cycle (damped Jacobi, aggregates of 2 per axis) on a box
    padded to powers of two with uncoupled cells."""

    def __init__(self, op):
        self.levels = []
        while op[0].numel() > 512:
            d = _diag(op)
            n = op[0].shape
            f = [2 if m > 2 else 1 for m in n]
            self.levels.append((op, torch.where(d > 0, 0.85 / d.clamp(min=1e-300), 0.0), f))
            nxt = []
            for a, c in enumerate(op):
                g = f[2 - a]
                c = c.narrow(2 - a, 0, n[2 - a]).unflatten(2 - a, (n[2 - a] // g, g)).select(3 - a, g - 1)
                for e in range(3):
                    if e != 2 - a:
                        c = c.unflatten(e, (n[e] // f[e], f[e])).sum(e + 1) / f[e]
                nxt.append(c / g ** 2)
            op = nxt
        m = op[0].numel()
        eye = torch.eye(m, dtype=torch.float64, device=DEV)
        M = torch.stack([_apply(op, eye[i].view(op[0].shape)).flatten() for i in range(m)])
        w, v = torch.linalg.eigh(M)
        self.bottom = (v * torch.where(w > 1e-10 * w.max(), 1 / w, 0.0)) @ v.T

    def __call__(self, b, l=0):
        if l == len(self.levels):
            return (self.bottom @ b.flatten()).view(b.shape)
        op, dinv, f = self.levels[l]
        x = dinv * b
        for _ in range(2):
            x += dinv * (b - _apply(op, x))
        r = b - _apply(op, x)
        for e in range(3):
            r = r.unflatten(e, (r.shape[e] // f[e], f[e])).mean(e + 1)
        e = self(r, l + 1)
        for a in range(3):
            e = e.repeat_interleave(f[a], a)
        x += e
        for _ in range(3):
            x += dinv * (b - _apply(op, x))
        return x


class _Exact:
    def __init__(self, case, c):
        self.n = (case["nz"], case["ny"], case["nx"])
        P = [2 ** math.ceil(math.log2(m)) for m in self.n]
        self.pad = [0, P[2] - self.n[2], 0, P[1] - self.n[1], 0, P[0] - self.n[0]]
        self.op = [torch.nn.functional.pad(c[a] * float(self.n[2 - a]) ** 2, self.pad) for a in range(3)]
        self.mg = _Multigrid(self.op)

    def solve(self, b):
        """Mean-free x with M x = b - mean(b), to the rounding floor of CG."""
        r = torch.nn.functional.pad(b - b.mean(), self.pad)
        x = torch.zeros_like(r)
        d, rz, bb, best = None, None, float((r * r).sum()), math.inf
        for _ in range(200):
            z = self.mg(r)
            new = float((r * z).sum())
            d = z if d is None else z + (new / rz) * d
            rz = new
            q = _apply(self.op, d)
            al = rz / float((d * q).sum())
            x += al * d
            r -= al * q
            if float((r * r).sum()) <= 1e-30 * bb:
                break
        x = x[:self.n[0], :self.n[1], :self.n[2]]
        return x - x.mean()


def _padded_p(case, x):
    """p as the solver returns it from p = 0: the interior, and the first
    ghost layer wrapped in a periodic direction."""
    p = torch.zeros([m + 2 * NG for m in x.shape], dtype=x.dtype, device=x.device)
    p[NG:-NG, NG:-NG, NG:-NG] = x
    if case["per_x"]:
        p[NG:-NG, NG:-NG, NG - 1] = x[:, :, -1]
        p[NG:-NG, NG:-NG, -NG] = x[:, :, 0]
    return p


def _exact_free(case, rho, c, b):
    """FREE_ITERS sweeps of SOR with weight 1.2 on the liquid cells, cells of
    even index sum first; gas cells stay at 0."""
    up = [c[a] * float((case["nx"], case["ny"], case["nz"])[a]) ** 2 for a in range(3)]
    dn = [torch.roll(up[a], 1, 2 - a) for a in range(3)]
    d = _diag(up)
    i = [torch.arange(m, device=DEV) for m in rho.shape]
    odd = (i[0].view(-1, 1, 1) + i[1].view(1, -1, 1) + i[2]) % 2
    live = ~_gas(rho)
    p = torch.zeros_like(rho)
    for _ in range(FREE_ITERS):
        for colour in (0, 1):
            t = b.clone()
            for a in range(3):
                t += up[a] * torch.roll(p, -1, 2 - a) + dn[a] * torch.roll(p, 1, 2 - a)
            p = torch.where(live & (odd == colour), -0.2 * p + 1.2 / d * t, p)
    return p


def exact(case, seed):
    rho, vel = _fields(case, seed)
    b, c = _rhs(case, vel), _faces(case, rho)
    if case["kind"] == "free":
        return _padded_p(case, _exact_free(case, rho, c, b))
    if case["kind"] != "step":
        del vel
    E = _Exact(case, c)
    x = E.solve(b)
    if case["kind"] == "grad":
        lam = E.solve(x - _target(case, seed))
        dc = torch.stack([-float(E.n[2 - a]) ** 2 * (x - torch.roll(x, -1, 2 - a)) * (lam - torch.roll(lam, -1, 2 - a))
                          for a in range(3)])
        return dict(p=x, dc=torch.where(c > 0, dc, 0.0), db=lam)
    if case["kind"] == "host":
        return _padded_p(case, x).cpu().numpy()
    if case["kind"] == "solve":
        return x
    out = dict(p=x)
    for a, name in enumerate("uvw"):
        v = vel[a] - c[a] * (torch.roll(x, -1, 2 - a) - x) * float(E.n[2 - a])
        o = _pad(vel[a], case["per_x"], "zero")
        o[NG:-NG, NG:-NG, NG:-NG] = v
        out[name] = o
    return out
