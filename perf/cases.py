"""Performance cases: the work that users of this framework have it do, through
its public entry points, from the smallest 2D run to the largest pressure
system.

Whole calls
  step    the two-phase step (Solver.problem_init, Solver.step): a short run
          of one reinitialisation interval from a given state, 2D and 3D
  batch   the same for a stack of independent 2D cases (BatchSolver)
  m3      the two-bubble MPLS_RisingBubble step (M3Solver.setup, M3Solver.step)
Parts that programs call by themselves
  poisson the variable-coefficient pressure solve (ppe_sor_init, ppe_solve_rhs)
  adjoint the differentiable WENO5 advection, forward and backward, in FP64
          and FP32 (adjoint.advect)
  uccd    the level-set advection with the upwind-CCD source
  redis   the reinitialisation of a level set that is no distance function
  curv    CCD normals and curvature
  blocks  the WENO5 advection on a multi-block layout with halo exchange

Every pass starts from the same inputs, which are copied into the solver's
fields on the device first, as a program that restarts from a stored state
does, so that a pass can be repeated.
"""
import math

import torch

from fortrancfd_amd import Case, Solver
from fortrancfd_amd.adjoint import advect
from fortrancfd_amd.blocks import Blocks
from fortrancfd_amd.solver import BatchSolver, M3Solver

F64 = torch.float64


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # one small 2D rising bubble, the reference's own CPU configuration: latency and launches
        {"name": "step2d_64x128", "kind": "step", "dim": 2, "nx": 64, "ny": 128, "nz": 1, "mixed": False,
         "half": False, "steps": 5},
        # a parameter study: 16 2D cases of one grid in one context
        {"name": "batch2d_16x128x256", "kind": "batch", "n": 16, "nx": 128, "ny": 256, "mixed": True, "steps": 5},
        # an ordinary 3D run in full precision
        {"name": "step3d_76x92x132_fp64", "kind": "step", "dim": 3, "nx": 76, "ny": 92, "nz": 132, "mixed": False,
         "half": False, "steps": 5},
        # the headline workload: 256^3 cells, FP32 cycles inside FP64 flexible CG
        {"name": "step3d_256", "kind": "step", "dim": 3, "nx": 256, "ny": 256, "nz": 256, "mixed": True,
         "half": True, "steps": 5},
        # the two-bubble problem on the reference's own grid, 140 x 140 x 280
        {"name": "m3_140x140x280", "kind": "m3", "unit": 35, "steps": 5},
        # the standalone pressure system: a small one in FP64 with odd extents, the largest one in mixed precision
        {"name": "poisson_97x81x113_fp64", "kind": "poisson", "nx": 97, "ny": 81, "nz": 113, "mixed": False,
         "half": False},
        {"name": "poisson_512_mixed", "kind": "poisson", "nx": 512, "ny": 512, "nz": 512, "mixed": True,
         "half": True},
        # differentiable advection: training-like forward and backward passes in both precisions
        {"name": "adjoint_128_fp64", "kind": "adjoint", "nx": 128, "ny": 128, "nz": 128, "f32": False, "steps": 8,
         "every": 4},
        {"name": "adjoint_101x87x117_fp32", "kind": "adjoint", "nx": 101, "ny": 87, "nz": 117, "f32": True,
         "steps": 8, "every": 4},
        # the advection's other source on a large 2D grid
        {"name": "uccd2d_1031x777", "kind": "uccd", "dim": 2, "nx": 1031, "ny": 777, "nz": 1, "steps": 4},
        # reinitialisation and curvature of a 3D level set
        {"name": "redis_curv_160x144x200", "kind": "redis", "nx": 160, "ny": 144, "nz": 200},
        # the multi-block layer: 2 x 2 x 2 blocks, a halo exchange after every stage
        {"name": "blocks_2x2x2_160x150x170", "kind": "blocks", "nx": 160, "ny": 150, "nz": 170, "gx": 2, "gy": 2,
         "gz": 2, "steps": 4},
    ]


def _size(rng, lo, hi):
    """log-uniform whole number; even and odd ones alike"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box_size(rng, lo, hi):
    """the same for the grids of flows, whose extents users take as multiples of four (the pressure multigrid pairs
    cells)"""
    return 4 * _size(rng, lo // 4, hi // 4)


def draw(rng):
    kind = rng.choice(["step2", "step3", "batch", "m3", "poisson", "poisson", "adjoint", "adjoint", "uccd", "redis",
                       "blocks"])
    if kind == "step2":
        n = _box_size(rng, 48, 300)
        return {"kind": "step", "dim": 2, "nx": n, "ny": 2 * n + 4 * rng.randint(-3, 3), "nz": 1,
                "mixed": rng.random() < 0.5, "half": False, "steps": 5}
    if kind == "step3":
        mixed = rng.random() < 0.5
        return {"kind": "step", "dim": 3, "nx": _box_size(rng, 40, 180), "ny": _box_size(rng, 40, 180),
                "nz": _box_size(rng, 60, 200), "mixed": mixed, "half": mixed and rng.random() < 0.5, "steps": 5}
    if kind == "batch":
        n = _box_size(rng, 48, 200)
        return {"kind": "batch", "n": rng.randint(3, 20), "nx": n, "ny": 2 * n, "mixed": rng.random() < 0.7,
                "steps": 5}
    if kind == "m3":
        return {"kind": "m3", "unit": 2 * rng.randint(6, 17), "steps": 5}
    if kind == "poisson":
        mixed = rng.random() < 0.5
        return {"kind": "poisson", "nx": _size(rng, 40, 320), "ny": _size(rng, 40, 320), "nz": _size(rng, 40, 320),
                "mixed": mixed, "half": mixed and rng.random() < 0.5}
    if kind == "adjoint":
        steps = rng.randint(3, 10)
        return {"kind": "adjoint", "nx": _size(rng, 32, 150), "ny": _size(rng, 32, 150), "nz": _size(rng, 32, 150),
                "f32": rng.random() < 0.5, "steps": steps, "every": rng.randint(2, 5)}
    if kind == "uccd":
        if rng.random() < 0.5:
            return {"kind": "uccd", "dim": 2, "nx": _size(rng, 64, 1400), "ny": _size(rng, 64, 1400), "nz": 1,
                    "steps": 4}
        return {"kind": "uccd", "dim": 3, "nx": _size(rng, 32, 180), "ny": _size(rng, 32, 180),
                "nz": _size(rng, 32, 180), "steps": 4}
    if kind == "redis":
        return {"kind": "redis", "nx": _size(rng, 40, 200), "ny": _size(rng, 40, 200), "nz": _size(rng, 40, 200)}
    return {"kind": "blocks", "nx": _size(rng, 48, 200), "ny": _size(rng, 48, 200), "nz": _size(rng, 48, 200),
            "gx": rng.randint(1, 3), "gy": rng.randint(1, 3), "gz": rng.randint(1, 3), "steps": 4}


# ------------------------------------------------------------- grids and inputs

def _rng(seed):
    g = torch.Generator()
    g.manual_seed(int(seed) * 7919 + 17)
    return lambda lo, hi: lo + (hi - lo) * float(torch.rand((), generator=g, dtype=F64))


def _grid(case):
    """the framework's grid of a case of kinds step, poisson, adjoint, uccd, redis, blocks"""
    k = case["kind"]
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    kw = dict(nx=nx, ny=ny, nz=nz)
    if k == "step":
        kw.update(cfl=0.1, cfl_r=0.1, redis_interval=5, picard_iters=4, ppe_tol=1e-10,
                  ppe_precision=int(case["mixed"]), ppe_max_cycles=200, ppe_rho_half=int(case["half"]))
        if case["dim"] == 2:
            return Case(dim=2, xend=1.0, yend=ny / nx, gvec=(0.0, -1.0, 0.0), **kw)
        # 256^3 is the benchmark's [0,1]^2 x [0,2] box (dz = 2 dx); other grids have cubic cells
        z = 2.0 if nx == ny == nz else nz / nx
        return Case(dim=3, xend=1.0, yend=ny / nx, zend=z, gvec=(0.0, 0.0, -1.0), **kw)
    if k == "poisson":
        return Case(dim=3, xend=1.0, yend=ny / nx, zend=nz / nx, ppe_max_cycles=200,
                    ppe_precision=int(case["mixed"]), ppe_rho_half=int(case["half"]), **kw)
    if k == "uccd":
        return Case(dim=case["dim"], xend=1.0, yend=ny / nx, zend=nz / nx, cfl=0.2, ls_scheme=1, **kw)
    if k == "redis":
        return Case(dim=3, xend=1.0, yend=ny / nx, zend=nz / nx, cfl_r=0.1, **kw)
    # adjoint, blocks: the deformation field's unit cube
    return Case(dim=3, xend=1.0, yend=1.0, zend=1.0, cfl=0.3 if k == "adjoint" else 0.2, **kw)


def _axes(c, face=None, dev="cuda"):
    """broadcastable coordinates x, y[, z] of the ghosted box; on axis `face` those of the high faces"""
    out = []
    dims = [(c.nx, c.xstart, c.dx), (c.ny, c.ystart, c.dy)] + ([(c.nz, c.zstart, c.dz)] if c.dim == 3 else [])
    for a, (n, start, h) in enumerate(dims):
        i = torch.arange(-c.ghc, n + c.ghc, dtype=F64, device=dev)
        shape = [1] * c.dim
        shape[c.dim - 1 - a] = -1
        out.append((start + (i + (1.0 if face == a else 0.5)) * h).reshape(shape))
    return out


def _full(c, a):
    """a contiguous flat ghosted array of a broadcastable field"""
    return a.expand(c.shape).contiguous().reshape(-1)


def _clamped(c, a):
    """the field of a broadcastable interior formula with zero-gradient ghosts"""
    a = a.expand(c.shape)
    for ax in range(c.dim):
        n = a.shape[ax]
        i = torch.clamp(torch.arange(n, device=a.device), c.ghc, n - c.ghc - 1)
        a = a.index_select(ax, i)
    return a.contiguous().reshape(-1)


def _sphere(c, centre, radius):
    d = sum((x - x0) ** 2 for x, x0 in zip(_axes(c), centre))
    return torch.sqrt(d) - radius


def _bubble(c, u):
    """a bubble in the lower half of a case's box: signed distance, positive in the heavy fluid"""
    w = [c.xend - c.xstart, c.yend - c.ystart] + ([c.zend - c.zstart] if c.dim == 3 else [])
    lo = min(w)
    centre = [x * u(0.45, 0.55) for x in w]
    return _sphere(c, centre, lo * u(0.18, 0.26))


def _velocity(c, u, amp):
    """discretely divergence-free MAC velocity of no-penetration vortices: u = d psi/dy, v = -d psi/dx of a stream
    function at the cell corners that vanishes on the walls, in 3D modulated along z (ghosts follow the solver's
    rules)"""
    pi = math.pi
    lx, ly = c.xend - c.xstart, c.yend - c.ystart
    xf, yf = _axes(c, 0)[0], _axes(c, 1)[1]
    psi = 0.0
    for m in (1, 2):
        for n in (1, 2):
            psi = psi + u(-1.0, 1.0) / (m * n) * torch.sin(m * pi * xf / lx) * torch.sin(n * pi * yf / ly)
    psi = amp * psi * min(lx, ly) / (2.0 * pi)
    z = 1.0
    if c.dim == 3:
        z = 1.0 + 0.5 * torch.cos(pi * u(0.5, 1.5) * _axes(c)[2] / (c.zend - c.zstart))
    U = (psi - torch.roll(psi, 1, dims=c.dim - 2)) / c.dy * z
    V = -(psi - torch.roll(psi, 1, dims=c.dim - 1)) / c.dx * z
    out = {"u": _full(c, U), "v": _full(c, V)}
    if c.dim == 3:
        out["w"] = torch.zeros_like(out["u"])
    return out


def _cell_velocity(c, u, amp):
    """smooth cell velocity with zero-gradient ghosts, the deformation field with seeded amplitudes"""
    pi = math.pi
    s = [torch.sin(pi * x / (b - a)) for x, (a, b) in zip(_axes(c), _box(c))]
    t = [torch.sin(2 * pi * x / (b - a)) for x, (a, b) in zip(_axes(c), _box(c))]
    a = [amp * u(0.8, 1.2) for _ in range(3)]
    if c.dim == 2:
        return [_clamped(c, a[0] * s[0] ** 2 * t[1]), _clamped(c, -a[1] * t[0] * s[1] ** 2)]
    return [_clamped(c, 2 * a[0] * s[0] ** 2 * t[1] * t[2]), _clamped(c, -a[1] * t[0] * s[1] ** 2 * t[2]),
            _clamped(c, -a[2] * t[0] * t[1] * s[2] ** 2)]


def _box(c):
    return [(c.xstart, c.xend), (c.ystart, c.yend)] + ([(c.zstart, c.zend)] if c.dim == 3 else [])


def _batch(case, u):
    """rising bubbles of seeded radius, density ratio and Eoetvoes number on one grid, with one time step within
    every case's explicit capillary limit"""
    nx, ny = case["nx"], case["ny"]
    par = [(u(0.15, 0.3), 1.0 / u(10.0, 1000.0), u(1.0, 100.0)) for _ in range(case["n"])]
    dx = 1.0 / nx
    cfl = min([0.1] + [0.5 * math.sqrt((1.0 - r12) / math.log(1.0 / r12) * we * dx ** 3 / (2.0 * math.pi)) / dx
                       for _, r12, we in par])
    cs = [Case(dim=2, nx=nx, ny=ny, nz=1, xend=1.0, yend=2.0, gvec=(0.0, -1.0, 0.0), rho_12=r12, mu_12=0.01,
               re=1.0e4, we=we, fr=1.0, cfl=cfl, cfl_r=0.1, redis_interval=5, ppe_tol=1e-10,
               ppe_precision=int(case["mixed"])) for _, r12, we in par]
    return cs, [r for r, _, _ in par]


def _two_bubbles(case):
    n = case["unit"]
    return Case(dim=3, nx=4 * n, ny=4 * n, nz=8 * n, xend=4.0, yend=4.0, zend=8.0, cfl=0.005, cfl_r=0.5, ls_w=1.5,
                rho_12=0.001, mu_12=0.01, re=67.27, we=16.0, fr=1.0, gvec=(0.0, 0.0, -1.0), ppe_tol=1e-10,
                ppe_precision=1, ppe_max_cycles=100)


def _poisson_fields(c, u, seed):
    """a sphere of density 1 in a fluid of 1000, joined by the smoothed Heaviside over 1.5 cells, and a uniform
    random source of zero mean"""
    w = [b - a for a, b in _box(c)]
    x = _sphere(c, [v * u(0.45, 0.55) for v in w], min(w) * u(0.25, 0.35)) / (1.5 * c.dx)
    h = 0.5 * (1.0 + x + torch.sin(math.pi * x) / math.pi)
    h = torch.where(x > 1, torch.ones_like(x), torch.where(x < -1, torch.zeros_like(x), h))
    rho = _full(c, 1.0 + 999.0 * h)
    del x, h
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) + 12345)
    f = torch.rand(c.size, generator=g, dtype=F64, device="cuda").mul_(2.0).sub_(1.0)
    inner = c.interior(f)
    inner -= inner.mean()
    return rho, f


def _not_a_distance(c, u):
    """the level set of a bubble stretched by a smooth positive factor"""
    phi = _bubble(c, u)
    f = 1.0
    for x, (a, b) in zip(_axes(c), _box(c)):
        f = f + u(0.1, 0.3) * torch.sin(math.pi * u(0.7, 2.3) * x / (b - a))
    return _clamped(c, phi * f)


# -------------------------------------------------------------------- prepare

def prepare(case, seed):
    k, u = case["kind"], _rng(seed)
    st = {"kind": k, "case": case}
    if k == "step":
        c = _grid(case)
        st["solver"] = Solver(c)
        st["in"] = {"phi": _full(c, _bubble(c, u)), **_velocity(c, u, 0.2)}
        st["in"]["p"] = torch.zeros_like(st["in"]["phi"])
        st["names"] = ["phi", "p", "u", "v"] + (["w"] if c.dim == 3 else [])
    elif k == "batch":
        cs, radii = _batch(case, u)
        c = cs[0]
        st["solver"] = BatchSolver(cs)
        phi, vel = [], []
        for r in radii:
            phi.append(_full(c, _sphere(c, (0.5, 0.5), r)))
            vel.append(_velocity(c, u, 0.2))
        st["in"] = {"phi": torch.cat(phi), "u": torch.cat([v["u"] for v in vel]),
                    "v": torch.cat([v["v"] for v in vel])}
        st["in"]["p"] = torch.zeros_like(st["in"]["phi"])
        st["names"] = ["phi", "p", "u", "v"]
    elif k == "m3":
        c = _two_bubbles(case)
        st["solver"] = M3Solver(c)
        r = [0.5 * u(0.96, 1.04) for _ in range(2)]
        x = [2.0 + u(-0.1, 0.1) for _ in range(2)]
        p1, p2 = (_full(c, -_sphere(c, (x[b], 2.0, (1.0, 2.5)[b]), r[b])) for b in range(2))
        st["in"] = {"phi1": p1, "phi2": p2, "phi": torch.maximum(p1, p2), **_velocity(c, u, 0.05)}
        st["in"]["p"] = torch.zeros_like(p1)
        st["names"] = ["phi", "phi1", "phi2", "p", "u", "v", "w"]
    elif k == "poisson":
        c = _grid(case)
        st["solver"] = Solver(c)
        rho, f = _poisson_fields(c, u, seed)
        st["solver"].push_device("rho", rho.data_ptr())
        st["solver"].push_device("ppe_src", f.data_ptr())
        torch.cuda.synchronize()
        st["in"] = {"p": torch.zeros_like(f)}
        st["names"] = ["p"]
    elif k == "adjoint":
        c = _grid(case)
        st["solver"] = Solver(c)
        dt = torch.float32 if case["f32"] else F64
        st["phi0"] = _clamped(c, _sphere(c, [u(0.3, 0.4) for _ in range(3)], 0.15)).to(dt).requires_grad_(True)
        st["A"] = torch.tensor(u(0.9, 1.1), dtype=dt, device="cuda", requires_grad=True)
        x, y, z = _axes(c)
        st["bar"] = _clamped(c, torch.cos(3 * x + u(0, 3)) * torch.sin(2 * y + u(0, 3)) * torch.cos(4 * z)).to(dt)
    elif k == "uccd":
        c = _grid(case)
        st["solver"] = Solver(c)
        for n, a in zip(("nu", "nv", "nw"), _cell_velocity(c, u, 0.5)):
            st["solver"].push_device(n, a.data_ptr())
            torch.cuda.synchronize()
        st["in"] = {"phi": _clamped(c, _bubble(c, u))}
        st["names"] = ["phi"]
    elif k == "redis":
        c = _grid(case)
        st["solver"] = Solver(c)
        st["in"] = {"phi": _not_a_distance(c, u)}
        st["names"] = ["phi", "nx", "ny", "nz", "curv"]
    else:
        c = _grid(case)
        st["blocks"] = b = Blocks(c, case["gx"], case["gy"], case["gz"])
        st["phi0"] = _clamped(c, _bubble(c, u))
        st["vel"] = []
        for a in _cell_velocity(c, u, 0.5):
            st["vel"].append(b.new_stack())
            b.scatter(a, st["vel"][-1])
            b.sync(st["vel"][-1])
        st["stack"] = b.new_stack()
        st["out"] = torch.zeros(c.size, dtype=F64, device="cuda")
    if "names" in st:
        n = next(iter(st["in"].values()))
        st["out"] = {m: torch.zeros_like(n) for m in st["names"]}
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------------ run

def run(st):
    k, case = st["kind"], st["case"]
    if k == "adjoint":
        phi = advect(st["phi0"], st["A"], st["solver"], case["steps"], 3.0, case["every"])
        g = torch.autograd.grad(phi, [st["phi0"], st["A"]], st["bar"])
        return {"phi": phi.detach(), "grad_phi0": g[0], "grad_A": g[1]}
    if k == "blocks":
        b = st["blocks"]
        b.scatter(st["phi0"], st["stack"])
        b.sync(st["stack"])
        for _ in range(case["steps"]):
            b.level_set_rk3_solver(st["stack"], *st["vel"])
        b.gather(st["stack"], st["out"])
        return st["out"]
    s = st["solver"]
    for n, a in st["in"].items():
        s.push_device(n, a.data_ptr())
    more = {}
    if k in ("step", "batch"):
        s.problem_init(False)
        for _ in range(case["steps"]):
            s.step()
    elif k == "m3":
        s.set_time(0.0, 0)
        s.setup()
        for _ in range(case["steps"]):
            s.step()
    elif k == "poisson":
        s.ppe_sor_init()
        s.ppe_solve_rhs(1e-10, int(case["mixed"]))
    elif k == "uccd":
        for _ in range(case["steps"]):
            s.level_set_rk3_solver()
    else:
        more["pseudo_steps"] = s.level_set_rk3_redis(1)
        s.curv()
    for n, a in st["out"].items():
        s.pull_device(n, a.data_ptr())
    return {**st["out"], **more}


# ----------------------------------------------------------------------- work

def _cells(case):
    if case["kind"] == "batch":
        return case["n"] * case["nx"] * case["ny"]
    if case["kind"] == "m3":
        return 128 * case["unit"] ** 3
    return case["nx"] * case["ny"] * case.get("nz", 1)


def work(case):
    """What one pass cannot do without: every input read once and every output written once per step, and the
    arithmetic of its explicit parts (a WENO5 reconstruction is about 75 operations; two to a face and direction).
    The sweeps of the pressure iteration, which depend on the method, are counted as one application of its
    operator to the accuracy asked for."""
    k, n = case["kind"], _cells(case)
    d = 2 if (k == "batch" or case.get("dim") == 2) else 3
    steps = case.get("steps", 1)
    if k in ("step", "batch", "m3"):
        # phi, velocity and pressure in and out, the momentum source of the previous step in and of this step out
        fields = 2 * (2 + d) + 2 * d + (2 if k == "m3" else 0)
        return {"bytes": 8.0 * n * fields * steps, "flops": n * steps * (3 * d * 150.0 + 4 * d * 50.0)}
    if k == "poisson":
        return {"bytes": 8.0 * 3 * n, "flops": 30.0 * n}
    if k == "adjoint":
        # forward: phi and velocity in, phi out; backward: the states again, the adjoint and the velocity's in and out
        b = 4.0 if case["f32"] else 8.0
        return {"bytes": b * n * steps * (5 + 1 + 3 + 2 + 6), "flops": n * steps * (2 * 3 * 490.0 + 3 * 1500.0)}
    if k == "uccd":
        return {"bytes": 8.0 * n * (2 + d) * steps, "flops": n * steps * 3 * d * 80.0}
    if k == "redis":
        return {"bytes": 8.0 * 6 * n, "flops": n * (31 * 3 * 530.0 + 6 * 40.0)}
    return {"bytes": 8.0 * n * 5 * steps, "flops": n * steps * 3 * 490.0}


# ------------------------------------------------------------------ tolerance

def tolerance(case):
    """About four times the largest difference seen over the listed cases and 150 drawn ones: for the flow steps
    and the pressure solve between solves to the default 1e-10 and to 2e-12 or less, for the others between the
    framework and exact()."""
    k = case["kind"]
    if k in ("step", "batch", "m3"):
        return {"rel": 1.6e-10, "max": 1.5e-8}
    if k == "poisson":
        return {"rel": 1.2e-8, "max": 2.5e-8}
    if k == "adjoint":
        return {"rel": 3.7e-6, "max": 4e-4} if case["f32"] else {"rel": 1.2e-14, "max": 8e-13}
    if k == "uccd":
        return {"rel": 2e-15, "max": 2.4e-14}
    if k == "redis":
        return {"rel": 4.5e-11, "max": 3e-9}
    return {"rel": 5e-16, "max": 5e-15}


# ---------------------------------------------------------------------- exact

def _dim_of(axis, nd):
    return nd - 1 - axis


def _shifted(a, axis, offsets, pos):
    """a at clamp(pos + o) along an axis, for each offset"""
    d = _dim_of(axis, a.dim())
    n = a.shape[d]
    return [a.index_select(d, torch.clamp(pos + o, 0, n - 1)) for o in offsets]


def _weno(g, eps):
    """left-biased WENO5-JS value of five samples (smoothness indicators times 12, weights 1, 6, 3)"""
    b1 = 13 * (g[0] - 2 * g[1] + g[2]) ** 2 + 3 * (g[0] - 4 * g[1] + 3 * g[2]) ** 2
    b2 = 13 * (g[1] - 2 * g[2] + g[3]) ** 2 + 3 * (g[1] - g[3]) ** 2
    b3 = 13 * (g[2] - 2 * g[3] + g[4]) ** 2 + 3 * (3 * g[2] - 4 * g[3] + g[4]) ** 2
    a1, a2, a3 = 1 / (eps + b1) ** 2, 6 / (eps + b2) ** 2, 3 / (eps + b3) ** 2
    return (a1 * (2 * g[0] - 7 * g[1] + 11 * g[2]) + a2 * (-g[1] + 5 * g[2] + 2 * g[3]) +
            a3 * (2 * g[2] + 5 * g[3] - g[4])) / (6 * (a1 + a2 + a3))


def _advection(phi, vel, h):
    """- div of the upwind-split WENO5 flux of an interior array"""
    out = torch.zeros_like(phi)
    for axis in range(phi.dim()):
        d = _dim_of(axis, phi.dim())
        n = phi.shape[d]
        u = vel[axis]
        f = torch.arange(-1, n, device=phi.device)
        sp = _shifted(0.5 * (u + u.abs()) * phi, axis, (-2, -1, 0, 1, 2), f)
        sm = _shifted(0.5 * (u - u.abs()) * phi, axis, (3, 2, 1, 0, -1), f)
        F = _weno(sp, 1e-13) + _weno(sm, 1e-13)
        out = out - (F.narrow(d, 1, n) - F.narrow(d, 0, n)) / h[axis]
    return out


def _rk3(phi, L, dt):
    l0 = L(phi)
    p1 = phi + dt * l0
    l1 = L(p1)
    p2 = p1 + dt * (l1 - 3 * l0) / 4
    return p2 + dt * (8 * L(p2) - l0 - l1) / 12


def _ghosted(c, a):
    """interior array -> flat ghosted array with zero-gradient ghosts"""
    for ax in range(a.dim()):
        n = a.shape[ax]
        a = a.index_select(ax, torch.clamp(torch.arange(-c.ghc, n + c.ghc, device=a.device), 0, n - 1))
    return a.contiguous().reshape(-1)


def _steps(c):
    return (c.dx, c.dy, c.dz)


def _exact_adjoint(case, seed):
    """the run differentiated step by step by autograd in 64 bits"""
    st = prepare(case, seed)
    c, A = st["solver"].case, float(st["A"].detach())
    pi = math.pi
    x, y, z = (a.narrow(_dim_of(q, 3), c.ghc, (c.nx, c.ny, c.nz)[q]) for q, a in enumerate(_axes(c)))
    shape = (c.nz, c.ny, c.nx)
    s, t = [torch.sin(pi * a) for a in (x, y, z)], [torch.sin(2 * pi * a) for a in (x, y, z)]
    uhat = [a.expand(shape).contiguous() for a in (2 * s[0] ** 2 * t[1] * t[2], -t[0] * s[1] ** 2 * t[2],
                                                   -t[0] * t[1] * s[2] ** 2)]
    ct = [math.cos(pi * n * c.dt / 3.0) for n in range(case["steps"])]
    step = lambda p, a, n: _rk3(p, lambda q: _advection(q, [a * ct[n] * v for v in uhat], _steps(c)), c.dt)
    inner = lambda a: c.interior(a.detach().to(F64)).clone()
    states = [inner(st["phi0"])]
    with torch.no_grad():
        for n in range(case["steps"]):
            states.append(step(states[-1], A, n))
    # the result's ghosts are copies of interior cells: their cotangents belong to those
    bar = st["bar"].to(F64).reshape(c.shape)
    for ax in range(3):
        n, g = bar.shape[ax] - 2 * c.ghc, c.ghc
        lo, hi = bar.narrow(ax, 0, g).sum(ax, keepdim=True), bar.narrow(ax, n + g, g).sum(ax, keepdim=True)
        bar = bar.narrow(ax, g, n).clone()
        bar.narrow(ax, 0, 1).add_(lo)
        bar.narrow(ax, n - 1, 1).add_(hi)
    gA = torch.zeros((), dtype=F64, device="cuda")
    for n in reversed(range(case["steps"])):
        p = states[n].requires_grad_(True)
        a = torch.tensor(A, dtype=F64, device="cuda", requires_grad=True)
        bar, ga = torch.autograd.grad(step(p, a, n), [p, a], bar)
        gA += ga
    full = torch.zeros(c.shape, dtype=F64, device="cuda")
    c.interior(full).copy_(bar)
    return {"phi": _ghosted(c, states[-1].detach()), "grad_phi0": full.reshape(-1), "grad_A": gA}


def _line_operators(kind, n, h):
    """first- and second-derivative matrices of the combined compact scheme on a line of n points: the 2x2 block
    tridiagonal system of (f', f'') solved for every unit source"""
    M = torch.zeros(2 * n, 2 * n, dtype=F64)
    R = torch.zeros(2 * n, n, dtype=F64)
    c1, c2, c3 = -1.93596119008109, 1.99692238016218, -0.06096119008109
    b1, b2, b3 = 0.1251282341599089, -0.2487176584009104, 0.0001282341599089
    for i in range(1, n - 1):
        e, q = 2 * i, 2 * i + 1
        if kind == "ccd":
            first = {(-1, 0): 7 / 16, (0, 0): 1.0, (1, 0): 7 / 16, (-1, 1): h / 16, (1, 1): -h / 16}
            src = {-1: -15 / 16 / h, 1: 15 / 16 / h}
        elif kind == "up":
            first = {(-1, 0): 0.875, (0, 0): 1.0, (-1, 1): b1 * h, (0, 1): b2 * h, (1, 1): b3 * h}
            src = {-1: c1 / h, 0: c2 / h, 1: c3 / h}
        else:
            first = {(0, 0): 1.0, (1, 0): 0.875, (-1, 1): -b3 * h, (0, 1): -b2 * h, (1, 1): -b1 * h}
            src = {-1: -c3 / h, 0: -c2 / h, 1: -c1 / h}
        for (o, w), v in first.items():
            M[e, 2 * (i + o) + w] = v
        for o, v in src.items():
            R[e, i + o] = v
        M[q, 2 * i - 2], M[q, 2 * i + 2] = -9 / 8 / h, 9 / 8 / h
        M[q, 2 * i - 1], M[q, 2 * i + 1], M[q, 2 * i + 3] = -1 / 8, 1.0, -1 / 8
        R[q, i - 1], R[q, i], R[q, i + 1] = 3 / h ** 2, -6 / h ** 2, 3 / h ** 2
    for i, s in ((0, 1), (n - 1, -1)):
        e, q, m = 2 * i, 2 * i + 1, 2 * (i + s)
        M[e, e], M[e, m], M[e, m + 1] = 1.0, 2.0, -s * h
        M[q, q], M[q, m], M[q, m + 1] = 1.0, -s * 2.5 / h, 8.5
        for o, v in enumerate((-3.5, 4.0, -0.5)):
            R[e, i + s * o] = s * v / h
        for o, v in enumerate((34 / 3, -83 / 4, 10.0, -7 / 12)):
            R[q, i + s * o] = v / h ** 2
    X = torch.linalg.solve(M.cuda(), R.cuda())
    return X[0::2].contiguous(), X[1::2].contiguous()


def _along(c, D, a, axis):
    """a line operator on the ghosted lines of an interior array with zero-gradient ghosts; interior rows"""
    d = _dim_of(axis, a.dim())
    n = a.shape[d]
    g = c.ghc
    i = torch.clamp(torch.arange(-g, n + g, device=a.device), 0, n - 1)
    b = a.movedim(d, 0)
    return (D[g:g + n] @ b.index_select(0, i).reshape(n + 2 * g, -1)).reshape(b.shape).movedim(0, d).contiguous()


def _exact_uccd(case, seed):
    st = prepare(case, seed)
    c = st["solver"].case
    vel = []
    for n in ("nu", "nv", "nw")[:c.dim]:
        t = torch.zeros(c.size, dtype=F64, device="cuda")
        st["solver"].pull_device(n, t.data_ptr())
        st["solver"].sync()
        vel.append(c.interior(t).clone())
    h = _steps(c)
    sizes = (c.nx, c.ny, c.nz)
    ops = [[_line_operators(k, sizes[a] + 2 * c.ghc, h[a])[0] for k in ("up", "down")] for a in range(c.dim)]

    def L(p):
        s = 0.0
        for a in range(c.dim):
            s = s - vel[a] * torch.where(vel[a] > 0, _along(c, ops[a][0], p, a), _along(c, ops[a][1], p, a))
        return s

    phi = c.interior(st["in"]["phi"]).clone()
    for _ in range(case["steps"]):
        phi = _rk3(phi, L, c.dt)
    return {"phi": _ghosted(c, phi)}


def _heaviside(phi, w):
    x = phi / w
    band = (x <= 1 - 1e-12) & (x >= -1 + 1e-12)
    H = torch.where(band, 0.5 * (1 + x + torch.sin(math.pi * x) / math.pi), (x > 0).to(F64)).clamp(0.0, 1.0)
    return H, torch.where(band, 0.5 * (1 + torch.cos(math.pi * x)) / w, torch.zeros_like(x))


def _exact_redis(case, seed):
    st = prepare(case, seed)
    c = st["solver"].case
    h, w, r12 = _steps(c), c.ls_wid, c.rho_12
    phi = c.interior(st["in"]["phi"]).clone()
    S = 2 * _heaviside(phi, w)[0] - 1

    def gradient(p):
        g = 0.0
        for a in range(3):
            n = p.shape[_dim_of(a, 3)]
            at = torch.arange(n, device=p.device)
            D = (p - _shifted(p, a, (-1,), at)[0]) / h[a]
            m = _weno(_shifted(D, a, (-2, -1, 0, 1, 2), at), 1e-10)
            q = _weno(_shifted(D, a, (3, 2, 1, 0, -1), at), 1e-10)
            up = torch.maximum(-q.clamp(max=0), m.clamp(min=0))
            dn = torch.maximum(q.clamp(min=0), -m.clamp(max=0))
            g = g + torch.where(S >= 0, up, dn) ** 2
        return torch.sqrt(g)

    def box(a):
        for ax in range(3):
            n = a.shape[ax]
            at = torch.arange(n, device=a.device)
            a = a + a.index_select(ax, (at - 1).clamp(min=0)) + a.index_select(ax, (at + 1).clamp(max=n - 1))
        return a

    def L(p):
        g = gradient(p)
        H, d = _heaviside(p, w)
        lam = (2 * (1 - r12) * H + r12) * d
        num, den = lam * S * (g - 1), g * d * lam
        num, den = 51 * num + box(num), 51 * den + box(den)
        s1 = torch.where(den.abs() > 1e-12, num / den * d, torch.zeros_like(den))
        return S - (S - s1) * g

    t, it = 0.0, 0
    while True:
        new = _rk3(phi, L, c.rdt)
        err, phi = float((new - phi).abs().max()), new
        it, t = it + 1, t + c.rdt
        if t > 3 * c.dx or err <= 1e-5:
            break
    n = [a + 2 * c.ghc for a in (c.nx, c.ny, c.nz)]
    D = [_line_operators("ccd", n[a], h[a]) for a in range(3)]
    f = [_along(c, D[a][0], phi, a) for a in range(3)]
    ff = [_along(c, D[a][1], phi, a) for a in range(3)]
    fxy, fxz, fyz = _along(c, D[1][0], f[0], 1), _along(c, D[2][0], f[0], 2), _along(c, D[2][0], f[1], 2)
    k = ((ff[1] + ff[2]) * f[0] ** 2 + (ff[0] + ff[2]) * f[1] ** 2 + (ff[0] + ff[1]) * f[2] ** 2 -
         2 * (fxy * f[0] * f[1] + fxz * f[0] * f[2] + fyz * f[1] * f[2])) / \
        (f[0] ** 2 + f[1] ** 2 + f[2] ** 2 + 1e-12) ** 1.5
    out = {m: _ghosted(c, a) for m, a in zip(("phi", "nx", "ny", "nz", "curv"), [phi, *f, k])}
    return {**out, "pseudo_steps": it}


def _exact_blocks(case, seed):
    c, u = _grid(case), _rng(seed)
    phi = c.interior(_clamped(c, _bubble(c, u))).clone()
    vel = [c.interior(a).clone() for a in _cell_velocity(c, u, 0.5)]
    for _ in range(case["steps"]):
        phi = _rk3(phi, lambda p: _advection(p, vel, _steps(c)), c.dt)
    out = torch.zeros(c.shape, dtype=F64, device="cuda")   # the gather writes the interior
    c.interior(out).copy_(phi)
    return out.reshape(-1)


def _exact_poisson(case, seed):
    """conjugate gradients with the diagonal as preconditioner, to the rounding of the residual"""
    c, u = _grid(case), _rng(seed)
    rho, f = (c.interior(a).clone() for a in _poisson_fields(c, u, seed))
    face, h = [], _steps(c)
    for a in range(3):
        d = _dim_of(a, 3)
        n = rho.shape[d]
        face.append(2 / (rho.narrow(d, 0, n - 1) + rho.narrow(d, 1, n - 1)) / h[a] ** 2)

    def A(p):   # minus the operator: positive semi-definite
        out = torch.zeros_like(p)
        for a in range(3):
            d = _dim_of(a, 3)
            n = p.shape[d]
            q = face[a] * (p.narrow(d, 1, n - 1) - p.narrow(d, 0, n - 1))
            out.narrow(d, 0, n - 1).sub_(q)
            out.narrow(d, 1, n - 1).add_(q)
        return out

    diag = torch.zeros_like(rho)
    for a in range(3):
        d = _dim_of(a, 3)
        n = rho.shape[d]
        diag.narrow(d, 0, n - 1).add_(face[a])
        diag.narrow(d, 1, n - 1).add_(face[a])
    x = torch.zeros_like(f)
    r = -(f - f.mean())
    norm = float(r.norm())
    z = r / diag
    p = z.clone()
    rz = (r * z).sum()
    for it in range(20000):
        q = A(p)
        al = rz / (p * q).sum()
        x += al * p
        r -= al * q
        if it % 50 == 49 and float(r.norm()) < 1e-13 * norm:
            break
        z = r / diag
        new = (r * z).sum()
        p.mul_(new / rz).add_(z)
        rz = new
    return {"p": _ghosted(c, x - x.mean())}


def exact(case, seed):
    """Plain torch in 64 bits.  Not for whole steps (a restatement of the full solver; their parts are the other
    cases) and not where it would take too long or too much memory."""
    k, n = case["kind"], _cells(case)
    if k == "adjoint":
        return _exact_adjoint(case, seed) if n <= 3_500_000 else None
    if k == "uccd":
        return _exact_uccd(case, seed)
    if k == "redis":
        return _exact_redis(case, seed)
    if k == "blocks":
        return _exact_blocks(case, seed)
    if k == "poisson":
        return _exact_poisson(case, seed) if n <= 4_000_000 else None
    return None
