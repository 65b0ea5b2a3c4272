"""Timed workloads of sgnx: what a user's program has it do, through the public
entry points of the `sgnx` package, on inputs made on the GPU from a seed.

Kinds of pass
  rhs       dU = R(U, t) on device arrays (SGN2D.rhs_device)
  adaptive  an adaptive BS3(2) run of a few accepted steps from a given state
            (SGN2D.integrateAdaptive); returns the state it reaches
  batch     the same for an uneven ensemble advanced together (Batch)
  vjp       one vector-Jacobian product of the right-hand side
            (SGN2D.rhs_vjp_device), as a Newton or sensitivity code calls it
  gradient  a taped adaptive run and its reverse sweep (SGN2D.tapeBegin*,
            integrateAdaptive, adjoint_device): the cotangents of the initial
            state and of the still depth

Grids run from 8x6 elements (25 nodes each, five FP64 variables per node) to
2000x1000. Beds: a slope with a shoal, a basin with mounds, a continental
margin with per-point roughness. Sides: periodic, a channel (periodic in x,
walls in y), closed walls, an incident wave on the left with walls elsewhere, a
margin (walls in x, periodic in y).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "sgn-hyperbolic-gpu_amd"))

import sgnx  # noqa: E402

G, GAMMA, ALPHA = 9.81, 1.5, 3.0
SIDES = {"periodic": ("periodic",) * 4, "channel": ("periodic", "periodic", "wall", "wall"),
         "walls": ("wall",) * 4, "inflow": ("inflow", "wall", "wall", "wall"),
         "margin": ("wall", "wall", "periodic", "periodic")}
RUN = {"atol": 1e-8, "rtol": 1e-6, "cfl": 0.5}      # the solver's usual tolerances
# a taped run starts inside a wave period: at t = 0 the incident ghost ties with
# the fluid at rest in the flux's max of wave speeds, which has no derivative there
TAPE_T0 = 0.1
INVERSION = {"atol": 1e-10, "rtol": 1e-8, "cfl": 0.5}   # those of a gauge inversion


def listed():
    return [
        # the smallest call: the gate grid a new build is checked on
        {"name": "rhs-8x6", "kind": "rhs", "nx": 8, "ny": 6, "sides": "periodic", "bed": "basin"},
        # a small channel, the size of a laptop run
        {"name": "rhs-128x64", "kind": "rhs", "nx": 128, "ny": 64, "sides": "channel",
         "bed": "basin"},
        # an ordinary grid whose sizes fit no tile
        {"name": "rhs-387x191", "kind": "rhs", "nx": 387, "ny": 191, "sides": "periodic",
         "bed": "basin"},
        # the production right-hand side
        {"name": "rhs-1024x512", "kind": "rhs", "nx": 1024, "ny": 512, "sides": "inflow",
         "bed": "shoal"},
        # a short run of the small channel: launches and the host's part count
        {"name": "adaptive-128x64", "kind": "adaptive", "nx": 128, "ny": 64, "sides": "channel",
         "bed": "basin", "steps": 20},
        # the production run: incident waves over a shoal, the fluid at rest at first
        {"name": "adaptive-1024x512", "kind": "adaptive", "nx": 1024, "ny": 512,
         "sides": "inflow", "bed": "shoal", "steps": 10},
        # the largest single grid: an uplift over a rough continental margin
        {"name": "adaptive-2000x1000", "kind": "adaptive", "nx": 2000, "ny": 1000,
         "sides": "margin", "bed": "margin", "steps": 5},
        # a parameter sweep of members that cannot fill the GPU alone
        {"name": "batch-24-small", "kind": "batch", "members": 24, "nx_min": 32, "nx_max": 128,
         "sides": "inflow", "bed": "shoal", "steps": 10},
        # the production sweep's sizes
        {"name": "batch-8-mixed", "kind": "batch", "members": 8, "nx_min": 128, "nx_max": 512,
         "sides": "inflow", "bed": "shoal", "steps": 5},
        # one product of the production grid
        {"name": "vjp-1024x512", "kind": "vjp", "nx": 1024, "ny": 512, "sides": "inflow",
         "bed": "shoal"},
        # a gauge inversion's gradient under a budget of held states
        {"name": "gradient-256x128", "kind": "gradient", "nx": 256, "ny": 128, "sides": "walls",
         "bed": "basin", "steps": 30, "states": 10, "gauges": 20},
        # a gradient of the reached state with every step's stage inputs kept, ragged grid
        {"name": "gradient-603x301", "kind": "gradient", "nx": 603, "ny": 301, "sides": "inflow",
         "bed": "shoal", "steps": 8, "states": 0, "gauges": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rhs", "rhs", "adaptive", "adaptive", "batch", "vjp", "gradient"])
    sides = rng.choice(["periodic", "channel", "walls", "inflow", "margin"])
    bed = {"inflow": "shoal", "margin": "margin"}.get(sides, "basin")
    if kind == "batch":
        lo = _log_int(rng, 16, 128)
        return {"kind": kind, "members": rng.randint(3, 24), "nx_min": lo,
                "nx_max": lo + _log_int(rng, 8, 256), "sides": "inflow", "bed": "shoal",
                "steps": rng.randint(3, 10)}
    nx = _log_int(rng, 8, {"rhs": 2000, "adaptive": 2000, "vjp": 1200, "gradient": 700}[kind])
    ny = 4 + int(nx * rng.uniform(0.4, 1.0))
    case = {"kind": kind, "nx": nx, "ny": min(ny, 1000), "sides": sides, "bed": bed}
    if kind == "adaptive":
        case["steps"] = rng.randint(3, 20) if nx < 1100 else rng.randint(2, 4)
    if kind == "gradient":
        case["steps"] = rng.randint(4, 24) if nx < 400 else rng.randint(2, 8)
        case["states"] = rng.choice([0, rng.randint(2, 8)])
        case["gauges"] = rng.choice([0, rng.randint(1, 20)])
    return case


# ---- inputs --------------------------------------------------------------------------------
# one element: GLL points of degree 4, local node a + 5 b; arrays [ey, ex, b, a]
_S = math.sqrt(3.0 / 7.0)
XI = (-1.0, -_S, 0.0, _S, 1.0)


def _extent(case, nx, ny):
    if case["bed"] == "margin":
        return 2.0e5, 2.0e5 * ny / nx
    return 96.0, 96.0 * ny / nx


def _coords(nx, ny, lx, ly, dev):
    xi = 0.5 * (torch.tensor(XI, dtype=torch.float64, device=dev) + 1.0)
    ex = torch.arange(nx, dtype=torch.float64, device=dev)
    ey = torch.arange(ny, dtype=torch.float64, device=dev)
    x = (ex[:, None] + xi) * (lx / nx)
    y = (ey[:, None] + xi) * (ly / ny)
    return x[None, :, None, :], y[:, None, :, None]


def _mesh_points(nx, ny, dev):
    """The index of every node among the grid's distinct points, per axis."""
    a = torch.arange(5, device=dev)
    return ((4 * torch.arange(ny, device=dev)[:, None] + a)[:, None, :, None],
            (4 * torch.arange(nx, device=dev)[:, None] + a)[None, :, None, :])


def _slow_wavenumber(omega, H):
    """k of the slow branch of the relaxed system at frequency omega (bisection)."""
    def cp(k):
        q = k * H
        J = 1.0 + q * q / (2.0 * GAMMA)
        mu = (q / ALPHA) ** 2 / (2.0 * GAMMA)
        half = 0.5 * (J + mu)
        return math.sqrt(G * H / (half + math.sqrt(max(half * half - mu, 0.0))))
    lo, hi = 0.0, omega / math.sqrt(G * H)
    while hi * cp(hi) < omega:
        hi *= 2.0
    for _ in range(80):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if mid * cp(mid) < omega else (lo, mid)
    return hi


def _inflow(ny, H=0.45, period=1.0, amp=0.01):
    """Ghost coefficients of a 1 s, 1 cm incident wave: (base, sin, cos) per variable."""
    omega = 2.0 * math.pi / period
    cp = omega / _slow_wavenumber(omega, H)
    q = cp * cp / H - G
    row = [[H, amp, 0.0], [0.0, cp * amp, 0.0], [0.0, 0.0, 0.0],
           [0.0, 0.0, -GAMMA * q * amp / omega], [0.0, H * q * amp, 0.0]]
    return torch.tensor(row, dtype=torch.float64).repeat(ny * 5, 1, 1), omega


def _fields(case, nx, ny, seed, moving, dev):
    """Still depth and state [5, ny, nx, 5, 5] of one grid, continuous across elements."""
    g = torch.Generator().manual_seed(1000003 * (seed % 999983) + 1009 * nx + ny)

    def u(lo, hi):
        return lo + (hi - lo) * float(torch.rand((), generator=g, dtype=torch.float64))

    lx, ly = _extent(case, nx, ny)
    x, y = _coords(nx, ny, lx, ly, dev)
    per_x = case["sides"] in ("periodic", "channel")
    per_y = case["sides"] in ("periodic", "margin")

    def hump(w):
        xc, yc = u(0.2, 0.8) * lx, u(0.2, 0.8) * ly
        return torch.exp(-((x - xc) / w) ** 2 - ((y - yc) / w) ** 2)

    if case["bed"] == "shoal":
        h0 = 0.45
        slope = torch.clamp(h0 - (x - 40.0) / 20.0, 0.10, h0)
        xc, yc, r, crest = u(18.0, 30.0), u(0.3, 0.7) * ly, u(1.5, 6.0), u(0.3, 0.9)
        H = slope - crest * h0 * torch.exp(-((x - xc) / r) ** 2 - ((y - yc) / r) ** 2)
    elif case["bed"] == "margin":
        h0 = 4000.0
        H = 50.0 + 1975.0 * (1.0 - torch.tanh((x - u(0.55, 0.75) * lx) / u(5e3, 15e3)))
        gd = torch.Generator(device=dev).manual_seed(seed % (1 << 31))
        rough = torch.rand((4 * ny + 1, 4 * nx + 1), generator=gd, dtype=torch.float64,
                           device=dev) * 0.04 - 0.02
        if per_y:
            rough[-1] = rough[0]
        iy, ix = _mesh_points(nx, ny, dev)
        H = H * (1.0 + rough[iy, ix])
    else:
        h0 = 0.5
        H = torch.full((1, 1, 1, 1), h0, dtype=torch.float64, device=dev)
        for _ in range(6):
            H = H - u(0.02, 0.06) * hump(u(2.0, 6.0))
    H = H.expand(ny, nx, 5, 5).contiguous()
    eta = torch.zeros_like(H)
    if case["bed"] == "margin":
        amp, sx, sy = u(0.5, 2.0), u(5e3, 2e4), u(1e4, 4e4)
        eta = eta + amp * torch.exp(-((x - u(0.2, 0.4) * lx) / sx) ** 2
                                    - ((y - u(0.3, 0.7) * ly) / sy) ** 2)
    elif case["sides"] != "inflow" or moving:
        for _ in range(8):
            eta = eta + u(0.005, 0.03) * hump(u(2.0, 6.0))
    U = torch.zeros((5, ny, nx, 5, 5), dtype=torch.float64, device=dev)
    U[0] = H + eta
    if moving:
        s = math.sqrt(h0 * G) * 0.05
        for v, amp in ((1, s), (2, s), (3, 0.3 * s), (4, 0.1 * s * s)):
            # whole waves along a periodic axis, half waves between walls
            kx = (2 if per_x else 1) * math.pi * int(u(1, 6)) / lx
            ky = (2 if per_y else 1) * math.pi * int(u(1, 6)) / ly
            U[v] = U[0] * amp * (torch.sin(kx * x + (u(0, 6.2) if per_x else 0.0))
                                 * torch.cos(ky * y + (u(0, 6.2) if per_y else 0.0)))
    par = (G, ALPHA * math.sqrt(G * h0), GAMMA, 0.0)
    return H, U, par, lx, ly


def _weights(n, seed, dev):
    gd = torch.Generator(device=dev).manual_seed(7 + seed % (1 << 31))
    return torch.randn(n, generator=gd, dtype=torch.float64, device=dev)


def _misfit(case, seed, dev):
    """A smooth cotangent of the reached state, as a misfit to a target state has."""
    nx, ny = case["nx"], case["ny"]
    g = torch.Generator().manual_seed(seed % (1 << 31) + 3)
    x, y = _coords(nx, ny, 1.0, 1.0, dev)
    W = torch.zeros((5, ny, nx, 5, 5), dtype=torch.float64, device=dev)
    for v in range(5):
        for _ in range(3):
            a, kx, ky = torch.rand(3, generator=g, dtype=torch.float64).tolist()
            W[v] += (a - 0.5) * (torch.cos(math.pi * int(1 + 4 * kx) * x)
                                 * torch.cos(math.pi * int(1 + 4 * ky) * y))
    return W.reshape(-1)


def _members(case, seed):
    g = torch.Generator().manual_seed(seed % (1 << 31) + 11)
    n = case["members"]
    # the ensemble's sizes are the case's, spread evenly; the beds are the seed's
    nx = [round(case["nx_min"] + (case["nx_max"] - case["nx_min"]) * (i + 0.5) / n)
          for i in range(n)]
    seeds = torch.randint(1 << 30, (n,), generator=g).tolist()
    return [(a, max(5, a // 2), s) for a, s in zip(nx, seeds)]


def _gauge_nodes(case, nd, seed):
    g = torch.Generator().manual_seed(seed % (1 << 31) + 5)
    return torch.randint(nd, (case["gauges"],), generator=g).sort().values


# ---- the program's side --------------------------------------------------------------------
class _Buffer:
    """The resident state of a solver, as torch reads it without a copy. The
    tensor holds this object, and so the solver whose memory it shows."""

    def __init__(self, s):
        self.owner = s
        self.__cuda_array_interface__ = {"shape": (s.nTotal(),), "typestr": "<f8",
                                         "data": (s.state_ptr(), False), "version": 3}


def _resident(s):
    return torch.as_tensor(_Buffer(s), device="cuda")


def _solver(case, nx, ny, seed, moving):
    H, U, par, lx, ly = _fields(case, nx, ny, seed, moving, "cuda")
    inflow = None
    if case["sides"] == "inflow":
        table, omega = _inflow(ny)
        inflow = (table.reshape(-1).numpy(), omega)
    s = sgnx.SGN2D(4, nx, ny, lx, ly, sgnx.Params(*par), bc=SIDES[case["sides"]], inflow=inflow)
    torch.cuda.synchronize()
    s.setDepth(H.data_ptr(), device=True)
    return s, U.reshape(-1)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        made = [_solver(case, nx, ny, sd, False) for nx, ny, sd in _members(case, seed)]
        solvers, states = [m[0] for m in made], [m[1] for m in made]
        for s, U in made:
            _resident(s).copy_(U)
        dt0 = [s.cflTimeStep(cfl=RUN["cfl"]) for s in solvers]
        opts = sgnx.RkOpts(atol=RUN["atol"], rtol=RUN["rtol"], max_accepted=case["steps"])
        return {"kind": kind, "batch": sgnx.Batch(solvers), "solvers": solvers, "U0": states,
                "dt0": dt0, "opts": opts}
    s, U = _solver(case, case["nx"], case["ny"], seed, kind in ("rhs", "vjp"))
    st = {"kind": kind, "s": s, "U0": U, "t": 0.0}
    if kind in ("rhs", "vjp"):
        st["t"] = 0.3
        st["out"] = torch.empty_like(U)
    if kind == "vjp":
        st["W"] = _weights(U.numel(), seed, "cuda")
        st["theta"] = torch.empty(s.nDof(), dtype=torch.float64, device="cuda")
    if kind in ("adaptive", "gradient"):
        _resident(s).copy_(U)
        r = INVERSION if kind == "gradient" else RUN
        st["dt0"] = s.cflTimeStep(cfl=r["cfl"])
        st["opts"] = sgnx.RkOpts(atol=r["atol"], rtol=r["rtol"], max_accepted=case["steps"])
    if kind == "gradient":
        st["steps"], st["states"] = case["steps"], case["states"]
        st["nodes"] = None
        st["Ubar"], st["gbar"] = None, None
        if case["gauges"]:
            st["nodes"] = _gauge_nodes(case, s.nDof(), seed).numpy()
            st["gbar"] = _weights(case["steps"] * case["gauges"], seed, "cuda")
        else:
            st["Ubar"] = _misfit(case, seed, "cuda")
        st["U0bar"] = torch.empty_like(U)
        st["theta"] = torch.empty(s.nDof(), dtype=torch.float64, device="cuda")
    return st


def run(st):
    kind = st["kind"]
    if kind == "batch":
        for s, U in zip(st["solvers"], st["U0"]):
            _resident(s).copy_(U)
        stats = st["batch"].integrateAdaptive(0.0, 1e9, st["dt0"], st["opts"])
        return {"U": [_resident(s) for s in st["solvers"]],
                "steps": [[q.accepted, q.rejected] for q in stats],
                "t": [q.tReached for q in stats]} if len(stats) <= 16 else \
               {"U": torch.cat([_resident(s) for s in st["solvers"]]),
                "t": torch.tensor([q.tReached for q in stats], dtype=torch.float64),
                "steps": torch.tensor([[q.accepted, q.rejected] for q in stats])}
    s = st["s"]
    if kind == "rhs":
        s.rhs_device(st["U0"].data_ptr(), st["out"].data_ptr(), st["t"])
        return st["out"]
    if kind == "vjp":
        s.rhs_vjp_device(st["U0"].data_ptr(), st["W"].data_ptr(), st["out"].data_ptr(),
                         st["theta"].data_ptr(), st["t"])
        return {"Ubar": st["out"], "theta": st["theta"]}
    _resident(s).copy_(st["U0"])
    if kind == "adaptive":
        q = s.integrateAdaptive(0.0, 1e9, st["dt0"], st["opts"])
        return {"U": _resident(s), "t": q.tReached, "accepted": q.accepted,
                "rejected": q.rejected}
    if st["nodes"] is not None:
        s.setGauges(st["nodes"], st["steps"])
    if st["states"]:
        s.tapeBeginPlan(st["steps"], st["states"])
    else:
        s.tapeKeepStages(True)
        s.tapeBegin(st["steps"])
    q = s.integrateAdaptive(TAPE_T0, 1e9, st["dt0"], st["opts"])
    s.tapeEnd()
    s.adjoint_device(st["Ubar"].data_ptr() if st["Ubar"] is not None else 0,
                     st["gbar"].data_ptr() if st["gbar"] is not None else 0,
                     st["U0bar"].data_ptr(), st["theta"].data_ptr())
    return {"U0bar": st["U0bar"], "theta": st["theta"], "accepted": q.accepted}


# floating-point operations of one right-hand side at one node: the two
# derivative sums of five fluxes and of the depth (120), the lifts and their
# quotients (85), fluxes, quotients and sources at the node (60), and its share
# of 10 interface nodes per element (35); a product differentiates each term
# once with respect to both of its factors
RHS_FLOPS, VJP_FLOPS = 300, 700


def work(case):
    kind = case["kind"]
    if kind == "batch":
        nodes = sum(25 * a * b for a, b, _ in _members(case, 0))
    else:
        nodes = 25 * case["nx"] * case["ny"]
    if kind == "rhs":       # U and the still depth in, dU out
        return {"bytes": 88 * nodes, "flops": RHS_FLOPS * nodes}
    if kind == "vjp":       # U, W and the still depth in, both cotangents out
        return {"bytes": 136 * nodes, "flops": VJP_FLOPS * nodes}
    # a step takes u, k1 and the still depth to uNew and k4
    steps = case["steps"]
    step = {"bytes": 168 * nodes, "flops": 3 * RHS_FLOPS * nodes}
    if kind in ("adaptive", "batch"):
        return {"bytes": steps * step["bytes"], "flops": steps * step["flops"]}
    # and a reversed one u, its cotangent and that of the depth to the latter two
    return {"bytes": steps * (step["bytes"] + 144 * nodes),
            "flops": steps * (step["flops"] + (2 * RHS_FLOPS + 3 * VJP_FLOPS) * nodes)}


# ---- the same in plain torch, 64 bits --------------------------------------------------------
def _operators(dev):
    """Derivative matrix and the derivatives of the left and right correction
    functions (Radau, DG) at the GLL points of degree 4."""
    def legendre(n, x):
        p, q = 1.0, x
        if n == 0:
            return p, 0.0
        dp, dq = 0.0, 1.0
        for k in range(2, n + 1):
            p, q, dp, dq = q, ((2 * k - 1) * x * q - (k - 1) * p) / k, dq, \
                ((2 * k - 1) * (q + x * dq) - (k - 1) * dp) / k
        return q, dq
    w = [1.0 / math.prod(XI[j] - XI[k] for k in range(5) if k != j) for j in range(5)]
    D = [[(w[j] / w[i]) / (XI[i] - XI[j]) if i != j else 0.0 for j in range(5)] for i in range(5)]
    for i in range(5):
        D[i][i] = -sum(D[i])
    d4, d5 = [legendre(4, x)[1] for x in XI], [legendre(5, x)[1] for x in XI]
    gl = [0.5 * (a - b) for a, b in zip(d4, d5)]
    gr = [0.5 * (a + b) for a, b in zip(d4, d5)]
    return tuple(torch.tensor(v, dtype=torch.float64, device=dev) for v in (D, gl, gr))


class _Exact:
    def __init__(self, case, nx, ny, H, par, lx, ly):
        self.nx, self.ny = nx, ny
        self.sides = SIDES[case["sides"]]
        self.g, self.c, self.gamma, _ = par
        self.jx, self.jy = 0.5 * lx / nx, 0.5 * ly / ny
        self.hx, self.hy = lx / nx, ly / ny
        self.D, self.gl, self.gr = _operators(H.device)
        self.inflow = None
        if case["sides"] == "inflow":
            table, self.omega = _inflow(ny)
            self.inflow = table.reshape(ny, 5, 5, 3).to(H.device)

    def ddx(self, f):
        return sum(f[..., k:k + 1] * self.D[:, k] for k in range(5))

    def ddy(self, f):
        return sum(f[..., k:k + 1, :] * self.D[:, k, None] for k in range(5))

    def flux(self, U, Hl, n):
        h, m = U[0], U[n]
        u, v, w, p = (U[k] / h for k in range(1, 5))
        F = [m, m * u, m * v, m * w, m * (p + self.c ** 2)]
        F[n] = F[n] + 0.5 * self.g * (h * h - Hl * Hl) + h * p
        return torch.stack(F)

    def speed(self, U, n):
        return (U[n] / U[0]).abs() + torch.sqrt(
            torch.clamp(self.g * U[0] + U[4] / U[0] + self.c ** 2, min=0.0))

    def lines(self, lo, hi, axis, n, t):
        """Lower and upper states of every interface line along `axis`."""
        first, last = hi.narrow(axis, 0, 1), lo.narrow(axis, lo.shape[axis] - 1, 1)
        a, b = (0, 1) if n == 1 else (2, 3)
        if self.sides[a] == "periodic":
            return torch.cat([last, lo], axis), torch.cat([hi, first], axis)

        def mirror(W):
            return torch.stack([-W[k] if k == n else W[k] for k in range(5)])
        left = mirror(first)
        if self.sides[a] == "inflow":
            q = self.inflow
            g = q[..., 0] + math.sin(self.omega * t) * q[..., 1] + math.cos(self.omega * t) * q[..., 2]
            left = g.permute(2, 0, 1).reshape(5, self.ny, 1, 5)
        return torch.cat([left, lo], axis), torch.cat([hi, mirror(last)], axis)

    def line_depth(self, lo, hi, axis, a):
        first, last = hi.narrow(axis, 0, 1), lo.narrow(axis, lo.shape[axis] - 1, 1)
        if self.sides[a] == "periodic":
            return 0.5 * (torch.cat([last, lo], axis) + torch.cat([hi, first], axis))
        return 0.5 * (torch.cat([first, lo], axis) + torch.cat([hi, last], axis))

    def faces(self, UL, UR, Hf, n):
        """Flux jumps F* - F and depth jumps h* - h on the two sides of each line."""
        FL, FR = self.flux(UL, Hf, n), self.flux(UR, Hf, n)
        lam = torch.maximum(self.speed(UL, n), self.speed(UR, n))
        Fs = 0.5 * (FL + FR) - 0.5 * lam * (UR - UL)
        hs = 0.5 * (UL[0] + UR[0])
        return Fs - FL, Fs - FR, hs - UL[0], hs - UR[0]

    def rhs(self, U, H, t):
        g2, c2 = self.gamma, self.c ** 2
        nx, ny = self.nx, self.ny
        Hx, Hy = self.ddx(H) / self.jx, self.ddy(H) / self.jy
        # x lines: [5, ny, nx + 1, b]; y lines: [5, ny + 1, nx, a]
        UL, UR = self.lines(U[..., :, 4], U[..., :, 0], 2, 1, t)
        lo, hi, hlo, hhi = self.faces(UL, UR, self.line_depth(H[..., 4], H[..., 0], 1, 0), 1)
        Fx = (self.ddx(self.flux(U, H, 1)) + hi[:, :, :nx, :, None] * self.gl
              + lo[:, :, 1:, :, None] * self.gr) / self.jx
        hx = (self.ddx(U[0]) + hhi[:, :nx, :, None] * self.gl + hlo[:, 1:, :, None] * self.gr) / self.jx
        UL, UR = self.lines(U[..., 4, :], U[..., 0, :], 1, 2, t)
        lo, hi, hlo, hhi = self.faces(UL, UR, self.line_depth(H[..., 4, :], H[..., 0, :], 0, 2), 2)
        gl, gr = self.gl[:, None], self.gr[:, None]
        Fy = (self.ddy(self.flux(U, H, 2)) + hi[:, :ny, :, None, :] * gl
              + lo[:, 1:, :, None, :] * gr) / self.jy
        hy = (self.ddy(U[0]) + hhi[:ny, :, None, :] * gl + hlo[1:, :, None, :] * gr) / self.jy
        u, v, w, p = (U[k] / U[0] for k in range(1, 5))
        bath = self.g * (U[0] - H) + g2 * p
        S = torch.stack([torch.zeros_like(H), bath * Hx, bath * Hy, g2 * p,
                         c2 * (u * hx + v * hy) - 2.0 * c2 * (w + u * Hx + v * Hy)])
        return S - Fx - Fy

    def cfl_step(self, U, cfl):
        lam = max(float(self.speed(U, 1).max()), float(self.speed(U, 2).max()))
        return cfl * min(self.hx, self.hy) / 9.0 / lam

    def candidate(self, U, H, t, dt, k1):
        k2 = self.rhs(U + 0.5 * dt * k1, H, t + 0.5 * dt)
        k3 = self.rhs(U + 0.75 * dt * k2, H, t + 0.75 * dt)
        return U + dt * (2.0 / 9.0 * k1 + 1.0 / 3.0 * k2 + 4.0 / 9.0 * k3), k2, k3

    def adaptive(self, U, H, steps, r, t=0.0):
        """Accepted steps from t: the state, the time and (input, t, dt) of each."""
        dt, err_prev, tape = self.cfl_step(U, r["cfl"]), 1.0, []
        k1, rejected = self.rhs(U, H, t), 0
        while len(tape) < steps:
            new, k2, k3 = self.candidate(U, H, t, dt, k1)
            k4 = self.rhs(new, H, t + dt)
            e = dt * ((2.0 / 9.0 - 7.0 / 24.0) * k1 + (1.0 / 3.0 - 0.25) * k2
                      + (4.0 / 9.0 - 1.0 / 3.0) * k3 - 0.125 * k4)
            e = e / (r["atol"] + r["rtol"] * torch.maximum(U.abs(), new.abs()))
            err = max(float(torch.sqrt(e.square().mean())), 1e-300)
            fac = 0.9 * err ** (-0.7 / 3.0)
            if err <= 1.0:
                tape.append((U, t, dt))
                U, k1, t, err_prev = new, k4, t + dt, err
            else:
                rejected += 1
            dt *= min(max(fac * err_prev ** (0.4 / 3.0), 0.2), 5.0)
        return U, t, rejected, tape


def _exact_of(case, nx, ny, seed, moving):
    H, U, par, lx, ly = _fields(case, nx, ny, seed, moving, "cuda")
    return _Exact(case, nx, ny, H, par, lx, ly), H, U


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        got = []
        for nx, ny, sd in _members(case, seed):
            E, H, U = _exact_of(case, nx, ny, sd, False)
            got.append(E.adaptive(U, H, case["steps"], RUN))
        U, t = [g[0].reshape(-1) for g in got], [g[1] for g in got]
        n = [[case["steps"], g[2]] for g in got]
        if len(got) <= 16:
            return {"U": U, "steps": n, "t": t}
        return {"U": torch.cat(U), "steps": torch.tensor(n),
                "t": torch.tensor(t, dtype=torch.float64)}
    E, H, U = _exact_of(case, case["nx"], case["ny"], seed, kind in ("rhs", "vjp"))
    if kind == "rhs":
        return E.rhs(U, H, 0.3).reshape(-1)
    if kind == "vjp":
        U.requires_grad_(True)
        H.requires_grad_(True)
        W = _weights(U.numel(), seed, "cuda").view_as(U)
        gu, gh = torch.autograd.grad(E.rhs(U, H, 0.3), (U, H), W)
        return {"Ubar": gu.reshape(-1), "theta": gh.reshape(-1)}
    r = INVERSION if kind == "gradient" else RUN
    UN, t, rejected, tape = E.adaptive(U, H, case["steps"], r,
                                       TAPE_T0 if kind == "gradient" else 0.0)
    if kind == "adaptive":
        return {"U": UN.reshape(-1), "t": t, "accepted": case["steps"], "rejected": rejected}
    lam, th = torch.zeros_like(U), torch.zeros_like(H)
    gbar = nodes = None
    if case["gauges"]:
        nodes = _gauge_nodes(case, H.numel(), seed).cuda()
        gbar = _weights(case["steps"] * case["gauges"], seed, "cuda").view(case["steps"], -1)
    else:
        lam = _misfit(case, seed, "cuda").view_as(U)
    H.requires_grad_(True)
    for m in range(len(tape) - 1, -1, -1):
        u, t, dt = tape[m]
        if gbar is not None:
            lam[0].view(-1).index_add_(0, nodes, gbar[m])
            th.view(-1).index_add_(0, nodes, gbar[m], alpha=-1.0)
        u = u.detach().requires_grad_(True)
        new = E.candidate(u, H, t, dt, E.rhs(u, H, t))[0]
        lam, gh = torch.autograd.grad(new, (u, H), lam)
        lam, th = lam.clone(), th + gh
    return {"U0bar": lam.reshape(-1), "theta": th.reshape(-1), "accepted": case["steps"]}
