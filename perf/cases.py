"""The work a user of this package has it do, as a set of timed cases.

Each case is one call pattern on the public API (Simulator, simulate_to_time,
advance_steps, Ensemble, Server, adjoint_gradient) at a size and with options
that the package's own workloads, tests and benchmark use, or ragged sizes
between them.  listed() names the cases, draw() makes more of the same ranges,
prepare() builds what a program holds before the call, run() is the call, and
exact() is the same scheme in 64-bit torch operations without this package's
kernels.

Kinds:
  callback   simulate_to_time with a callback: the host steps the grid one
             perform_step at a time and reads the state at output times.
  scenario   set_current_state, simulate_to_time to an end time, read the
             state: one whole (short) run, 1D or 2D.
  advance    advance_steps by a fixed count and read the state: a long run
             between two outputs, the state kept on the device.
  ensemble   Ensemble.advance_steps over members of uneven size, then every
             member's state.
  serving    requests submitted together to a Server, waited for and fetched.
  adjoint    adjoint_gradient of a run: objective and all gradients.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "volumefluxes.jl_amd"))

import volumefluxes as VF  # noqa: E402

G = 9.81
RHO = 1.0
THETA = 1.2
MANNING = 0.03
RAIN = 0.036            # m/h, as ConstantRain takes it (1e-5 m/s)
INFILTRATION = 15 / 1000.0 / 3600
HORTON = (1.977e-4, 3.272e-5, 2.43e-3)      # f0, fc, k
CFL = 0.25


def _grid_case(name, kind, nx, ny, **more):
    case = {"name": name, "kind": kind, "nx": nx, "ny": ny, "dx": 1.0, "dy": 1.0, "dtype": "f64", "stepper": "rk2",
            "bc": "wall", "rec": "linear", "rain": True, "infiltration": "none", "friction": True,
            "cutoff": 1e-5, "kappa": 1e-4}
    case.update(more)
    return case


def listed():
    return [
        # The smallest call: a small grid driven step by step from the host, as
        # any run with an output callback is; latency and launches count.
        _grid_case("callback_64x48", "callback", 64, 48, max_dt=0.02, span=0.39),
        # The 1D Stoker dam break of the tests and the benchmark: 1024 cells to
        # t = 20 s, device-resident, hundreds of very small steps.
        _grid_case("stoker_1d_1024", "scenario", 1024, 0, dx=1000.0 / 1024, rain=False, friction=False, span=20.0,
                   cutoff=1e-5, kappa=1e-5),
        # The bay example's configuration: ForwardEuler, NeumannBC, Horton
        # infiltration, rain and friction on 107 x 145 cells whose spacing is
        # no power of two, flooded from one side.
        _grid_case("bay_107x145_euler", "scenario", 107, 145, dx=451.0 / 107, dy=601.0 / 145, stepper="euler",
                   bc="neumann", infiltration="horton", cutoff=8e-2, kappa=1e-5, span=12.0),
        # A mid-size survey grid with a spacing that is no power of two and a
        # constant infiltration: RungeKutta2, walls.
        _grid_case("survey_333x221", "scenario", 333, 221, dx=1.7, dy=1.3, infiltration="constant", span=6.0),
        # A mid-size terrain run between two outputs: too small to fill the GPU.
        _grid_case("terrain_512", "advance", 512, 512, steps=300),
        # Float32 storage at a ragged size around a million cells.
        _grid_case("terrain_1100x900_f32", "advance", 1100, 900, dtype="f32", steps=300),
        # ForwardEuler on a large periodic grid, non-square.
        _grid_case("terrain_1500x1000_euler", "advance", 1500, 1000, stepper="euler", bc="periodic", steps=300),
        # The benchmark's grid and options: 2048^2, Float64, RungeKutta2.
        _grid_case("terrain_2048", "advance", 2048, 2048, steps=300),
        # Large survey grid, spacing no power of two, constant infiltration.
        _grid_case("survey_1777x1409", "advance", 1777, 1409, dx=2.5, dy=2.5, infiltration="constant", steps=200),
        # The ensemble workload in small: members of uneven, non-square sizes.
        {"name": "ensemble_16", "kind": "ensemble", "members": 16, "steps": 200, "low": 128, "high": 1024},
        # Flood scenarios submitted together: dam breaks and terrains.
        {"name": "serving_16", "kind": "serving", "requests": 16, "low": 64, "high": 512, "span": 2.0},
        # Gradient of a run with respect to bottom, friction and initial state,
        # the benchmark's grid size and checkpoint spacing.
        _grid_case("adjoint_512", "adjoint", 512, 512, steps=100, every=20),
    ]


def _log_size(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["callback", "scenario", "scenario", "advance", "advance", "advance", "ensemble", "serving",
                       "adjoint", "adjoint"])
    options = {"dtype": rng.choice(["f64", "f64", "f32"]), "stepper": rng.choice(["rk2", "rk2", "euler"]),
               "bc": rng.choice(["wall", "wall", "periodic", "neumann"]),
               "rec": rng.choice(["linear", "linear", "linear", "none"]), "rain": rng.random() < 0.7,
               "friction": rng.random() < 0.8, "infiltration": rng.choice(["none", "none", "constant"])}
    if rng.random() < 0.5:
        options["dx"] = round(rng.uniform(0.5, 4.0), 2)
        options["dy"] = round(rng.uniform(0.5, 4.0), 2)
    name = "drawn"
    if kind == "callback":
        case = _grid_case(name, kind, _log_size(rng, 32, 160), _log_size(rng, 32, 160), **options)
        case["max_dt"] = 0.01 * min(case["dx"], case["dy"])
        case["span"] = case["max_dt"] * (rng.randint(10, 30) - 0.5)
    elif kind == "scenario":
        if rng.random() < 0.3:
            nx = _log_size(rng, 200, 4000)
            case = _grid_case(name, kind, nx, 0, dx=1000.0 / nx, rain=False, friction=False, kappa=1e-5)
            case["span"] = 48.0 * rng.uniform(50, 400) / nx
        else:
            case = _grid_case(name, kind, _log_size(rng, 64, 400), _log_size(rng, 64, 400), **options)
            case["span"] = 0.03 * min(case["dx"], case["dy"]) * rng.uniform(50, 200)
    elif kind == "advance":
        nx, ny = _log_size(rng, 256, 2300), _log_size(rng, 256, 2300)
        case = _grid_case(name, kind, nx, ny, **options)
        case["steps"] = max(50, min(300, int(8e8 / (nx * ny))))
    elif kind == "ensemble":
        case = {"name": name, "kind": kind, "members": rng.randint(4, 16), "steps": rng.choice([64, 120, 200]),
                "low": 128, "high": rng.choice([256, 512, 1024])}
    elif kind == "serving":
        case = {"name": name, "kind": kind, "requests": rng.randint(4, 16), "low": 64,
                "high": rng.choice([128, 256, 512]), "span": round(rng.uniform(0.5, 2.0), 2)}
    else:
        nx, ny = _log_size(rng, 64, 512), _log_size(rng, 64, 512)
        for k in ("dtype", "stepper", "bc", "rec", "infiltration"):
            options.pop(k)
        case = _grid_case(name, kind, nx, ny, **options)
        case["bc"] = rng.choice(["wall", "wall", "periodic"])
        case["steps"] = rng.randint(20, 100)
        case["every"] = rng.choice([10, 20, 25])
    del case["name"]
    return case


# ------------------------------------------------------------------ inputs

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _bottom_and_state(case, seed):
    """Corner bottom (nxT+1, nyT+1) and interior state (nx, ny, 3) as Float64
    numpy arrays, x fastest: a slope with 32 seeded bumps scaled to the
    domain, water to a level that leaves about a third of the cells dry, and
    a raised surface on one side that sets it in motion."""
    rng = np.random.default_rng(seed)
    nx, ny, dx, dy = case["nx"], case["ny"], case["dx"], case["dy"]
    if ny == 0:                                        # 1D dam break on a flat bottom
        U = np.zeros((nx, 2))
        left = 0.005 * (1.0 + 0.2 * rng.random()) * 400
        U[:, 0] = np.where((np.arange(nx) + 0.5) < nx * (0.45 + 0.1 * rng.random()), left, 0.2 * left)
        return None, U
    low = max(2.0, min(nx * dx, ny * dy) / 40)
    high = max(low, max(nx * dx, ny * dy) / 8)
    amp, width = rng.uniform(0.5, 5.0, 32), rng.uniform(low, high, 32)
    cx, cy = rng.uniform(0, nx * dx, 32), rng.uniform(0, ny * dy, 32)
    dev = _device()
    x = (torch.arange(nx + 5, dtype=torch.float64, device=dev) - 2) * dx
    y = (torch.arange(ny + 5, dtype=torch.float64, device=dev) - 2) * dy
    B = (1e-3 * x)[None, :].repeat(ny + 5, 1)
    for a, w, px, py in zip(amp, width, cx, cy):
        B += a * torch.exp(-((y - py) ** 2) / (2 * w * w))[:, None] * torch.exp(-((x - px) ** 2) / (2 * w * w))[None, :]
    Bc = 0.25 * (((B[:-1, :-1] + B[:-1, 1:]) + B[1:, :-1]) + B[1:, 1:])[2:-2, 2:-2]
    level = float(torch.sort(Bc.reshape(-1)).values[int(0.65 * nx * ny)])
    px, py, s = nx * dx * rng.uniform(0.2, 0.8), ny * dy * rng.uniform(0.2, 0.8), 0.15 * max(nx * dx, ny * dy)
    xc, yc = x[2:2 + nx] + dx / 2, y[2:2 + ny] + dy / 2
    swell = 0.5 * torch.exp(-((yc - py) ** 2) / (2 * s * s))[:, None] * torch.exp(-((xc - px) ** 2) / (2 * s * s))[None, :]
    w = torch.maximum(Bc, level + swell)
    U = torch.zeros((3, ny, nx), dtype=torch.float64, device=dev)
    U[0] = w
    return B.cpu().numpy().T, U.cpu().numpy().T


_BC = {"wall": VF.WallBC, "periodic": VF.PeriodicBC, "neumann": VF.NeumannBC}


def _simulator(case, B):
    nx, ny = case["nx"], case["ny"]
    bc = _BC[case["bc"]]()
    backend = VF.make_hip_backend(np.float64 if case["dtype"] == "f64" else np.float32)
    more = dict(depth_cutoff=case["cutoff"], desingularizing_kappa=case["kappa"])
    rec = VF.LinearReconstruction() if case["rec"] == "linear" else VF.NoReconstruction()
    stepper = VF.RungeKutta2() if case["stepper"] == "rk2" else VF.ForwardEulerStepper()
    if ny == 0:
        grid = VF.CartesianGrid(nx, gc=2, boundary=bc, extent=[[0.0, nx * case["dx"]]])
        eq = VF.ShallowWaterEquations1D(**more)
        system = VF.ConservedSystem(backend, rec, VF.CentralUpwind(eq), eq, grid, [])
        return VF.Simulator(backend, system, stepper, grid, cfl=CFL)
    grid = VF.CartesianGrid(nx, ny, gc=2, boundary=bc, extent=[[0.0, nx * case["dx"]], [0.0, ny * case["dy"]]])
    eq = VF.ShallowWaterEquations(VF.BottomTopography2D(B, backend, grid), **more)
    sources = [VF.SourceTermBottom()]
    if case["infiltration"] == "horton":
        sources.append(VF.HortonInfiltration(grid))
    elif case["infiltration"] == "constant":
        sources.append(VF.ConstantInfiltration(INFILTRATION))
    if case["rain"]:
        sources.append(VF.ConstantRain(RAIN))
    friction = VF.ImplicitFriction(Cz=MANNING ** 2) if case["friction"] else None
    system = VF.ConservedSystem(backend, rec, VF.CentralUpwind(eq), eq, grid, sources, friction)
    return VF.Simulator(backend, system, stepper, grid, cfl=CFL)


def _members(case, seed):
    """The sizes and scenarios of an ensemble's members."""
    rng = np.random.default_rng(seed + 17)
    sides = [s for s in (128, 256, 512, 768, 1024) if case["low"] <= s <= case["high"]]
    sizes = np.random.default_rng(case["members"] * 7 + case["high"])       # the same work for every seed
    for _ in range(case["members"]):
        nx, ny = int(sizes.choice(sides)), int(sizes.choice(sides))
        yield _grid_case("member", "advance", nx, ny, steps=case["steps"]), int(rng.integers(1 << 30))


def _requests(case, seed):
    """The requests of a serving case: square grids of ragged sides, half of
    them dam breaks on a flat bottom (no rain), half terrains."""
    rng = np.random.default_rng(seed + 29)
    sizes = np.random.default_rng(case["requests"] * 11 + case["high"])
    for k in range(case["requests"]):
        n = int(round(math.exp(sizes.uniform(math.log(case["low"]), math.log(case["high"])))))
        flat = k % 2 == 0
        yield (_grid_case("request", "scenario", n, n, rain=not flat, span=case["span"] * sizes.uniform(0.5, 1.0)),
               int(rng.integers(1 << 30)), flat)


def _request_inputs(case, seed, flat):
    B, U = _bottom_and_state(case, seed)
    if flat:
        B = np.zeros_like(B)
        U = np.zeros_like(U)
        U[:, :, 0] = np.where((np.arange(case["nx"]) + 0.5)[:, None] < 0.5 * case["nx"], 2.0, 1.0 + (seed % 97) / 200)
    return B, U


def _target(case, seed, B, U):
    """The depth an adjoint's objective compares with: the initial depth with
    a smooth seeded change."""
    rng = np.random.default_rng(seed + 3)
    nx, ny = case["nx"], case["ny"]
    Bc = (0.25 * (((B[:-1, :-1] + B[1:, :-1]) + B[:-1, 1:]) + B[1:, 1:]))[2:-2, 2:-2]
    kx, ky, p = rng.uniform(1, 4), rng.uniform(1, 4), rng.uniform(0, 6)
    wave = np.sin(kx * np.arange(nx) / nx + p)[:, None] * np.cos(ky * np.arange(ny) / ny)[None, :]
    return np.asfortranarray((U[:, :, 0] - Bc) * (1.0 + 0.1 * wave))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        sims = []
        for member, s in _members(case, seed):
            B, U = _bottom_and_state(member, s)
            sim = _simulator(member, B)
            VF.set_current_state(sim, U)
            sims.append(sim)
        return {"case": case, "sims": sims, "ensemble": VF.Ensemble(sims)}
    if kind == "serving":
        todo = []
        for request, s, flat in _requests(case, seed):
            B, U = _request_inputs(request, s, flat)
            sim = _simulator(request, B)
            todo.append((sim.system, sim.grid, np.asfortranarray(U), request["span"]))
            del sim
        return {"case": case, "server": VF.Server(16 << 30), "todo": todo}
    B, U = _bottom_and_state(case, seed)
    sim = _simulator(case, B)
    VF.set_current_state(sim, U)
    state = {"case": case, "sim": sim, "U": U}
    if kind == "adjoint":
        state["target"] = _target(case, seed, B, U)
    return state


# --------------------------------------------------------------------- run

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "ensemble":
        state["ensemble"].advance_steps(case["steps"])
        return [VF.current_state(sim) for sim in state["sims"]]
    if kind == "serving":
        server = state["server"]
        ids = [server.submit(system, grid, U, span) for system, grid, U, span in state["todo"]]
        for i in ids:
            server.wait(i)
        return [server.fetch(i)[0] for i in ids]
    sim = state["sim"]
    if kind == "advance":
        VF.advance_steps(sim, case["steps"])
        return VF.current_state(sim)
    VF.set_current_state(sim, state["U"])              # the other kinds are whole runs from the initial state
    sim.t = 0.0
    if kind == "adjoint":
        return VF.adjoint_gradient(sim, case["steps"], state["target"], checkpoint_every=case["every"])
    if kind == "callback":
        heights = []
        writer = VF.IntervalWriter(case["span"] / 4, lambda t, s: heights.append(VF.current_interior_state(s).h))
        VF.simulate_to_time(sim, case["span"], callback=writer, maximum_timestep=case["max_dt"])
        return {"heights": heights, "state": VF.current_state(sim), "dt": sim.current_timestep}
    VF.simulate_to_time(sim, case["span"])
    return VF.current_state(sim)


# -------------------------------------------------------------------- work

def _steps(case):
    """Steps of one pass: given, or the end time over the CFL step of the wave
    speeds these inputs reach (about 5 m/s in 1D, 6 m/s in 2D)."""
    if case["kind"] in ("advance", "adjoint"):
        return case["steps"]
    if case["kind"] == "callback":
        return case["span"] / case["max_dt"]
    d = case["dx"] if case["ny"] == 0 else min(case["dx"], case["dy"])
    return case["span"] * (5.0 if case["ny"] == 0 else 6.0) / (CFL * d)


def _grid_work(case):
    """A step reads the state and the bottom once per stage and writes the
    state once per stage (136 bytes per cell with RK2 in Float64, the stage's
    right-hand side among it); about 400 floating operations per cell and
    stage.  The reverse pass of an adjoint reads both stages' states and
    right-hand sides and reads and writes the adjoint once per stage."""
    cells = case["nx"] * max(1, case["ny"])
    es = 8 if case["dtype"] == "f64" else 4
    stages = 2 if case["stepper"] == "rk2" else 1
    per = 8 * stages + es * (15 if stages == 2 else 6)
    flops = 400 * stages
    if case["kind"] == "adjoint":
        per += 8 * stages + es * 24
        flops += 1000 * stages
    steps = _steps(case)
    return per * cells * steps, flops * cells * steps


def work(case):
    if case["kind"] == "ensemble":
        parts = [_grid_work(m) for m, _ in _members(case, 0)]
    elif case["kind"] == "serving":
        parts = [_grid_work(m) for m, _, _ in _requests(case, 0)]
    else:
        parts = [_grid_work(case)]
    return {"bytes": float(sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


# ------------------------------------------------------------------- exact

def _max(x, y):
    return torch.where(x > y, x, y)


def _min(x, y):
    return torch.where(x < y, x, y)


class _Scheme:
    """The scheme on (3, nyT, nxT) Float64 tensors, out of place, so that it
    can be differentiated."""

    def __init__(self, case, B, Cz=MANNING ** 2):
        self.c = case
        self.one_d = case["ny"] == 0
        self.B = B                                     # (nyT+1, nxT+1); None: zero
        self.Cz = Cz if case["friction"] else None
        if B is None:
            self.Bc = 0.0
        else:
            self.Bc = 0.25 * (((B[:-1, :-1] + B[:-1, 1:]) + B[1:, :-1]) + B[1:, 1:])

    def desingularize(self, h):
        k = self.c["kappa"]
        a = torch.abs(h)
        thin = _max(a, _min(h * h / (2 * k) + k / 2.0, torch.full_like(h, k)))
        return torch.where(a >= k, h, torch.where(h < 0, -thin, thin))

    def side(self, d, s):
        wet = s[0] > self.c["cutoff"]
        h = torch.where(wet, s[0], torch.ones_like(s[0]))
        hs = self.desingularize(h)
        u, v = s[1] / hs, s[2] / hs
        c = torch.sqrt(G * h)
        n = u if d == 0 else v
        p = 0.5 * RHO * G * (h * h)
        if d == 0:
            f = [RHO * h * u, RHO * h * u * u + p, RHO * h * u * v]
        else:
            f = [RHO * h * v, RHO * h * u * v, RHO * h * v * v + p]
        zero = torch.zeros_like(h)
        f = torch.stack([torch.where(wet, x, zero) for x in f])
        return f, torch.where(wet, n + c, zero), torch.where(wet, n - c, zero)

    def faces(self, d, m, q):
        fm, em, lm = self.side(d, m)
        fp, ep, lp = self.side(d, q)
        zero = torch.zeros_like(em)
        ap, am = _max(_max(ep, em), zero), _min(_min(lp, lm), zero)
        da = ap - am
        still = torch.abs(da) < self.c["kappa"]
        da = torch.where(still, torch.ones_like(da), da)
        F = (ap * fm - am * fp) / da + (ap * am) / da * (q - m)
        F = torch.where(still, torch.zeros_like(F), F)
        dry = still | ((m[0] < self.c["cutoff"]) & (q[0] < self.c["cutoff"]))
        return F, torch.where(dry, zero, _max(torch.abs(ap), torch.abs(am)))

    def direction(self, d, U):
        """Flux difference, bottom term and largest speed of one direction, on
        the interior."""
        c = self.c
        if d == 1:
            U = U.transpose(1, 2)
        B = None if self.B is None else (self.B if d == 0 else self.B.transpose(0, 1))
        U = U[:, 2:-2, :] if not self.one_d else U
        if B is None:
            bl = br = torch.zeros_like(U[0])
        else:
            f = 0.5 * (B[2:-3, :] + B[3:-2, :])
            bl, br = f[:, :-1], f[:, 1:]
        if c["rec"] == "linear":
            mid, left, right = U[:, :, 1:-1], U[:, :, :-2], U[:, :, 2:]
            fwd, bwd = right - mid, mid - left
            a, b, e = THETA * fwd, (fwd + bwd) / 2.0, THETA * bwd
            low, high = _min(_min(a, b), e), _max(_max(a, b), e)
            zero = torch.zeros_like(a)
            s = torch.where((a > 0) & (b > 0) & (e > 0), low, torch.where((a < 0) & (b < 0) & (e < 0), high, zero))
            w, bl, br = mid[0], bl[:, 1:-1], br[:, 1:-1]
            s0 = torch.where(w - 0.5 * s[0] < bl, 2.0 * (w - bl), torch.where(w + 0.5 * s[0] < br, 2.0 * (br - w), s[0]))
            s = torch.cat([s0[None], s[1:]])
            L, R = mid - 0.5 * s, mid + 0.5 * s
            L = torch.cat([(L[0] - bl)[None], L[1:]])
            R = torch.cat([(R[0] - br)[None], R[1:]])
        else:
            mid = U[:, :, 1:-1]
            if B is None:
                h = mid[0]
            else:
                Bc = self.Bc if d == 0 else self.Bc.transpose(0, 1)
                h = mid[0] - Bc[2:-2, 1:-1]
            bl, br = bl[:, 1:-1], br[:, 1:-1]
            L = R = torch.cat([h[None], mid[1:]])
        F, speed = self.faces(d, R[:, :, :-1], L[:, :, 1:])
        delta = c["dx"] if d == 0 else c["dy"]
        inv = 1.0 / delta
        change = -(inv * (F[:, :, 1:] - F[:, :, :-1]))
        bottom = -G * ((br - bl) / delta)[:, 1:-1] * ((R[0] + L[0])[:, 1:-1] / 2.0)
        fastest = speed.reshape(-1)[torch.argmax(speed.detach())]
        if d == 1:
            change, bottom = change.transpose(1, 2), bottom.transpose(0, 1)
        return change, bottom, fastest

    def rhs(self, U, t):
        c = self.c
        x, bx, ax = self.direction(0, U)
        if self.one_d:
            inner, ay = x, None
        else:
            y, by, ay = self.direction(1, U)
            if self.B is None:
                inner = x + y
            else:
                inner = torch.stack([x[0] + y[0], (x[1] + bx) + y[1], (x[2] + y[2]) + by])
        R = torch.nn.functional.pad(inner, (2, 2, 0, 0) if self.one_d else (2, 2, 2, 2))
        w = R[0]
        if c["infiltration"] == "horton":
            w = w - (HORTON[1] + (HORTON[0] - HORTON[1]) * math.exp(-HORTON[2] * t))
        elif c["infiltration"] == "constant":
            w = w - INFILTRATION
        if c["rain"]:
            w = w + RAIN / 3600
        return torch.cat([w[None], R[1:]]), ax, ay

    def finish(self, X, o, dt):
        """Implicit friction from X, the dry clamp and the boundary condition."""
        c = self.c
        if self.Cz is not None:
            hs = self.desingularize(X[0] - self.Bc)
            u, v = X[1] / hs, X[2] / hs
            q = u * u + v * v
            moving = q > 0
            speed = torch.where(moving, torch.sqrt(torch.where(moving, q, torch.ones_like(q))), torch.zeros_like(q))
            D = 1 - dt * (-self.Cz * speed / (hs * hs))
            o = torch.stack([o[0], o[1] / D, o[2] / D])
        Bc = self.Bc + torch.zeros_like(o[0])
        dry = o[0] - Bc < c["cutoff"]
        zero = torch.zeros_like(o[0])
        o = torch.stack([torch.where(dry, _max(o[0], Bc), o[0]), torch.where(dry, zero, o[1]),
                         torch.where(dry, zero, o[2])])
        return self.boundary(o)

    def boundary(self, U):
        U = self.lines(U, 2, 1)
        return U if self.one_d else self.lines(U.transpose(1, 2), 2, 2).transpose(1, 2)

    def lines(self, U, gc, normal):
        inner = slice(0, 1) if self.one_d else slice(gc, -gc)
        N = U.shape[2]
        cols = [U[:, inner, i] for i in range(gc)], [U[:, inner, N - gc + g] for g in range(gc)]
        flip = torch.ones((3, 1), dtype=U.dtype, device=U.device)
        if self.c["bc"] == "wall":
            flip[normal] = -1.0

        def at(i):
            return cols[0][i] if i < gc else cols[1][i - (N - gc)] if i >= N - gc else U[:, inner, i]

        for g in range(1, gc + 1):
            if self.c["bc"] == "wall":
                pairs = (g - 1, 2 * gc - g), (N - gc + g - 1, N - gc - g)
            elif self.c["bc"] == "periodic":
                pairs = (g - 1, N + g - 2 * gc - 1), (N - (gc - g) - 1, gc + g - 1)
            else:
                pairs = (g - 1, 2 * gc - g), (N - (gc - g) - 1, N - g)
            for to, of in pairs:
                v = at(of) * flip
                if to < gc:
                    cols[0][to] = v
                else:
                    cols[1][to - (N - gc)] = v
        V = U.clone()
        for g in range(gc):
            V[:, inner, g] = cols[0][g]
            V[:, inner, N - gc + g] = cols[1][g]
        return V

    def step(self, U, t, limit):
        R, ax, ay = self.rhs(U, t)
        dt = self.c["dx"] / ax
        if ay is not None:
            dy = self.c["dy"] / ay
            dt = torch.where(dt < dy, dt, dy)
        dt = CFL * dt
        if limit < float(dt.detach()):
            dt = torch.full_like(dt, limit)
        U1 = self.finish(U, U + dt * R, dt)
        if self.c["stepper"] != "rk2":
            return U1, dt
        R, _, _ = self.rhs(U1, t)
        return self.finish(U1, 0.5 * (U + (U1 + dt * R)), dt), dt


def _start(case, B, U, dev):
    """The scheme and the full initial state, ghost cells filled."""
    u = torch.from_numpy(np.ascontiguousarray(U.T)).to(dev)
    if case["ny"] == 0:
        full = torch.zeros((3, 1, case["nx"] + 4), dtype=torch.float64, device=dev)
        full[:2, 0, 2:-2] = u
        b = None
    else:
        full = torch.zeros((3, case["ny"] + 4, case["nx"] + 4), dtype=torch.float64, device=dev)
        full[:, 2:-2, 2:-2] = u
        b = torch.from_numpy(np.ascontiguousarray(B.T)).to(dev)
    return full, b


def _as_state(case, U):
    if case["ny"] == 0:
        return U[:2, 0, :].transpose(0, 1)
    return U.permute(2, 1, 0)


def _exact_run(case, B, U0, dev, writer=None):
    U, b = _start(case, B, U0, dev)
    scheme = _Scheme(case, b)
    U = scheme.boundary(U)
    if case["kind"] == "advance":
        for k in range(case["steps"]):
            U, dt = scheme.step(U, 0.0, math.inf)
        return U, dt
    t, dt = 0.0, None
    while t < case["span"]:
        U, dt = scheme.step(U, t, min(case["span"] - t, case.get("max_dt", math.inf)))
        t += float(dt)
        if writer is not None:
            writer(t, float(dt), U)
    return U, dt


#: Cell-steps that the tensor operations take in about ten seconds.
MOST_CELL_STEPS = 3e8


def exact(case, seed):
    dev = _device()
    cells = sum(m["nx"] * max(1, m["ny"]) * _steps(m) for m in
                ([m for m, _ in _members(case, seed)] if case["kind"] == "ensemble" else
                 [m for m, _, _ in _requests(case, seed)] if case["kind"] == "serving" else [case]))
    if case["kind"] == "adjoint":
        cells *= 8
    if cells > MOST_CELL_STEPS:
        return None
    if case["kind"] != "adjoint":
        with torch.no_grad():
            return _exact_forward(case, seed, dev)
    from torch.utils.checkpoint import checkpoint
    B, U0 = _bottom_and_state(case, seed)
    full, b = _start(case, B, U0, dev)
    target = torch.from_numpy(np.ascontiguousarray(_target(case, seed, B, U0).T)).to(dev)
    u0 = full[:, 2:-2, 2:-2].clone().requires_grad_(True)
    b.requires_grad_(True)
    Cz = torch.tensor(MANNING ** 2, dtype=torch.float64, device=dev, requires_grad=True)

    def begin(u):
        return _Scheme(case, b, Cz).boundary(torch.nn.functional.pad(u, (2, 2, 2, 2)))

    def step(U, bb, cz):
        return _Scheme(case, bb, cz).step(U, 0.0, math.inf)[0]

    U = begin(u0)
    for _ in range(case["steps"]):
        U = checkpoint(step, U, b, Cz, use_reentrant=False)
    Bc = 0.25 * (((b[:-1, :-1] + b[:-1, 1:]) + b[1:, :-1]) + b[1:, 1:])
    J = (((U[0] - Bc)[2:-2, 2:-2] - target) ** 2).sum()
    J.backward()
    dCz = float(Cz.grad) if Cz.grad is not None else 0.0
    return {"J": float(J.detach()), "dJ_dB": b.grad.transpose(0, 1), "dJ_dCz": dCz,
            "dJ_dU0": u0.grad.permute(2, 1, 0)}


def _exact_forward(case, seed, dev):
    if case["kind"] == "ensemble":
        return [_as_state(m, _exact_run(m, *_bottom_and_state(m, s), dev)[0]) for m, s in _members(case, seed)]
    if case["kind"] == "serving":
        return [_as_state(m, _exact_run(m, *_request_inputs(m, s, flat), dev)[0])[2:-2, 2:-2]
                for m, s, flat in _requests(case, seed)]
    heights, due = [], [0.0]

    def writer(t, dt, U):
        if t + dt >= due[0]:
            heights.append(U[0, 2:-2, 2:-2].transpose(0, 1).clone())
            due[0] += case["span"] / 4

    U, dt = _exact_run(case, *_bottom_and_state(case, seed), dev, writer if case["kind"] == "callback" else None)
    if case["kind"] == "callback":
        return {"heights": heights, "state": _as_state(case, U), "dt": float(dt)}
    return _as_state(case, U)
