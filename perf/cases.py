"""The work that programs on this framework have it do, as timed cases.

Families (each listed case says what it stands for):

* ``cavity``, ``box``, ``duct`` and ``step``: SIMPLEC iterations of a
  ``SteadySolver`` followed by the report and the fields, as a program that
  monitors its run reads them. Paired and plain float state, closed and open
  domains, laminar and k-omega SST.
* ``pressure``: assembly, refresh and solve of the pressure-correction
  operator to 1e-6, with the V-cycle, the K-cycle, or FGMRES with an FP64
  dense coarse level.
* ``momentum``: three convection-diffusion systems in one batched BiCGStab.
* ``learned``: the learned coarse correction's network, forward (inference)
  and backward (loss and gradient).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import kutta_amd as ka
from kutta_amd import meshes

KCYCLE = dict(pre_sweeps=1, post_sweeps=1, coarse_sweeps=4, max_levels=5, k_min_rows=50000)
SPEED, RHO, MU = 20.0, 1.225, 1.7894e-5  # the step's air

_device = None
_plans: dict = {}


def device() -> ka.Device:
    global _device
    if _device is None:
        _device = ka.Device(0)
    return _device


def tensor(buffer: ka.Buffer) -> torch.Tensor:
    """A float32 device array as a torch tensor over the same memory."""
    class View:
        __cuda_array_interface__ = {"shape": (buffer.n,), "typestr": "<f4", "data": (buffer.ptr, False),
                                    "version": 2, "strides": None}
        owner = buffer
    return torch.as_tensor(View(), device="cuda")


# ------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # The smallest 2-D cavity a user starts with: host latency and launches.
        dict(name="cavity_32", family="cavity", nx=32, ny=32, nz=1, re=1000.0, paired=True, iterations=5),
        # The laminar lid-driven cavity benchmark, 128 x 128 at Re = 1000.
        dict(name="cavity_128", family="cavity", nx=128, ny=128, nz=1, re=1000.0, paired=True, iterations=5),
        # An open square duct in the plain float state, odd sizes.
        dict(name="duct_float_61x27x23", family="duct", nx=61, ny=27, nz=23, re=50.0, paired=False, iterations=5),
        # The 3-D lid-driven box of the finite-volume benchmark.
        dict(name="box_80", family="box", nx=80, ny=80, nz=80, re=100.0, paired=True, iterations=4),
        # k-omega SST behind a backward-facing step, walls graded to y+ = 1.
        dict(name="step_sst_8", family="step", nz=8, growth=1.15, iterations=4),
        # One pressure correction of a small tetrahedral mesh.
        dict(name="pressure_tet_10k", family="pressure", nx=12, ny=12, nz=12, method="v"),
        # The same on a ragged mid-size box.
        dict(name="pressure_tet_80k", family="pressure", nx=27, ny=23, nz=21, method="v"),
        # The pressure-operator benchmark: 998,250 perturbed tetrahedra.
        dict(name="pressure_tet_1m", family="pressure", nx=55, ny=55, nz=55, method="v"),
        # The K-cycle variant for large meshes (the operator exceeds the caches).
        dict(name="pressure_kcycle_3m", family="pressure", nx=80, ny=80, nz=80, method="k"),
        # The mixed-precision variant: FGMRES over an FP64 dense coarse level.
        dict(name="pressure_mixed_197k", family="pressure", nx=32, ny=32, nz=32, method="mixed"),
        # The three momentum components of one outer iteration, batched.
        dict(name="momentum_150k", family="momentum", nx=61, ny=47, nz=53),
        # One pass of the learned correction's network each way, on a graph of
        # the size of the second AMG level of a million-cell mesh.
        dict(name="learned_64k", family="learned", nx=40, ny=41, nz=39, layers=3),
    ]


def _size(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng) -> dict:
    family = rng.choice(["cavity", "duct", "box", "step", "v", "v", "k", "mixed", "momentum", "learned"])
    if family == "cavity":
        return dict(family="cavity", nx=_size(rng, 24, 200), ny=_size(rng, 24, 200), nz=1,
                    re=rng.choice([100.0, 400.0, 1000.0]), paired=rng.random() < 0.75, iterations=5)
    if family == "duct":
        return dict(family="duct", nx=_size(rng, 24, 90), ny=_size(rng, 10, 40), nz=_size(rng, 10, 40),
                    re=rng.choice([20.0, 50.0]), paired=rng.random() < 0.5, iterations=5)
    if family == "box":
        return dict(family="box", nx=_size(rng, 20, 80), ny=_size(rng, 20, 80), nz=_size(rng, 20, 80),
                    re=100.0, paired=rng.random() < 0.75, iterations=4)
    if family == "step":
        return dict(family="step", nz=rng.randint(1, 8), growth=rng.choice([1.15, 1.2, 1.25]), iterations=4)
    if family in ("v", "k", "mixed"):
        top = {"v": 50, "k": 60, "mixed": 36}[family]
        low = {"v": 7, "k": 26, "mixed": 14}[family]
        return dict(family="pressure", nx=_size(rng, low, top), ny=_size(rng, low, top), nz=_size(rng, low, top),
                    method=family)
    if family == "momentum":
        return dict(family="momentum", nx=_size(rng, 16, 90), ny=_size(rng, 16, 90), nz=_size(rng, 16, 90))
    return dict(family="learned", nx=_size(rng, 10, 48), ny=_size(rng, 10, 48), nz=_size(rng, 10, 48),
                layers=rng.choice([1, 2, 3, 4]))


def _key(case: dict) -> tuple:
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _plan(case: dict, make, part="plan"):
    """What a program builds once per mesh and keeps for all its solves."""
    key = (part, _key(case))
    if key not in _plans:
        _plans[key] = make()
    return _plans[key]


# ------------------------------------------------------------------ SIMPLEC
FIELDS = ("u", "v", "w", "p")
SST_FIELDS = FIELDS + ("k", "omega")
REPORTED = ("u_raw", "v_raw", "continuity_raw", "maximum_velocity", "pseudo_time_step")


def _wave(points, rng, amplitude):
    """A smooth random field of the cell centroids."""
    out = np.zeros(len(points))
    for _ in range(4):
        k, phase = rng.integers(1, 4, 3), rng.uniform(0, 2 * np.pi)
        out += np.sin(np.pi * (points @ k) + phase)
    return amplitude * out / 4


def _prepare_simplec(case, seed):
    rng = np.random.default_rng(seed)
    family = case["family"]
    if family == "step":
        first = meshes.first_cell_height(SPEED, MU / RHO, 0.5)
        mesh = _plan(case, lambda: meshes.backward_step(meshes.StepGeometry(), first=first, growth=case["growth"],
                                                        largest=0.02, nz=case["nz"]))
        turbulence = ka.IntensityViscosityRatio(0.01, 10.0)
        conditions = {"inlet": ka.VelocityInlet((SPEED, 0.0, 0.0), turbulence),
                      "outlet": ka.PressureOutlet(0.0, None, False, turbulence),
                      "wall": ka.Wall(), "symmetry": ka.Symmetry()}
        settings = ka.SolverSettings(density=RHO, viscosity=MU, monitor_interval=20)
        solver = ka.SteadySolver.from_mesh(device(), mesh, conditions, settings, ka.SstSettings())
        k = 1.5 * (0.01 * SPEED) ** 2
        x = solver.centroids()
        velocity = np.stack([SPEED * (1 + _wave(x, rng, 0.02)), SPEED * _wave(x, rng, 0.01),
                             SPEED * _wave(x, rng, 0.01)], 1)
        solver.initialize_fields(velocity, 0.0, k, RHO * k / (MU * 10.0))
        names = SST_FIELDS
    else:
        extent = (1.0, 1.0, 1.0)
        if family == "duct":
            conditions = {p: ka.Wall() for p in ka.PATCHES}
            conditions["xmin"] = ka.VelocityInlet((1.0, 0.0, 0.0))
            conditions["xmax"] = ka.PressureOutlet()
            extent = (2.0, 1.0, 1.0)
            settings = ka.SolverSettings(viscosity=1.0 / case["re"], paired_state=case["paired"])
        else:
            conditions = ka.cavity_conditions()
            settings = ka.SolverSettings(viscosity=1.0 / case["re"], momentum_relaxation=1.0,
                                         monitor_interval=100 if family == "cavity" else 20,
                                         paired_state=case["paired"])
        solver = ka.SteadySolver(device(), case["nx"], case["ny"], case["nz"], conditions, settings, extent)
        x = solver.centroids()
        velocity = np.stack([_wave(x, rng, 0.1), _wave(x, rng, 0.1),
                             _wave(x, rng, 0.1) if case["nz"] > 1 else np.zeros(len(x))], 1)
        if family == "duct":
            velocity[:, 0] += 1.0
        solver.initialize(velocity, 0.0)
        names = FIELDS
    solver.iterate(2)  # past the start: the pressure plan exists, as in a running program
    return {"solver": solver, "count": case["iterations"], "names": names}


def _run_simplec(state):
    solver = state["solver"]
    solver.iterate(state["count"])
    report = solver.report()
    return {"fields": {name: solver.field(name) for name in state["names"]},
            "report": [report[name] for name in REPORTED]}


# ----------------------------------------------------------------- pressure
def _pressure_plan(case):
    problem = ka.PressureProblem(device(), case["nx"], case["ny"], case["nz"])
    base = dict(aggregation_passes=2, structure=ka.OperatorStructure.SymmetricMMatrix)
    kind = ka.SolverKind.AmgPcg
    if case["method"] == "k":
        options = ka.AmgOptions(cycle=ka.AmgCycle.K, **KCYCLE, **base)
    else:
        options = ka.AmgOptions(**base)
    if case["method"] == "mixed":
        kind = ka.SolverKind.AmgFgmres
    solver = ka.make_amg_solver(kind, device(), problem.host, options)
    if case["method"] == "mixed":
        solver.set_direct(8192)
    solver.refresh(problem)
    solver.autotune_tail(problem)
    return {"problem": problem, "solver": solver, "x": device().alloc(problem.n_rows)}


def _pressure_rhs(problem, seed):
    b = np.random.default_rng(seed).standard_normal(problem.n_rows)
    b -= b.mean()
    b = b.astype(np.float32)
    if problem.reference >= 0:
        b[problem.reference] = 0
    return b


def _prepare_pressure(case, seed):
    plan = _plan(case, lambda: _pressure_plan(case))
    return {**plan, "b": device().upload(_pressure_rhs(plan["problem"], seed))}


def _run_pressure(state):
    problem, solver, x = state["problem"], state["solver"], state["x"]
    problem.assemble(problem.reference)
    solver.refresh(problem)
    x.fill(np.float32(0))
    solver.solve(problem, x, state["b"], ka.SolveControl(1e-6, 0.0, 2000))
    return tensor(x)


# ----------------------------------------------------------------- momentum
def _grid_links(nx, ny, nz, steps):
    """(row, column, step index) of each link of a grid along `steps`."""
    ids = np.arange(nx * ny * nz).reshape(nz, ny, nx)
    rows, cols, which = [], [], []
    for k, (dx, dy, dz) in enumerate(steps):
        a = ids[max(0, -dz):nz - max(0, dz), max(0, -dy):ny - max(0, dy), max(0, -dx):nx - max(0, dx)]
        b = ids[max(0, dz):nz - max(0, -dz), max(0, dy):ny - max(0, -dy), max(0, dx):nx - max(0, -dx)]
        rows.append(a.reshape(-1))
        cols.append(b.reshape(-1))
        which.append(np.full(a.size, k))
    return np.concatenate(rows), np.concatenate(cols), np.concatenate(which)


def _pattern(n, rows, cols):
    """CSR pattern (columns sorted) of links and a diagonal: row_ptr, columns,
    diagonal positions, and the order that sorts links-then-diagonal values."""
    r, c = np.concatenate([rows, np.arange(n)]), np.concatenate([cols, np.arange(n)])
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    row_ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    return row_ptr, c.astype(np.int32), np.nonzero(r == c)[0].astype(np.int32), order


def _float32(v):
    return v.astype(np.float32).astype(np.float64)


FACES = [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]


def _momentum_arrays(case, seed):
    """Upwind convection-diffusion systems of a velocity that varies over the
    grid, one diagonal relaxation for each component."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    rng = np.random.default_rng(seed)

    def grid():
        rows, cols, which = _grid_links(nx, ny, nz, FACES)
        return rows, np.array(FACES)[which], np.unravel_index(rows, (nz, ny, nx)), _pattern(n, rows, cols)
    rows, direction, (z, y, x), (row_ptr, col, diag, order) = _plan(case, grid, "grid")
    phase = rng.uniform(0, 2 * np.pi, 3)
    speed = np.stack([np.sin(2 * np.pi * y / ny + phase[0]), np.sin(2 * np.pi * z / nz + phase[1]),
                      np.sin(2 * np.pi * x / nx + phase[2])], 1)
    outflow = 2.0 * (speed * direction).sum(1)
    off = -(1.0 + np.maximum(-outflow, 0.0))
    systems = []
    for k in range(3):
        diagonal = np.bincount(rows, -off, n) * (1.02 + 0.05 * k) + 0.05
        systems.append((row_ptr, col, diag, _float32(np.concatenate([off, diagonal])[order]),
                        rng.standard_normal(n).astype(np.float32)))
    return systems


def _prepare_momentum(case, seed):
    systems = _momentum_arrays(case, seed)
    hosts = [ka.CsrMatrixHost(*s[:4]) for s in systems]
    plan = _plan(case, lambda: {
        "solvers": [ka.make_solver(ka.SolverKind.BicgstabJacobi, device(), h) for h in hosts],
        "xs": [device().alloc(hosts[0].n_rows) for _ in hosts]})
    return {**plan, "matrices": [ka.upload(device(), h) for h in hosts],
            "bs": [device().upload(s[4]) for s in systems]}


def _run_momentum(state):
    for solver, matrix, x in zip(state["solvers"], state["matrices"], state["xs"]):
        solver.refresh(matrix)
        x.fill(np.float32(0))
    ka.solve_batched(state["solvers"], state["matrices"], state["xs"], state["bs"], ka.SolveControl(1e-6, 0.0, 500))
    return [tensor(x) for x in state["xs"]]


# ------------------------------------------------------------------ learned
EDGES = FACES + [(1, 1, 0), (-1, -1, 0), (0, 1, 1), (0, -1, -1), (1, 0, 1), (-1, 0, -1)]


def _learned_arrays(case, seed):
    """A symmetric M-matrix on a 13-point grid graph, a residual and a target."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    rng = np.random.default_rng(seed)
    rows, cols, which = _grid_links(nx, ny, nz, EDGES)
    up = which % 2 == 0  # each link once; its reverse is the next step's
    weight = rng.uniform(0.1, 1.0, int(up.sum()))
    r, c = np.concatenate([rows[up], cols[up]]), np.concatenate([cols[up], rows[up]])
    off = -np.concatenate([weight, weight])
    row_ptr, col, diag, order = _pattern(n, r, c)
    val = _float32(np.concatenate([off, np.bincount(r, -off, n) + 0.05])[order])
    residual, target = rng.standard_normal((2, n)).astype(np.float32)
    return (row_ptr, col, diag, val), residual, 0.3 * target


def _prepare_learned(case, seed):
    arrays, residual, target = _learned_arrays(case, seed)
    net = ka.LearnedNetwork(device(), case["layers"], seed=seed % 1000)
    matrix = ka.upload(device(), ka.CsrMatrixHost(*arrays))
    net.set_graph(matrix)
    n = len(residual)
    return {"net": net, "matrix": matrix, "r": device().upload(residual), "target": device().upload(target),
            "e": device().alloc(n), "n": n}


def _run_learned(state):
    net = state["net"]
    net.infer(state["r"], state["e"])
    loss, gradient, y = net.gradient(state["r"], state["target"], state["n"])
    return {"correction": tensor(state["e"]), "loss": loss, "gradient": gradient, "y": y}


# ---------------------------------------------------------------- interface
_PREPARE = {"pressure": _prepare_pressure, "momentum": _prepare_momentum, "learned": _prepare_learned}
_RUN = {"pressure": _run_pressure, "momentum": _run_momentum, "learned": _run_learned}


def prepare(case: dict, seed: int) -> dict:
    state = _PREPARE.get(case["family"], _prepare_simplec)(case, seed)
    return {"family": case["family"], **state}


def run(state: dict):
    return _RUN.get(state["family"], _run_simplec)(state)


def _step_cells(case) -> int:
    per_layer = {1.15: 50736, 1.2: 39124, 1.25: 32856}  # cells of one spanwise layer
    return per_layer[case["growth"]] * case["nz"]


def work(case: dict) -> dict:
    """Iterative methods are priced by their own iterations: each reads its
    operator and its vectors once per iteration (a V-cycle: the hierarchy,
    1.6 times the fine level), however many launches that takes."""
    family = case["family"]
    if family == "learned":
        n = case["nx"] * case["ny"] * case["nz"]
        layers, links = case["layers"], 13
        # Per node: the graph once a direction, the features and targets, and
        # each layer's activations and their gradients kept and read once.
        return {"bytes": n * (2 * 8 * links + 40 + layers * 5 * 128),
                "flops": n * layers * (4 * 2 * 64 * 128 + 3 * 2 * 64 * links)}
    if family == "momentum":
        n = case["nx"] * case["ny"] * case["nz"]
        steps = 25  # BiCGStab steps to 1e-6, two products each
        return {"bytes": 3 * steps * n * (2 * 56 + 60), "flops": 3 * steps * n * 2 * (2 * 7 + 10)}
    if family == "pressure":
        n = 6 * case["nx"] * case["ny"] * case["nz"]
        steps = 16 if case["method"] == "k" else 20 if case["method"] == "mixed" else 1.3 * math.log2(n)
        sweeps = 4 if case["method"] == "k" else 12
        out = {"bytes": steps * 1.6 * n * (5 * 8 + 24) + n * 60, "flops": steps * 1.6 * n * sweeps * 2 * 5}
        if case["method"] == "mixed":
            m = n / 60  # rows of the dense level, inverted in FP64 at each refresh
            out["flops"] += 2 * m ** 3
            out["bytes"] += (steps + 1) * 8 * m * m
        return out
    # A SIMPLEC iteration: the state, geometry and coefficients of every cell
    # and face once, three momentum systems of about 5 BiCGStab steps and
    # about 15 pressure iterations; with SST two more equations.
    n = _step_cells(case) if family == "step" else case["nx"] * case["ny"] * case["nz"]
    per_cell = 1200 + 3 * 5 * 170 + 15 * 1.2 * (7 * 8 + 24)
    if family == "step":
        per_cell += 800 + 2 * 5 * 170
    return {"bytes": case["iterations"] * n * per_cell, "flops": case["iterations"] * n * 2000.0}


def tolerance(case: dict):
    """Measured: each case run again with its inputs off by one unit in the
    last place; four times what that changes. SIMPLEC iterations from a start
    amplify such a change to the size of the fields within a few iterations
    (limiters, automatic time step), so only the same bits say anything."""
    family = case["family"]
    if family == "learned":
        return {"rel": 1e-2}  # bfloat16 activations and weights
    if family == "pressure":
        return {"rel": 5e-6 if case["method"] == "mixed" else 2e-6, "max": 2e-5}
    if family == "momentum":
        return {"rel": 2e-5, "max": 2e-4}
    return "exact"


def _sparse64(n, row_ptr, col, val):
    return torch.sparse_csr_tensor(torch.as_tensor(np.asarray(row_ptr, np.int64)).cuda(),
                                   torch.as_tensor(np.asarray(col, np.int64)).cuda(),
                                   torch.as_tensor(np.asarray(val, np.float64)).cuda(), size=(n, n))


def _cg64(a, diagonal, b, steps=8000):
    x, r = torch.zeros_like(b), b.clone()
    z = r / diagonal
    p, rho, stop = z.clone(), torch.dot(r, z), 1e-11 * float(b.norm())
    for k in range(steps):
        q = a @ p
        alpha = rho / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        if k % 50 == 0 and float(r.norm()) <= stop:
            break
        z = r / diagonal
        rho, last = torch.dot(r, z), rho
        p = z + (rho / last) * p
    return x


def _bicgstab64(a, diagonal, b, steps=2000):
    x, r = torch.zeros_like(b), b.clone()
    shadow, p, stop = r.clone(), r.clone(), 1e-11 * float(b.norm())
    rho = torch.dot(shadow, r)
    for k in range(steps):
        ph = p / diagonal
        v = a @ ph
        alpha = rho / torch.dot(shadow, v)
        s = r - alpha * v
        sh = s / diagonal
        t = a @ sh
        omega = torch.dot(t, s) / torch.dot(t, t)
        x += alpha * ph + omega * sh
        r = s - omega * t
        if float(r.norm()) <= stop:
            break
        rho, last = torch.dot(shadow, r), rho
        p = r + (rho / last) * (alpha / omega) * (p - omega * v)
    return x


def _learned64(case, seed):
    """The network, its loss and its gradient in FP64 by autograd."""
    (row_ptr, col, diag, val), residual, target = _learned_arrays(case, seed)
    n, layers = len(residual), case["layers"]
    theta_host = ka.LearnedNetwork(device(), layers, seed=seed % 1000).parameters()  # an input: the initial weights
    as64 = lambda v: torch.as_tensor(np.asarray(v, np.float64)).cuda()  # noqa: E731
    rows = torch.as_tensor(np.repeat(np.arange(n), np.diff(row_ptr))).cuda()
    cols = torch.as_tensor(np.asarray(col, np.int64)).cuda()
    v, d = as64(val), as64(val[diag])
    weight = torch.where(rows == cols, torch.zeros_like(v), v.abs() / d[rows])
    l1 = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(
        0, rows, torch.where(rows == cols, torch.zeros_like(v), v.abs()))
    r, t, mean = as64(residual), as64(target), d.mean()
    rms = (r * r).mean().sqrt()
    scale = rms / mean
    theta = as64(theta_host).requires_grad_(True)
    x = torch.stack([r / rms, d / mean, l1 / mean, torch.ones_like(r)], 1)
    h = torch.relu(x @ theta[:256].reshape(4, 64) + theta[256:320])
    at = 320
    for _ in range(layers):
        own, near = theta[at:at + 4096].reshape(64, 64), theta[at + 4096:at + 8192].reshape(64, 64)
        m = torch.zeros_like(h).index_add(0, rows, weight[:, None] * h[cols])
        h = torch.relu(h @ own + m @ near + theta[at + 8192:at + 8256])
        at += 8256
    y = h @ theta[at:at + 64] + theta[at + 64]
    loss = ((y - t / scale) ** 2).mean()
    loss.backward()
    return {"correction": (y * scale).detach(), "loss": float(loss), "gradient": theta.grad, "y": y.detach()}


def exact(case: dict, seed: int):
    """In 64 bits by plain torch; None for whole SIMPLEC iterations."""
    family = case["family"]
    if family == "learned":
        return _learned64(case, seed)
    if family == "momentum":
        out = []
        for row_ptr, col, diag, val, b in _momentum_arrays(case, seed):
            a = _sparse64(len(b), row_ptr, col, val)
            out.append(_bicgstab64(a, torch.as_tensor(val[diag]).cuda(), torch.as_tensor(b.astype(np.float64)).cuda()))
        return out
    if family == "pressure":
        problem = _plan(case, lambda: _pressure_plan(case))["problem"]  # for its operator, an input of the solve
        val = problem["values"].astype(np.float64)
        a = _sparse64(problem.n_rows, problem["row_ptr"], problem["col"], val)
        b = torch.as_tensor(_pressure_rhs(problem, seed).astype(np.float64)).cuda()
        return _cg64(a, torch.as_tensor(val[problem["diag"]]).cuda(), b)
    return None
