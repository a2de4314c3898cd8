"""The work a user of this library has it do, as cases that can be timed and
checked: one traversal on device tensors, time loops on the device and from
the host, remeshing every step, ensembles, and gradients.

listed() names the cases, draw() gives more of the same ranges, prepare()
makes what a program holds before the call (inputs, meshes, handles), run() is
one pass through the public entry points, work() the bytes and operations a
pass cannot do without, and exact() the same outputs from plain PyTorch in 64
bits.

Scenes (the inputs of a mesh's cells, made from the seed):
  tsunami  the 1000 km square of the tsunami scenario: rough bathymetry with a
           coastal shelf, an elliptical source, here travelling outwards
  radial   a dam break of varying place and height on a flat bed
  beach    a closed basin with a sloping, bumpy, partly dry bed
"""
import math
import random

import numpy as np
import torch

from samoa_amd import _native, host, swe
from samoa_amd.adjoint import GaugeInversion
from samoa_amd.inversion import gauges_near

G = 9.80665
COURANT = 0.45
SCALING = {"tsunami": 1.0e6, "radial": 1.0, "beach": 1.0e3}
DRYTOL = {"tsunami": 1.0e-3, "radial": 0.01, "beach": 1.0e-3}
WALLS = {"tsunami": swe.BC_OUTFLOW, "radial": swe.BC_WALL, "beach": swe.BC_WALL}
SOLVERS = {"aug_riemann": swe.SOLVER_AUG_RIEMANN, "fwave": swe.SOLVER_FWAVE,
           "llfbath": swe.SOLVER_LLF_BATH}


def listed():
    return [
        # a host program's own time loop on a small basin: one synchronous
        # traversal with refinement flags, and the state back for its outputs
        {"name": "host_loop_d8", "kind": "traverse", "scene": "radial", "depth": 8},
        # the radial dam break at its full size (32,768 cells), 100 steps
        # between two outputs, the dt chain on the device
        {"name": "radial_run_d14", "kind": "run", "scene": "radial", "depth": 14, "steps": 100,
         "toleranced": False},
        # a mid-sized tsunami between two outputs in the toleranced arithmetic
        {"name": "tsunami_run_tol_d18", "kind": "run", "scene": "tsunami", "depth": 18,
         "steps": 100, "toleranced": True},
        # one traversal of a large frozen mesh on the caller's device tensors
        {"name": "tsunami_step_d21", "kind": "step", "scene": "tsunami", "depth": 21,
         "rings": 0, "radius": 0.0, "solver": "aug_riemann", "toleranced": False,
         "forward": True, "flags": False},
        # the same in the toleranced arithmetic, backward, on a mesh refined
        # around a moving front (cells of several depths, a ragged count)
        {"name": "tsunami_step_graded_tol", "kind": "step", "scene": "tsunami", "depth": 17,
         "rings": 4, "radius": 0.21, "solver": "aug_riemann", "toleranced": True,
         "forward": False, "flags": True},
        # a basin with a beach and walls, refined, with refinement flags: the
        # f-wave solver
        {"name": "beach_step_fwave_graded", "kind": "step", "scene": "beach", "depth": 14,
         "rings": 3, "radius": 0.3, "solver": "fwave", "toleranced": False,
         "forward": True, "flags": True},
        # many small meshes of uneven size advanced together
        {"name": "ensemble_run_16", "kind": "ensemble", "scenarios": 16, "dmin": 12, "dmax": 16,
         "mix": 5, "steps": 100, "toleranced": False},
        # the adaptive tsunami remeshed before every step, between two outputs
        {"name": "adaptive_d16_26", "kind": "adaptive", "dmin": 16, "dmax": 26, "tol": 1.5e-3,
         "steps": 100, "toleranced": False},
        # the same at an everyday size, on a coarse base mesh
        {"name": "adaptive_d10_18", "kind": "adaptive", "dmin": 10, "dmax": 18, "tol": 8.0e-3,
         "steps": 50, "toleranced": False},
        # one adjoint traversal of a depth-20 inversion
        {"name": "adjoint_step_d20", "kind": "adjoint", "scene": "tsunami", "depth": 20,
         "solver": "aug_riemann", "forward": True},
        # a gauge misfit and its gradient (forward and reverse sweep)
        {"name": "gauge_gradient_d15", "kind": "gradient", "depth": 15, "steps": 30,
         "gauges": 32, "checkpoints": False},
        # a host that keeps its state in host memory: in, one step, out
        {"name": "host_buffers_d16", "kind": "host_buffers", "scene": "tsunami", "depth": 16},
    ]


def draw(rng):
    kind = rng.choice(["traverse", "run", "run", "step", "step", "step", "ensemble", "adaptive",
                       "adjoint", "gradient", "host_buffers"])
    scene = rng.choice(["tsunami", "radial", "beach"])
    tol = rng.random() < 0.35
    if kind == "traverse":
        return {"kind": kind, "scene": scene, "depth": rng.randint(4, 12)}
    if kind == "run":
        depth = rng.randint(9, 18)
        return {"kind": kind, "scene": scene, "depth": depth, "steps": rng.randint(11, 100),
                "toleranced": tol}
    if kind == "step":
        solver = rng.choice(["aug_riemann", "aug_riemann", "fwave", "llfbath"])
        rings = rng.randint(0, 4)
        return {"kind": kind, "scene": "tsunami" if solver == "llfbath" else scene,
                "depth": rng.randint(10, 20 - rings), "rings": rings,
                "radius": round(rng.uniform(0.05, 0.3), 3) if rings else 0.0, "solver": solver,
                "toleranced": tol and solver != "llfbath", "forward": rng.random() < 0.5,
                "flags": rng.random() < 0.5}
    if kind == "ensemble":
        dmin = rng.randint(8, 13)
        return {"kind": kind, "scenarios": rng.randint(3, 16), "dmin": dmin,
                "dmax": dmin + rng.randint(1, 3), "mix": rng.randint(0, 10 ** 6),
                "steps": rng.randint(11, 100), "toleranced": tol}
    if kind == "adaptive":
        dmin = rng.randint(8, 14)
        return {"kind": kind, "dmin": dmin, "dmax": dmin + rng.randint(5, 8),
                "tol": round(2.0 ** rng.uniform(-8.0, -5.0), 5), "steps": rng.randint(20, 100),
                "toleranced": tol}
    if kind == "adjoint":
        return {"kind": kind, "scene": rng.choice(["tsunami", "beach"]),
                "depth": rng.randint(10, 20), "solver": rng.choice(["aug_riemann", "fwave"]),
                "forward": rng.random() < 0.5}
    if kind == "gradient":
        return {"kind": kind, "depth": rng.randint(9, 15), "steps": rng.randint(8, 30),
                "gauges": rng.randint(3, 40), "checkpoints": rng.random() < 0.5}
    return {"kind": kind, "scene": scene, "depth": rng.randint(9, 16)}


# -- inputs -------------------------------------------------------------------

def _state(scene, mesh, seed, moving=True):
    """(eta, hu, hv, b) of a scene at the cells of a mesh."""
    rng = random.Random(int(seed) * 7919 + 13)
    if scene == "tsunami":
        eta, hu, hv, b = host.tsunami(mesh, seed=int(seed) % (1 << 31), drytol=DRYTOL[scene])
        if moving:
            p = host.tsunami_draw(int(seed) % (1 << 31))
            x = mesh.coords.mean(axis=1) * SCALING[scene]
            h = np.maximum(eta - b, 0.0)
            wet = h > DRYTOL[scene]
            rx, ry = x[:, 0] - p["x0"], x[:, 1] - p["y0"]
            r = np.sqrt(rx * rx + ry * ry) + 1.0
            a = np.where(wet, 0.5 * np.sqrt(G * h) * eta / r, 0.0)
            hu, hv = a * rx, a * ry
        return eta, hu, hv, b
    x = mesh.coords.mean(axis=1)
    cx, cy = 0.5 + rng.uniform(-0.15, 0.15), 0.5 + rng.uniform(-0.15, 0.15)
    r = np.hypot(x[:, 0] - cx, x[:, 1] - cy)
    z = np.zeros(mesh.n)
    if scene == "radial":
        return np.where(r < 0.1, rng.uniform(8.0, 12.0), 5.0), z, z.copy(), z.copy()
    k = [rng.uniform(5.0, 25.0) for _ in range(4)]
    b = -20.0 + 26.0 * x[:, 0] + 1.5 * np.sin(k[0] * x[:, 0] + k[1]) * np.cos(k[2] * x[:, 1] + k[3])
    eta = rng.uniform(1.0, 3.0) * np.exp(-((r / 0.12) ** 2))
    h = np.maximum(eta - b, 0.0)
    wet = h > DRYTOL[scene]
    a = np.where(wet, 0.3 * np.sqrt(G * h) * eta, 0.0)
    hu, hv = a * (x[:, 0] - cx) / (r + 1e-9), a * (x[:, 1] - cy) / (r + 1e-9)
    return np.where(wet, eta, np.minimum(b, 0.0)), hu, hv, b


def _params(scene, mesh_depths, solver="aug_riemann"):
    return dict(scaling=SCALING[scene], dry_tolerance=DRYTOL[scene], courant=COURANT,
                min_depth=max(0, int(mesh_depths.min()) - 2),
                max_depth=int(mesh_depths.max()) + 2,
                solver=SOLVERS[solver], boundary=WALLS[scene])


def _graded(depth, rings, radius):
    """A uniform mesh refined `rings` times in ever thinner bands around a
    circle, by the library's own remeshing: depths of a moving front."""
    mesh = host.mesh_uniform(depth)
    if not rings:
        return mesh
    with swe.EulerTimestep(mesh, min_depth=depth, max_depth=depth + rings) as op:
        z = np.zeros(mesh.n)
        op.upload(z, z, z, z)
        coords = mesh.coords
        for k in range(rings):
            x = coords.mean(axis=1)
            near = np.abs(np.hypot(x[:, 0] - 0.47, x[:, 1] - 0.52) - radius) < 0.12 / (1 + k)
            op.adapt(near.astype(np.int8))
            d, p, nbr = op.download_mesh()
            coords = host.coords_from_depths(d)[1]
    return swe.Mesh(d, p, nbr, coords)


def _source(seed):
    """A source of about 1 m (the scenario draws 0.5 to 2 m and axis ratios
    from 1 to 3): the refined mesh's size does not depend much on the seed."""
    for s in range(64 * (int(seed) % (1 << 24)), 1 << 31):
        p = host.tsunami_draw(s)
        if 0.95 < p["amplitude"] < 1.15 and 1.5 < p["ratio"] < 2.5:
            return s


def _adaptive_cells(case):
    """About the cells of the adaptive run's refined mesh: the base mesh, and
    inside the source's ellipse cells as wide as the elevation takes to vary
    by tol."""
    return int((2 << case["dmin"]) + 10.0 / case["tol"] ** 2)


def _capacity(case):
    return 2 * _adaptive_cells(case) + 4096


def _dev(a):
    return torch.tensor(np.ascontiguousarray(a), device="cuda")


def _mesh_and_state(case, seed):
    mesh = _graded(case["depth"], case.get("rings", 0), case.get("radius", 0.0))
    st = _state(case["scene"], mesh, seed)
    # the initialisation's dt estimate is in unit-square units
    dt = host.initial_dt(mesh, st, COURANT) * SCALING[case["scene"]]
    return mesh, st, dt


def _ensemble(case, seed):
    rng = random.Random(case["mix"])
    depths = [rng.randint(case["dmin"], case["dmax"]) for _ in range(case["scenarios"])]
    meshes = {d: host.mesh_uniform(d) for d in sorted(set(depths))}
    ms = [meshes[d] for d in depths]
    states = [_state("tsunami", m, seed * 64 + s, moving=False) for s, m in enumerate(ms)]
    dt0 = np.array([host.initial_dt(m, st, COURANT) for m, st in zip(ms, states)])
    return ms, states, dt0


def _gradient_inputs(case, seed):
    mesh = host.mesh_uniform(case["depth"])
    seed = int(seed) % (1 << 31)
    eta, _, _, b = host.tsunami(mesh, seed=seed, drytol=1e-3)
    src = host.tsunami_draw(seed)
    target = host.tsunami(mesh, seed=seed, drytol=1e-3, amplitude=1.25 * src["amplitude"])[0]
    z = np.zeros(mesh.n)
    dt = host.initial_dt(mesh, (eta, z, z, b), COURANT) * SCALING["tsunami"]
    gauges = gauges_near(mesh, src["x0"], src["y0"], 1.5e5, case["gauges"], seed=2024)
    return mesh, eta, b, target, dt, gauges


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("traverse", "run", "step", "adjoint", "host_buffers"):
        mesh, st, dt = _mesh_and_state(case, seed)
        op = swe.EulerTimestep(mesh, **_params(case["scene"], mesh.depth,
                                               case.get("solver", "aug_riemann")))
        if case.get("toleranced"):
            op.set_arithmetic(swe.ARITH_TOLERANCED)
        s.update(op=op, mesh=mesh, dt=dt, t=0.0, forward=case.get("forward", True))
        if kind in ("traverse", "run"):
            op.upload(*st)
        elif kind == "host_buffers":
            s["host"] = st
        else:
            s["stream"] = torch.cuda.Stream()
            s["q"] = [_dev(a) for a in st]
            s["out"] = [torch.empty_like(s["q"][0]) for _ in range(3)]
            s["cfl"] = torch.zeros(1, dtype=torch.float64, device="cuda")
            s["nref"] = torch.zeros(1, dtype=torch.int64, device="cuda")
            if kind == "step":
                s["refine"] = torch.zeros(mesh.n, dtype=torch.int8, device="cuda")
            else:
                # the forward traversal whose adjoint is taken, and dL/dQ'
                g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
                s["dtd"] = torch.full((1,), dt, dtype=torch.float64, device="cuda")
                s["masks"] = torch.empty(mesh.n, dtype=torch.int8, device="cuda")
                s["lam"] = [torch.randn(mesh.n, dtype=torch.float64, device="cuda", generator=g)
                            for _ in range(3)]
                s["gb"] = torch.zeros_like(s["q"][0])
                torch.cuda.synchronize()
                op.forward_device(*[a.data_ptr() for a in s["q"] + s["out"]], s["dtd"].data_ptr(),
                                  s["forward"], masks=s["masks"].data_ptr(),
                                  stream=s["stream"].cuda_stream)
    elif kind == "ensemble":
        ms, states, dt0 = _ensemble(case, seed)
        s["op"] = swe.Batch(ms, [dict(scaling=SCALING["tsunami"], dry_tolerance=DRYTOL["tsunami"],
                                      courant=COURANT) for _ in ms])
        if case["toleranced"]:
            s["op"].set_arithmetic(swe.ARITH_TOLERANCED)
        for i, st in enumerate(states):
            s["op"].upload(i, *st)
        s.update(dt=dt0, t=np.zeros(len(ms)), forward=False)
    elif kind == "adaptive":
        mesh = host.mesh_uniform(case["dmin"])
        op = swe.EulerTimestep(mesh, scaling=SCALING["tsunami"], dry_tolerance=DRYTOL["tsunami"],
                               courant=COURANT, min_depth=case["dmin"], max_depth=case["dmax"])
        if case["toleranced"]:
            op.set_arithmetic(swe.ARITH_TOLERANCED)
        z = np.zeros(mesh.n)
        op.upload(z, z, z, z)
        n, dt = host.tsunami_adaptive_setup(op, _source(seed), case["tol"], case["dmax"],
                                            DRYTOL["tsunami"], COURANT)
        # the host's arrays for an output, with room for the mesh to grow
        cap = _capacity(case)
        s.update(op=op, dt=dt, t=0.0, forward=False, k=0,
                 state=[np.zeros(cap) for _ in range(4)],
                 mesh=[np.zeros(cap, np.int8), np.zeros(cap, np.int8),
                       np.zeros(3 * cap, np.int32)])
    else:
        mesh, eta, b, target, dt, gauges = _gradient_inputs(case, seed)
        steps = case["steps"]
        prob = GaugeInversion(mesh, gauges, steps,
                              dict(scaling=SCALING["tsunami"], dry_tolerance=1e-3, courant=COURANT),
                              checkpoint_every=math.ceil(math.sqrt(steps)) if case["checkpoints"]
                              else "all")
        s.update(op=prob, eta=_dev(eta), b=_dev(b))
        prob.record_dt(s["eta"], s["b"], dt)
        s["target"] = prob.gauge_series(_dev(target), s["b"]).detach()
    torch.cuda.synchronize()
    return s


# -- one pass -----------------------------------------------------------------

def run(s):
    return {"traverse": _run_traverse, "run": _run_run, "step": _run_step,
            "ensemble": _run_ensemble, "adaptive": _run_adaptive, "adjoint": _run_adjoint,
            "gradient": _run_gradient, "host_buffers": _run_host_buffers}[s["kind"]](s)


def _run_traverse(s):
    res = s["op"].traverse(s["dt"], s["forward"], flags=True)
    s["dt"] = COURANT * res.dt_cfl
    s["forward"] = not s["forward"]
    eta, hu, hv, _ = s["op"].download()
    return eta, hu, hv, res.dt_cfl, res.n_refine, res.refine


def _run_run(s):
    n = s["case"]["steps"]
    s["t"], s["dt"] = s["op"].run(n, s["dt"], s["forward"], time=s["t"])
    s["forward"] ^= n % 2 == 1
    return (*s["op"].download()[:3], s["t"], s["dt"])


def _run_step(s):
    flags = s["case"]["flags"]
    s["op"].step_device(*[a.data_ptr() for a in s["q"] + s["out"]], s["dt"], s["forward"],
                        s["cfl"].data_ptr(), n_refine=s["nref"].data_ptr(),
                        refine=s["refine"].data_ptr() if flags else 0,
                        stream=s["stream"].cuda_stream)
    return (*s["out"], s["cfl"], s["nref"], s["refine"])


def _run_ensemble(s):
    n = s["case"]["steps"]
    s["t"], s["dt"] = s["op"].run(n, s["dt"], s["forward"], time=s["t"])
    s["forward"] ^= n % 2 == 1
    parts = [s["op"].download(i)[:3] for i in range(s["op"].n_scen)]
    return (*[np.concatenate(x) for x in zip(*parts)], s["t"], s["dt"])


def _run_adaptive(s):
    c = s["case"]
    s["dt"], s["t"], s["forward"], cells = host.adaptive_loop(
        s["op"], c["steps"], 1, c["tol"] / 2.0, c["tol"] / 16.0, s["k"], s["dt"], s["t"],
        s["forward"])
    s["k"] += c["steps"]
    if s["op"].n > s["state"][0].shape[0]:
        raise RuntimeError("the mesh outgrew the output arrays")
    lib, h = _native.load(), s["op"]._h
    _native.check("swe_download_mesh", lib.swe_download_mesh(h, *[a.ctypes.data for a in s["mesh"]]))
    _native.check("swe_download", lib.swe_download(h, *[a.ctypes.data for a in s["state"]]))
    return (*s["state"], *s["mesh"], s["t"], cells)


def _run_adjoint(s):
    s["op"].adjoint_device(*[a.data_ptr() for a in s["q"]], s["masks"].data_ptr(),
                           *[a.data_ptr() for a in s["lam"] + s["out"]], s["gb"].data_ptr(),
                           s["dtd"].data_ptr(), s["forward"], stream=s["stream"].cuda_stream)
    return (*s["out"], s["gb"])


def _run_gradient(s):
    eta = s["eta"].detach().requires_grad_()
    b = s["b"].detach().requires_grad_()
    series = s["op"].gauge_series(eta, b)
    ((series - s["target"]) ** 2).sum().backward()
    return series.detach(), eta.grad, b.grad


def _run_host_buffers(s):
    s["op"].upload(*s["host"])
    res = s["op"].traverse(s["dt"], True)
    eta, hu, hv, _ = s["op"].download()
    return eta, hu, hv, res.dt_cfl, res.n_refine


# -- what a pass cannot do without ----------------------------------------------

# per cell of one traversal: eta, hu, hv, b in and eta, hu, hv out; neighbours,
# plotter type and depth in.  About 250 operations a solve, 1.5 solves a cell,
# and the update.
STEP_BYTES, TOPOLOGY_BYTES, STEP_FLOPS = 56, 14, 420


def _cells(case):
    n = 2 << case["depth"]
    if not case.get("rings"):
        return n
    # bands of half width 0.12 / (1 + k) around a circle, each refined once
    # more (a cell of the band becomes two)
    area = lambda w: math.pi * ((case["radius"] + w) ** 2 - max(0.0, case["radius"] - w) ** 2)  # noqa: E731
    return int(n * (1.0 + sum(2 ** k * min(1.0, area(0.12 / (1 + k)))
                              for k in range(case["rings"]))))


def work(case):
    kind = case["kind"]
    step = STEP_BYTES + TOPOLOGY_BYTES
    if kind == "ensemble":
        rng = random.Random(case["mix"])
        n = sum(2 << rng.randint(case["dmin"], case["dmax"]) for _ in range(case["scenarios"]))
        return {"bytes": n * (step * case["steps"] + 32), "flops": n * STEP_FLOPS * case["steps"]}
    if kind == "adaptive":
        n = _adaptive_cells(case)
        # a remeshing reads and writes the state and the topology once
        return {"bytes": n * ((step + 2 * 46) * case["steps"] + 46),
                "flops": n * STEP_FLOPS * case["steps"]}
    n = _cells(case)
    if kind == "run":
        return {"bytes": n * (step * case["steps"] + 24), "flops": n * STEP_FLOPS * case["steps"]}
    if kind == "step":
        return {"bytes": n * (step + (1 if case["flags"] else 0)), "flops": n * STEP_FLOPS}
    if kind == "traverse":
        return {"bytes": n * (step + 1 + 24), "flops": n * STEP_FLOPS}
    if kind == "host_buffers":
        return {"bytes": n * (step + 32 + 24), "flops": n * STEP_FLOPS}
    adjoint = 32 + 24 + 24 + 16 + 1 + TOPOLOGY_BYTES
    if kind == "adjoint":
        return {"bytes": n * adjoint, "flops": n * 2.5 * STEP_FLOPS}
    return {"bytes": n * (step + 1 + adjoint) * case["steps"],
            "flops": n * 3.5 * STEP_FLOPS * case["steps"]}


# -- the same outputs from plain PyTorch, 64 bits ---------------------------------

def _tables():
    """Outward unit normals [17, 3, 2] by plotter type + 8, and sqrt(1/2)**k at
    k + 1 (the legs of depth k; the hypotenuse is the leg of depth k - 1)."""
    normal = np.zeros((17, 3, 2))
    for p in list(range(-8, 0)) + list(range(1, 9)):
        a = math.pi / 4.0 * abs(p)
        c, s = math.cos(a), math.sin(a)
        J = np.array([[c, -s], [s, c]] if p > 0 else [[-s, c], [c, s]])
        Ji = np.linalg.inv(np.trunc(1.5 * J))
        for k, e in enumerate(((-1.0, 0.0), (1.0, 1.0), (0.0, -1.0))):
            v = np.array(e) @ Ji
            normal[p + 8, k] = v / math.hypot(*v)
    return normal, np.sqrt(0.5) ** np.arange(-1, 63)


def _sqrt(x):
    """sqrt with derivative 0 at 0 (a dry side)."""
    pos = x > 0.0
    return torch.where(pos, torch.sqrt(torch.where(pos, x, torch.ones_like(x))),
                       torch.zeros_like(x))


def _min(a, b):
    """min whose derivative goes to the operand taken (ties: the second)."""
    return torch.where(a < b, a, torch.zeros_like(a) + b)


def _max(a, b):
    return torch.where(a > b, a, torch.zeros_like(a) + b)


def _ok(x, cond):
    """x where cond holds, else a harmless 1 (the branch is not taken)."""
    return torch.where(cond, x, torch.ones_like(x))


def _middle_speeds(hL, hR, uL, uR, cL, cR, drytol):
    """Speeds of the two waves at the middle state and its depth (one step of
    the root search), cL = sqrt(g hL) and cR = sqrt(g hR)."""
    W = torch.where
    right_low = hR < hL
    lo, hi = W(right_low, hR, hL), W(right_low, hL, hR)
    clo, chi = W(right_low, cR, cL), W(right_low, cL, cR)
    du = uR - uL
    dry = lo <= drytol
    los, his = _ok(lo, ~dry), _ok(hi, ~dry)
    fmin = du + 2.0 * (clo - chi)
    fmax = du + (hi - lo) * _sqrt(((0.5 * G) * (his + los)) / (his * los))
    two_rare = ~dry & (fmin > 0.0)
    two_shock = ~dry & ~(fmin > 0.0) & (fmax <= 0.0)
    mixed = ~dry & ~(fmin > 0.0) & (fmax > 0.0)
    t = _max(-du + 2.0 * (cL + cR), 0.0)
    hm_r = t * t / (16.0 * G)
    cm = _sqrt(_ok(G * hm_r, two_rare))
    r1, r2 = (uL + 2.0 * cL) - 3.0 * cm, (uR - 2.0 * cR) + 3.0 * cm
    h0, hLs, hRs = _ok(hi, two_shock), _ok(hL, two_shock), _ok(hR, two_shock)
    gL = _sqrt((0.5 * G) * (1.0 / h0 + 1.0 / hLs))
    gR = _sqrt((0.5 * G) * (1.0 / h0 + 1.0 / hRs))
    f0 = (du + (h0 - hLs) * gL) + (h0 - hRs) * gR
    df = ((gL - (G * (h0 - hLs)) / ((4.0 * h0 * h0) * gL)) + gR) - \
        (G * (h0 - hRs)) / ((4.0 * h0 * h0) * gR)
    q = _sqrt(h0) - f0 / _ok((2.0 * _sqrt(h0)) * df, two_shock)
    hm_s = _ok(q * q, two_shock)
    cm = _sqrt(G * hm_s)
    s1 = (uL - (hm_s - hLs) * _sqrt((0.5 * G) * (1.0 / hm_s + 1.0 / hLs))) - cm
    s2 = (uR + (hm_s - hRs) * _sqrt((0.5 * G) * (1.0 / hm_s + 1.0 / hRs))) + cm
    slope = (fmax - fmin) / _ok(hi - lo, mixed)
    hm_m = los - fmin / _ok(slope, mixed)
    cm = _sqrt(_ok(G * hm_m, mixed))
    left = hL > hR
    m1 = W(left, (uL + 2.0 * cL) - 3.0 * cm, (uR - 2.0 * cR) + cm)
    m2 = W(left, (uL + 2.0 * cL) - cm, (uR - 2.0 * cR) + 3.0 * cm)
    d = ((uR + uL) - 2.0 * cR) + 2.0 * cL
    zero = torch.zeros_like(hL)
    return (W(dry, d, W(two_rare, r1, W(two_shock, s1, m1))),
            W(dry, d, W(two_rare, r2, W(two_shock, s2, m2))),
            W(dry, zero, W(two_rare, hm_r, W(two_shock, hm_s, hm_m))))


def _geoclaw(L, R, drytol, solver):
    """Net updates of both sides and the largest speed, in the edge frame;
    L, R = (h, normal momentum, tangential momentum, b)."""
    W = torch.where
    (hL, pL, tL, bL), (hR, pR, tR, bR) = L, R
    zero, one = torch.zeros_like(hL), torch.ones_like(hL)
    wetL, wetR = hL > drytol, hR > drytol
    active = wetL | wetR
    uL, vL = W(wetL, pL / _ok(hL, wetL), zero), W(wetL, tL / _ok(hL, wetL), zero)
    uR, vR = W(wetR, pR / _ok(hR, wetR), zero), W(wetR, tR / _ok(hR, wetR), zero)
    hL, pL, hR, pR = W(wetL, hL, zero), W(wetL, pL, zero), W(wetR, hR, zero), W(wetR, pR, zero)
    cl, cr = _sqrt(G * hL), _sqrt(G * hR)
    starR = _middle_speeds(hL, hL, uL, -uL, cl, cl, drytol)[2]
    starL = _middle_speeds(hR, hR, -uR, uR, cr, cr, drytol)[2]
    wallR = wetL & ~wetR & (_max(hL, starR) + bL < bR)
    clipR = wetL & ~wetR & ~wallR & (hL + bL < bR)
    wallL = wetR & ~wetL & (_max(hR, starL) + bR < bL)
    clipL = wetR & ~wetL & ~wallL & (hR + bR < bL)
    (hR, pR, uR, vR, bR), (hL, pL, uL, vL, bL) = (
        (W(wallR, hL, hR), W(wallR, -pL, pR), W(wallR, -uL, uR), W(wallR, vL, vR),
         W(wallR, bL, W(clipR, hL + bL, bR))),
        (W(wallL, hR, hL), W(wallL, -pR, pL), W(wallL, -uR, uL), W(wallL, vR, vL),
         W(wallL, bR, W(clipL, hR + bR, bL))))
    walls = (W(wallL, zero, one), W(wallL | wallR, zero, one), W(wallR, zero, one))
    dh, dp, db = hR - hL, pR - pL, bR - bL
    dphi = ((dp * (uL + uR) - (uL * uR) * dh) +
            ((0.5 * G) * (((bR + hR) - bL) - hL)) * (hR + hL)) - ((0.5 * G) * (hR + hL)) * db
    cL, cR = _sqrt(G * hL), _sqrt(G * hR)
    roe = (cL * uL + cR * uR) / _ok(cR + cL, active)
    croe = _sqrt((G * 0.5) * (hR + hL))
    e1 = _min(uL - cL, roe - croe)
    e2 = _max(uR + cR, roe + croe)
    if solver == "fwave":
        dec = dphi + ((G * 0.5) * (hR + hL)) * db
        span = _ok(e2 - e1, active)
        b1, b2 = (e2 * dp - dec) / span, (dec - e1 * dp) / span
        speeds = (e1, 0.5 * (e1 + e2), e2)
        f0, f2 = (b1, b1 * e1, b1 * vL), (b2, b2 * e2, b2 * vR)
        f1 = (zero, zero, ((pR * vR - pL * vL) - f0[2]) - f2[2])
    else:
        s1, s2, _ = _middle_speeds(hL, hR, uL, uR, cL, cR, drytol)
        l0, l2 = _min(e1, s2), _max(e2, s1)
        span = _ok(l2 - l0, active)
        hll = _max((((pL - pR) + l2 * hR) - l0 * hL) / span, 0.0)
        l1 = 0.5 * (l0 + l2)
        l1 = W(torch.abs(l1) < 1.0e-20, zero, l1)
        eps = 1.0e-6
        hbar = _max(0.5 * (hL + hR), 0.0)
        bar = 0.25 * ((uL + uR) * (uL + uR)) - G * hbar
        tilde = _max(uL * uR, 0.0) - G * hbar
        sonic = ((torch.abs(bar) <= eps) | (bar * tilde <= eps) | ((bar * l0) * l2 <= eps) |
                 (_min(torch.abs(l0), torch.abs(l2)) < eps) |
                 ((l0 < 0.0) & (s1 > 0.0)) | ((l2 > 0.0) & (s2 < 0.0)) |
                 ((uL + cL) * (uR + cR) < 0.0) | ((uL - cL) * (uR - cR) < 0.0))
        bars = _ok(bar, ~sonic & active)
        ddh = W(sonic, -db, ((db * G) * hbar) / bars)
        sub, sup, sdn = (l0 < -eps) & (l2 > eps), l0 >= eps, l2 <= -eps
        sup = ~sub & sup
        sdn = ~sub & ~sup & sdn
        top = (hll * (l2 - l0)) / _ok(l2, sub | sdn)
        bot = (hll * (l2 - l0)) / _ok(l0, sub | sup)
        ddh = W(sub, _max(_min(ddh, top), bot),
                W(sup, _max(_min(ddh, bot), -hL),
                  W(sdn, _max(_min(ddh, hR), top), ddh)))
        ddphi = W(sonic, -((G * hbar) * db), -((((db * G) * hbar) * tilde) / bars))
        kL, kR = -(hL * db), -(hR * db)
        ddphi = _min(ddphi, G * _max(kL, kR))
        ddphi = _max(ddphi, G * _min(kL, kR))
        x0, x2 = dh - ddh, dphi - ddphi
        q0, q2 = l0 * l0, l2 * l2
        det = _ok(l0 - l2, active)
        b0 = (-(x0 * l2) + dp) / det
        b1 = ((dp * q2 - l2 * x2) - x0 * (l0 * q2 - l2 * q0) + (l0 * x2 - dp * q0)) / det
        b2 = (-dp + x0 * l0) / det
        speeds = (l0, l1, l2)
        f0 = (b0 * l0, b0 * q0, (b0 * l0) * vL)
        f2 = (b2 * l2, b2 * q2, (b2 * l2) * vR)
        f1 = (zero, b1, (((hR * uR) * vR - (hL * uL) * vL) - f0[2]) - f2[2])
    speeds = [s * w for s, w in zip(speeds, walls)]
    left, right = [], []
    for m in range(3):
        a, c = zero, zero
        for f, w, s in zip((f0, f1, f2), walls, speeds):
            x = f[m] * w
            a = a + W(s < 0.0, x, W(s > 0.0, zero, 0.5 * x))
            c = c + W(s > 0.0, x, W(s < 0.0, zero, 0.5 * x))
        left.append(W(active, a, zero))
        right.append(W(active, c, zero))
    fastest = _max(_max(torch.abs(speeds[0]), torch.abs(speeds[1])),
                            torch.abs(speeds[2]))
    return left, right, W(active, fastest, zero)


def _llfbath(nx, ny, L, R, drytol):
    """Local Lax-Friedrichs with bathymetry, a wall against a dry side."""
    W = torch.where
    (eL, pL, qL, bL), (eR, pR, qR, bR) = L, R
    zero = torch.zeros_like(eL)
    dryL, dryR = eL - bL < drytol, eR - bR < drytol
    hL, hR = _max(eL - bL, 0.0), _max(eR - bR, 0.0)
    uL = nx * (pL / _ok(eL - bL, ~dryL)) + ny * (qL / _ok(eL - bL, ~dryL))
    uR = nx * (pR / _ok(eR - bR, ~dryR)) + ny * (qR / _ok(eR - bR, ~dryR))
    sL, sR = _sqrt(G * hL) + torch.abs(uL), _sqrt(G * hR) + torch.abs(uR)
    a = _max(sL, sR)
    fh = 0.5 * ((hL * uL + hR * uR) + a * (eL - eR))
    pr = (0.5 * G) * (hL * hL + hR * hR)
    fu = 0.5 * (((pL * uL + pR * uR) + pr * nx) + a * (pL - pR))
    fv = 0.5 * (((qL * uL + qR * uR) + pr * ny) + a * (qL - qR))
    src = ((0.25 * G) * (hL + hR)) * (bR - bL)
    prL, prR = ((0.5 * G) * hL) * hL, ((0.5 * G) * hR) * hR
    wL, wR = dryR & ~dryL, dryL & ~dryR
    any_dry = dryL | dryR
    fL = (W(any_dry, zero, fh),
          W(any_dry, W(wL, ((0.5 * uL) * pL + prL * nx) + (0.5 * sL) * pL, zero), fu + src * nx),
          W(any_dry, W(wL, ((0.5 * uL) * qL + prL * ny) + (0.5 * sL) * qL, zero), fv + src * ny),
          W(dryL, zero, sL))
    fR = (W(any_dry, zero, -fh),
          W(any_dry, W(wR, (-((0.5 * uR) * pR) - prR * nx) + (0.5 * sR) * pR, zero), -fu + src * nx),
          W(any_dry, W(wR, (-((0.5 * uR) * qR) - prR * ny) + (0.5 * sR) * qR, zero), -fv + src * ny),
          W(dryR, zero, sR))
    return fL, fR


class _Plain:
    """A mesh (or several, end to end) for the plain step."""

    def __init__(self, mesh, scene, solver="aug_riemann", n_scen=1, scen=None):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        normal, leg = _tables()
        n = mesh.n
        self.scene, self.solver, self.n_scen, self.scen = scene, solver, n_scen, scen
        if scen is not None:
            self.scen = torch.tensor(scen, device=dev)
        nbr = torch.tensor(np.asarray(mesh.nbr, np.int64).reshape(n, 3), device=dev)
        cell = torch.arange(n, device=dev)[:, None].expand(n, 3)
        self.bnd = nbr < 0
        self.o = torch.where(self.bnd, cell, nbr)
        self.lower = self.bnd | (cell < self.o)
        self.upper = self.bnd | (cell > self.o)
        pt = torch.tensor(np.asarray(mesh.plotter, np.int64), device=dev) + 8
        nt = torch.tensor(normal, device=dev)[pt]
        self.nx, self.ny = nt[..., 0], nt[..., 1]
        d = torch.tensor(np.asarray(mesh.depth, np.int64), device=dev)
        self.depth = d
        S = SCALING[scene]
        self.vol = (S * S) * torch.pow(torch.full_like(d, 0.5, dtype=torch.float64), d + 1)
        legs = torch.tensor(leg, device=dev)
        self.len = (S * legs[d + 1], S * legs[d], S * legs[d + 1])

    def step(self, eta, hu, hv, b, dt, forward):
        """One traversal; dt a number, or one per scenario.  Returns the new
        state, the CFL minimum (per scenario) and |sum of the depth fluxes|."""
        W, drytol = torch.where, DRYTOL[self.scene]
        own = [a[:, None].expand(-1, 3) for a in (eta, hu, hv, b)]
        oth = [a[self.o] for a in (eta, hu, hv, b)]
        if WALLS[self.scene] == swe.BC_WALL:
            m = 2.0 * (own[1] * self.nx + own[2] * self.ny)
            oth[1] = W(self.bnd, own[1] - m * self.nx, oth[1])
            oth[2] = W(self.bnd, own[2] - m * self.ny, oth[2])
        is_left = self.lower if forward else self.upper
        L = [W(is_left, x, y) for x, y in zip(own, oth)]
        R = [W(is_left, y, x) for x, y in zip(own, oth)]
        nx, ny = W(is_left, self.nx, -self.nx), W(is_left, self.ny, -self.ny)
        if self.solver == "llfbath":
            fL, fR = _llfbath(nx, ny, L, R, drytol)
        else:
            turn = lambda q: (q[0] - q[3], nx * q[1] + ny * q[2], nx * q[2] - ny * q[1], q[3])  # noqa: E731
            l, r, s = _geoclaw(turn(L), turn(R), drytol, self.solver)
            back = lambda f: (f[0], f[1] * nx - f[2] * ny, f[1] * ny + f[2] * nx, s)  # noqa: E731
            fL, fR = back(l), back(r)
        order = (0, 1, 2) if forward else (2, 1, 0)
        total = []
        for x, y in zip(fL, fR):
            f = W(is_left, x, y)
            acc = torch.zeros_like(eta)
            for k in order:
                acc = acc + self.len[k] * f[:, k]
            total.append(acc)
        limit = self.vol / _ok(total[3], total[3] > 0.0)
        limit = W(total[3] > 0.0, limit, torch.full_like(limit, np.inf)).detach()
        if self.scen is None:
            cfl = limit.min()
            scale = -dt / self.vol
        else:
            cfl = torch.full((self.n_scen,), np.inf, dtype=torch.float64, device=limit.device)
            cfl = cfl.scatter_reduce(0, self.scen, limit, "amin")
            scale = -dt[self.scen] / self.vol
        dh, d1, d2 = scale * total[0], scale * total[1], scale * total[2]
        zero = torch.zeros_like(eta)
        wetting = (eta < b + drytol) & (dh > 0.0)
        e = W(wetting, b + drytol, eta) + dh
        u = W(wetting, zero, hu) + d1
        v = W(wetting, zero, hv) + d2
        drying = e < b + drytol
        e = W(drying, _min(b, 0.0), e)
        return e, W(drying, zero, u), W(drying, zero, v), cfl, torch.abs(total[0]).detach()


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    up = lambda st: [torch.tensor(np.ascontiguousarray(a), device=dev) for a in st]  # noqa: E731
    if kind == "adaptive":
        return None  # a remeshed run: minutes in plain code
    if kind == "gradient":
        return _exact_gradient(case, seed, dev)
    if kind == "ensemble":
        ms, states, dt0 = _ensemble(case, seed)
        off = np.cumsum([0] + [m.n for m in ms])
        nbr = np.concatenate([np.where(m.nbr < 0, -1, m.nbr + o) for m, o in zip(ms, off)])
        whole = swe.Mesh(np.concatenate([m.depth for m in ms]),
                         np.concatenate([m.plotter for m in ms]), nbr)
        scen = np.repeat(np.arange(len(ms)), [m.n for m in ms])
        p = _Plain(whole, "tsunami", n_scen=len(ms), scen=scen)
        q = up([np.concatenate(x) for x in zip(*states)])
        dt = torch.tensor(dt0, device=dev)
        return _exact_run(p, q, dt, False, case["steps"])
    mesh, st, dt = _mesh_and_state(case, seed)
    p = _Plain(mesh, case["scene"], case.get("solver", "aug_riemann"))
    q = up(st)
    forward = case.get("forward", True)
    if kind == "run":
        return _exact_run(p, q, torch.tensor(dt, dtype=torch.float64, device=dev), forward,
                          case["steps"])
    if kind == "adjoint":
        g = torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))
        lam = [torch.randn(mesh.n, dtype=torch.float64, device="cuda", generator=g)
               for _ in range(3)]
        q = [a.requires_grad_() for a in q]
        out = p.step(*q, dt, forward)
        return torch.autograd.grad(out[:3], q, lam)
    e, u, v, cfl, _ = p.step(*q, dt, forward)
    if kind == "host_buffers":
        return e, u, v, cfl, None
    return e, u, v, cfl if kind == "traverse" else cfl.reshape(1), None, None


def _exact_run(p, q, dt, forward, steps):
    t = torch.zeros_like(dt)
    for _ in range(steps):
        e, u, v, cfl, _ = p.step(*q, dt, forward)
        q = [e, u, v, q[3]]
        t, dt, forward = t + dt, COURANT * cfl, not forward
    return q[0], q[1], q[2], t, dt


def _exact_gradient(case, seed, dev):
    if (2 << case["depth"]) * case["steps"] > 3_000_000:
        return None  # its tape would not be kept in plain code
    mesh, eta, b, target, dt0, gauges = _gradient_inputs(case, seed)
    p = _Plain(mesh, "tsunami")
    g = torch.tensor(np.asarray(gauges), device=dev)
    z = torch.zeros(mesh.n, dtype=torch.float64, device=dev)
    eta, b, target = (torch.tensor(a, device=dev) for a in (eta, b, target))

    def series(e, bed, dts):
        q, rows, used = (e, z, z), [], []
        dt = torch.tensor(dt0, dtype=torch.float64, device=dev)
        for n in range(case["steps"]):
            dt = dt if dts is None else dts[n]
            used.append(dt)
            e1, u1, v1, cfl, _ = p.step(*q, bed, dt, n % 2 == 1)
            q = (e1, u1, v1)
            rows.append(e1[g])
            dt = COURANT * cfl
        return torch.stack(rows), used

    with torch.no_grad():
        _, dts = series(eta, b, None)
        want, _ = series(target, b, dts)
    eta.requires_grad_()
    b.requires_grad_()
    got, _ = series(eta, b, dts)
    ge, gb = torch.autograd.grad(((got - want) ** 2).sum(), (eta, b))
    return got.detach(), ge, gb
