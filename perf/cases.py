"""The solves this package is timed on: what a program that uses it has it do,
through the package's public entry points (``aither_amd.Solver``,
``aither_amd.Server``), over the range of sizes, schemes and precisions the
input files of the package's benchmark, tests and case generators use.

One pass of a case is

* ``calls: "run"``: one solve request as a program makes it with a case that
  is resident on the device: the initial field goes in (``set_state``), the
  outer steps run (``run``, a replayed graph), the field and the norms come
  out.  The field goes in again at every pass, so every pass is the same work.
* ``calls: "iterate"``: the reference's own main loop around this package:
  ``begin_step`` and ``iterate`` with the norms read after every nonlinear
  iteration, the field read at the end.  The solve goes on from pass to pass.
* ``calls: "serve"``: one batch step of a server that holds several cases,
  then every case's field.  The solves go on from pass to pass.

The arithmetic is double precision throughout (the single-precision operator
only steers the iteration), so there is no plain computation in higher
precision to hold the outputs against: ``exact`` gives None.
"""
import math
import os
import tempfile

import numpy as np

from aither_amd import Server, Solver, cases

T_INF = 288.15
GAMMA = (cases.AIR_N + 1.0) / cases.AIR_N


def _case(name, kind, ni, nj, nk, steps, calls="run", **opt):
    c = {"name": name, "kind": kind, "ni": ni, "nj": nj, "nk": nk, "steps": steps, "subits": 1, "calls": calls,
         "time": "implicitEuler", "cfl": 5.0, "recon": "thirdOrder", "limiter": "vanAlbada", "flux": "roe",
         "viscous": False, "visc_recon": "central", "solver": "lusgs", "sweeps": 1, "precision": "fp64", "beta": 5.0}
    c.update(opt)
    return c


# the multiblock laminar channel of the benchmark (eight blocks, BDF2 with
# subiterations, 5x5 blocks)
CHANNEL = dict(subits=20, time="bdf2", flux="ausm", viscous=True, solver="blusgs")
# the served solves (bump channels, minmod, single-precision operator)
SERVED = dict(limiter="minmod", cfl=20.0, precision="fp32")


def listed():
    return [
        # the smallest calls: a 24^3 bump channel driven iteration by
        # iteration with the norms read each time, as the reference's main
        # loop does; launches and latency count
        _case("bump_24_iterate", "bump", 24, 24, 24, 5, calls="iterate", limiter="minmod", cfl=20.0),
        # one steady request of the serving stream alone
        _case("bump_40_fp32", "bump", 40, 40, 40, 60, **SERVED),
        # the served stream: eight requests of different sizes resident on
        # the device, 20 iterations each in shared launches
        _case("serve_8_fp32", "serve", 24, 40, 8, 20, calls="serve", **SERVED),
        # the isentropic vortex at its standard size: scalar LU-SGS, Roe
        _case("vortex_64", "box", 64, 64, 64, 100),
        # ragged block, AUSMPW+, single-precision operator
        _case("euler_97x61x43_fp32", "box", 97, 61, 43, 60, flux="ausm", precision="fp32", beta=2.0),
        # fifth-order reconstruction on a ragged block
        _case("weno_57x49x38", "box", 57, 49, 38, 40, recon="weno", flux="ausm", cfl=2.0, beta=2.0),
        # explicit time integration: the residual is the iteration
        _case("explicit_96", "box", 96, 96, 96, 60, time="explicitEuler", cfl=0.3),
        # a laminar channel with the scalar solver, two sweeps, fourth-order
        # viscous face states, moving isothermal wall
        _case("laminar_48_sweeps2", "bump", 48, 48, 48, 40, viscous=True, visc_recon="centralFourth", sweeps=2),
        # point-Jacobi block solver on a laminar channel
        _case("laminar_44_bdplur", "bump", 44, 44, 44, 30, viscous=True, solver="bdplur", sweeps=4),
        # the multiblock channel at a quarter of its resolution
        _case("channel_16k", "channel", 24, 16, 8, 2, **CHANNEL),
        # an odd-sized multiblock channel with the single-precision operator
        _case("channel_ragged_fp32", "channel", 59, 39, 19, 3, precision="fp32", **CHANNEL),
        # the benchmark's multiblock channel, 1,032,192 cells
        _case("channel_1M", "channel", 96, 64, 32, 8, **CHANNEL),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "box", "bump", "bump", "serve", "channel", "channel"])
    c = _case("", kind, 0, 0, 0, rng.randint(20, 60))
    del c["name"]
    c["precision"] = rng.choice(["fp64", "fp32"])
    if kind == "channel":
        c.update(CHANNEL)
        c.update(ni=_logint(rng, 16, 88), nj=_logint(rng, 12, 60), nk=_logint(rng, 6, 32), steps=rng.randint(1, 3),
                 flux=rng.choice(["ausm", "roe"]), sweeps=rng.choice([1, 1, 2]))
    elif kind == "serve":
        lo = rng.randint(16, 32)
        c.update(SERVED)
        c.update(ni=lo, nj=lo + rng.randint(4, 24), nk=rng.randint(2, 12), calls="serve", steps=20,
                 precision=rng.choice(["fp64", "fp32"]))
    elif kind == "bump":
        n = _logint(rng, 16, 72)
        viscous = rng.random() < 0.5
        c.update(ni=n, nj=n, nk=n, limiter=rng.choice(["minmod", "vanAlbada"]), viscous=viscous,
                 visc_recon=rng.choice(["central", "centralFourth"]), cfl=5.0 if viscous else 20.0,
                 solver=rng.choice(["lusgs", "lusgs", "blusgs", "dplur", "bdplur"]), sweeps=rng.choice([1, 2]),
                 calls=rng.choice(["run", "run", "iterate"]))
        if c["calls"] == "iterate":
            c["steps"] = rng.randint(3, 10)
    else:
        explicit = rng.random() < 0.2
        c.update(beta=2.0, ni=_logint(rng, 17, 110), nj=_logint(rng, 17, 90), nk=_logint(rng, 13, 72),
                 recon=rng.choice(["thirdOrder", "thirdOrder", "weno", "wenoZ", "constant"]),
                 flux=rng.choice(["roe", "ausm"]), limiter=rng.choice(["vanAlbada", "minmod"]),
                 time="explicitEuler" if explicit else "implicitEuler", cfl=0.3 if explicit else 2.0,
                 solver=rng.choice(["lusgs", "lusgs", "lusgs", "blusgs"]))
    return c


# ---- the case files, in the reference's formats

def _numerics(c, name, p_inf, rho_inf, u_inf, states, extra=""):
    return f"""gridName: {name}
equationSet: {"navierStokes" if c["viscous"] else "euler"}
viscousFaceReconstruction: {c["visc_recon"]}
timeIntegration: {c["time"]}
cflStart: {c["cfl"]}
cflMax: {c["cfl"]}
nonlinearIterations: {c["subits"]}
iterations: {c["steps"]}
faceReconstruction: {c["recon"]}
limiter: {c["limiter"]}
inviscidFlux: {c["flux"]}
referenceTemperature: {T_INF!r}
referenceDensity: {rho_inf!r}
referenceLength: 1.0
initialConditions: <icState(tag=-1; pressure={p_inf!r}; density={rho_inf!r}; velocity=[{u_inf!r}, 0.0, 0.0])>
matrixSolver: {c["solver"]}
matrixSweeps: {c["sweeps"]}
matrixRelaxation: 1.0
boundaryStates: <characteristic(tag=1; pressure={p_inf!r}; density={rho_inf!r}; velocity=[{u_inf!r}, 0.0, 0.0]){states}>
{extra}"""


def _surfaces(ni, nj, nk, types):
    lim = ((0, 0, 0, nj, 0, nk), (ni, ni, 0, nj, 0, nk), (0, ni, 0, 0, 0, nk), (0, ni, nj, nj, 0, nk),
           (0, ni, 0, nj, 0, 0), (0, ni, 0, nj, nk, nk))
    rows = [f"{t} {' '.join(map(str, r))} {tag}" for (t, tag), r in zip(types, lim)]
    return "2 2 2\n" + "\n".join(rows) + "\n"


def _write(work, name, c, blocks, surfaces, p_inf, rho_inf, u_inf, states="", extra=""):
    cases.write_plot3d(os.path.join(work, name + ".xyz"), blocks)
    text = _numerics(c, name, p_inf, rho_inf, u_inf, states, extra)
    text += f"boundaryConditions: {len(blocks)}\n" + "".join(surfaces)
    path = os.path.join(work, name + ".inp")
    with open(path, "w") as f:
        f.write(text)
    return path


def _box(work, c, rng):
    """the isentropic vortex on a Mach 0.5 free stream (strength `beta`, core moved by
    the seed)"""
    ni, nj, nk = c["ni"], c["nj"], c["nk"]
    h = 10.0 / max(ni, nj)
    g = [(np.arange(n + 1) * h) for n in (ni, nj, nk)]
    x, y, z = np.meshgrid(*g, indexing="ij")
    xc, yc, zc = cases.cell_centres(x, y, z)
    rho, u, v, w, p, fs = cases.vortex_state(xc, yc, beta=c["beta"], x0=h * ni * rng.uniform(0.45, 0.55),
                                             y0=h * nj * rng.uniform(0.45, 0.55))
    path = _write(work, "box", c, [(x, y, z)], [_surfaces(ni, nj, nk, [("characteristic", 1)] * 6)], fs["p_inf"],
                  fs["rho_inf"], fs["u_inf"])
    w = 1.0e-3 * fs["u_inf"] * rng.uniform(-1, 1, w.shape)
    return path, [np.stack([a.transpose(2, 1, 0).reshape(-1) for a in (rho, u, v, w, p)], axis=1)]


def _free_stream(dims, rng, rho, u, p, eps=1.0e-3):
    out = []
    for ni, nj, nk in dims:
        W = np.empty((ni * nj * nk, 5))
        W[:, 0], W[:, 4] = rho, p
        W[:, 1:4] = eps * u * rng.uniform(-1.0, 1.0, (len(W), 3))
        W[:, 1] += u
        out.append(W)
    return out


def _bump(work, c, rng, n, name="bump"):
    """a channel with a sine bump on its lower wall; height and Mach by the
    seed; viscous: a small channel with an adiabatic lower and a moving
    isothermal upper wall, Reynolds number of order 1e3"""
    hl, mach = float(rng.uniform(0.02, 0.10)), float(rng.uniform(0.2, 0.8))
    i, j, k = np.meshgrid(*[np.arange(n + 1)] * 3, indexing="ij")
    x = 3.0 * i / n
    yw = hl * np.sin(np.pi * np.clip(x - 1.0, 0.0, 1.0)) ** 2
    y, z = yw + (1.0 - yw) * j / n, 1.0 * k / n
    s = 2.0e-4 if c["viscous"] else 1.0
    rho = 1.225
    p = rho * cases.air_gas_constant() * T_INF
    u = mach * math.sqrt(GAMMA * p / rho)
    lo, hi = (("viscousWall", 3), ("viscousWall", 4)) if c["viscous"] else (("slipWall", 2), ("slipWall", 2))
    states = (f", viscousWall(tag=3), viscousWall(tag=4; temperature=300.0; velocity=[{0.3 * u!r}, 0.0, 0.0])"
              if c["viscous"] else "")
    types = [("characteristic", 1), ("characteristic", 1), lo, hi, ("slipWall", 2), ("slipWall", 2)]
    path = _write(work, name, c, [(s * x, s * y, s * z)], [_surfaces(n, n, n, types)], p, rho, u, states)
    return path, _free_stream([(n, n, n)], rng, rho, u, p)


def _channel_dims(c):
    cols = [c["ni"]] * 3 + [max(2, c["ni"] // 2)]
    rows = [c["nj"], max(2, c["nj"] // 2)]
    return cols, rows, [(cc, rr, c["nk"]) for rr in rows for cc in cols]


def _channel(work, c, rng):
    """the laminar channel of ``cases.channel_case``: 4 x 2 blocks, no-slip
    lower wall, wall-normal stretching 1.1, spanwise periodic, Mach 0.3,
    Re 1e6; uniform free stream with 1e-3 velocity perturbations"""
    cols, rows, dims = _channel_dims(c)
    nk = c["nk"]
    xs = np.linspace(0.0, 4.0, sum(cols) + 1)
    ys = np.concatenate([[0.0], np.cumsum(1.0e-5 * 1.1 ** np.arange(sum(rows)))])
    zs = np.linspace(0.0, 0.5, nk + 1)
    u = 0.3 * math.sqrt(GAMMA * cases.air_gas_constant() * T_INF)
    rho = 1.0e6 * (1.458e-6 * T_INF ** 1.5 / (T_INF + 110.4)) / u
    p = rho * cases.air_gas_constant() * T_INF
    x0, y0 = np.concatenate([[0], np.cumsum(cols)]), np.concatenate([[0], np.cumsum(rows)])
    blocks, surfaces = [], []
    for r in range(2):
        for q in range(4):
            blocks.append(np.meshgrid(xs[x0[q]:x0[q + 1] + 1], ys[y0[r]:y0[r + 1] + 1], zs, indexing="ij"))
            here = q + 4 * r
            surfaces.append(_surfaces(cols[q], rows[r], nk, [
                ("characteristic", 1) if q == 0 else ("interblock", 2000 + here - 1),
                ("characteristic", 1) if q == 3 else ("interblock", 1000 + here + 1),
                ("viscousWall", 3) if r == 0 else ("interblock", 4000 + q),
                ("characteristic", 1) if r == 1 else ("interblock", 3000 + q + 4),
                ("periodic", 7), ("periodic", 8)]))
    states = ", viscousWall(tag=3), periodic(startTag=7; endTag=8; translation=[0.0, 0.0, 0.5])"
    path = _write(work, "channel", c, blocks, surfaces, p, rho, u, states, "timeStep: 1.0e-5\n")
    return path, _free_stream(dims, rng, rho, u, p)


def _scaled(info, fields):
    """SI fields as the library takes them (nondimensional primitives)"""
    r, a = info.r_ref, info.a_ref
    scale = np.array([1.0 / r, 1.0 / a, 1.0 / a, 1.0 / a, 1.0 / (r * a * a)])
    return [np.ascontiguousarray(W * scale) for W in fields]


def _serve_sizes(c):
    """`nk` request sizes from ni^3 to nj^3"""
    m = c["nk"]
    return [c["ni"] + ((c["nj"] - c["ni"]) * q) // max(1, m - 1) for q in range(m)]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    fp32 = case["precision"] == "fp32"
    with tempfile.TemporaryDirectory() as work:
        if case["kind"] == "serve":
            srv = Server(max_slots=64, precision=1 if fp32 else 0)
            slots = []
            for q, n in enumerate(_serve_sizes(case)):
                path, _ = _bump(work, case, rng, n, name=f"r{q}")
                slots.append(srv.admit(path, 1.0e-200, 2 ** 30))
            return {"case": case, "server": srv, "slots": slots}
        make = {"box": _box, "channel": _channel}.get(case["kind"])
        path, fields = make(work, case, rng) if make else _bump(work, case, rng, case["ni"])
        solver = Solver(path)
    if fp32 and case["time"] != "explicitEuler":
        solver.set_implicit_precision(Solver.FP32)
    fields = _scaled(solver.info, fields)
    for b, W in enumerate(fields):
        solver.set_state(W, b)
    if case["calls"] == "run":
        solver.run(0, 0)  # captures the iteration, as a program does before its loop
    return {"case": case, "solver": solver, "fields": fields, "step": 0}


def _norms(n):
    return np.array(list(n.l2[:5]) + [n.linf, n.matrix_resid])


def run(state):
    case = state["case"]
    if case["calls"] == "serve":
        srv = state["server"]
        srv.step(case["steps"])
        return [srv.state(s) for s in state["slots"]]
    s = state["solver"]
    if case["calls"] == "run":
        for b, W in enumerate(state["fields"]):
            s.set_state(W, b)
        n = s.run(0, case["steps"])
    else:
        for nn in range(state["step"], state["step"] + case["steps"]):
            s.begin_step(nn)
            for mm in range(case["subits"]):
                n = s.iterate(nn, mm)
        state["step"] += case["steps"]
    return {"state": [s.get_state(b) for b in range(s.info.num_blocks)], "norms": _norms(n)}


def cells(case):
    if case["kind"] == "channel":
        return sum(i * j * k for i, j, k in _channel_dims(case)[2])
    if case["kind"] == "serve":
        return sum(n ** 3 for n in _serve_sizes(case))
    return case["ni"] * case["nj"] * case["nk"]


def work(case):
    """Per cell and nonlinear iteration.  Bytes: the state (5 doubles) and the
    cell's metrics (three face vectors of 4 doubles, volume, widths: 16
    doubles) once for the residual and once for every pass of the implicit
    solver, the old time levels, the update vector written by each pass and
    read by the next pass and the state update, the new state.  Operations:
    three faces of reconstruction and flux, and the implicit products."""
    explicit = case["time"] == "explicitEuler"
    block = case["solver"] in ("blusgs", "bdplur")
    passes = 0 if explicit else case["sweeps"] * (1 if "dplur" in case["solver"] else 2)
    du = 4 if case["precision"] == "fp32" else 8
    old = 0 if explicit else (80 if case["time"] == "bdf2" else 40)
    nbytes = (1 + passes) * 168 + old + passes * 10 * du + 40
    if case["viscous"]:
        nbytes += 48  # the centre distances of three faces, for the residual and the operator
    flops = {"thirdOrder": 900, "constant": 500}.get(case["recon"], 6000) + (900 if case["viscous"] else 0)
    flops += passes * (600 if block else 350) + (700 if block and not explicit else 0)
    n = cells(case) * case["steps"] * case["subits"]
    return {"bytes": float(nbytes * n), "flops": float(flops * n)}


def exact(case, seed):
    return None
