"""What users of this framework have it do, as timed cases.

A case is a dict of plain values; `prepare` makes what a program holds before the call (a
domain on the GPU with its fields, or host arrays), `run` is one pass through the public
entry points.  Seven kinds of work:

  step      momentum_FC3 time steps of one two-phase wave tank (3-D, or 2-D x-z with ny = 1),
            FP64 or mixed-precision projection, with or without viscous terms (D20)
  vortex    level-set benchmark steps in the unit cube (transport, reinit, void momentum)
  reini     the initial reinitialisation of a distorted level set, on stretched nodes
  solve     one pressure Poisson solve on the tank's variable-density operator
  operator  the same solve on a matrix and right-hand side that the caller holds on the host
            (the drop-in use of solver::start)
  batch     many uneven 2-D tanks, stepped together by the iteration-level scheduler
  serve     a stream of tank requests through the server, host arrays in and out

Tanks are those of reef3d_amd.cases: still-water depth 0.6 of the height, linear waves with
amplitude 1 to 10 % of the depth and wave lengths of 1 to 4 m, cells of 1 to 5 cm, a time
step of a quarter cell per wave speed, the projection solved to 1e-10 of its first residual.
The seed gives the amplitude and the wave length (and the solution of `solve`, `operator`).
"""
import math

import numpy as np

from reef3d_amd import Batch, Domain, Server
from reef3d_amd import cases as tanks

RHO = (1000.0, 1.205)
RTOL, MAXITER = 1e-10, 20000
TANK_FIELDS = ("phi", "u", "v", "w", "press")
# iterations of one solve to 1e-10 that the work of a case is counted with (300 to 450 on the
# large 3-D tank)
ITERS = 370


def listed():
    return [
        # the benchmark tank: the largest single domain, FP64 as the reference solves it
        dict(name="tank_512x64x128", kind="step", nx=512, ny=64, nz=128, dx=0.02, precision="fp64", graphs=True,
             D20=0, steps=2, restart=False),
        # an ordinary 3-D tank of the served stream, mixed precision
        dict(name="tank_224x40x96_mixed", kind="step", nx=224, ny=40, nz=96, dx=0.03, precision="mixed", graphs=True,
             D20=0, steps=2, restart=True),
        # a 2-D tank of the batched workload run alone: ragged width, launch by launch
        dict(name="tank_1150x157_2d", kind="step", nx=1150, ny=1, nz=157, dx=0.02, precision="fp64", graphs=False,
             D20=0, steps=1, restart=True),
        # the smallest tank (set-up checks, teaching cases): latency only
        dict(name="tank_40x8x24", kind="step", nx=40, ny=8, nz=24, dx=0.05, precision="fp64", graphs=False, D20=0,
             steps=4, restart=True),
        # a viscous tank with the implicit diffusion solves of each velocity component
        dict(name="tank_96x24x48_viscous", kind="step", nx=96, ny=24, nz=48, dx=0.04, precision="fp64", graphs=False,
             D20=2, steps=2, restart=True),
        # the level-set benchmark at its published size
        dict(name="vortex_128", kind="vortex", n=128, steps=64),
        # the initial reinitialisation of a run, vertically stretched, odd sizes
        dict(name="reini_203x45x97", kind="reini", nx=203, ny=45, nz=97, dx=0.02, stretch=1.4, F49=1),
        # pressure solves: an odd mid-sized 3-D tank in FP64, the benchmark tank in mixed precision
        dict(name="solve_193x37x101", kind="solve", nx=193, ny=37, nz=101, dx=0.02, precision="fp64", graphs=False),
        dict(name="solve_512x64x128_mixed", kind="solve", nx=512, ny=64, nz=128, dx=0.02, precision="mixed",
             graphs=True),
        # the reference's own solver call with its matrix on the host
        dict(name="operator_320x96_2d", kind="operator", nx=320, ny=1, nz=96, dx=0.02),
        # uneven 2-D tanks in one batch, graph replay, mixed precision
        dict(name="batch_8_2d", kind="batch", tanks=8, nx=256, nz=64, dx=0.02, precision="mixed", graphs=True, steps=1),
        # requests through the server, 2-D and one 3-D
        dict(name="serve_6", kind="serve", requests=6, nx=256, nz=64, dx=0.03, precision="mixed", steps=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step3", "step3", "step2", "step2", "vortex", "reini", "solve3", "solve2", "operator", "batch",
                       "serve"])
    dx = round(rng.uniform(0.01, 0.05), 4)
    precision = rng.choice(["fp64", "mixed"])
    graphs = rng.random() < 0.5
    if kind == "step3":
        return dict(kind="step", nx=_log(rng, 32, 320), ny=_log(rng, 5, 64), nz=_log(rng, 16, 128), dx=dx,
                    precision=precision, graphs=graphs, D20=rng.choice([0, 0, 0, 1, 2]), steps=1, restart=True)
    if kind == "step2":
        return dict(kind="step", nx=_log(rng, 128, 2048), ny=1, nz=_log(rng, 32, 256), dx=dx, precision=precision,
                    graphs=graphs, D20=rng.choice([0, 0, 0, 1, 2]), steps=1, restart=True)
    if kind == "vortex":
        return dict(kind="vortex", n=_log(rng, 24, 140), steps=32)
    if kind == "reini":
        return dict(kind="reini", nx=_log(rng, 48, 320), ny=_log(rng, 8, 64), nz=_log(rng, 24, 128), dx=dx,
                    stretch=round(rng.uniform(1.0, 1.6), 3), F49=rng.choice([1, 0]))
    if kind == "solve3":
        return dict(kind="solve", nx=_log(rng, 48, 512), ny=_log(rng, 8, 64), nz=_log(rng, 24, 128), dx=dx,
                    precision=precision, graphs=graphs)
    if kind == "solve2":
        return dict(kind="solve", nx=_log(rng, 128, 2048), ny=1, nz=_log(rng, 32, 256), dx=dx, precision=precision,
                    graphs=graphs)
    if kind == "operator":
        if rng.random() < 0.5:
            return dict(kind="operator", nx=_log(rng, 64, 512), ny=1, nz=_log(rng, 32, 128), dx=dx)
        return dict(kind="operator", nx=_log(rng, 24, 128), ny=_log(rng, 5, 32), nz=_log(rng, 16, 64), dx=dx)
    if kind == "batch":
        return dict(kind="batch", tanks=rng.randint(2, 10), nx=_log(rng, 128, 400), nz=_log(rng, 32, 96), dx=dx,
                    precision=precision, graphs=graphs, steps=1)
    return dict(kind="serve", requests=rng.randint(2, 8), nx=_log(rng, 96, 300), nz=_log(rng, 32, 80), dx=dx,
                precision=precision, steps=1)


# ------------------------------------------------------------------ inputs
def _spec(nx, ny, nz, dx, rng):
    depth = 0.6 * nz * dx
    return dict(nx=nx, ny=ny, nz=nz, jdir=0 if ny == 1 else 1, dx=dx, depth=depth,
                amp=float(rng.uniform(0.01, 0.1)) * depth, wavelength=float(rng.uniform(1.0, 4.0)))


def _load(D, f):
    """The initial state of a run: fields, ghost layers, density and viscosity."""
    for n in TANK_FIELDS:
        D.put(n, f[n])
    D.start4("phi", 52)
    D.start1("u", 10)
    D.start2("v", 11)
    D.start3("w", 12)
    D.start4("press", 40)
    D.fluid_update()


def _tank_domain(case, spec, f):
    D20 = case.get("D20", 0)
    D = Domain(**tanks.tank_kwargs(spec, f, RTOL, MAXITER), D20=D20,
               visc=(0.01, 0.002) if D20 else (1.0e-6, 1.4938e-5))
    if case["precision"] == "mixed":
        D.solver_config("mixed")
    if case["graphs"]:
        D.set_control("graphs", 1)
    return D


def _sizes(case, count):
    """The uneven 2-D tanks of a batch or a stream: 1 to 4 times the case's width, 1 to 2.5
    times its height, odd ones among them."""
    return [(case["nx"] * (1 + (5 * q) % 4) + q, 1, case["nz"] * (2 + (3 * q) % 4) // 2 + q % 3) for q in range(count)]


def _interior(a):
    return a[3:-3, 3:-3, 3:-3]


def _couplings(spec, phi):
    """The six couplings (+x, -x, +y, -y, +z, -z) of the projection's operator on a uniform
    grid: 1 / (face density * dx^2), the face density from the smoothed Heaviside function of
    the mean phi of the two cells."""
    psi, dx2 = 2.1 * spec["dx"], spec["dx"] ** 2

    def face(axis, side):
        nb = np.roll(phi, -side, axis)
        m = _interior(0.5 * (phi + nb))
        H = np.where(m > psi, 1.0, np.where(m < -psi, 0.0, 0.5 * (1.0 + m / psi + np.sin(math.pi * m / psi) / math.pi)))
        return 1.0 / ((RHO[0] * H + RHO[1] * (1.0 - H)) * dx2)
    T = [face(2, 1), face(2, -1), face(1, 1), face(1, -1), face(0, 1), face(0, -1)]
    if spec["jdir"] == 0:
        T[2] = T[3] = np.zeros_like(T[0])
    return T


def _solution(spec, seed):
    """A pressure correction: a few smooth modes and some cell noise, interior shape (z, y, x)."""
    rng = np.random.default_rng([seed, 7])
    x = (np.arange(spec["nx"]) + 0.5) / spec["nx"]
    y = (np.arange(spec["ny"]) + 0.5) / spec["ny"]
    z = (np.arange(spec["nz"]) + 0.5) / spec["nz"]
    p = np.zeros((spec["nz"], spec["ny"], spec["nx"]))
    for _ in range(4):
        a, b, c = rng.integers(1, 6, 3)
        my = np.sin(math.pi * b * y) if spec["jdir"] else np.ones(1)
        p += rng.standard_normal() * (np.sin(math.pi * c * z)[:, None, None] * my[None, :, None]
                                      * np.sin(math.pi * a * x)[None, None, :])
    return 100.0 * (p + 0.01 * rng.standard_normal(p.shape))


def _apply(T, p):
    out = sum(T) * p
    out[:, :, :-1] -= T[0][:, :, :-1] * p[:, :, 1:]
    out[:, :, 1:] -= T[1][:, :, 1:] * p[:, :, :-1]
    out[:, :-1] -= T[2][:, :-1] * p[:, 1:]
    out[:, 1:] -= T[3][:, 1:] * p[:, :-1]
    out[:-1] -= T[4][:-1] * p[1:]
    out[1:] -= T[5][1:] * p[:-1]
    return out


def _rows(T):
    """M.p, M.n, M.s, M.w, M.e, M.t, M.b of matrix_diag in vec order (i outermost, k
    innermost); couplings out of the domain are folded away, the diagonal keeps them."""
    off = [-t for t in T]
    off[0][:, :, -1] = 0.0
    off[1][:, :, 0] = 0.0
    off[2][:, -1] = 0.0
    off[3][:, 0] = 0.0
    off[4][-1] = 0.0
    off[5][0] = 0.0
    n, s, w, e, t, b = off
    return [np.ascontiguousarray(a.transpose(2, 1, 0)).ravel() for a in (sum(T), n, s, w, e, t, b)]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "vortex":
        n = case["n"]
        f = tanks.vortex3d(n)
        # the benchmark's sphere, moved by up to a cell
        x = [0.5 * (f["XN"][:-1] + f["XN"][1:])[2:2 + n + 6] - 0.35 + float(rng.uniform(-1, 1)) / n for _ in range(3)]
        f["phi"] = 0.15 - np.sqrt(x[0][None, None, :] ** 2 + x[1][None, :, None] ** 2 + x[2][:, None, None] ** 2)
        dt = 0.25 / n
        D = Domain(n, n, n, f["XN"], f["YN"], f["ZN"], 1.0 / n, 1.0 / n, dt=dt)
        return dict(case=case, D=D, f=f, dt=dt)
    if kind == "reini":
        nx, ny, nz, dx = case["nx"], case["ny"], case["nz"], case["dx"]
        f = tanks.wave_tank(nx, ny, nz, dx, 0.6 * nz * dx, float(rng.uniform(0.02, 0.06)) * nz * dx,
                            float(rng.uniform(1.0, 4.0)))
        # nodes that widen away from the still-water level by up to `stretch`
        k = np.arange(-5, nz + 6)
        d = dx * (1.0 + (case["stretch"] - 1.0) * np.abs(k[:-1] + 0.5 - 0.6 * nz) / (0.6 * nz))
        ZN = np.concatenate([[0.0], np.cumsum(d)])
        ZN -= ZN[5]
        # a level set with the wave's interface and gradients between 0.5 and 2
        phi = f["phi"] * (1.0 + 0.5 * np.tanh(f["phi"] / (4.0 * dx))) * float(rng.uniform(0.8, 1.2))
        D = Domain(nx, ny, nz, f["XN"], f["YN"], ZN, dx, float(d.mean()), top_group=3, g=(0.0, 0.0, -9.81),
                   F49=case["F49"])
        return dict(case=case, D=D, phi=phi, maxlength=max(nx, ny, nz) * dx)
    if kind in ("step", "solve", "operator"):
        spec = _spec(case["nx"], case["ny"], case["nz"], case["dx"], rng)
        f = tanks.tank_fields(spec)
        if kind == "step":
            D = _tank_domain(case, spec, f)
            _load(D, f)
            D.sync()
            return dict(case=case, D=D, f=f if case["restart"] else None)
        T = _couplings(spec, f["phi"])
        b = _apply(T, _solution(spec, seed))
        if kind == "operator":
            D = Domain(**tanks.tank_kwargs(spec, f, RTOL, MAXITER))
            return dict(case=case, D=D, M=_rows(T), b=np.ascontiguousarray(b.transpose(2, 1, 0)).ravel())
        D = _tank_domain(case, spec, f)
        D.put("phi", f["phi"])
        rhs = np.zeros(D.shape)
        _interior(rhs)[...] = b
        D.put("work1", rhs)
        D.sync()
        return dict(case=case, D=D)
    specs = [_spec(*s, case["dx"], rng) for s in _sizes(case, case["tanks" if kind == "batch" else "requests"])]
    if kind == "batch":
        B, ids, fields = Batch(), [], []
        for sp in specs:
            f = tanks.tank_fields(sp)
            ids.append(B.add(**tanks.tank_kwargs(sp, f, RTOL, MAXITER)))
            fields.append(f)
        B.solver_config(case["precision"])
        B.set_control("graphs", 1 if case["graphs"] else 0)
        return dict(case=case, B=B, ids=ids, fields=fields)
    # a stream: the last request is a small 3-D tank
    specs[-1] = _spec(case["nx"] // 2, max(4, case["nz"] // 4), case["nz"], case["dx"], rng)
    S = Server(precision=case["precision"], N44=-RTOL, N46=MAXITER)
    return dict(case=case, S=S, specs=specs, fields=[tanks.tank_fields(sp) for sp in specs])


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        D = state["D"]
        if state["f"] is not None:
            _load(D, state["f"])
        for _ in range(case["steps"]):
            _, vol = D.momentum_fc3()
        out = {n: D.get(n) for n in TANK_FIELDS if n != "v" or case["ny"] > 1}
        return dict(out, volumes=vol)
    if kind == "vortex":
        D, t = state["D"], 0.0
        D.put("phi", state["f"]["phi"])
        for n in ("u", "v", "w"):
            D.zero(n)
        D.start4("phi", 52)
        for _ in range(case["steps"]):
            D.vortex_step(t, volumes=False)
            t += state["dt"]
        return D.get("phi")
    if kind == "reini":
        D = state["D"]
        D.put("phi", state["phi"])
        D.reini_ini("phi", maxlength=state["maxlength"], F43=0.55, DXM=case["dx"])
        return D.get("phi")
    if kind == "solve":
        D = state["D"]
        D.zero("work0")
        (D.solver if case["precision"] == "fp64" else D.solver_mixed)("work0", "work1", -RTOL, MAXITER)
        return _interior(D.get("work0"))
    if kind == "operator":
        D = state["D"]
        D.zero("work0")
        D.solver_start(5, state["M"], state["b"], "work0", -RTOL, MAXITER)
        return _interior(D.get("work0"))
    if kind == "batch":
        B = state["B"]
        for tid, f in zip(state["ids"], state["fields"]):
            for n in TANK_FIELDS:
                B.put(tid, n, f[n])
        for n, k, gcv in (("phi", 4, 52), ("u", 1, 10), ("v", 2, 11), ("w", 3, 12), ("press", 4, 40)):
            B.ghost_fill(n, k, gcv)
        B.fluid_update()
        B.run(case["steps"])
        return [{n: B.get(t, n) for n in ("phi", "u", "w", "press")} for t in state["ids"]]
    S = state["S"]
    ids = []
    for sp, f in zip(state["specs"], state["fields"]):
        ids.append(S.submit(sp["nx"], sp["ny"], sp["nz"], f["XN"], f["YN"], f["ZN"], sp["dx"], sp["dx"], f["dt"],
                            case["steps"], *(f[n] for n in TANK_FIELDS), jdir=sp["jdir"], top_group=3))
    out = []
    for r in ids:
        if S.wait(r) != "done":
            raise RuntimeError("a served request failed")
        out.append({n: S.result(r, n) for n in ("phi", "u", "w", "press")})
        S.release(r)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _solve_bytes(cells, precision, iters=ITERS):
    """BiCGStab with its vectors in memory: per iteration r, p, v, r0 in and p, v out; r, v in
    and t out; x, p, r, v, t, r0 in and x, r out."""
    return cells * iters * 17 * (8 if precision == "fp64" else 4)


def _step_bytes(cells, precision, steps, jdir):
    """Per step: level-set transport 136, nine reinit iterations of 64, the predictors 184
    (120 in 2-D) a stage, right-hand side and correction 112 a stage, fluid update 24 bytes a
    cell, and three solves."""
    stage = (184 if jdir else 120) + 112
    return steps * (cells * (136 + 9 * 64 + 3 * stage + 24) + 3 * _solve_bytes(cells, precision))


def work(case):
    kind = case["kind"]
    if kind == "vortex":
        cells = case["n"] ** 3
        # transport 40 + 48 + 48, three reinit iterations of 64, velocity writes and updates 72
        return dict(bytes=float(cells * case["steps"] * (136 + 192 + 72)), flops=float(cells * case["steps"] * 7500))
    if kind == "reini":
        cells = case["nx"] * case["ny"] * case["nz"]
        it = 2 * int(max(case["nx"], case["ny"], case["nz"]) / 0.55)
        return dict(bytes=float(cells * it * 64), flops=float(cells * it * 3 * 600))
    if kind == "step":
        cells = case["nx"] * case["ny"] * case["nz"]
        b = _step_bytes(cells, case["precision"], case["steps"], case["ny"] > 1)
        return dict(bytes=float(b), flops=float(cells * case["steps"] * (27 * 600 + 3 * ITERS * 60)))
    if kind in ("solve", "operator"):
        cells = case["nx"] * case["ny"] * case["nz"]
        extra = 64 * cells if kind == "operator" else 0
        return dict(bytes=float(_solve_bytes(cells, case.get("precision", "fp64")) + extra), flops=float(cells * ITERS * 60))
    sizes = _sizes(case, case["tanks" if kind == "batch" else "requests"])
    if kind == "serve":
        sizes[-1] = (case["nx"] // 2, max(4, case["nz"] // 4), case["nz"])
    cells = sum(a * b * c for a, b, c in sizes)
    return dict(bytes=float(_step_bytes(cells, case["precision"], case["steps"], 0)),
                flops=float(cells * case["steps"] * (27 * 600 + 3 * ITERS * 60)))


def exact(case, seed):
    """The solution the right-hand side of a solve was made from.  Time steps and
    reinitialisations have none: an independent 64-bit oracle of a whole step runs for
    minutes, and the reinitialisation picks one-sided differences by comparing nearly equal
    values, so it has no value that is exact beyond those choices."""
    if case["kind"] not in ("solve", "operator"):
        return None
    rng = np.random.default_rng(seed)
    return _solution(_spec(case["nx"], case["ny"], case["nz"], case["dx"], rng), seed)
