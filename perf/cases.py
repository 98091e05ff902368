"""The work that programs have this framework do, as cases to time and compare.

A case is one pass through the public entry points of euler2d_cudafortran_amd:
a batch of time steps on a run or on a caller's own buffers, the host-driven
loop, one adjoint step, or the gradient of a rollout.  Inputs are made on the
GPU from a seed: the diagonal discontinuity with 16 Gaussian bumps in density
and pressure and a smooth velocity field, which gives shocks, contacts,
rarefactions and smooth flow at once.  `exact` restates the scheme
(pkestene/euler2d_cudaFortran, serial_ref/m_run.f90 and m_utils.f90) in plain
torch in 64 bits, the gradients by torch's own reverse mode.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import euler2d_cudafortran_amd as e2d
from euler2d_cudafortran_amd.autograd import GodunovRollout, interior_mask, record_dts

GAMMA, CFL, SMALLR, SMALLC, NITER = 1.4, 0.8, 1e-7, 1e-7, 10
FP32_STATE = ("fp32", "fp32_native")  # 4 bytes per stored value; fp64 and mixed store 8


def listed():
    return [
        # A serving loop that owns its buffers, at the 128^2 grid of the reference's parameter
        # file: the smallest call, where launches and one wavefront's latency are the time.
        _case("noalloc_128_fp64", "noalloc", 128, 128, "fp64", 20),
        # The reference's own main loop (dt on the host every step) on a small ragged grid with
        # three kinds of boundary.
        _case("loop_250x130_fp64", "loop", 250, 130, "fp64", 10, bc="1231"),
        # A run of ordinary size on an odd grid in the reference's default precision, periodic,
        # with the sharper limiter.
        _case("steps_1000x610_fp32_mc", "steps", 1000, 610, "fp32", 10, bc="3333", slope=2),
        # The headline workload: 2048^2 FP64, the fused step, walls.
        _case("steps_2048_fp64", "steps", 2048, 2048, "fp64", 10),
        # The same in FP32, the headline's other side.
        _case("steps_2048_fp32", "steps", 2048, 2048, "fp32", 10),
        # The precision variant at its configured size, the largest grid: FP64 state and update,
        # FP32 flux arithmetic.
        _case("steps_4096_mixed", "steps", 4096, 4096, "mixed", 6),
        # The quickest variant on a large odd grid with open boundaries.
        _case("steps_3001x1537_fp32_native", "steps", 3001, 1537, "fp32_native", 6, bc="2222"),
        # implementationVersion 1 at the headline size: every stage stored, to be looked at.
        _case("materialised_2048_fp64", "steps", 2048, 2048, "fp64", 4, impl=1),
        # implementationVersion 2, the reference's default version, on a ragged grid.
        _case("flux_store_1500x1100_fp64", "steps", 1500, 1100, "fp64", 6, impl=2, bc="1122"),
        # One adjoint step with a dense adjoint field at the headline size.
        _case("adjoint_step_2048_fp64", "adjoint_step", 2048, 2048, "fp64", 1),
        # The gradient of a misfit through the torch harness at the 512^2 configuration's size
        # (recorded forward, checkpointed reverse sweep), with fewer steps.
        _case("gradient_512_fp64", "gradient", 512, 512, "fp64", 60, nsnap=6),
        # The checkpointed reverse sweep in FP32 at the large rollout's grid, with fewer steps.
        _case("rollout_2048_fp32", "rollout", 2048, 2048, "fp32", 16, nsnap=6),
    ]


def _case(name, kind, nx, ny, precision, steps, impl=0, bc="1111", slope=1, nsnap=0):
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "precision": precision, "steps": steps, "impl": impl,
            "bc": bc, "slope": slope, "nsnap": nsnap}


def draw(rng):
    """Grids from 64 to 4096 cells a side (half of them up to 4 times as wide as high or the
    other way round), every precision, version, boundary kind and limiter that the listed cases
    stand for; the steps are as many as keep the pass below the largest listed case."""
    kind = rng.choice(["noalloc", "loop", "steps", "steps", "steps", "steps", "adjoint_step", "gradient", "rollout"])
    largest = 4096 if kind in ("noalloc", "steps") else (2048 if kind in ("adjoint_step", "loop") else 1024)
    n = math.exp(rng.uniform(math.log(64), math.log(largest)))
    aspect = math.exp(rng.uniform(-math.log(2), math.log(2))) if rng.random() < 0.5 else 1.0
    nx, ny = (max(48, min(largest, int(n * a))) for a in (aspect, 1 / aspect))
    if rng.random() < 0.25:  # powers of two are common grids
        nx = ny = 2 ** min(int(math.log2(largest)), max(6, round(math.log2(n))))
    precision = "fp64" if kind == "gradient" else rng.choice(["fp64", "fp64", "fp32", "fp32_native", "mixed"])
    impl = rng.choice([0, 0, 1, 2]) if kind == "steps" else 0
    bc = rng.choice(["1111", "1111", "2222", "3333", "".join(rng.choice("123") for _ in range(4))])
    slope = rng.choice([1, 1, 2])
    cells = nx * ny
    if kind == "adjoint_step":
        steps = 1
    elif kind in ("gradient", "rollout"):
        steps = max(2, min(rng.randrange(10, 40), 8_000_000 // cells))
    else:
        most = (8_000_000 if impl else 40_000_000) // cells
        steps = max(2, min(rng.randrange(4, 30), most))
    nsnap = rng.randrange(3, 9) if kind in ("gradient", "rollout") else 0
    case = _case("", kind, nx, ny, precision, steps, impl, bc, slope, nsnap)
    del case["name"]
    return case


# ---------------------------------------------------------------------------
# what a program has in hand, and the pass

def prepare(case, seed):
    nx, ny = case["nx"], case["ny"]
    p = e2d.HydroParams(nx=nx, ny=ny, gamma0=GAMMA, cfl=CFL, smallr=SMALLR, smallc=SMALLC, niter_riemann=NITER,
                        slope_type=case["slope"], implementation_version=case["impl"],
                        precision=e2d.PRECISIONS[case["precision"]])
    for side, kind in zip(("xmin", "xmax", "ymin", "ymax"), case["bc"]):
        setattr(p, "boundary_type_" + side, int(kind))
    u0 = _initial(case, seed)
    if case["kind"] == "noalloc":
        pitch = -(-(nx + 4) // 64) * 64
        u = _padded(u0, pitch)
        return {"params": p, "case": case, "n": 0, "pitch": pitch, "u": u, "u2": torch.zeros_like(u),
                "invdt": torch.zeros(1, dtype=torch.float64, device="cuda")}
    run = e2d.HydroRun(p)
    _, pitch = run.device_buffer(0)
    u = _padded(u0, pitch)
    torch.cuda.synchronize()
    run.copy_to_buffer(0, u.data_ptr())
    run.make_boundaries(0)
    state = {"run": run, "case": case}
    if case["kind"] in ("steps", "loop"):
        state["out"] = [_buffer(run, b)[:, :, :nx + 4] for b in (0, 1)]
        return state
    if case["kind"] == "adjoint_step":
        lam = _padded(_field(case, seed, dense=True), pitch)
        state.update(dt=run.compute_dt(0), lam=lam, out=torch.zeros_like(lam))
        torch.cuda.synchronize()
        return state
    if case["kind"] == "gradient":
        state["dts"] = record_dts(run, u, case["steps"])
        state.update(u0=u.requires_grad_(True), inner=interior_mask(run, u)[0],
                     target=_padded(_target(case, seed), pitch))
        return state
    # rollout: the frozen dt sequence of a forward run
    dts = []
    for n in range(case["steps"]):
        dts.append(run.compute_dt(n % 2))
        run.godunov_unsplit(n, dts[-1])
    run.synchronize()
    lam = _padded(_field(case, seed, dense=False), pitch)
    state.update(dts=dts, u0=u, lam=lam, out=torch.zeros_like(lam))
    torch.cuda.synchronize()
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "noalloc":
        u, u2 = state["u"], state["u2"]
        e2d.run_steps_noalloc(state["params"], u.data_ptr(), u2.data_ptr(), state["pitch"], case["steps"], state["n"],
                              state["invdt"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        state["n"] += case["steps"]
        return {"u": u[:, :, :case["nx"] + 4], "u2": u2[:, :, :case["nx"] + 4], "invdt": state["invdt"]}
    r = state["run"]
    if kind == "steps":
        # a batch of steps, then the conservation sums and the next dt, which programs log
        r.run_steps(case["steps"])
        sums = r.sums(r.current())
        return {"u": state["out"][0], "u2": state["out"][1], "sums": sums, "dt": r.get_dt()}
    if kind == "loop":
        dts = []
        for _ in range(case["steps"]):
            dts.append(r.compute_dt(r.nStep % 2))
            r.godunov_unsplit(r.nStep, dts[-1])
            r.nStep += 1
        return {"u": state["out"][0], "u2": state["out"][1], "sums": r.sums(r.current()),
                "dts": np.array(dts, dtype=np.float64)}
    if kind == "adjoint_step":
        r.adjoint_step(0, state["dt"], state["lam"].data_ptr(), state["out"].data_ptr())
        r.synchronize()
        return {"lam": state["out"][:, :, :case["nx"] + 4]}
    if kind == "gradient":
        u_n = GodunovRollout.apply(state["u0"], r, state["dts"], case["nsnap"])
        misfit = torch.where(state["inner"], (u_n[0] - state["target"]) ** 2, 0.0).sum()
        (grad,) = torch.autograd.grad(misfit, state["u0"])
        return {"misfit": misfit.detach(), "grad": grad[:, :, :case["nx"] + 4]}
    r.copy_to_buffer(0, state["u0"].data_ptr())
    r.adjoint_rollout(0, state["dts"], case["nsnap"], state["lam"].data_ptr(), state["out"].data_ptr())
    return {"lam": state["out"][:, :, :case["nx"] + 4]}


def work(case):
    """Bytes: the 4 conserved variables read and written once per cell and step; version 1 also
    writes its 9 stage arrays and version 2 its 3, which are what those versions are for; an
    adjoint step reads the state and the adjoint field (always 8 bytes a value) and writes the
    adjoint field.  Operations: those of the scheme, one Newton iteration per Riemann problem,
    a division or a square root counted as one."""
    cells, steps = case["nx"] * case["ny"], case["steps"]
    value = 4 if case["precision"] in FP32_STATE else 8
    stage = 4 if case["precision"] != "fp64" else 8
    forward = 4 * 2 * value
    if case["impl"] == 1:
        forward += 4 * 9 * stage
    elif case["impl"] == 2:
        forward += 4 * 3 * stage
    ops, adjoint, adjoint_ops = 440, 4 * (value + 16), 1100
    if case["kind"] == "adjoint_step":
        return {"bytes": cells * adjoint, "flops": cells * adjoint_ops}
    if case["kind"] in ("gradient", "rollout"):
        return {"bytes": cells * steps * (forward + adjoint), "flops": cells * steps * (ops + adjoint_ops)}
    return {"bytes": cells * steps * forward, "flops": cells * steps * ops}


def tolerance(case):
    """About four times what these paths differ by from the same scheme with its sums in another
    order (`exact`).  64 bits: the state 3e-16 and single cells more, where a Newton iteration
    stops one step earlier or later; an adjoint field 1e-15.  32 bits: the state 8e-8; an adjoint
    field 2e-4 to 8e-3, because a limiter or an upwind branch goes the other way in some cells,
    which it shows in full."""
    adjoint = case["kind"] in ("adjoint_step", "gradient", "rollout")
    if case["precision"] == "fp64":
        return {"rel": 1e-14, "max": 1e-10} if adjoint else {"rel": 2e-15, "max": 1e-11}
    if adjoint:
        return {"rel": 0.03, "max": 0.999}
    return {"rel": 4e-7, "max": 1e-3}


# ---------------------------------------------------------------------------
# inputs

class _Device:
    """A run's device buffer for torch: no copy; the run lives as long as the tensor."""

    def __init__(self, run, buf):
        self.run = run
        ptr, pitch = run.device_buffer(buf)
        double = run.params.precision in (e2d.PREC_FP64, e2d.PREC_MIXED)
        self.__cuda_array_interface__ = {"shape": (4, run.params.jsize, pitch), "typestr": "<f8" if double else "<f4",
                                         "data": (ptr, False), "version": 2}


def _buffer(run, buf):
    return torch.as_tensor(_Device(run, buf), device="cuda")


def _padded(a, pitch):
    out = torch.zeros((a.shape[0], a.shape[1], pitch) if a.dim() == 3 else (a.shape[0], pitch), dtype=a.dtype,
                      device=a.device)
    out[..., :a.shape[-1]] = a
    return out


def _centres(case):
    """Cell centres, ghost cells included, as a row of x and a column of y."""
    x = (torch.arange(case["nx"] + 4, dtype=torch.float64, device="cuda") - 1.5) / case["nx"]
    y = (torch.arange(case["ny"] + 4, dtype=torch.float64, device="cuda") - 1.5) / case["ny"]
    return x[None, :], y[:, None]


def _waves(rng, x, y, modes=3):
    f = torch.zeros((y.shape[0], x.shape[1]), dtype=torch.float64, device="cuda")
    for _ in range(modes):
        kx, ky = (int(k) for k in rng.integers(1, 4, 2))
        a, b, c = (float(v) for v in (rng.normal(), rng.uniform(), rng.uniform()))
        f += a * torch.sin(2 * math.pi * (kx * x + b)) * torch.cos(2 * math.pi * (ky * y + c))
    return f / modes


def _initial(case, seed):
    """(4, ny+4, nx+4) conserved variables rho, E, rho u, rho v in the storage type."""
    rng = np.random.default_rng([seed, 1])
    x, y = _centres(case)
    left = x + y < 1
    rho = torch.where(left, 1.0, 0.125).to(torch.float64)
    p = torch.where(left, 1.0, 0.1).to(torch.float64)
    for _ in range(16):  # amplitudes in [0.1, 2], widths in [0.02, 0.1]
        cx, cy, ar, ap, s = (float(v) for v in rng.uniform([0, 0, 0.1, 0.1, 0.02], [1, 1, 2, 2, 0.1]))
        w = torch.exp(-((x - cx) ** 2 + (y - cy) ** 2) / (2 * s * s))
        rho, p = rho + ar * w, p + ap * w
    u, v = 0.2 * _waves(rng, x, y), 0.2 * _waves(rng, x, y)
    a = torch.stack([rho, p / (GAMMA - 1) + 0.5 * rho * (u * u + v * v), rho * u, rho * v])
    return a.float() if case["precision"] in FP32_STATE else a


def _target(case, seed):
    x, y = _centres(case)
    return 1 + 0.3 * _waves(np.random.default_rng([seed, 2]), x, y)


def _field(case, seed, dense):
    """An adjoint field, zero on ghost cells: noise in every variable, or a smooth misfit of rho."""
    out = torch.zeros((4, case["ny"] + 4, case["nx"] + 4), dtype=torch.float64, device="cuda")
    if dense:
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        out[:, 2:-2, 2:-2] = torch.randn((4, case["ny"], case["nx"]), dtype=torch.float64, device="cuda", generator=g)
    else:
        x, y = _centres(case)
        out[0, 2:-2, 2:-2] = (1 + _waves(np.random.default_rng([seed, 3]), x, y))[2:-2, 2:-2]
    return out


# ---------------------------------------------------------------------------
# the scheme in plain torch, 64 bits; arrays are (variable, y, x), variables
# rho, p | E, u | rho u, v | rho v

SMALLP = SMALLC ** 2 / GAMMA
GAMMA6 = (GAMMA + 1) / (2 * GAMMA)
CONV_TOL = float(np.float32(1e-6))


def _ghosts(u, case):
    """Fills the ghost cells of u in place, corners left alone."""
    nx, ny, bc = case["nx"], case["ny"], case["bc"]
    for side in range(4):
        for k in range(2):
            n = nx if side < 2 else ny
            ghost = k if side % 2 == 0 else n + 2 + k
            if bc[side] == "1":
                source = 3 - k if side % 2 == 0 else n + 1 - k
            elif bc[side] == "2":
                source = 2 if side % 2 == 0 else n + 1
            else:
                source = n + k if side % 2 == 0 else 2 + k
            sign = torch.ones((4, 1), dtype=u.dtype, device=u.device)
            if bc[side] == "1":
                sign[2 if side < 2 else 3] = -1
            if side < 2:
                u[:, 2:-2, ghost] = sign * u[:, 2:-2, source].clone()
            else:
                u[:, ghost, 2:-2] = sign * u[:, source, 2:-2].clone()


def _larger(a, b):
    return torch.where(a > b, a, b)


def _size(a):
    return torch.where(a >= 0, a, -a)


def _primitive(u):
    rho = _larger(u[0], torch.full_like(u[0], SMALLR))
    vx, vy = u[2] / rho, u[3] / rho
    p = (GAMMA - 1) * rho * (u[1] / rho - 0.5 * (vx * vx + vy * vy))
    return torch.stack([rho, _larger(p, rho * SMALLP), vx, vy])


def _slope(minus, centre, plus, slope_type):
    dl, dr, dc = slope_type * (centre - minus), slope_type * (plus - centre), 0.5 * (plus - minus)
    lim = torch.where(_size(dl) < _size(dr), _size(dl), _size(dr))
    lim = torch.where(dl * dr <= 0, torch.zeros_like(lim), lim)
    lim = torch.where(lim < _size(dc), lim, _size(dc))
    return torch.where(dc >= 0, lim, -lim)


def _riemann(l, r, normal):
    """Flux of the two-shock solver's state at x/t = 0; l, r (4, ...) primitive, `normal` 2 or 3."""
    t = 5 - normal
    rl, rr = (_larger(s[0], torch.full_like(s[0], SMALLR)) for s in (l, r))
    pl, pr = _larger(l[1], rl * SMALLP), _larger(r[1], rr * SMALLP)
    ul, ur = l[normal], r[normal]
    cl, cr = GAMMA * pl * rl, GAMMA * pr * rr
    wl, wr = torch.sqrt(cl), torch.sqrt(cr)
    p = (wr * pl + wl * pr + wl * wr * (ul - ur)) / (wl + wr)
    p = _larger(p, torch.zeros_like(p))
    more = torch.ones_like(p, dtype=torch.bool)
    for _ in range(NITER):
        wwl = torch.sqrt(cl * (1 + GAMMA6 * (p - pl) / pl))
        wwr = torch.sqrt(cr * (1 + GAMMA6 * (p - pr) / pr))
        zl, zr = 2 * wwl ** 3 / (wwl * wwl + cl), 2 * wwr ** 3 / (wwr * wwr + cr)
        usl, usr = ul - (p - pl) / wwl, ur + (p - pr) / wwr
        delp = _larger(zr * zl / (zr + zl) * (usl - usr), -p)
        new = p + delp
        p, more = torch.where(more, new, p), more & (_size(delp / (new + SMALLR * SMALLP)) > CONV_TOL)
        if not bool(more.any()):
            break
    wl = torch.sqrt(cl * (1 + GAMMA6 * (p - pl) / pl))
    wr = torch.sqrt(cr * (1 + GAMMA6 * (p - pr) / pr))
    us = 0.5 * (ul + (pl - p) / wl + ur - (pr - p) / wr)
    right = us >= 0
    sign = torch.where(right, 1.0, -1.0).to(p.dtype)
    ro, uo, po, wo = (torch.where(right, a, b) for a, b in ((rl, rr), (ul, ur), (pl, pr), (wl, wr)))
    small = torch.full_like(p, SMALLC)
    co = _larger(torch.sqrt(_size(GAMMA * po / ro)), small)
    rs = _larger(ro / (1 + ro * (po - p) / (wo * wo)), torch.full_like(p, SMALLR))
    cs = _larger(torch.sqrt(_size(GAMMA * p / rs)), small)
    spout, spin, shock = co - sign * uo, cs - sign * us, wo / ro - sign * uo
    spout, spin = (torch.where(p >= po, shock, s) for s in (spout, spin))
    frac = 0.5 * (1 + (spout + spin) / _larger(spout - spin, SMALLC + _size(spout + spin)))
    g = [frac * a + (1 - frac) * b for a, b in ((rs, ro), (p, po), (us, uo))]
    g = [torch.where(spout < 0, b, a) for a, b in zip(g, (ro, po, uo))]
    rho, p, un = (torch.where(spin > 0, b, a) for a, b in zip(g, (rs, p, us)))
    ut = torch.where(right, l[t], r[t])
    mass = rho * un
    energy = p / (GAMMA - 1) + 0.5 * rho * (un * un + ut * ut)
    f = [mass, un * (energy + p), None, None]
    f[normal], f[t] = mass * un + p, mass * ut
    return torch.stack(f)


def _step(u, dt, case):
    """New interior (4, ny, nx) of the filled state u."""
    nx, ny, st = case["nx"], case["ny"], case["slope"]
    dtdx, dtdy = dt * nx, dt * ny
    q = _primitive(u)
    c = q[:, 1:-1, 1:-1]
    dx = _slope(q[:, 1:-1, :-2], c, q[:, 1:-1, 2:], st)
    dy = _slope(q[:, :-2, 1:-1], c, q[:, 2:, 1:-1], st)
    r, p, vx, vy = c
    div = dx[2] + dy[3]
    s = torch.stack([-vx * dx[0] - vy * dy[0] - div * r,
                     -vx * dx[1] - vy * dy[1] - div * GAMMA * p,
                     -vx * dx[2] - vy * dy[2] - dx[1] / r,
                     -vx * dx[3] - vy * dy[3] - dy[1] / r])

    def face(dq, dtd, side):
        f = c + side * 0.5 * dq + 0.5 * dtd * s
        return torch.cat([_larger(f[:1], torch.full_like(f[:1], SMALLR)), f[1:]])

    xm, xp, ym, yp = face(dx, dtdx, -1), face(dx, dtdx, 1), face(dy, dtdy, -1), face(dy, dtdy, 1)
    fx = _riemann(xp[:, 1:-1, :-1], xm[:, 1:-1, 1:], 2) * dtdx
    fy = _riemann(yp[:, :-1, 1:-1], ym[:, 1:, 1:-1], 3) * dtdy
    return u[:, 2:-2, 2:-2] + (fy[:, :-1] - fy[:, 1:]) + (fx[:, :, :-1] - fx[:, :, 1:])


def _rate(u, case):
    """Largest CFL rate over the window of the reference's compute_dt (0-based [2, n])."""
    q = _primitive(u[:, 2:case["ny"] + 1, 2:case["nx"] + 1])
    c = torch.sqrt(GAMMA * q[1] / q[0])
    return float(((c + _size(q[2])) * case["nx"] + (c + _size(q[3])) * case["ny"]).max())


def _forward(case, seed, keep=False):
    """Both buffers after the steps, the dt of each step, the running invDt with the last state
    in it, and with `keep` the filled input state of each step."""
    first = _initial(case, seed).double()
    bufs = [first, torch.zeros_like(first)]
    _ghosts(first, case)
    invdt, dts, states = 0.0, [], []
    for n in range(case["steps"]):
        u, new = bufs[n % 2], bufs[1 - n % 2]
        invdt = max(invdt, _rate(u, case))
        dts.append(CFL / invdt)
        _ghosts(u, case)
        if keep:
            states.append(u.clone())
        new[:, 2:-2, 2:-2] = _step(u, dts[-1], case)
    last = bufs[case["steps"] % 2]
    return bufs, dts, max(invdt, _rate(last, case)), states


def _reverse(u, lam, dt, case):
    """J^T lam on the interior, as a full array, for the step from state u."""
    full = u.clone()
    inner = full[:, 2:-2, 2:-2].clone().requires_grad_(True)
    with torch.enable_grad():
        v = full.clone()
        v[:, 2:-2, 2:-2] = inner
        _ghosts(v, case)
        (g,) = torch.autograd.grad(_step(v, dt, case), inner, lam[:, 2:-2, 2:-2])
    out = torch.zeros_like(lam)
    out[:, 2:-2, 2:-2] = g
    return out


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "adjoint_step":
        u = _initial(case, seed).double()
        _ghosts(u, case)
        return {"lam": _reverse(u, _field(case, seed, dense=True), CFL / _rate(u, case), case)}
    if kind in ("gradient", "rollout"):
        bufs, dts, _, states = _forward(case, seed, keep=True)
        last = bufs[case["steps"] % 2]
        if kind == "gradient":
            d = (last[0] - _target(case, seed))[2:-2, 2:-2]
            lam = torch.zeros_like(last)
            lam[0, 2:-2, 2:-2] = 2 * d
        else:
            lam = _field(case, seed, dense=False)
        for u, dt in zip(reversed(states), reversed(dts)):
            lam = _reverse(u, lam, dt, case)
        return {"misfit": (d * d).sum(), "grad": lam} if kind == "gradient" else {"lam": lam}
    bufs, dts, invdt, _ = _forward(case, seed)
    out = {"u": bufs[0], "u2": bufs[1]}
    if kind == "noalloc":
        return {**out, "invdt": torch.tensor([invdt], dtype=torch.float64)}
    sums = bufs[case["steps"] % 2][:, 2:-2, 2:-2].sum(dim=(1, 2)).cpu().numpy()
    if kind == "steps":
        return {**out, "sums": sums, "dt": CFL / invdt}
    return {**out, "sums": sums, "dts": np.array(dts, dtype=np.float64)}
