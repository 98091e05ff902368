"""Tangent-linear and adjoint of the step on the GPU (FP64, frozen dt).

* dot-product identity <J v, w> = <v, J^T w> (tangent = dual numbers through
  the forward kernel, adjoint = hand-written reverse kernels), on
  discontinuous states, for all boundary and slope types;
* tangent against 4-point finite differences of the forward step;
* the checkpointed rollout adjoint: independent of the number of snapshots
  (bit for bit), consistent with the chained tangent, and against finite
  differences of a rollout objective.
"""
import numpy as np
import pytest

import euler2d_cudafortran_amd as e2d

pytestmark = pytest.mark.gpu

# variants whose reverse passes run in float
FLOAT_PRECS = (e2d.PREC_FP32, e2d.PREC_FP32_NATIVE, e2d.PREC_MIXED)


def _params(nx, ny=None, **kw):
    p = e2d.HydroParams(nx=nx, ny=nx if ny is None else ny)
    for k, v in kw.items():
        setattr(p, k, v)
    return p


def _interior(nx, ny):
    m = np.zeros((nx + 4, ny + 4, 4), dtype=bool)
    m[2:nx + 2, 2:ny + 2, :] = True
    return m


def _smooth_field(nx, ny, rng, modes=4):
    x = (np.arange(nx + 4) - 1.5) / nx
    y = (np.arange(ny + 4) - 1.5) / ny
    X, Y = np.meshgrid(x, y, indexing="ij")
    f = np.zeros_like(X)
    for _ in range(modes):
        kx, ky = rng.integers(1, 4, 2)
        f += rng.normal() * np.sin(2 * np.pi * (kx * X + rng.uniform())) * np.cos(2 * np.pi * (ky * Y + rng.uniform()))
    return f / modes


def _smooth_state(nx, ny, seed, gamma=1.4):
    rng = np.random.default_rng(seed)
    rho = 1.0 + 0.3 * _smooth_field(nx, ny, rng)
    u = 0.2 * _smooth_field(nx, ny, rng)
    v = 0.2 * _smooth_field(nx, ny, rng)
    p = 1.0 + 0.3 * _smooth_field(nx, ny, rng)
    U = np.stack([rho, p / (gamma - 1) + 0.5 * rho * (u * u + v * v), rho * u, rho * v], axis=-1)
    return U


def _evolved_diag(run, steps):
    run.init("diag")
    run.make_boundaries(0)
    run.run_steps(steps)
    return run.download(run.current())


@pytest.mark.parametrize("bc,st", [((1, 1, 1, 1), 1), ((2, 2, 2, 2), 2), ((3, 3, 3, 3), 0), ((1, 2, 3, 1), 1)])
def test_dot_product_single_step(gpu_lib, bc, st):
    nx, ny = 96, 80
    p = _params(nx, ny, boundary_type_xmin=bc[0], boundary_type_xmax=bc[1], boundary_type_ymin=bc[2],
                boundary_type_ymax=bc[3], slope_type=st)
    rng = np.random.default_rng(7)
    mask = _interior(nx, ny)
    with e2d.HydroRun(p) as run:
        U = _evolved_diag(run, 30)
        run.upload(0, U)
        dt = run.compute_dt(0)
        v = np.where(mask, rng.normal(size=mask.shape), 0.0)
        w = np.where(mask, rng.normal(size=mask.shape), 0.0)
        dv, djv, dw, djw = (run.field_alloc() for _ in range(4))
        run.field_upload(dv, v)
        run.field_upload(dw, w)
        run.tangent_step(0, dt, dv, djv)
        run.upload(0, U)
        run.adjoint_step(0, dt, dw, djw)
        jv, jtw = run.field_download(djv), run.field_download(djw)
        for d in (dv, djv, dw, djw):
            run.field_free(d)
    lhs = float(np.sum(jv[mask] * w[mask]))
    rhs = float(np.sum(v[mask] * jtw[mask]))
    rel = abs(lhs - rhs) / max(abs(lhs), abs(rhs))
    print(f"dot test bc={bc} slope_type={st}: <Jv,w>={lhs:.15e} <v,J^T w>={rhs:.15e} rel={rel:.2e}")
    assert rel <= 1e-10


def _forward(run, U, dt):
    run.upload(0, U)
    run.godunov_unsplit(0, dt)
    return run.download(1)


def _perturbed_diag(run, seed, amp=1e-3, gamma=1.4):
    """The diagonal problem with seeded uniform perturbations of amplitude amp
    in rho and p on the interior (no exact ties in the limiters)."""
    run.init("diag")
    U = run.download(0)
    nx, ny = U.shape[0] - 4, U.shape[1] - 4
    inner = _interior(nx, ny)[..., 0]
    rng = np.random.default_rng(seed)
    U0 = U.copy()
    U0[..., 0] = np.where(inner, U[..., 0] + amp * rng.random(inner.shape), U[..., 0])
    U0[..., 1] = np.where(inner, ((gamma - 1) * U[..., 1] + amp * rng.random(inner.shape)) / (gamma - 1), U[..., 1])
    return U0


# the finite differences of the tangent and gradient checks: 4-point central
# differences of the step (or rollout) evaluated by the oracle in binary128
# at eps = 1e-10, every decision (limiters, the solver's branches, maxima and
# Newton counts) frozen at the unperturbed run's.  That map, the step as
# executed, is smooth and is what the tangent and adjoint differentiate; at
# that step neither truncation (eps^4) nor roundoff (1e-34 / eps) shows in a
# double.  Measured on the CPU: the binary128 quotients at eps 1e-8 .. 1e-12
# round to the same doubles.
QUAD_EPS = 1e-10


@pytest.mark.parametrize("st,bc,state", [(0, (3, 3, 3, 3), "smooth"), (1, (3, 3, 3, 3), "smooth"),
                                         (2, (3, 3, 3, 3), "smooth"), (1, (1, 2, 3, 1), "smooth"),
                                         (1, (1, 1, 1, 1), "shocked"), (2, (1, 3, 2, 1), "shocked")])
def test_tangent_vs_quad_finite_differences(gpu_lib, st, bc, state):
    """One step: the GPU tangent (dual numbers through the fused kernel)
    against the binary128 finite differences of the oracle's step, on a
    smooth state with flow and on the perturbed diagonal problem after 30
    steps (shocks and contacts, no exact ties); relative L2 over the
    interior, bar 1e-10."""
    from oracle_lib import Oracle
    nx, ny = 64, 48
    p = _params(nx, ny, slope_type=st, boundary_type_xmin=bc[0], boundary_type_xmax=bc[1],
                boundary_type_ymin=bc[2], boundary_type_ymax=bc[3])
    mask = _interior(nx, ny)
    rng = np.random.default_rng(12 + st)
    V = np.stack([_smooth_field(nx, ny, rng) for _ in range(4)], axis=-1)
    V = np.where(mask, V, 0.0)
    with e2d.HydroRun(p) as run:
        if state == "smooth":
            U = _smooth_state(nx, ny, 11)
        else:
            U0 = _perturbed_diag(run, 5)
            run.upload(0, U0)
            run.run_steps(30)
            U = run.download(run.current())
        run.upload(0, U)
        dt = run.compute_dt(0)
        dv, djv = run.field_alloc(), run.field_alloc()
        run.field_upload(dv, V)
        run.upload(0, U)
        run.tangent_step(0, dt, dv, djv)
        jv = run.field_download(djv)
    o = Oracle(nx, ny, bc=bc, slope_type=st, precision="f128")
    fd = o.fd(U, V, [dt], QUAD_EPS, freeze=True)
    err = np.linalg.norm((fd - jv)[mask]) / np.linalg.norm(fd[mask])
    print(f"tangent vs binary128 FD, slope_type={st} bc={bc} {state}: relative L2 error {err:.2e}")
    assert err <= 1e-10


def _record_forward(run, U0, nsteps):
    run.upload(0, U0)
    run.nStep = 0
    dts = []
    for n in range(nsteps):
        dt = run.compute_dt(n % 2)
        dts.append(dt)
        run.godunov_unsplit(n, dt)
    return np.array(dts)


def _beta(c, r):
    from math import comb
    return comb(c + r, c) if r >= 0 else 0


def _split(l, s):
    """Griewank and Walther's binomial split: the largest m in the range that
    gives the least number of forward steps (c = s + 1 kept states)."""
    c, r = s + 1, 1
    while _beta(c, r) < l:
        r += 1
    lo = max(l - _beta(c - 1, r), _beta(c, r - 2) + 1)
    hi = min(_beta(c, r - 1), l - _beta(c - 1, r - 1) - 1)
    return min(max(hi if hi >= lo else lo, 1), l - 1)


def _first_descent_steps(nsteps, nsnap):
    """Forward steps of the reverse sweep's first descent, i.e. what a
    recorded forward saves the sweep."""
    a, s, done = 0, nsnap - 1, 0
    while nsteps - a > 1 and s > 0:
        m = _split(nsteps - a, s)
        done, a, s = done + m, a + m, s - 1
    return done


def _least_forward_steps(l, c):
    """The least number of forward steps that reverses l steps keeping c states
    (the first included), r l - beta(c+1, r-1) for the least r with
    beta(c, r) >= l (Griewank and Walther, Algorithm 799: revolve, ACM TOMS 26 (2000))."""
    r = 1
    while _beta(c, r) < l:
        r += 1
    return r * l - _beta(c + 1, r - 1)


def test_recorded_forward_rollout(gpu_lib):
    """e2d_rollout_forward: the same final state as the plain steps, the same
    gradient bit for bit, and the first descent's forward steps saved; a
    different starting state or dt sequence falls back to the full recompute."""
    nx, ny, nsteps = 64, 48, 24
    mask = _interior(nx, ny)
    rng = np.random.default_rng(5)
    with e2d.HydroRun(_params(nx, ny)) as run:
        U0 = _evolved_diag(run, 10)
        run.init("diag")
        dts = _record_forward(run, U0, nsteps)
        run.upload(0, U0)
        for n in range(nsteps):
            run.godunov_unsplit(n, dts[n])
        UT = run.download(nsteps % 2)
        lam_n = np.where(mask, rng.normal(size=mask.shape), 0.0)
        d_n, d_0 = run.field_alloc(), run.field_alloc()
        run.field_upload(d_n, lam_n)
        for nsnap in (1, 3, 6, nsteps):
            run.upload(0, U0)
            nf_plain = run.adjoint_rollout(0, dts, nsnap, d_n, d_0)
            plain = run.field_download(d_0)
            run.upload(0, U0)
            run.rollout_forward(0, dts, nsnap)
            assert np.array_equal(run.download(nsteps % 2), UT)
            run.upload(0, U0)
            nf_rec = run.adjoint_rollout(0, dts, nsnap, d_n, d_0)
            assert np.array_equal(run.field_download(d_0), plain), f"nsnap={nsnap}"
            assert nf_rec == nf_plain - _first_descent_steps(nsteps, nsnap), (nsnap, nf_rec, nf_plain)
            assert nf_plain == _least_forward_steps(nsteps, nsnap), (nsnap, nf_plain)
            assert np.array_equal(run.download(0)[mask], U0[mask])  # the starting state is back
            print(f"nsnap={nsnap}: {nf_plain} recomputed steps plain, {nf_rec} after a recorded forward")
        # a recording made from another starting state, or for other dts, is not used
        U1 = U0.copy()
        U1[10, 10, 0] *= 1.0 + 1e-12
        run.upload(0, U1)
        nf1 = run.adjoint_rollout(0, dts, 6, d_n, d_0)
        g1 = run.field_download(d_0)
        run.upload(0, U0)
        run.rollout_forward(0, dts, 6)
        run.upload(0, U1)
        assert run.adjoint_rollout(0, dts, 6, d_n, d_0) == nf1
        assert np.array_equal(run.field_download(d_0), g1)
        run.upload(0, U0)
        run.rollout_forward(0, dts, 6)
        run.upload(0, U0)
        dts2 = list(dts)
        dts2[-1] *= 0.5
        nf2 = run.adjoint_rollout(0, dts2, 6, d_n, d_0)
        assert nf2 == nf1


def test_rollout_snapshots_and_tangent_chain(gpu_lib):
    nx, ny, nsteps = 64, 64, 24
    mask = _interior(nx, ny)
    rng = np.random.default_rng(21)
    with e2d.HydroRun(_params(nx, ny)) as run:
        U0 = _evolved_diag(run, 10)
        run.init("diag")  # corners of both buffers as the run starts
        dts = _record_forward(run, U0, nsteps)
        lam_n = np.where(mask, rng.normal(size=mask.shape), 0.0)
        d_n, d_0 = run.field_alloc(), run.field_alloc()
        run.field_upload(d_n, lam_n)
        results = {}
        for nsnap in (1, 3, 6, nsteps):
            run.upload(0, U0)
            nf = run.adjoint_rollout(0, dts, nsnap, d_n, d_0)
            results[nsnap] = (run.field_download(d_0), nf)
            print(f"nsnap={nsnap}: {nf} forward steps recomputed")
        # tangent chained through the same states
        v0 = np.where(mask, rng.normal(size=mask.shape), 0.0)
        dv, dw = run.field_alloc(), run.field_alloc()
        run.field_upload(dv, v0)
        run.upload(0, U0)
        for n in range(nsteps):
            state = run.download(n % 2)
            run.tangent_step(n % 2, dts[n], dv, dw)
            run.upload(n % 2, state)
            run.godunov_unsplit(n, dts[n])
            dv, dw = dw, dv
        vn = run.field_download(dv)
    ref = results[nsteps][0]
    for nsnap, (lam0, _) in results.items():
        assert np.array_equal(lam0, ref), f"nsnap={nsnap} differs"
    assert results[1][1] > results[3][1] > results[nsteps][1]
    lhs = float(np.sum(vn[mask] * lam_n[mask]))
    rhs = float(np.sum(v0[mask] * ref[mask]))
    rel = abs(lhs - rhs) / max(abs(lhs), abs(rhs))
    print(f"rollout dot test: {lhs:.15e} vs {rhs:.15e}, rel {rel:.2e}")
    assert rel <= 1e-10


def test_rollout_gradient_vs_quad_finite_differences(gpu_lib):
    """J = sum of rho over cells with centres in [0.6,0.8]^2 after a 40-step
    rollout (64^2, periodic, smooth initial state with flow); gradient with
    respect to the initial rho and p (E = p/(gamma-1) + kinetic) from the
    checkpointed adjoint, against the binary128 finite difference of J along
    that direction (the oracle's rollout with the frozen dt sequence); bar
    1e-10."""
    from oracle_lib import Oracle
    nx, ny, nsteps, gamma = 64, 64, 40, 1.4
    bc = (3, 3, 3, 3)
    mask = _interior(nx, ny)
    xc = (np.arange(nx + 4) - 2 + 0.5) / nx
    box = np.zeros_like(mask)
    sel = (xc >= 0.6) & (xc <= 0.8)
    box[np.ix_(sel, sel, [0])] = True
    U0 = _smooth_state(nx, ny, 31)
    rng = np.random.default_rng(32)
    drho = _smooth_field(nx, ny, rng)
    dp = _smooth_field(nx, ny, rng)
    dU = np.zeros_like(U0)
    rho, u, v = U0[..., 0], U0[..., 2] / U0[..., 0], U0[..., 3] / U0[..., 0]
    dU[..., 0] = drho
    dU[..., 1] = dp / (gamma - 1) + 0.5 * drho * (u * u + v * v)
    dU[..., 2] = drho * u
    dU[..., 3] = drho * v
    dU = np.where(mask, dU, 0.0)
    with e2d.HydroRun(_params(nx, ny, boundary_type_xmin=bc[0], boundary_type_xmax=bc[1],
                              boundary_type_ymin=bc[2], boundary_type_ymax=bc[3])) as run:
        run.init("diag")
        dts = _record_forward(run, U0, nsteps)
        lam_n = np.where(box, 1.0, 0.0)
        d_n, d_0 = run.field_alloc(), run.field_alloc()
        run.field_upload(d_n, lam_n)
        run.upload(0, U0)
        run.adjoint_rollout(0, dts, 5, d_n, d_0)
        lam0 = run.field_download(d_0)
    o = Oracle(nx, ny, bc=bc, precision="f128")
    fd = o.fd(U0, dU, dts, QUAD_EPS, weight=box.astype(np.float64), freeze=True)
    ad = float(np.sum(lam0[mask] * dU[mask]))
    rel = abs(fd - ad) / abs(fd)
    print(f"rollout gradient: adjoint {ad:.15e}, binary128 finite difference {fd:.15e}, rel {rel:.2e}")
    assert rel <= 1e-10


def test_c4_adjoint_512(gpu_lib):
    """512^2 FP64, 400 steps, diagonal-discontinuity IC with seeded uniform
    perturbations of amplitude 1e-3 in rho and p, reflective walls, 20
    snapshots; J = sum of rho over cells with centres in [0.6,0.8]^2.

    * dot test of the rollout: the chained tangent against the checkpointed
      adjoint, <J_N...J_1 v, e_box> = <v, lam_0>, relative error <= 1e-10;
    * directional derivative along a smooth (rho, p) direction against the
      4-point finite difference of the oracle's rollout in long double with
      every decision frozen at the unperturbed run's (limiters, solver
      branches and maxima, Newton counts), eps = 1e-6: the map as executed,
      which the adjoint linearises, is smooth, so the quotient carries only
      truncation (eps^4) and long-double roundoff (1e-19 / eps); bar 1e-10.
      Left free, the map is only piecewise smooth along the direction: over
      400 steps the limiters meet hundreds of kinks within 2 eps at eps 1e-8
      and the solver's sampling has jumps, so free differences stall near
      1e-8..1e-10 (measured at eps 1e-7, 1e-8, 1e-9, 1e-10: 1.7e-8, 9.3e-8,
      1.6e-8, 7.9e-10 with the solver's decisions frozen and the limiters
      free; on the CPU at 128^2 x 100 steps the fully frozen long-double
      quotient at eps 1e-6 agrees with the binary128 one to 2e-14)."""
    nx, nsteps, gamma = 512, 400, 1.4
    mask = _interior(nx, nx)
    xc = (np.arange(nx + 4) - 2 + 0.5) / nx
    sel = (xc >= 0.6) & (xc <= 0.8)
    box = np.zeros_like(mask)
    box[np.ix_(sel, sel, [0])] = True
    rng = np.random.default_rng(2024)
    with e2d.HydroRun(_params(nx)) as run:
        run.init("diag")
        U = run.download(0)
        U0 = U.copy()
        inner = mask[..., 0]
        rho = U[..., 0] + 1e-3 * rng.random(inner.shape)
        p = (gamma - 1) * U[..., 1] + 1e-3 * rng.random(inner.shape)
        U0[..., 0] = np.where(inner, rho, U[..., 0])
        U0[..., 1] = np.where(inner, p / (gamma - 1), U[..., 1])
        dts = _record_forward(run, U0, nsteps)
        d_n, d_0 = run.field_alloc(), run.field_alloc()
        run.field_upload(d_n, np.where(box, 1.0, 0.0))
        run.upload(0, U0)
        nf = run.adjoint_rollout(0, dts, 20, d_n, d_0)
        lam0 = run.field_download(d_0)
        print(f"C4 rollout: {nf} forward steps for {nsteps} adjoint steps with 20 snapshots")

        v0 = np.where(mask, rng.normal(size=mask.shape), 0.0)
        dv, dw = run.field_alloc(), run.field_alloc()
        run.field_upload(dv, v0)
        run.upload(0, U0)
        for n in range(nsteps):
            state = run.download(n % 2)
            run.tangent_step(n % 2, dts[n], dv, dw)
            run.upload(n % 2, state)
            run.godunov_unsplit(n, dts[n])
            dv, dw = dw, dv
        vn = run.field_download(dv)
        lhs, rhs = float(np.sum(vn[box])), float(np.sum(v0[mask] * lam0[mask]))
        rel_dot = abs(lhs - rhs) / abs(rhs)
        print(f"C4 dot test: {lhs:.15e} vs {rhs:.15e}, rel {rel_dot:.2e}")
        assert rel_dot <= 1e-10

        X, Y = np.meshgrid((np.arange(nx + 4) - 1.5) / nx, (np.arange(nx + 4) - 1.5) / nx, indexing="ij")
        dU = np.zeros_like(U0)
        dU[..., 0] = np.sin(2 * np.pi * (X + 0.13)) * np.cos(2 * np.pi * (Y + 0.29))
        dU[..., 1] = np.cos(2 * np.pi * (X - Y + 0.41)) / (gamma - 1)
        dU = np.where(mask, dU, 0.0)

    from oracle_lib import Oracle
    o = Oracle(nx, precision="f80")
    fd = o.fd(U0, dU, dts, 1e-6, weight=box.astype(np.float64), freeze=True)
    ad = float(np.sum(lam0[mask] * dU[mask]))
    rel = abs(fd - ad) / abs(fd)
    print(f"C4 gradient: adjoint {ad:.15e}, frozen long-double finite difference {fd:.15e}, rel {rel:.2e}")
    assert rel <= 1e-10


def _adjoint_step_all_precisions(U, nx, dt, lam, **kw):
    out = {}
    for prec in (e2d.PREC_FP64,) + FLOAT_PRECS:
        with e2d.HydroRun(_params(nx, precision=prec, **kw)) as run:
            run.init("diag")
            run.upload(0, U)
            a, b = run.field_alloc(), run.field_alloc()
            run.field_upload(a, lam)
            run.adjoint_step(0, dt, a, b)
            out[prec] = run.field_download(b)
    return out


def test_fp32_adjoint_step_against_fp64_first_order(gpu_lib):
    """The FP32 and mixed adjoints (reverse passes in float, lam accumulated in
    double) against the FP64 adjoint on the same float-representable smooth
    state with flow, first-order reconstruction (slope_type 0, so no limiter
    subgradient can flip): they differ by FP32 rounding only."""
    nx = 96
    mask = _interior(nx, nx)
    U = _smooth_state(nx, nx, 41).astype(np.float32).astype(np.float64)
    lam = np.where(mask, np.random.default_rng(42).normal(size=mask.shape), 0.0)
    out = _adjoint_step_all_precisions(U, nx, 2e-3, lam, slope_type=0, boundary_type_xmin=3, boundary_type_xmax=3,
                                       boundary_type_ymin=3, boundary_type_ymax=3)
    ref = out[e2d.PREC_FP64][mask]
    for prec in FLOAT_PRECS:
        err = np.linalg.norm(out[prec][mask] - ref) / np.linalg.norm(ref)
        print(f"precision {prec}: adjoint step vs fp64, relative L2 {err:.2e}")
        assert err <= 1e-5


def test_fp32_adjoint_step_against_fp64_minmod(gpu_lib):
    """Same comparison on the benchmark configuration (diagonal problem after
    30 FP32 steps, minmod): where |dl| and |dr| of the limiter differ by less
    than FP32 resolves (nearly linear profiles), the float forward takes the
    other subgradient, so the adjoints differ beyond rounding (measured
    relative L2 2.9e-3 at 128^2)."""
    nx = 128
    mask = _interior(nx, nx)
    with e2d.HydroRun(_params(nx, precision=e2d.PREC_FP32)) as run:
        U = _evolved_diag(run, 30)
    lam = np.where(mask, np.random.default_rng(3).normal(size=mask.shape), 0.0)
    out = _adjoint_step_all_precisions(U, nx, 1e-3, lam)
    ref = out[e2d.PREC_FP64][mask]
    for prec in FLOAT_PRECS:
        err = np.linalg.norm(out[prec][mask] - ref) / np.linalg.norm(ref)
        print(f"precision {prec}: adjoint step vs fp64 (minmod, diagonal problem), relative L2 {err:.2e}")
        assert err <= 1e-2


def test_fp32_rollout_against_fp64(gpu_lib):
    """C5 at reduced size (256^2, 200 steps, 10 snapshots): gradient of
    J = sum over the interior of (rho_T - rho_target)^2 from the FP32 and mixed
    forward/adjoint against the FP64 one, same frozen dt sequence (measured
    relative L2 8.3e-4 / 8.4e-4)."""
    nx, nsteps = 256, 200
    mask = _interior(nx, nx)
    X, Y = np.meshgrid((np.arange(nx + 4) - 1.5) / nx, (np.arange(nx + 4) - 1.5) / nx, indexing="ij")
    target = 1 + 0.3 * np.sin(2 * np.pi * (X + 0.1)) * np.cos(2 * np.pi * (2 * Y + 0.3))
    grads, dts = {}, None
    for prec in (e2d.PREC_FP64,) + FLOAT_PRECS:
        with e2d.HydroRun(_params(nx, precision=prec)) as run:
            run.init("diag")
            U0 = run.download(0)
            if dts is None:
                dts = _record_forward(run, U0, nsteps)
            run.upload(0, U0)
            for n in range(nsteps):
                run.godunov_unsplit(n, dts[n])
            uT = run.download(nsteps % 2)
            lam = np.zeros_like(uT)
            lam[..., 0] = np.where(mask[..., 0], 2 * (uT[..., 0] - target), 0.0)
            a, b = run.field_alloc(), run.field_alloc()
            run.field_upload(a, lam)
            run.upload(0, U0)
            run.adjoint_rollout(0, dts, 10, a, b)
            grads[prec] = run.field_download(b)[mask]
    ref = grads[e2d.PREC_FP64]
    for prec in FLOAT_PRECS:
        err = np.linalg.norm(grads[prec] - ref) / np.linalg.norm(ref)
        print(f"precision {prec}: rollout gradient vs fp64, relative L2 {err:.2e}")
        assert err <= 1e-2


# C5 gradient bounds: relative L2 of each float variant's gradient against
# the FP64 gradient; measured on MI355X: fp32 2.35e-3, fp32_native 2.32e-3,
# mixed 2.35e-3 (the limiters' subgradients, which the float forward resolves
# differently where |dl| and |dr| nearly tie, dominate; the state's precision
# barely enters); bounds about twice those
C5_BOUNDS = {e2d.PREC_FP32: 5e-3, e2d.PREC_FP32_NATIVE: 5e-3, e2d.PREC_MIXED: 5e-3}


def test_c5_adjoint_2048(gpu_lib):
    """Configuration C5: 2048^2 diagonal problem, 2000 steps, binomial
    checkpointing with 45 snapshots in HBM, J = sum over the interior of
    (rho_T - rho_target)^2 with a seeded smooth target, the frozen dt sequence
    of the FP64 run.
    * FP64: revolve's least forward-step count for 45 states (4,872); after a
      recorded forward (e2d_rollout_forward) 2,875 recomputed steps and the
      same gradient bit for bit;
    * the float variants (forward and adjoint in float arithmetic, lam
      accumulated in FP64) against the FP64 gradient: relative L2 within the
      stated bounds."""
    nx, nsteps, nsnap = 2048, 2000, 45
    mask = _interior(nx, nx)
    inner = mask[..., 0]
    X, Y = np.meshgrid((np.arange(nx + 4) - 1.5) / nx, (np.arange(nx + 4) - 1.5) / nx, indexing="ij")
    rng = np.random.default_rng(2048)
    k = rng.integers(1, 4, size=(3, 2))
    ph = rng.uniform(size=(3, 2))
    target = 1.0 + 0.3 * sum(np.sin(2 * np.pi * (k[m, 0] * X + ph[m, 0])) *
                             np.cos(2 * np.pi * (k[m, 1] * Y + ph[m, 1])) for m in range(3)) / 3

    def misfit_lam(uT):
        lam = np.zeros_like(uT)
        lam[..., 0] = np.where(inner, 2.0 * (uT[..., 0] - target), 0.0)
        return lam

    with e2d.HydroRun(_params(nx)) as run:
        run.init("diag")
        U0 = run.download(0)
        print("C5: recording the FP64 dt sequence", flush=True)
        dts = _record_forward(run, U0, nsteps)

    grads = {}
    for prec in (e2d.PREC_FP64,) + FLOAT_PRECS:
        with e2d.HydroRun(_params(nx, precision=prec)) as run:
            print(f"C5: precision {prec}, forward and checkpointed adjoint", flush=True)
            run.upload(0, U0)
            for n in range(nsteps):
                run.godunov_unsplit(n, dts[n])
            lam_n, lam_0 = run.field_alloc(), run.field_alloc()
            run.field_upload(lam_n, misfit_lam(run.download(nsteps % 2)))
            run.upload(0, U0)
            nf = run.adjoint_rollout(0, dts, nsnap, lam_n, lam_0)
            grads[prec] = run.field_download(lam_0)[mask]
            assert nf == 4872, nf
            if prec == e2d.PREC_FP64:
                run.upload(0, U0)
                run.rollout_forward(0, dts, nsnap)
                run.upload(0, U0)
                nf_rec = run.adjoint_rollout(0, dts, nsnap, lam_n, lam_0)
                print(f"C5 fp64: recorded forward, {nf_rec} forward steps recomputed", flush=True)
                assert nf_rec == 2875, nf_rec
                assert np.array_equal(run.field_download(lam_0)[mask], grads[prec])
    ref = grads[e2d.PREC_FP64]
    errs = {prec: float(np.linalg.norm(grads[prec] - ref) / np.linalg.norm(ref)) for prec in FLOAT_PRECS}
    print(f"C5 gradient relative L2 against fp64: {errs}", flush=True)
    for prec in FLOAT_PRECS:
        assert errs[prec] <= C5_BOUNDS[prec], (prec, errs[prec])


@pytest.mark.parametrize("prec", [e2d.PREC_FP64, e2d.PREC_FP32, e2d.PREC_FP32_NATIVE, e2d.PREC_MIXED])
def test_marching_adjoint_equals_separate_passes(gpu_lib, prec, monkeypatch):
    """The three kernel sequences of the adjoint step give the same bits: the
    fused marching kernel (face bars and the gather in registers, segment seams
    through a small buffer), the marching kernel plus a marching gather (bars
    of q and of the slopes through HBM) and the gather passes
    (E2D_ADJOINT_PASSES=separate, face bars through HBM as well), on odd sizes,
    thin grids, every boundary type, and row segments of 1, 2, 3 and 5 rows
    (the last segment of a grid may be shorter than the others), and plans
    that mix long and short segments (rows, short rows, percent of rows in
    long segments; fused only); and each in place (lam_out = lam_in, which
    runs march where fused was chosen)."""
    cases = [((1, 1, 1, 1), (96, 80), None), ((3, 3, 3, 3), (61, 37), None), ((1, 3, 2, 1), (130, 7), None),
             ((2, 2, 2, 2), (4, 4), None), ((1, 1, 3, 3), (64, 200), None), ((1, 1, 1, 1), (96, 80), "3"),
             ((3, 1, 2, 3), (70, 21), "2"), ((1, 2, 3, 1), (33, 45), "1"), ((2, 3, 1, 1), (50, 60), "5"),
             ((1, 1, 1, 1), (96, 80), ("5", "2", "60")), ((3, 1, 2, 3), (70, 21), ("4", "1", "50")),
             ((1, 1, 3, 3), (64, 200), ("7", "3", "75")), ((2, 2, 2, 2), (40, 9), ("3", "2", "0"))]
    for bc, (nx, ny), seg_rows in cases:
        plan = seg_rows if isinstance(seg_rows, tuple) else (seg_rows, None, None)
        for name, v in zip(("E2D_ADJOINT_SEG_ROWS", "E2D_ADJOINT_SHORT_ROWS", "E2D_ADJOINT_LONG_PCT"), plan):
            if v is None:
                monkeypatch.delenv(name, raising=False)
            else:
                monkeypatch.setenv(name, v)
        p = _params(nx, ny, precision=prec, boundary_type_xmin=bc[0], boundary_type_xmax=bc[1],
                    boundary_type_ymin=bc[2], boundary_type_ymax=bc[3])
        lam = np.random.default_rng(nx * ny).normal(size=(nx + 4, ny + 4, 4))
        res = {}
        for mode in ("separate", "march", "fused"):
            monkeypatch.setenv("E2D_ADJOINT_PASSES", mode)
            with e2d.HydroRun(p) as run:
                U = _evolved_diag(run, 25)
                run.upload(0, U)
                dt = run.compute_dt(0)
                a, b = run.field_alloc(), run.field_alloc()
                run.field_upload(a, lam)
                run.adjoint_step(0, dt, a, b)
                res[mode] = run.field_download(b)
                # in place (lam_out aliasing lam_in): interior bit-identical, ghost
                # cells keep lam_in's values
                run.adjoint_step(0, dt, a, a)
                res[mode + " in place"] = run.field_download(a)
        interior = np.zeros(lam.shape, bool)
        interior[2:-2, 2:-2] = True
        for mode in ("march", "fused"):
            assert np.array_equal(res["separate"], res[mode]), f"{mode} bc={bc} {nx}x{ny} seg_rows={seg_rows}"
        for mode in ("separate", "march", "fused"):
            got = res[mode + " in place"]
            assert np.array_equal(got[interior], res["separate"][interior]), f"{mode} in place bc={bc} {nx}x{ny}"
            assert np.array_equal(got[~interior], lam[~interior]), f"{mode} in place ghosts bc={bc} {nx}x{ny}"


# a single strip and two (58 columns each), tiles higher than the grid, rows that do not divide
@pytest.mark.parametrize("rows", [1, 2, 6, 7, 10])
@pytest.mark.parametrize("nx, ny, bc, st", [(4, 4, (1, 1, 1, 1), 1), (54, 9, (1, 2, 3, 1), 2), (57, 31, (3, 3, 2, 1), 1),
                                            (121, 23, (2, 1, 3, 3), 0)])
def test_adjoint_tiles_equal_the_march(gpu_lib, monkeypatch, nx, ny, bc, st, rows):
    """The adjoint step on tiles gives the marching kernels' lam and leaves the input state with
    the same filled ghost cells, bit for bit, in every precision."""
    mask = _interior(nx, ny)
    rng = np.random.default_rng(nx + rows)
    u = _smooth_state(nx, ny, 7)
    u[nx // 2:, :, :2] *= 0.3  # a jump
    lam = np.where(mask, rng.normal(size=mask.shape), 0.0)
    lam[:, ny // 2] = 0.0
    kw = dict(zip(("boundary_type_xmin", "boundary_type_xmax", "boundary_type_ymin", "boundary_type_ymax"), bc))
    for prec in (e2d.PREC_FP64, e2d.PREC_FP32, e2d.PREC_FP32_NATIVE, e2d.PREC_MIXED):
        got = []
        for tile in (0, rows):
            monkeypatch.setenv("E2D_ADJOINT_TILE_ROWS", str(tile))
            with e2d.HydroRun(_params(nx, ny, precision=prec, slope_type=st, **kw)) as run:
                run.upload(0, u)
                dt = run.compute_dt(0)
                a, b = run.field_alloc(), run.field_alloc()
                run.field_upload(a, lam)
                run.adjoint_step(0, dt, a, b)
                got.append((run.field_download(b), run.download(0)))
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]), prec


@pytest.mark.parametrize("prec", [e2d.PREC_FP64, e2d.PREC_FP32, e2d.PREC_FP32_NATIVE, e2d.PREC_MIXED])
def test_adjoint_beside_nonfinite_cells(gpu_lib, monkeypatch, prec):
    """A state with NaN and infinite cells: the marching kernels and the tiles give the separate
    passes' lam (these take the limiter as e2d_pointwise does), NaN where they have one."""
    nx, ny = 130, 41
    u = _smooth_state(nx, ny, 7)
    u[nx // 2:, :, :2] *= 0.3
    for k, (v, bad) in enumerate([(2, np.nan), (3, np.nan), (2, np.inf), (3, -np.inf), (1, np.inf), (0, np.inf)]):
        u[6 + 20 * k, 4 + 9 * (k % 4), v] = bad
        u[7 + 20 * k, 24 - 4 * (k % 4):26 - 4 * (k % 4), v] = bad
    lam = np.where(_interior(nx, ny), np.random.default_rng(3).normal(size=u.shape), 0.0)
    res = {}
    for mode, tile in (("separate", 0), ("march", 0), ("fused", 0), ("fused", 2), ("fused", 7)):
        monkeypatch.setenv("E2D_ADJOINT_PASSES", mode)
        monkeypatch.setenv("E2D_ADJOINT_TILE_ROWS", str(tile))
        with e2d.HydroRun(_params(nx, ny, precision=prec)) as run:
            run.upload(0, u)
            a, b = run.field_alloc(), run.field_alloc()
            run.field_upload(a, lam)
            run.adjoint_step(0, 1e-4, a, b)
            res[mode, tile] = run.field_download(b)
    want = res.pop(("separate", 0))
    assert 0 < np.isnan(want).sum() < 0.1 * want.size
    for k, got in res.items():
        assert np.array_equal(got, want, equal_nan=True), (k, int((~((got == want) | np.isnan(want))).sum()))


@pytest.mark.parametrize("n0, bc", [(0, (1, 2, 3, 1)), (1, (3, 3, 1, 2))])
def test_rollout_leaves_the_start_with_filled_ghosts(gpu_lib, n0, bc):
    """After an adjoint rollout, recorded or not, the buffer it started from holds the starting state
    with its ghost cells filled and its corners as they were, whatever the numbers of steps and
    snapshots, and whatever the ghost cells held."""
    nx, ny = 40, 30
    kw = dict(zip(("boundary_type_xmin", "boundary_type_xmax", "boundary_type_ymin", "boundary_type_ymax"), bc))
    u = _smooth_state(nx, ny, 7)
    u[~_interior(nx, ny)] *= 0.5
    with e2d.HydroRun(_params(nx, ny, **kw)) as run:
        run.upload(n0, u)
        run.make_boundaries(n0)
        want = run.download(n0)
        assert not np.array_equal(u, want)
        a, b = run.field_alloc(), run.field_alloc()
        run.field_upload(a, np.where(_interior(nx, ny), 1.0, 0.0))
        for nsteps in (1, 2, 3, 4, 7):
            for nsnap in (1, 2, 3, 5):
                for record in (False, True):
                    run.upload(n0, u)
                    if record:
                        run.rollout_forward(n0, np.full(nsteps, 2e-3), nsnap)
                        run.upload(n0, u)
                    run.adjoint_rollout(n0, np.full(nsteps, 2e-3), nsnap, a, b)
                    assert np.array_equal(run.download(n0), want), (nsteps, nsnap, record)
