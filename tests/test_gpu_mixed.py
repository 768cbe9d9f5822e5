"""Mixed precision (FP32 reconstruction + Riemann flux; FP64 state, pressure
recovery, flux differencing, RK sum, CT) against the FP64 path.  The FP64
path is the parity-checked one; here the L1 error of the mixed path is
measured and bounded."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def l1rel(a, b):
    return float(np.abs(a - b).sum() / np.abs(b).sum())


def run(p, steps, precision, dt):
    from qasmhd_amd import capi
    with capi.solver_for(p, precision=precision) as s:
        s.upload(p.state)
        # fixed dt: both precisions take identical time steps
        s.run(steps, flg=0, dt=dt, history=False)
        return s.download()


def pressure(st, gam):
    ro = st[0]
    v2 = (st[1] ** 2 + st[2] ** 2 + st[3] ** 2) / ro
    return (gam - 1) * (st[7] - 0.5 * (v2 + st[4] ** 2 + st[5] ** 2 + st[6] ** 2))


@pytest.mark.parametrize("case", ["khi", "turb"])
def test_mixed_l1_error(case):
    from qasmhd_amd import capi, problems
    if case == "khi":
        p = problems.kelvin_helmholtz(n=128)
        steps, tol = 200, 1e-5
    else:
        p = problems.turbulence2d(n=128, seed=3)
        steps, tol = 100, 1e-4
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    a = run(p, steps, 0, dt)
    b = run(p, steps, 1, dt)
    assert np.isfinite(b).all()
    I = (slice(4, -4), slice(4, -4))
    e_ro = l1rel(b[0][I], a[0][I])
    e_pr = l1rel(pressure(b, p.gam)[I], pressure(a, p.gam)[I])
    _say("mixed vs fp64 %s: L1(rho) %.3e  L1(p) %.3e" % (case, e_ro, e_pr))
    assert e_ro < tol and e_pr < tol


@pytest.mark.parametrize("rmn", [1, 3])
def test_mixed_across_units(rmn):
    """The same flow in units whose speeds are 2^k times larger: FP32 scales
    exactly but for the range of its reciprocals, and the WCNS smoothness
    denominators (of pressures squared, to the fourth power) run from far
    below to above 2^120, where the weights take the division instead of the
    estimate.  The error against the FP64 path keeps the bound it has in the
    first units (test_mixed_l1_error)."""
    from qasmhd_amd import capi, problems
    p = problems.turbulence2d(n=64, seed=3)
    with capi.solver_for(p, rmn=rmn) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    for k in (0, 8, 12, 13, 14):  # (at 2^15 the denominators overflow FP32)
        q = p.copy()
        f = 2.0 ** k
        q.state[1:7] *= f
        q.state[7] *= f * f
        out = []
        for precision in (0, 1):
            with capi.solver_for(q, rmn=rmn, precision=precision) as s:
                s.upload(q.state)
                s.run(20, flg=0, dt=dt / f, history=False)
                out.append(s.download())
        I = (slice(4, -4), slice(4, -4))
        e = l1rel(out[1][0][I], out[0][0][I])
        _say("mixed vs fp64, speeds x 2^%d, rmn %d: L1(rho) %.3e" % (k, rmn, e))
        assert np.isfinite(out[1]).all() and e < 1e-4


@pytest.mark.parametrize("jump", [1e3, 1.1e4, 1.4e4, 1.8e4, 3e4])
@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
def test_mixed_wcns3_flat_beside_a_jump(rmn, jump):
    """ODR 3 where the pressure is flat up to a jump: one smoothness measure
    is zero, the weights' sum is the jump squared over the FP32 eps (1e-30),
    and from a jump of 1.07e4 on the sum lies above 2^126, past which the FP32
    reciprocal estimate gives 0; from 1.84e4 on it overflows FP32.
    The stencil must stay on the flat side, as in FP64: both pressures'
    differences are a few FP32 roundings (6e-8 each) after three steps."""
    from qasmhd_amd import capi
    n = 32
    st = np.zeros((8, n + 8, n + 8))
    st[0], st[4], st[5] = 1.0, 30.0, 20.0
    pr = np.full((n + 8, n + 8), 3e4)
    pr[:, (n + 8) // 2:] += jump
    pr[(n + 8) // 2:] += jump
    st[7] = pr / (5.0 / 3.0 - 1.0) + 0.5 * (900.0 + 400.0)
    out = []
    for precision in (0, 1):
        with capi.Solver(st.shape[1:], 1.0 / n, 1.0 / n, rmn=rmn, odr=3, precision=precision) as s:
            s.upload(st)
            s.run(3, flg=0, dt=0.2 / n / 400.0, history=False)
            out.append(s.download())
    I = (slice(4, -4), slice(4, -4))
    e = [l1rel(out[1][m][I], out[0][m][I]) for m in (0, 7)]
    _say("mixed odr 3, flat beside a jump of %g, rmn %d: L1(rho) %.2e L1(en) %.2e" % (jump, rmn, *e))
    assert max(e) < 1e-6


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
@pytest.mark.parametrize("odr", [1, 2, 3])
def test_mixed_across_units_at_lower_orders(odr, rmn):
    """test_mixed_across_units at ODR 1 to 3: each order's error stays at the
    size it has in the first units."""
    from qasmhd_amd import capi, problems
    p = problems.turbulence2d(n=32, seed=3)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    I = (slice(4, -4), slice(4, -4))
    for k in (0, 4, 8, 11):
        q = p.copy()
        f = 2.0 ** k
        q.state[1:7] *= f
        q.state[7] *= f * f
        out = []
        for precision in (0, 1):
            with capi.solver_for(q, rmn=rmn, odr=odr, precision=precision) as s:
                s.upload(q.state)
                s.run(4, flg=0, dt=dt / f, history=False)
                out.append(s.download())
        e = [l1rel(out[1][m][I], out[0][m][I]) for m in (0, 7)]
        _say("mixed vs fp64, odr %d, rmn %d, speeds x 2^%d: L1(rho) %.2e L1(en) %.2e" % (odr, rmn, k, *e))
        assert max(e) < 1e-6


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
@pytest.mark.parametrize("odr", [1, 2, 3])
def test_mixed_at_small_speeds(odr, rmn):
    """Units in which the speeds are 2^k and the densities 2^b (pressures stay
    above the positivity floor): below 2^-31 the squares of the squared speeds
    are FP32 denormals, which the root estimate takes for 0, so the operators
    must serve there.  Same error as in the first units; at 2^-33 the
    denormals keep 9 bits of those squares, which is 1e-3 of a quarter of the
    squared speed in a dissipation that acts on differences of 1e-4.  (Roe's
    mean field energy underflows from 2^-32 on.)"""
    from qasmhd_amd import capi, problems
    p = problems.turbulence2d(n=32, seed=3)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    I = (slice(4, -4), slice(4, -4))
    for k, b in ((-10, 20), (-28, 60), (-31, 64)) + (((-33, 70),) if rmn else ()):
        q = p.copy()
        f, d = 2.0 ** k, 2.0 ** b
        q.state[0] *= d
        q.state[1:4] *= f * d
        q.state[4:7] *= f * np.sqrt(d)
        q.state[7] *= f * f * d
        out = []
        for precision in (0, 1):
            with capi.solver_for(q, rmn=rmn, odr=odr, precision=precision) as s:
                s.upload(q.state)
                s.run(4, flg=0, dt=dt / f, history=False)
                out.append(s.download())
        e = [l1rel(out[1][m][I], out[0][m][I]) for m in (0, 7)]
        _say("mixed vs fp64, odr %d, rmn %d, speeds 2^%d, densities 2^%d: L1(rho) %.2e L1(en) %.2e" % (odr, rmn, k, b, *e))
        assert max(e) < 1e-6


@pytest.mark.parametrize("n,ny", [(64, 48), (320, 300), (520, 516)])
@pytest.mark.parametrize("odr", [1, 2, 3, 4])
def test_mixed_l1_error_by_size_and_order(odr, n, ny):
    """The three forms of the corner EMF (fused, one and two corners a thread)
    at every order: an FP32 rounding's error against FP64 after 4 steps."""
    from qasmhd_amd import capi, problems
    p = problems.turbulence2d(n=n, ny=ny, seed=3)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    out = []
    for precision in (0, 1):
        with capi.solver_for(p, odr=odr, precision=precision) as s:
            s.upload(p.state)
            s.run(4, flg=0, dt=dt, history=False)
            out.append(s.download())
    I = (slice(4, -4), slice(4, -4))
    e = [l1rel(out[1][m][I], out[0][m][I]) for m in (0, 4, 5, 7)]
    _say("mixed vs fp64, odr %d, %d x %d: L1 of ro, bx, by, en %.2e %.2e %.2e %.2e" % (odr, n, ny, *e))
    assert max(e) < 1e-6


def test_mixed_l1_error_vs_oracle(oracle):
    """The mixed path's L1 error measured against the oracle itself (the
    CPU restatement of the reference) rather than through the FP64 HIP
    path: KH 128^2, MLAU, 200 steps at a fixed dt; the FP64 HIP result is
    the oracle's bit for bit in the same run."""
    from qasmhd_amd import capi, problems
    p = problems.kelvin_helmholtz(n=128)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    steps = 200
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam, cfl=p.cfl, rmn=p.rmn, odr=p.odr, r_k=p.r_k,
                          ctw=p.ctw, dn=p.dn)
    ref = p.state.copy()
    oracle.run(cfg, ref, steps, 0, dt=dt)
    a = run(p, steps, 0, dt)
    b = run(p, steps, 1, dt)
    assert np.array_equal(a, ref)
    I = (slice(4, -4), slice(4, -4))
    e_ro = l1rel(b[0][I], ref[0][I])
    e_pr = l1rel(pressure(b, p.gam)[I], pressure(ref, p.gam)[I])
    _say("mixed vs oracle khi: L1(rho) %.3e  L1(p) %.3e" % (e_ro, e_pr))
    assert np.isfinite(b).all() and e_ro < 1e-5 and e_pr < 1e-5


def test_mixed_3d_runs(oracle):
    from qasmhd_amd import capi, problems
    p = problems.turbulence3d(n=16, seed=2, nmodes=8)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    a = run(p, 4, 0, dt)
    b = run(p, 4, 1, dt)
    e = l1rel(b[0], a[0])
    _say("mixed vs fp64 3d: L1(rho) %.3e" % e)
    assert np.isfinite(b).all() and e < 1e-5


def test_mixed_full_size_khi():
    """The low-Mach Kelvin-Helmholtz workload at its full size and length
    (2048^2, M = 0.01, MLAU / WCNS-4 / CT / RK3, 2000 steps at one fixed dt):
    mean |rho_mixed - rho_fp64| and mean |p_mixed - p_fp64| over the
    interior at most 1e-6 (rho = 1 and p = 1/gam, so absolute and relative
    L1 coincide up to the factor gam for p)."""
    from qasmhd_amd import capi, problems
    p = problems.kelvin_helmholtz(n=2048)
    with capi.solver_for(p) as s:
        s.upload(p.state)
        dt = s.cfl_dt()
    _say("case: mixed vs fp64, KH 2048^2, 2000 steps, fp64 run")
    a = run(p, 2000, 0, dt)
    _say("  mixed run")
    b = run(p, 2000, 1, dt)
    assert np.isfinite(b).all()
    I = (slice(4, -4), slice(4, -4))
    e_ro = float(np.abs(b[0][I] - a[0][I]).mean())
    e_pr = float(np.abs(pressure(b, p.gam)[I] - pressure(a, p.gam)[I]).mean())
    _say("  L1(rho) %.3e  L1(p) %.3e" % (e_ro, e_pr))
    assert e_ro <= 1e-6 and e_pr <= 1e-6


def test_mixed_full_size_3d():
    """The 3D turbulence workload at its full size and length (512^3, 200
    steps at one fixed dt) in mixed precision against FP64: L1(rho) and
    L1(p) at most 1e-6 (tests/gpu_mixed3d_full_check.py, fresh process)."""
    import os
    import subprocess
    _say("case: mixed vs fp64 3D 512^3, 200 steps (subprocess)")
    script = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gpu_mixed3d_full_check.py")
    r = subprocess.run([sys.executable, "-u", script], capture_output=True, text=True, timeout=280)
    _say(r.stdout[-3000:])
    if r.returncode != 0:
        _say(r.stderr[-3000:])
    assert r.returncode == 0
    assert "OK" in r.stdout
