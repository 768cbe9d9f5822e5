"""HIP path vs the reference (golden fixtures) and the oracle, through the C
ABI.  FP64 parity is bit-exact: array equality of float64 values."""
import os
import sys

import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu

S1 = np.load(os.path.join(GOLDEN, "steps_1d.npz"))
S2 = np.load(os.path.join(GOLDEN, "steps_2d.npz"))


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def qas():
    from qasmhd_amd import capi
    capi.load()
    return capi


@pytest.mark.parametrize("name", [str(n) for n in S2["names"]])
def test_2d_golden(qas, name):
    c = S2["cfg_" + name]
    rmn, odr, r_k, ctw = (int(v) for v in c[:4])
    dn = np.zeros((3, 8), dtype=int)
    dn[0], dn[1] = c[4:12], c[12:20]
    st = S2["in"]
    _say("2d golden", name, st.shape)
    with qas.Solver(st.shape[1:], float(S2["dx"]), float(S2["dy"]), gam=float(S2["gam"]), rmn=rmn, odr=odr,
                    r_k=r_k, ctw=ctw, dn=dn) as s:
        s.upload(st)
        hist, _ = s.run(int(S2["nsteps"]), flg=1)
        out = s.download()
    assert np.array_equal(hist, S2["dt_" + name])
    assert np.array_equal(out, S2["out_" + name])


def test_2d_golden_long(qas):
    st = S2["long_in"]
    n = st.shape[-1] - 8
    d = 2 * np.pi / n
    _say("2d golden long", st.shape)
    with qas.Solver(st.shape[1:], d, d) as s:
        s.upload(st)
        hist, _ = s.run(40, flg=1)
        out = s.download()
    assert np.array_equal(hist, S2["long_dt"])
    assert np.array_equal(out, S2["long_out"])


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
def test_1d_brio_wu_golden(qas, rmn):
    st = S1["in"]
    _say("1d golden", rmn)
    with qas.Solver(st.shape[1:], float(S1["dx"]), gam=float(S1["gam"]), rmn=rmn, dn=S1["dn"]) as s:
        s.upload(st)
        dt0 = s.cfl_dt()
        assert dt0 == float(S1["dt0"])
        s.run(int(S1["steps_r%d" % rmn]), flg=0, dt=dt0, history=False)
        out = s.download()
    assert np.array_equal(out, S1["out_r%d" % rmn])


@pytest.mark.parametrize("seed,n,ny,rmn,odr", [(1, 40, 24, 1, 4), (2, 24, 48, 3, 4), (3, 32, 32, 2, 3),
                                               (4, 20, 36, 0, 2), (5, 64, 64, 1, 4)])
def test_2d_vs_oracle(qas, oracle, seed, n, ny, rmn, odr):
    from qasmhd_amd import problems
    # Roe at 2nd order with open/mirror walls breaks down (NaN in the oracle
    # too) at rms Mach 1.2 on this grid; that case runs at 0.8
    p = problems.turbulence2d(n=n, ny=ny, seed=seed, vrms=0.8 if (rmn, odr) == (0, 2) else 1.2)
    assert np.isfinite(p.state).all()
    dn = np.zeros((3, 8), dtype=int)
    if seed % 2 == 0:
        dn[0] = [2] * 8
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    _say("2d vs oracle", seed, n, ny, rmn, odr)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, dn=dn)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 10, 1)
    with qas.Solver(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, dn=dn) as s:
        s.upload(p.state)
        hist, dt_now = s.run(10, flg=1)
        out = s.download()
    assert np.isfinite(ref).all()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("rmn,odr,walls", [(1, 2, False), (3, 3, True), (2, 1, False)])
def test_2d_column_emf_vs_oracle(qas, oracle, rmn, odr, walls):
    """Domains of 512^2 corners and more compute two EMF corners of a column
    per thread (k_emf2d<ODR, FT, 2>): the same arithmetic per corner as the
    one-corner forms (fused with the CT up to 300^2 cells, k_emf2d<ODR, FT, 1>
    between, test_2d_separate_emf_and_ct_vs_oracle), for every ODR's
    interpolation; a ragged last column (an odd corner count along y) and
    walls."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=516, ny=518, seed=7, vrms=0.8)
    dn = np.zeros((3, 8), dtype=int)
    if walls:
        dn[0] = [2] * 8
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    ny_g, nx_g = p.state.shape[1:]
    assert (nx_g - 5) * (ny_g - 5) >= 512 * 512 and (ny_g - 5) % 2 == 1
    _say("2d column EMF vs oracle", rmn, odr, walls)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, dn=dn)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 2, 1)
    with qas.Solver(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, dn=dn) as s:
        s.upload(p.state)
        hist, dt_now = s.run(2, flg=1)
        out = s.download()
    assert np.isfinite(ref).all()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("rmn,odr,ctw,walls", [(1, 1, 1, False), (0, 2, 1, True), (2, 3, 0, True), (3, 4, 1, True),
                                               (1, 3, 1, False)])
def test_2d_separate_emf_and_ct_vs_oracle(qas, oracle, rmn, odr, ctw, walls):
    """Between 300^2 cells and 512^2 corners the corner EMF (one corner a
    thread) and the CT with the ghost fill are launches of their own: every
    ODR's interpolation, walls, with and without the upwind weight."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=330, ny=301, seed=8, vrms=0.8)
    dn = np.zeros((3, 8), dtype=int)
    if walls:
        dn[0] = [2] * 8
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    _say("2d separate EMF and CT vs oracle", rmn, odr, ctw, walls)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, ctw=ctw, dn=dn)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 2, 1)
    with qas.Solver(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, odr=odr, ctw=ctw, dn=dn) as s:
        s.upload(p.state)
        hist, dt_now = s.run(2, flg=1)
        out = s.download()
    assert np.isfinite(ref).all()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("nx,ny,rmn,walls", [(1400, 128, 1, False), (1401, 130, 3, True), (2601, 59, 2, True),
                                             (5000, 16, 0, False)])
def test_2d_runs_across_columns_and_rows_vs_oracle(qas, oracle, nx, ny, rmn, walls):
    """Shapes whose y sweep cuts its runs across column groups (short columns,
    enough tiles to fill the chip), the last bundle and the last column group
    partly empty, and runs of the x sweep across rows: bit-identical in each
    x-sweep workgroup size."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=nx, ny=ny, seed=3, vrms=0.8)
    dn = np.zeros((3, 8), dtype=int)
    if walls:
        dn[0] = [2] * 8
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
    _say("2d runs across columns and rows", nx, ny, rmn, walls)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, dn=dn)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 2, 1)
    assert np.isfinite(ref).all()
    for xwpb in (1, 2, 4):
        with qas.Solver(p.state.shape[1:], p.dx, p.dy, gam=p.gam, rmn=rmn, dn=dn) as s:
            s.set_shape(xwpb, 256)
            s.upload(p.state)
            hist, dt_now = s.run(2, flg=1)
            assert np.array_equal(hist, h_ref) and dt_now == dt_ref
            assert np.array_equal(s.download(), ref), xwpb


@pytest.mark.parametrize("nx,ny,nz,rmn,odr,walls", [(41, 40, 90, 1, 4, False), (41, 40, 90, 3, 4, True),
                                                    (300, 9, 17, 2, 2, True), (17, 130, 8, 0, 3, False)])
def test_3d_runs_chunks_and_ghosts_vs_oracle(qas, oracle, nx, ny, nz, rmn, odr, walls):
    """3D shapes whose y and z sweeps cut their runs across column groups
    (short columns, many planes) or by column, with partly empty last groups;
    edge and face marches with a partly empty last chunk; planes that do not
    divide into workgroups; every boundary kind: bit-identical."""
    rng = np.random.default_rng(nx + ny)
    shape = (nz + 8, ny + 8, nx + 8)
    z, y, x = np.meshgrid(*[2 * np.pi * (np.arange(n) - 4) / (n - 8) for n in shape], indexing="ij")
    f = [sum(rng.uniform(0.2, 0.5) * np.cos(a * x + b * y + c * z + rng.uniform(0, 6)) for a, b, c in
             ((1, 0, 1), (0, 1, 1), (1, 1, 0))) for _ in range(8)]
    st = np.stack([1.5 + 0.3 * f[0], f[1], f[2], f[3], f[4], f[5], f[6], 8.0 + f[7]])
    dn = np.zeros((3, 8), dtype=int)
    if walls:
        dn[0] = [2] * 8
        dn[1] = [1, 1, -1, 1, 1, -1, 1, 1]
        dn[2] = [-2 if m == 3 else 2 for m in range(8)]
    _say("3d runs, chunks and ghosts", nx, ny, nz, rmn, odr, walls)
    d = 2 * np.pi / max(nx, ny, nz)
    cfg = oracle.make_cfg(shape, d, d, d, rmn=rmn, odr=odr, dn=dn)
    ref = st.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 2, 1)
    assert np.isfinite(ref).all()
    with qas.Solver(shape, d, d, d, rmn=rmn, odr=odr, dn=dn) as s:
        s.upload(st)
        hist, dt_now = s.run(2, flg=1)
        out = s.download()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("rmn,odr,ctw,precision", [(1, 4, 1, 0), (1, 4, 0, 0), (3, 3, 1, 0), (0, 2, 1, 0), (2, 1, 1, 0),
                                                   (1, 4, 1, 1), (3, 3, 0, 1)])
def test_3d_large_domain_is_its_tiles(qas, oracle, rmn, odr, ctw, precision):
    """Above 45 MB a face-part array the edge EMFs come from the form with all
    three components in a thread.  A periodic domain laid side by side is
    periodic with the same period, cell for cell: the large domain's step must
    be the small one's (other EMF form; in FP64 the oracle's) repeated."""
    n, rep = (20, 28, 24), (9, 7, 8) if precision == 0 else (12, 7, 9)  # nz, ny, nx; partly empty last chunk
    rng = np.random.default_rng(5)
    shape = tuple(m + 8 for m in n)
    z, y, x = np.meshgrid(*[2 * np.pi * (np.arange(m) - 4) / (m - 8) for m in shape], indexing="ij")
    f = [sum(rng.uniform(0.2, 0.5) * np.cos(a * x + b * y + c * z + rng.uniform(0, 6)) for a, b, c in
             ((1, 0, 1), (0, 1, 1), (1, 1, 0))) for _ in range(8)]
    st = np.stack([1.5 + 0.3 * f[0], f[1], f[2], f[3], f[4], f[5], f[6], 8.0 + f[7]])
    inner = st[:, 4:-4, 4:-4, 4:-4]
    big = np.tile(inner, (1,) + rep)
    big = np.pad(big, ((0, 0),) + ((4, 4),) * 3, mode="wrap")
    st = np.pad(inner, ((0, 0),) + ((4, 4),) * 3, mode="wrap")
    assert big[0].size * (4 if precision else 8) >= 45000000 > st[0].size * 8
    _say("3d large domain is its tiles", rmn, odr, ctw, precision, big.shape)
    out = []
    for u in (st, big):
        with qas.Solver(u.shape[1:], 0.1, 0.12, 0.11, rmn=rmn, odr=odr, ctw=ctw, precision=precision) as s:
            s.upload(u)
            s.run(1, flg=0, dt=2e-3, history=False)
            out.append(s.download())
    if precision == 0:
        cfg = oracle.make_cfg(st.shape[1:], 0.1, 0.12, 0.11, rmn=rmn, odr=odr, ctw=ctw)
        ref = st.copy()
        oracle.run(cfg, ref, 1, 0, dt=2e-3)
        assert np.array_equal(out[0], ref)
    want = np.pad(np.tile(out[0][:, 4:-4, 4:-4, 4:-4], (1,) + rep), ((0, 0),) + ((4, 4),) * 3, mode="wrap")
    assert np.isfinite(out[0]).all() and np.array_equal(out[1], want)


@pytest.mark.parametrize("n", [8, 52, 53, 57, 112, 4097])
@pytest.mark.parametrize("dn", [0, 1, -1, 2, -2])
def test_1d_stage_and_ghosts_vs_oracle(qas, oracle, n, dn):
    """The 1D stage's one launch at the ends of its 60-cell wavefronts, with
    every boundary kind (bx is staggered along x, so its last face is kept
    though not evolved), and the CFL reduction in one workgroup or two
    launches: bit-identical, ghosts included."""
    rng = np.random.default_rng(n)
    x = 2 * np.pi * np.arange(n + 8) / n
    f = [rng.uniform(0.1, 0.3) * np.sin(x + rng.uniform(0, 6)) for _ in range(8)]
    st = np.stack([1.0 + f[0], f[1], f[2], f[3], 0.7 + f[4], 0.5 + f[5], f[6], 4.0 + f[7]])
    flags = np.zeros((3, 8), dtype=int)
    flags[0] = dn
    flags[0, [0, 7]] = abs(dn)          # density and energy keep their sign
    flags[0, 4] = 2 if dn == -2 else dn  # (a zero normal field would stop the run)
    _say("1d stage and ghosts", n, dn)
    cfg = oracle.make_cfg((n + 8,), 1.0 / n, gam=1.4, dn=flags)
    ref = st.copy()
    oracle.bound(cfg, ref)
    h_ref, dt_ref = oracle.run(cfg, ref, 3, 1)
    with qas.Solver((n + 8,), 1.0 / n, gam=1.4, dn=flags) as s:
        s.upload(st)
        s.bound()
        hist, dt_now = s.run(3, flg=1)
        out = s.download()
    if dn != -2:
        assert np.isfinite(ref).all()
    assert np.array_equal(hist, h_ref, equal_nan=True) and np.array_equal(dt_now, dt_ref, equal_nan=True)
    assert np.array_equal(out, ref, equal_nan=True)


def test_1d_context_holds_its_states_only(qas):
    """The 1D stage keeps its primitives in LDS: three states of 8 arrays on
    the device, and the small words."""
    n = 100000
    with qas.Solver((n + 8,), 1.0 / n) as s:
        assert 24 * 8 * (n + 8) <= s.device_bytes < 24 * 8 * (n + 8 + 64) + 16384


@pytest.mark.parametrize("shape", [(64,), (48, 40), (40, 2500), (16, 18, 20)])
@pytest.mark.parametrize("rmn", [1, 2])
def test_work_model_is_of_the_launches(qas, shape, rmn):
    """qas_kernel_model has work for the kernels a step launches and none for
    the others; the stage's work does not depend on how it is cut into
    launches but for the corner EMF's way through memory."""
    import ctypes as C
    sh = tuple(m + 8 for m in shape)
    st = np.zeros((8,) + sh)
    st[0], st[4], st[7] = 1.0, 0.5, 3.0
    work = []
    _say("work model", shape, rmn)
    with qas.Solver(sh, 0.1, 0.1, 0.1, rmn=rmn) as s:
        s.upload(st)
        s.bound()
        s.sync()
        s.lib.qas_prof_enable(s.ctx, (1 << 6) - 1, 64)
        s.step(1e-3)
        for kid in range(6):
            ms, n, fl, by = C.c_double(), C.c_longlong(), C.c_double(), C.c_double()
            assert s.lib.qas_prof_query(s.ctx, kid, C.byref(ms), C.byref(n)) == 0
            r = s.lib.qas_kernel_model(s.ctx, kid, C.byref(fl), C.byref(by))
            assert n.value in (0, 3) and (n.value > 0) == (r == 0 and fl.value > 0) == (r == 0 and by.value > 0), kid
            work.append((n.value, fl.value, by.value) if r == 0 else (0, 0.0, 0.0))
        s.lib.qas_prof_enable(s.ctx, 0, 0)
    cells = np.prod(sh, dtype=float)
    # every launch moves the state or more, and the stage at least 16 arrays
    assert sum(w[2] for w in work) > 16 * 8 * np.prod(shape) and all(w[2] < 8 * 60 * cells for w in work)
    pf = (C.c_double * 8)()
    s.lib.qas_point_flops(rmn, 4, pf)
    assert sum(w[1] for w in work) > len(shape) * np.prod(shape) * (min(pf[0], pf[1]) + pf[2])


@pytest.mark.parametrize("nsteps", [1, 255, 256, 300])
def test_history_through_pinned_buffer_or_direct(qas, oracle, nsteps):
    """The dt history comes back with dt in one wait where it fits the pinned
    buffer (255 steps) and by a copy of its own beyond: every entry."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=16, seed=5, vrms=0.3)
    _say("history", nsteps)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, nsteps, 1)
    with qas.solver_for(p) as s:
        s.upload(p.state)
        hist, dt_now = s.run(nsteps, flg=1)
        out = s.download()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


def test_step_and_bound_entry_points(qas, oracle):
    """qas_bound / qas_step / qas_cfl_dt individually == bound / ideal / setdt."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=24, seed=9)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam)
    ref = p.state.copy()
    ref[:, :4, :] = 123.0  # stale ghosts: bound must rewrite them
    st = ref.copy()
    oracle.bound(cfg, ref)
    dt = oracle.cfl_dt(cfg, ref)
    oracle.step(cfg, ref, dt)
    with qas.Solver(p.state.shape[1:], p.dx, p.dy, gam=p.gam) as s:
        s.upload(st)
        s.bound()
        b = s.download()
        d = s.cfl_dt()
        s.step(d)
        out = s.download()
    assert d == dt
    st2 = st.copy()
    oracle.bound(cfg, st2)
    assert np.array_equal(b, st2)
    assert np.array_equal(out, ref)


def test_2d_full_size_invariants(qas):
    """1024^2 turbulence (the benchmark workload), 20 steps: periodic totals
    of ro, mx, my, mz, bz, en conserved to round-off, and the 4th-order
    corner divergence of the face B stays at round-off (CT)."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=1024, seed=2)
    _say("2d 1024^2 invariants")

    def divb(st):
        bx, by = st[4], st[5]
        d = p.dx
        dbx = (27.0 * (bx[4:-4, 5:-3] - bx[4:-4, 4:-4]) - (bx[4:-4, 6:-2] - bx[4:-4, 3:-5])) / 24.0 / d
        dby = (27.0 * (by[5:-3, 4:-4] - by[4:-4, 4:-4]) - (by[6:-2, 4:-4] - by[3:-5, 4:-4])) / 24.0 / d
        return np.abs(dbx + dby).max()

    st0 = p.state
    tot0 = st0[:, 4:-4, 4:-4].sum(axis=(1, 2))
    d0 = divb(st0)
    with qas.Solver(st0.shape[1:], p.dx, p.dy, gam=p.gam) as s:
        s.upload(st0)
        s.run(20, flg=1, history=False)
        out = s.download()
    assert np.isfinite(out).all()
    tot = out[:, 4:-4, 4:-4].sum(axis=(1, 2))
    scale = np.abs(st0[:, 4:-4, 4:-4]).sum(axis=(1, 2)) + 1.0
    for m in (0, 1, 2, 3, 6, 7):
        assert abs(tot[m] - tot0[m]) / scale[m] < 1e-12, m
    bmax = np.abs(out[4:6]).max()
    assert divb(out) < 1e-11 * bmax / p.dx + 10 * d0


def test_3d_full_size_invariants():
    """The 3D turbulence workload at its full size and length (512^3, 200
    steps) in a fresh process (tests/gpu_turb3d_full_check.py: the state is
    built and checked with torch on the device): periodic totals of rho, m
    and E at round-off, div B at round-off, finite."""
    import subprocess
    _say("3d 512^3 invariants, 200 steps (subprocess)")
    script = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gpu_turb3d_full_check.py")
    r = subprocess.run([sys.executable, "-u", script], capture_output=True, text=True, timeout=280)
    print(r.stdout[-3000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0


@pytest.mark.parametrize("rmn,odr,bc", [(1, 4, "periodic"), (3, 4, "mixed"), (2, 3, "periodic"), (0, 4, "mixed")])
def test_3d_vs_oracle(qas, oracle, rmn, odr, bc):
    from qasmhd_amd import problems
    p = problems.turbulence3d(n=16, seed=7, nmodes=12)
    dn = np.zeros((3, 8), dtype=int)
    if bc == "mixed":
        dn[0] = [2] * 8
        dn[2] = [1, 1, 1, -1, 1, 1, -1, 1]
    _say("3d vs oracle", rmn, odr, bc)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, p.dz, gam=p.gam, rmn=rmn, odr=odr, dn=dn)
    ref = p.state.copy()
    h_ref, dt_ref = oracle.run(cfg, ref, 4, 1)
    with qas.Solver(p.state.shape[1:], p.dx, p.dy, p.dz, gam=p.gam, rmn=rmn, odr=odr, dn=dn) as s:
        s.upload(p.state)
        hist, dt_now = s.run(4, flg=1)
        out = s.download()
    assert np.array_equal(hist, h_ref) and dt_now == dt_ref
    assert np.array_equal(out, ref)


def test_cpp_driver_matches_oracle(oracle, tmp_path):
    """The C++ host driver (include/qasmhd_driver.hpp), used the way a
    reference problem uses MHD2D, gives the oracle's result bit for bit."""
    import subprocess
    exe = os.path.join(os.path.dirname(GOLDEN), "cpp", "_build", "ot2d_driver")
    if not os.path.exists(exe):
        pytest.skip("C++ driver not built (run __graft_entry__.build())")
    init, final = str(tmp_path / "init.bin"), str(tmp_path / "final.bin")
    _say("cpp driver")
    r = subprocess.run([exe, "32", "24", "6", "1", init, final], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    shape = (8, 32, 40)
    st0 = np.fromfile(init).reshape(shape)
    out = np.fromfile(final).reshape(shape)
    d = 2 * np.pi / 32, 2 * np.pi / 24
    cfg = oracle.make_cfg(shape[1:], d[0], d[1])
    ref = st0.copy()
    oracle.run(cfg, ref, 6, 1)
    assert np.array_equal(out, ref)


def test_cpp_driver_output_and_restart(oracle, tmp_path):
    """dout_ / bkup files of the C++ driver in the reference's formats
    (2D/SERIAL/OTvortex/mhd2d_class.cpp:62-112, common/common_func.c:281-344),
    and a restart from the backup continues the run bit for bit: 6 steps,
    backup, 6 more steps == 12 straight steps of the oracle."""
    import subprocess
    exe = os.path.join(os.path.dirname(GOLDEN), "cpp", "_build", "ot2d_driver")
    if not os.path.exists(exe):
        pytest.skip("C++ driver not built (run __graft_entry__.build())")
    out = tmp_path / "dat"
    out.mkdir()
    init, mid, fin = str(tmp_path / "init.bin"), str(tmp_path / "mid.bin"), str(tmp_path / "fin.bin")
    _say("cpp driver restart")
    r = subprocess.run([exe, "32", "24", "6", "1", init, mid, str(out)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    shape = (8, 32, 40)
    st0 = np.fromfile(init).reshape(shape)
    # dout_(0) at n == 0: the initial state and the text files
    assert np.array_equal(np.fromfile(str(out / "outdat_00000.dat")).reshape(shape), st0)
    assert (out / "offsets.dat").read_text() == "4 4\n"
    assert (out / "params.dat").read_text() == "%f\n" % (5.0 / 3.0)
    x = np.loadtxt(str(out / "x.dat"))
    assert x.size == 40 and abs(x[4]) < 1e-12
    # backup after 6 steps
    n, cnt = (int(v) for v in (out / "bkup_stamp.dat").read_text().split())
    assert n >= 6
    tdt = np.fromfile(str(out / "bkup_time.dat"))
    assert tdt.size == 3 and tdt[1] > 0
    assert np.array_equal(np.fromfile(str(out / "bkup_data_00000.dat")).reshape(shape),
                          np.fromfile(mid).reshape(shape))
    r = subprocess.run([exe, "32", "24", "6", "1", init, fin, str(out), "restart"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    d = 2 * np.pi / 32, 2 * np.pi / 24
    cfg = oracle.make_cfg(shape[1:], d[0], d[1])
    ref = st0.copy()
    oracle.run(cfg, ref, 12, 1)
    assert np.array_equal(np.fromfile(fin).reshape(shape), ref)


def test_cpp_driver_mpi_files_and_resume(oracle, tmp_path):
    """The MPI drivers' file set and backup cycle as one rank (mpi_files;
    2D/MPI/OTvortex/mhd2d_class.cpp exec_ and dout_): an output and a
    backup after every step, outdat_%05d_00000.dat in FP32 (a plain cast of
    each value, common/common_func.c:22-26), mpinum.dat "1 1"; a second run
    over the same directory resumes from the backup and ends where 12
    straight steps of the oracle do, bit for bit."""
    import subprocess
    exe = os.path.join(os.path.dirname(GOLDEN), "cpp", "_build", "ot2d_driver")
    if not os.path.exists(exe):
        pytest.skip("C++ driver not built (run __graft_entry__.build())")
    out = tmp_path / "dat"
    out.mkdir()
    init, mid, fin = str(tmp_path / "init.bin"), str(tmp_path / "mid.bin"), str(tmp_path / "fin.bin")
    _say("cpp driver, MPI file set")
    r = subprocess.run([exe, "32", "24", "6", "1", init, mid, str(out), "mpi"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    shape = (8, 32, 40)
    st0 = np.fromfile(init).reshape(shape)
    st6 = np.fromfile(mid).reshape(shape)
    assert (out / "mpinum.dat").read_text() == "1 1\n"
    assert (out / "offsets.dat").read_text() == "4 4\n"
    assert np.loadtxt(str(out / "x_00000.dat")).size == 40
    assert np.loadtxt(str(out / "y_00000.dat")).size == 32
    assert np.array_equal(np.fromfile(str(out / "outdat_00000_00000.dat"), dtype=np.float32).reshape(shape),
                          st0.astype(np.float32))
    assert np.array_equal(np.fromfile(str(out / "outdat_00006_00000.dat"), dtype=np.float32).reshape(shape),
                          st6.astype(np.float32))
    assert not (out / "outdat_00007_00000.dat").exists()
    assert (out / "bkup_stamp.dat").read_text().split() == ["6", "6"]
    assert np.array_equal(np.fromfile(str(out / "bkup_data_00000.dat")).reshape(shape), st6)
    assert len((out / "t.dat").read_text().split()) == 7
    # resume: the same command with 12 steps continues from step 6
    r = subprocess.run([exe, "32", "24", "12", "1", init, fin, str(out), "mpi"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    d = 2 * np.pi / 32, 2 * np.pi / 24
    cfg = oracle.make_cfg(shape[1:], d[0], d[1])
    ref = st0.copy()
    oracle.run(cfg, ref, 12, 1)
    st12 = np.fromfile(fin).reshape(shape)
    assert np.array_equal(st12, ref)
    assert (out / "bkup_stamp.dat").read_text().split() == ["12", "12"]
    assert np.array_equal(np.fromfile(str(out / "outdat_00012_00000.dat"), dtype=np.float32).reshape(shape),
                          ref.astype(np.float32))
    assert len((out / "t.dat").read_text().split()) == 13
    # the reference's own merge tool (2D/MPI/common/merge.c, built from its
    # source) reads the file set: merged outputs are the FP32 interiors
    from oracle import build as obuild
    merge = os.path.join(obuild.REFOUT, "merge2d")
    if os.access(merge, os.X_OK):
        (tmp_path / "merged").mkdir()
        r = subprocess.run([merge, "dat", "merged"], capture_output=True, text=True, timeout=120, cwd=str(tmp_path))
        assert r.returncode == 0, r.stderr
        mdir = tmp_path / "merged"
        assert np.loadtxt(str(mdir / "merge_x.dat")).size == 32
        assert np.loadtxt(str(mdir / "merge_y.dat")).size == 24
        for c, st in ((0, st0), (6, st6), (12, ref)):
            m = np.fromfile(str(mdir / ("merge_outdat_%05d.dat" % c)), dtype=np.float32).reshape(8, 24, 32)
            assert np.array_equal(m, st[:, 4:-4, 4:-4].astype(np.float32)), c


def test_launch_shapes_bit_identical(qas, oracle):
    """Every 2D launch shape (x-sweep wavefronts per workgroup, element-wise
    workgroup size) gives the oracle's result bit for bit; qas_tune picks
    one of them without changing the state, and qas_run tunes on its first
    call unless a shape was set."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=40, ny=56, seed=6)
    _say("launch shapes 40x56")
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam)
    ref = p.state.copy()
    href, _ = oracle.run(cfg, ref, 6, 1)
    for xwpb, ewb in ((1, 64), (2, 128), (4, 256), (1, 256), (4, 64)):
        with qas.solver_for(p) as s:
            s.set_shape(xwpb, ewb)
            s.upload(p.state)
            h, _ = s.run(6, flg=1)
            assert s.shape_now() == (xwpb, ewb)  # a set shape is not re-tuned
            assert np.array_equal(s.download(), ref), (xwpb, ewb)
            assert np.array_equal(h, href)
    with qas.solver_for(p) as s:
        s.upload(p.state)
        shp = s.tune()
        assert shp[0] in (1, 2, 4) and shp[1] in (64, 128, 256)
        bounded = p.state.copy()
        oracle.bound(cfg, bounded)  # the tuner fills the ghosts, nothing else
        assert np.array_equal(s.download(), bounded)
        h, _ = s.run(6, flg=1)
        assert np.array_equal(s.download(), ref)
    with qas.solver_for(p) as s:
        s.upload(p.state)
        h, _ = s.run(6, flg=1)  # tunes first
        assert np.array_equal(s.download(), ref)
        assert np.array_equal(h, href)


@pytest.mark.parametrize("nx,ny", [(292, 292), (320, 300)])
def test_launch_shapes_where_they_matter(qas, oracle, nx, ny):
    """The largest domain whose corner EMF and CT are one launch (its tuned
    shape has the default element-wise size, which no launch of it uses), and
    one with separate launches, whose workgroup size is ewb: the oracle's bits
    in every shape."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=nx, ny=ny, seed=6)
    _say("launch shapes", nx, ny)
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam)
    ref = p.state.copy()
    href, _ = oracle.run(cfg, ref, 2, 1)
    for xwpb, ewb in ((1, 64), (2, 128), (4, 256), (1, 256), (4, 64)):
        with qas.solver_for(p) as s:
            s.set_shape(xwpb, ewb)
            s.upload(p.state)
            h, _ = s.run(2, flg=1)
            assert s.shape_now() == (xwpb, ewb)
            assert np.array_equal(s.download(), ref) and np.array_equal(h, href), (xwpb, ewb)
    for _ in range(8):
        with qas.solver_for(p) as s:
            s.upload(p.state)
            xwpb, ewb = s.tune()
            assert xwpb in (1, 2, 4) and (ewb == 256 if (nx + 8) * (ny + 8) <= 300 * 300 else ewb in (64, 128, 256))


@pytest.mark.parametrize("nsteps", [7, 10])
def test_graph_replay_matches_direct_launches(qas, oracle, nsteps):
    """qas_run with captured 2-step graphs == host-launched steps == oracle,
    including the dt history, over an odd and an even step count and a
    second call that continues the running counter."""
    from qasmhd_amd import problems
    p = problems.turbulence2d(n=48, seed=4)
    _say("graphs", nsteps)
    outs = []
    for graphs in (1, 0):
        with qas.solver_for(p) as s:
            s.lib.qas_use_graphs(s.ctx, graphs)
            s.upload(p.state)
            h1, _ = s.run(nsteps, flg=1)
            h2, _ = s.run(5, flg=1)
            outs.append((s.download(), np.concatenate([h1, h2])))
    cfg = oracle.make_cfg(p.state.shape[1:], p.dx, p.dy, gam=p.gam)
    ref = p.state.copy()
    href, dt = oracle.run(cfg, ref, nsteps, 1)
    href2, _ = oracle.run(cfg, ref, 5, 1, dt=dt) if nsteps % 2 == 0 else (None, None)
    for out, h in outs:
        assert np.array_equal(h[:nsteps], href)
    assert np.array_equal(outs[0][0], outs[1][0])
    assert np.array_equal(outs[0][1], outs[1][1])
    if nsteps % 2 == 0:
        assert np.array_equal(outs[0][0], ref)
