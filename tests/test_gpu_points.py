"""Device per-point functions against vectors written by the reference's own
functions (tests/golden/unit_vectors.npz, made by tests/golden/make_golden.py
through oracle/ref/unit.cpp).  One GPU thread per vector, through the same
device functions the stage kernels inline (qas_device.hpp); bit-exact:
array equality of float64 values (NaN where the reference gives NaN).

References: interpol / l_interp common/common_interp.c:7-150; fcen / df1
common/common_interp.h:10-24; mhd_lrstate common/mhd_func.c:108-161 with
mhd_m_reconst / mhd_a_reconst common/mhd_eigen.c:513-665; riemann[RMN]
common/mhd_flux.c:7-698; mhd_cuct_weight common/mhd_func.c:56-76."""
import os

import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu

U = np.load(os.path.join(GOLDEN, "unit_vectors.npz"))


def _eq_nan(a, b):
    both = np.isnan(a) & np.isnan(b)
    return np.array_equal(np.where(both, 0, a), np.where(both, 0, b))


@pytest.fixture(scope="module")
def pts():
    from qasmhd_amd import capi
    return capi.points


@pytest.mark.parametrize("kind", [0, 1, 2, 3, 10, 11, 12, 13])
def test_interp(pts, kind):
    print("case: interp kind", kind, flush=True)
    fl, fr = pts.interp(kind, U["interp_in"])
    ref = U["interp_%d" % kind]
    assert np.array_equal(fl, ref[:, 0]) and np.array_equal(fr, ref[:, 1])


def test_rcp_inrange_is_the_division(pts):
    """The reciprocal the WCNS-4 weights take (qas_device.hpp rcp_inrange:
    the estimate, Newton steps and correction of the FP64 division without
    its operand scaling and fix-up) equals 1.0 / d bit for bit over the
    whole range where the kernels use it, 2^-767 <= |d| <= 2^1022:
    log-uniform random values of both signs, the range ends, powers of two
    and significands of all ones."""
    print("case: rcp_inrange vs 1.0 / d", flush=True)
    rng = np.random.default_rng(21)
    e = rng.uniform(-767.0, 1022.0, 2_000_000)
    d = np.exp2(e) * rng.choice([-1.0, 1.0], e.size)
    ends = np.array([2.0 ** -767, 2.0 ** 1022, np.nextafter(2.0 ** 1022, 0), np.nextafter(2.0 ** -767, 1),
                     1.0, 3.0, 24.0, 1e-40, 1e40, 2.0 ** 700, 0.65 * 2.0 ** -700])
    k = np.arange(-767, 1022)
    allones = (2.0 - 2.0 ** -52) * np.exp2(k.astype(float))
    d = np.concatenate([d, ends, -ends, np.exp2(k.astype(float)), allones, -allones])
    fast, div = pts.rcp(d)
    assert np.array_equal(fast.view(np.int64), div.view(np.int64))
    assert np.array_equal(div, 1.0 / d)      # the device division is IEEE (numpy: correctly rounded)


def test_wcns4_across_magnitudes(pts, oracle):
    """WCNS-4 on stencils scaled from 1e-300 to 1e300: the smoothness
    denominators cross the in-range test (2^700) of the device's fast
    reciprocal both ways, and constant stencils hit d = eps.  Bit-exact
    against the oracle's C restatement (plain divisions), NaN where it has
    NaN."""
    print("case: wcns4 over magnitudes", flush=True)
    rng = np.random.default_rng(8)
    base = rng.standard_normal((201 * 64, 5))
    scale = np.repeat(10.0 ** np.arange(-300, 301, 3), 64)[:, None]
    f5 = base * scale
    const = np.repeat(rng.standard_normal((64, 1)), 5, axis=1)
    smooth = np.cumsum(rng.standard_normal((64, 5)) * 1e-3, axis=1) + 1.0
    f5 = np.concatenate([f5, const, smooth, smooth * 1e120, smooth * 1e-120])
    fl, fr = pts.interp(3, f5)
    ol, or_ = oracle.interp(3, f5)
    assert _eq_nan(fl, ol) and _eq_nan(fr, or_)
    ok = ~np.isnan(ol)
    assert np.array_equal(fl[ok].view(np.int64), ol[ok].view(np.int64))
    assert np.array_equal(fr[ok].view(np.int64), or_[ok].view(np.int64))


@pytest.mark.parametrize("odr", [1, 2, 3, 4])
def test_fcen_df(pts, odr):
    print("case: fcen/df odr", odr, flush=True)
    assert np.array_equal(pts.f4(0, odr, U["f4_in"]), U["fcen_%d" % odr])
    assert np.array_equal(pts.f4(1, odr, U["f4_in"]), U["df_%d" % odr])


@pytest.mark.parametrize("odr", [1, 2, 3, 4])
def test_lrstate(pts, odr):
    print("case: lrstate odr", odr, flush=True)
    vl, vr = pts.lrstate(odr, U["lrstate_st"], U["lrstate_bn"], float(U["lrstate_gam"]))
    assert np.array_equal(vl, U["lrstate_%d_vl" % odr])
    assert np.array_equal(vr, U["lrstate_%d_vr" % odr])


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
@pytest.mark.parametrize("g", ["g53", "g2", "g14"])
def test_flux(pts, rmn, g):
    print("case: flux rmn", rmn, g, flush=True)
    f = pts.flux(rmn, U["flux_L"], U["flux_R"], U["flux_bn"], float(U["flux_gam_" + g]), U["flux_dv"])
    assert _eq_nan(f, U["flux_%d_%s" % (rmn, g)])


def test_cuct(pts):
    print("case: cuct", flush=True)
    assert np.array_equal(pts.cuct(U["cuct_c"], U["cuct_b"]), U["cuct"])


def test_df_across_magnitudes(pts, oracle):
    """The 4th-order difference's division by 24 (a product with the rounded
    1/24 and one exact residual step) on differences from 1e-280 to 1e280,
    signed zeros, infinities and NaN: the bits of the oracle's division."""
    print("case: df over magnitudes", flush=True)
    rng = np.random.default_rng(31)
    f4 = rng.standard_normal((281 * 512, 4)) * np.repeat(10.0 ** np.arange(-280, 281, 2), 512)[:, None]
    ints = rng.integers(-200, 200, (4096, 4)).astype(float)     # exact quotients and ties among them
    odd = np.array([[0.0, 0.0, 0.0, 0.0], [0.0, -0.0, -0.0, 0.0], [1.0, 2.0, 2.0, 1.0], [np.inf, 1.0, 2.0, 3.0],
                    [1.0, np.inf, 1.0, 1.0], [np.nan, 1.0, 1.0, 1.0]])
    f4 = np.concatenate([f4, ints, odd])
    out, ref = pts.f4(1, 4, f4), oracle.df(4, f4)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(out), nan)
    assert np.array_equal(out[~nan].view(np.int64), ref[~nan].view(np.int64))


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
def test_flux_across_magnitudes(pts, oracle, rmn):
    """The fluxes' reciprocals, quotients and roots without operand scaling,
    on states whose density, speed and pressure run over 1e-40 .. 1e40 (all
    intermediate values inside 2^-960 .. 2^960), on states at rest, without
    field, with equal sides, and with the contact at exactly the speed of a
    rotational wave: the oracle's values, NaN where it has NaN."""
    print("case: flux over magnitudes, rmn", rmn, flush=True)
    rng = np.random.default_rng(40 + rmn)
    n = 40000
    q = rng.uniform(0.5, 2.0, (2, n, 7)) * np.where(np.arange(7) % 6 == 0, 1.0, rng.choice([-1.0, 1.0], (2, n, 7)))
    bn = rng.uniform(-2.0, 2.0, n)
    dv = rng.uniform(-0.2, 0.2, (n, 2))
    a, b = 10.0 ** rng.uniform(-40, 40, n), 10.0 ** rng.uniform(-25, 25, n)
    scale = np.stack([a, b, b, b, np.sqrt(a) * b, np.sqrt(a) * b, a * b * b], axis=1)
    scale[:n // 4] = 1.0
    q = q * scale
    bn, dv = bn * scale[:, 4], dv * scale[:, 1:2]
    k = n // 64                      # special states, at scale 1
    q[1, :k] = q[0, :k]              # equal sides
    q[:, k:2 * k, 1:4] = 0.0         # at rest
    q[:, 2 * k:3 * k, 4:6] = 0.0     # no field
    bn[2 * k:3 * k] = 0.0
    q[1, 3 * k:4 * k] = q[0, 3 * k:4 * k]   # equal sides with v_n = |B_n| / sqrt(ro): ro = 1, 4
    q[:, 3 * k:4 * k, 0] = rng.choice([1.0, 4.0], k)
    bn[3 * k:4 * k] = rng.integers(1, 16, k) / 8.0
    q[:, 3 * k:4 * k, 1] = bn[3 * k:4 * k] / np.sqrt(q[0, 3 * k:4 * k, 0]) * rng.choice([-1.0, 1.0], k)
    out, ref = pts.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv), oracle.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv)
    assert _eq_nan(out, ref)


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
def test_flux_with_tiny_velocities_and_fields(pts, oracle, rmn):
    """Densities and pressures of order 1 with some velocities and field
    components from 1e-320 to 1e-50, as in the tails of a localised
    perturbation: their squares, the normal field's above all, are denormal or
    underflow.  The oracle's values."""
    print("case: flux, tiny velocities and fields, rmn", rmn, flush=True)
    rng = np.random.default_rng(50 + rmn)
    n = 40000
    for lo, hi in ((-100, -50), (-165, -140), (-200, -100), (-290, -200), (-320, -290)):
        q = rng.uniform(0.5, 2.0, (2, n, 7)) * np.where(np.arange(7) % 6 == 0, 1.0, rng.choice([-1.0, 1.0], (2, n, 7)))
        bn = rng.uniform(-2.0, 2.0, n)
        dv = rng.uniform(-0.2, 0.2, (n, 2))
        q[1, : n // 4] = q[0, : n // 4]  # equal sides but for what is tiny
        for a in (q[..., 1], q[..., 2], q[..., 3], q[..., 4], q[..., 5], bn):
            a *= np.where(rng.random(n) < 0.7, 10.0 ** rng.uniform(lo, hi, a.shape), 1.0)
        out, ref = pts.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv), oracle.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv)
        assert _eq_nan(out, ref), (lo, hi)


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
@pytest.mark.parametrize("side", ["left", "right", "both"])
@pytest.mark.parametrize("var", [0, 6])
def test_flux_of_broken_states(pts, oracle, rmn, side, var):
    """A negative density or pressure on either side: the oracle's values, NaN
    where it has NaN (a run that breaks down must show it)."""
    print("case: flux, negative variable", var, side, "rmn", rmn, flush=True)
    rng = np.random.default_rng(60 + rmn)
    n = 20000
    q = rng.uniform(0.5, 2.0, (2, n, 7)) * np.where(np.arange(7) % 6 == 0, 1.0, rng.choice([-1.0, 1.0], (2, n, 7)))
    bn = rng.uniform(-2.0, 2.0, n)
    bn[: n // 8] = 0.0
    dv = rng.uniform(-0.2, 0.2, (n, 2))
    for s in {"left": (0,), "right": (1,), "both": (0, 1)}[side]:
        q[s, :, var] *= -1.0
    out, ref = pts.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv), oracle.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv)
    assert _eq_nan(out, ref)


@pytest.mark.parametrize("rmn", [0, 1, 2, 3])
def test_flux_to_the_ends_of_its_range(pts, oracle, rmn):
    """Speeds of 1e-76 to 1e76 (their fourth powers are normal numbers) and
    densities of 1e-302 to 1e302: the oracle's values."""
    print("case: flux, ends of the range, rmn", rmn, flush=True)
    rng = np.random.default_rng(70 + rmn)
    n = 20000
    for d, v in [(1.0, 10.0 ** k) for k in (-76, -60, 60, 76)] + [(10.0 ** k, 1.0) for k in (-302, -290, 290, 302)]:
        q = rng.uniform(0.5, 2.0, (2, n, 7)) * np.where(np.arange(7) % 6 == 0, 1.0, rng.choice([-1.0, 1.0], (2, n, 7)))
        b = np.sqrt(d) * v
        q *= np.array([d, v, v, v, b, b, d * v * v])
        bn, dv = rng.uniform(-2.0, 2.0, n) * b, rng.uniform(-0.2, 0.2, (n, 2)) * v
        out, ref = pts.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv), oracle.flux(rmn, q[0], q[1], bn, 5.0 / 3.0, dv)
        assert np.isfinite(ref).any() and _eq_nan(out, ref), (d, v)
