"""The pair terms against extended precision (numpy's 80-bit long double).

FP64 mode: V and dV/dr at the bin radius x = k s, whose reciprocals and exponentials are
the kernels' own, are no further off than the reference's formulas in plain FP64 (IEEE
quotients and square root, the library's exponential): rms over 20 000 to 50 000 bins of
each range of x, within the 5 % that two such samples may differ by, over the sizes of the
terms that make them up.

Mixed mode: V of far pairs that share a wave with a pair of another kind takes the form
with the damping test.  Beyond x = 3 the repulsion, whose exponential is FP32, is below
1e-8 of the dispersion and its error below 1e-15; 1/k^2 is within 2^-46, so V is within
3 2^-46 and some fifty roundings of the coefficients and the sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble
YEARS = {1979: dict(eps=10.8, rm=2.9673, D=1.241314, al=13.353384, be=0.0, C6=1.3732412, C8=0.4253785, C10=0.1781,
                    A=0.5448504e6),
         1987: dict(eps=10.948, rm=2.9673, D=1.4826, al=10.43329537, be=-2.27965105, C6=1.36745214, C8=0.42123807,
                    C10=0.17473318, A=1.8443101e5),
         1995: dict(eps=10.956, rm=2.9683, D=1.438, al=10.5717543, be=-2.07758779, C6=1.35186623, C8=0.4149514,
                    C10=0.17151143, A=1.86924404e5)}
RANGES = [(0.05, 0.3), (0.3, 0.6), (0.6, 0.9), (0.9, 1.1), (1.1, 1.4), (1.5, 2.0), (2.0, 3.0), (3.0, 4.5), (4.5, 8.0)]


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


def _dr(p):
    return 1.0e-6 * p["rm"]


def _bins(p, lo, hi, n, seed):
    s = _dr(p) / p["rm"]
    return np.random.default_rng(seed).integers(int(lo / s), int(hi / s), n), s


def _v_terms(x, p, T):
    """Repulsion, dispersion and damping factor in type T, in valueV's order."""
    c = {k: T(v) for k, v in p.items()}
    rep = c["A"] * np.exp(-c["al"] * x + c["be"] * x * x)
    ix2 = T(1) / (x * x)
    ix6 = ix2 * ix2 * ix2
    disp = c["C6"] * ix6 + c["C8"] * ix6 * ix2 + c["C10"] * ix6 * ix2 * ix2
    t = c["D"] / x - T(1)
    return rep, disp, np.where(x < c["D"], np.exp(-t * t), T(1))


def _dv_terms(x, p, T):
    """The three terms of dV/dx in type T, in valuedVdr's order."""
    c = {k: T(v) for k, v in p.items()}
    rep = c["A"] * (-c["al"] + T(2) * c["be"] * x) * np.exp(-c["al"] * x + c["be"] * x * x)
    ix = T(1) / x
    ix2 = ix * ix
    ix6 = ix2 * ix2 * ix2
    ix7, ix8, ix10 = ix6 * ix, ix6 * ix2, ix6 * ix2 * ix2
    t = c["D"] * ix - T(1)
    F = np.where(x < c["D"], np.exp(-t * t), T(1))
    dF = np.where(x < c["D"], T(2) * c["D"] * ix2 * t * np.exp(-t * t), T(0))
    return (rep, (T(6) * c["C6"] * ix7 + T(8) * c["C8"] * (ix8 * ix) + T(10) * c["C10"] * (ix10 * ix)) * F,
            (c["C6"] * ix6 + c["C8"] * ix8 + c["C10"] * ix10) * dF)


def _rms(x):
    return float(np.sqrt(np.mean(np.square(x))))


@pytest.mark.parametrize("year", sorted(YEARS))
def test_v_fp64(gpu, year):
    p = YEARS[year]
    az = gpu.Aziz(year, 10.0 * p["rm"], 5.0 * p["rm"], v_mode=1)
    for i, (lo, hi) in enumerate(RANGES):
        k, s = _bins(p, lo, hi, 50000, year + i)
        x = k.astype(float) * s
        sep = np.zeros((len(k), 3))
        sep[:, 0] = (k + 0.5) * _dr(p)
        rep, disp, F = _v_terms(x.astype(LD), p, LD)
        want, size = LD(p["eps"]) * (rep - disp * F), LD(p["eps"]) * (rep + disp * F)
        r, d, f = _v_terms(x, p, np.float64)
        plain = _rms((p["eps"] * (r - d * f) - want) / size)
        got = _rms((az.V(sep) - want) / size)
        assert got <= 1.05 * plain, (lo, hi, got, plain)


@pytest.mark.parametrize("year", sorted(YEARS))
def test_dv_fp64(gpu, year):
    """Two beads per slice: gradVSquared = 2 (dV/dr)^2."""
    p, M, L = YEARS[year], 4000, 60.0
    ctx = gpu.Context(L, M, 2, 0.004, 6.0596, L, year=year, v_mode=1)
    for i, (lo, hi) in enumerate(RANGES):
        k, s = _bins(p, lo, hi, 5 * M, year + 50 + i)
        x = k.astype(float) * s
        t1, t2, t3 = _dv_terms(x.astype(LD), p, LD)
        c = LD(p["eps"]) / LD(p["rm"])
        want, size = np.abs(c * (t1 + t2 - t3)), c * (np.abs(t1) + t2 + np.abs(t3))
        t1, t2, t3 = _dv_terms(x, p, np.float64)
        sep = (k + 0.5) * _dr(p)
        plain = ((p["eps"] / p["rm"]) * (t1 + t2 - t3)) / sep * sep
        plain = _rms((np.sqrt((2.0 * plain * plain).astype(LD) / 2) - want) / size)
        got = np.empty(0)
        for b in range(5):
            beads = np.zeros((M, 2, 3))
            beads[:, 1, 0] = sep[b * M:(b + 1) * M]
            ctx.upload_path(beads)
            got = np.append(got, ctx.gradVSquared())
        got = _rms((np.sqrt(got.astype(LD) / 2) - want) / size)
        assert got <= 1.05 * plain, (lo, hi, got, plain)


def test_v_mixed_far_beside_others(gpu):
    p, M, L = YEARS[1979], 4000, 41.234
    dr, half = _dr(p), 0.5 * L
    assert 0.1 < (np.sqrt(0.75) * L / dr) % 1.0 < 0.9   # bead 2 is past the table from bead 0
    s = dr / p["rm"]
    k = np.random.default_rng(1).integers(int(3.0 / s), int(6.5 / s), 3 * M)
    r01 = (k + 0.5) * dr
    r12 = np.sqrt((half - r01) ** 2 + 2.0 * half ** 2)
    w = r12 / dr
    ok = (w % 1.0 > 0.1) & (w % 1.0 < 0.9)
    r01, k01, k12 = r01[ok][:M], k[ok][:M], np.floor(w[ok][:M])
    assert len(r01) == M
    beads = np.zeros((M, 3, 3))
    beads[:, 1, 0] = r01
    beads[:, 2] = -half
    ctx = gpu.Context(L, M, 3, 0.004, 6.0596, L)
    ctx.upload_path(beads)
    _, v = ctx.potentialAction(with_slices=True)
    got = np.asarray(v).reshape(M, -1)[:, -1]
    want = 0
    for kk in (k01, k12):
        rep, disp, F = _v_terms(kk.astype(LD) * LD(s), p, LD)
        want = want + LD(p["eps"]) * (rep - disp * F)
    assert np.abs((got - want) / want).max() <= 3 * 2.0 ** -46 + 50 * 2.0 ** -53
