"""The all-pairs kernel's bins at the edges where its short cuts hand over.

The exact modes take the bin from the mixed mode's |w| unless that lies within 1e-4
of a whole number: separations at whole multiples of dr and a few 1e-5 dr to either
side, beads on one point, and pairs at half the box must land in the oracle's bins.
One bin off moves V by dV/dr dr, about 1e-6 of it; the sums agree to rounding
(1e-12; 1e-9 where V is evaluated in closed form, 1e-6 with FP32 exponentials), so
the table and closed-form modes see a single wrong bin among the few pairs here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = {0: 1e-6, 1: 1e-9, 2: 1e-12}
RM = 2.9673


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


def _compare(orc, gpu, b, L, mode):
    M, N = b.shape[:2]
    ref = orc.State(L, M, N, 0.004, 6.0596, L)
    ref.set_beads(b)
    ctx = gpu.Context(L, M, N, 0.004, 6.0596, L, v_mode=mode)
    ctx.upload_path(b)
    a, r = ctx.potentialAction(), ref.total_action()
    assert abs(a - r) <= TOL[mode] * max(abs(r), 1e-3), (a, r)


@pytest.mark.parametrize("mode", [1, 2])   # the mixed mode's bin is its own within 1e-8 of a whole number
@pytest.mark.parametrize("x", [0.5, 0.9, 1.0, 1.2413, 1.5, 3.0, 5.0])
def test_bin_edges(orc, gpu, mode, x):
    """Two beads per slice inside the box, |r| = (k + e) dr, e around 0, along each axis and the diagonal."""
    L, dr = 30.0, 1e-6 * RM
    k = round(x * 1e6)
    e = np.array([-2e-4, -9.9e-5, -1e-5, -1e-7, 0.0, 1e-7, 1e-5, 9.9e-5, 2e-4, 0.5])
    dirs = np.array([[1, 0, 0], [0, 1, 0], [0, 0, 1], [1, 1, 1] / np.sqrt(3.0)])
    d = ((k + e)[:, None, None] * dr * dirs[None]).reshape(-1, 3)
    b = np.zeros((len(d), 2, 3))
    b[:, 1] = d
    b += np.random.default_rng(k).uniform(-5.0, 0.0, size=(len(d), 1, 3)) * (np.arange(len(d)) % 2)[:, None, None]
    _compare(orc, gpu, b, L, mode)


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("N", [2, 3, 7, 64, 65, 130])
def test_coincident_and_half_box(orc, gpu, mode, N):
    """Beads on one point (V = 0), a bead half the box away along one, two and three axes, corner pairs."""
    L = 12.0
    rng = np.random.default_rng(N)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(4, N, 3))
    b[0, 1] = b[0, 0]
    b[1, 1] = b[1, 0] - np.sign(b[1, 0]) * np.array([0.5 * L, 0, 0])
    b[2, 1] = b[2, 0] - np.sign(b[2, 0]) * np.array([0.5 * L, 0.5 * L, 0])
    b[3, 0], b[3, 1] = -0.5 * L, 0.0      # |r| = maxSep, past the table
    _compare(orc, gpu, b, L, mode)


@pytest.mark.parametrize("L", [100.0, 700.0, 7000.0])
def test_bins_of_large_boxes(gpu, L):
    """Up to 2e9 bins, the most an int holds: |r| = (k + e) dr at half the longest separations,
    e around 0.  V ~ k^-6, so one bin off moves it by 6/k of itself, 3e-9 and more."""
    dr, s = 1.0e-6 * RM, 1.0e-6 * RM / RM
    rng = np.random.default_rng(int(L))
    M = 3000
    k = rng.integers(int(0.3 * L / dr), int(0.49 * np.sqrt(3.0) * L / dr), M)
    e = rng.choice([-1.5e-4, -9e-5, -5e-5, -1e-5, -1e-6, 0.0, 1e-6, 1e-5, 5e-5, 9e-5, 1.5e-4], M)
    u = rng.uniform(0.9, 1.0, size=(M, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    b = np.zeros((M, 2, 3))
    b[:, 0] = -0.25 * L
    b[:, 1] = b[:, 0] + (k + e)[:, None] * dr * u
    # the reference's bin: separation, minimum image, norm, root and quotient in its order
    d = b[:, 1] - b[:, 0]
    d = d - L * np.floor(d * (1.0 / L) + 0.5)
    bins = (np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]) / dr).astype(np.int64)
    assert bins.max() < 2 ** 31 and len(set(bins - k)) > 1
    ctx = gpu.Context(L, M, 2, 0.004, 6.0596, L, v_mode=1)
    ctx.upload_path(b)
    v = ctx.potential_slices()[:, 1]
    x2 = (bins * s) ** -2.0
    want = -10.8 * (1.3732412 * x2 ** 3 + 0.4253785 * x2 ** 4 + 0.1781 * x2 ** 5)
    assert (np.abs(v / want - 1.0) < 2.0 / bins).all()
