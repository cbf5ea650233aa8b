"""The density modes of a q list in the matrix form (k_rho_matrix) and in the lane
form (k_rho_lattice) at the edges of both: table sizes (|n| <= 4, 8, 16, 20, 24, 32, 40) and
the blocks of 16 rows, 16 columns and 32 beads, permuted and repeated lists, lists
without their -q, and lists mixed with general q.

A list too sparse for the matrix form takes the lane form, and the two are equal
bit for bit by design (the same FP32 sums over 32 beads in the same order, the same
FP64 sums); every value is also compared with FP64 phasors.  Tolerance: a phasor
table entry is off by at most one FP32 product of two entries within 1 ulp (4 2^-24),
X Y Z by 12 2^-24, a 32-bead sum by 32 2^-24 of its terms more, so |d rho| <= 44 2^-24 N,
and with S = sum_m |rho|^2 / N, |rho| <= N: |dS| <= 2 M 44 2^-24 N = 5.3e-6 M N; the
same bound holds for F."""
import numpy as np
import pytest

from tests._oracle_util import isf_from_rho, lattice_rho

pytestmark = pytest.mark.gpu
BOUND = 5.3e-6


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


def _context(gpu, N, M, seed=5):
    L = 10.0
    rng = np.random.default_rng(seed)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    ctx = gpu.Context(L, M, N, 0.004, 6.0596, L)
    ctx.upload_path(b)
    return ctx, b, L


def _box(hx, hy, hz):
    r = [np.arange(-h, h + 1) for h in (hx, hy, hz)]
    return np.stack(np.meshgrid(*r, indexing="ij"), axis=-1).reshape(-1, 3)


def _q(n, L):
    return n * 2.0 * np.pi / L


def _check(ctx, b, L, n, N, M):
    s, f = ctx.ssf(_q(n, L)), ctx.isf(_q(n, L))
    ref = isf_from_rho(lattice_rho(b, n, L), N)
    assert np.abs(s - ref[:, 0]).max() <= BOUND * M * N
    assert np.abs(f - ref).max() <= BOUND * M * N
    return s, f


@pytest.mark.parametrize("N", [1, 3, 4, 31, 32, 33, 65, 100])
def test_bead_counts(gpu, N):
    M = 5
    ctx, b, L = _context(gpu, N, M)
    _check(ctx, b, L, _box(3, 3, 3), N, M)


@pytest.mark.parametrize("h", [(0, 0, 0), (1, 0, 0), (0, 0, 1), (2, 3, 4), (5, 4, 3), (8, 7, 9), (3, 9, 15),
                               (2, 2, 16), (4, 2, 17), (1, 1, 31), (1, 2, 33), (2, 20, 3), (21, 2, 2),
                               (3, 3, 24), (25, 1, 2), (40, 1, 1), (1, 40, 2), (2, 1, 40)])
def test_table_sizes(gpu, h):
    N, M = 37, 4
    ctx, b, L = _context(gpu, N, M)
    n = _box(*h)
    s, f = _check(ctx, b, L, n, N, M)
    # a few of them, far apart, take the lane form
    few = np.linspace(0, len(n) - 1, min(len(n), 9)).astype(int)
    assert np.array_equal(ctx.ssf(_q(n[few], L)), s[few])
    assert np.array_equal(ctx.isf(_q(n[few], L)), f[few])
    assert np.array_equal(ctx.ssf_noalloc(_q(n, L)), s)


@pytest.mark.parametrize("kind", ["shuffled", "reversed", "repeated", "half", "sparse", "mixed"])
def test_list_orders(gpu, kind):
    N, M = 50, 7
    ctx, b, L = _context(gpu, N, M)
    rng = np.random.default_rng(2)
    n = _box(6, 6, 6)
    s, f = _check(ctx, b, L, n, N, M)
    if kind == "mixed":
        k = rng.permutation(len(n))[:40]
        q = np.concatenate([_q(n[k[:20]], L), [[0.3, 0.1, 0.2]], _q(n[k[20:]], L), [[0.0, 0.05, 0.0]]])
        at = [i for i in range(42) if i not in (20, 41)]
        assert np.array_equal(ctx.ssf(q)[at], s[k]) and np.array_equal(ctx.isf(q)[at], f[k])
        one = ctx.isf(q[[20, 41]])
        assert np.array_equal(ctx.isf(q)[[20, 41]], one)
        return
    k = {"shuffled": rng.permutation(len(n)), "reversed": np.arange(len(n))[::-1],
         "repeated": rng.integers(0, len(n), 3 * len(n)), "half": np.arange(len(n) // 2 + 1),
         "sparse": rng.permutation(len(n))[:30]}[kind]
    assert np.array_equal(ctx.ssf(_q(n[k], L)), s[k])
    assert np.array_equal(ctx.isf(_q(n[k], L)), f[k])


@pytest.mark.parametrize("kind", ["list", "shuffled", "repeated", "repeated often"])
def test_pieces_into_pinned(gpu, kind):
    """F into page-locked memory (more than 4 MB) in several pieces: rows copied as they
    complete, whatever the list's order; the values of the pageable result."""
    N, M = 33, 96
    ctx, b, L = _context(gpu, N, M)
    n = _box(11, 11, 11)
    rng = np.random.default_rng(3)
    k = {"list": np.arange(len(n)), "shuffled": rng.permutation(len(n)),
         "repeated": np.concatenate([np.arange(len(n)), [5, 5, 700]]),       # copied by the host
         "repeated often": np.concatenate([np.arange(len(n)), rng.integers(0, len(n), 900)])}[kind]   # by the device
    q = _q(n[k], L)
    out = gpu.pinned_empty((len(k), M))
    out[:] = -1.0
    ctx.isf(q, out=out)
    # a list whose order scatters the pieces' rows is copied at the end
    assert ctx.kernel_time("isf_chunks")[1] == 2
    assert ctx.kernel_time("isf_dma")[1] == (2 if kind in ("list", "repeated") else 0)
    assert np.array_equal(out, ctx.isf(q))
    ref = isf_from_rho(lattice_rho(b, n[k][::97], L), N)
    assert np.abs(out[::97] - ref).max() <= BOUND * M * N


@pytest.mark.parametrize("nq", [1, 2, 33, 500, 2500])
def test_few_q_of_a_large_box(gpu, nq):
    """Lists that leave their box mostly empty find their modes by a hash table: q, -q and
    repeats of either, up to a table half full, against FP64 phasors and each other."""
    N, M = 20, 3
    ctx, b, L = _context(gpu, N, M)
    rng = np.random.default_rng(nq)
    n = rng.integers(-40, 41, size=(nq, 3))
    n[0] = (40, 40, 40)
    s, f = _check(ctx, b, L, n, N, M)
    k = rng.integers(0, nq, 4 * nq)
    sign = rng.choice([-1, 1], size=(4 * nq, 1))
    assert np.array_equal(ctx.ssf(_q(n[k] * sign, L)), s[k])
    assert np.array_equal(ctx.isf(_q(n[k] * sign, L)), f[k])


@pytest.mark.parametrize("M", [1, 2, 3, 7, 8, 9, 64, 126, 127, 128, 129, 511, 512])
def test_lags_and_parts(gpu, M):
    """Lags up to M / 2 and their mirror images, and S in eight parts, at every remainder."""
    N = 6
    ctx, b, L = _context(gpu, N, M)
    _check(ctx, b, L, _box(1, 1, 1), N, M)
