"""Delta V requests of more than 32 beads: the direct form with the bead list read
from pinned memory (up to 512 beads, slices of up to 1024), and the one-kernel form
beyond.  Packets, HIP launches and timed calls agree bit for bit; A_old and A_new
equal the per-bead sums to rounding (n 2^-52 of the largest partial sum, bounded by
1e-12 of the sum of magnitudes); committed beads and cells equal update_beads'."""
import numpy as np
import pytest

from tests.test_gpu_direct import LAMBDA, _context

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("n,M,N,cells", [(32, 40, 20, False), (33, 40, 20, False), (143, 143, 181, True),
                                         (512, 512, 17, False), (513, 520, 9, False), (40, 48, 1025, True),
                                         (33, 33, 1024, False)])
def test_long_requests(gpu, mode, n, M, N, cells):
    L = (N / 0.02198) ** (1.0 / 3.0)
    rc = 0.24 * L if cells else L
    rng = np.random.default_rng(n)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    sp = np.stack([rng.permutation(M)[:n], rng.integers(0, N, n)], axis=-1).astype(np.int32)
    new = rng.uniform(-0.5 * L, 0.5 * L, size=(n, 3))
    ctx = [_context(gpu, L, M, N, 0.004, rc, mode, b, packets=p) for p in (True, False, True)]
    ctx[2].set_timing(True, kinds=["delta_action"])
    out = [c.delta_action(sp, new) for c in ctx]
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
    vf = 0.004
    _, old = ctx[0].action_list(sp, per_bead=True)
    out2 = [c.delta_action(sp, new, commit=True) for c in ctx]
    assert all(np.array_equal(out[0], o) for o in out2)
    _, now = ctx[0].action_list(sp, per_bead=True)
    for got, v in ((out[0][0], old), (out[0][1], now)):
        assert abs(got - vf * v.sum()) <= 1e-12 * vf * np.abs(v).sum()
    ref = _context(gpu, L, M, N, 0.004, rc, mode, b, packets=True)
    ref.update_beads(sp, new)
    for c in ctx:
        assert np.array_equal(c.download_path(), ref.download_path())
        a, r = c.cell_lists(), ref.cell_lists()
        assert all(np.array_equal(a[k], r[k]) for k in ("grid", "bead_label", "num_labels"))


def test_lists_rewritten_in_place(gpu):
    """The list's block is written again for every request and read in place by the packet's
    kernel: requests of changing lengths, beads and positions, one after another, are those
    of a context that launches through HIP, bit for bit."""
    rng = np.random.default_rng(8)
    M, N = 512, 24
    L = (N / 0.02198) ** (1.0 / 3.0)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    a, h = (_context(gpu, L, M, N, 0.004, L, 0, b, packets=p) for p in (True, False))
    for k in range(60):
        n = int(rng.integers(33, M + 1))
        sp = np.stack([rng.permutation(M)[:n], rng.integers(0, N, n)], axis=-1).astype(np.int32)
        new = rng.uniform(-0.5 * L, 0.5 * L, size=(n, 3))
        commit = k % 5 == 4
        assert np.array_equal(a.delta_action(sp, new, commit=commit), h.delta_action(sp, new, commit=commit)), (k, n)
    assert a.kernel_time("delta_packets")[1] == 60 - 1   # the first long request goes through HIP
    assert h.kernel_time("delta_packets")[1] == 0
    assert np.array_equal(a.download_path(), h.download_path())
