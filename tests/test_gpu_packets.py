"""Actions, energies and Delta V with the gradient correction as packets on the device
queue against the same kernels launched through HIP: bit for bit, in every mode, for
repeated calls between moves, with links given and changed, and from two threads whose
contexts share the queue.  The counts of requests and actions sent show that the packets
are what ran: a kernel the queue refuses would go through HIP with the same values."""
import threading

import numpy as np
import pytest

from tests.test_gpu_direct import _context

pytestmark = pytest.mark.gpu

GSF = ((2.0 / 3.0, 4.0 / 3.0), (0.0, 2.0 / 9.0), 2)


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


def _walk(gpu, packets, mode, M, N, correction, seed):
    L = (N / 0.02198) ** (1.0 / 3.0)
    rng = np.random.default_rng(seed)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    ctx = _context(gpu, L, M, N, 0.004, L, mode, b, packets=packets)
    if correction:
        ctx.set_action_factors(*GSF)
    nxt = np.stack([(np.arange(M)[:, None] + 1) % M + np.zeros((1, N), int),
                    np.zeros((M, 1), int) + np.arange(N)], axis=-1).astype(np.int32)
    swap = nxt.copy()
    if N > 1:
        swap[M - 1, 0, 1], swap[M - 1, 1, 1] = 1, 0
    out = []
    for k in range(6):
        n = min(M, 7 + 5 * k)
        sp = np.stack([rng.permutation(M)[:n], rng.integers(0, N, n)], axis=-1).astype(np.int32)
        new = rng.uniform(-0.5 * L, 0.5 * L, size=(n, 3))
        out.append(np.asarray(ctx.delta_action(sp, new, commit=True)))
        a, v = ctx.potentialAction(with_slices=True)
        out += [np.asarray(a), np.asarray(v), np.asarray(ctx.potentialAction())]
        links = (None, nxt, swap)[k % 3]
        out.append(np.asarray(list(ctx.energy(next_links=links).values())))
        out.append(np.asarray(list(ctx.virial_energy(3, next_links=links).values())))
    sent = [ctx.kernel_time(k)[1] for k in ("delta_packets", "action_packets")]
    return out, ctx.download_path(), sent


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("M,N,correction", [(40, 64, True), (41, 65, False), (20, 300, True), (6, 1, True)])
def test_packets_equal_launches(gpu, mode, M, N, correction):
    a, pa, sent = _walk(gpu, True, mode, M, N, correction, M)
    b, pb, none = _walk(gpu, False, mode, M, N, correction, M)
    assert np.array_equal(pa, pb)
    # every request is one; an action is one where the walker's factors are on the device
    # already (energy and virial_energy ask for unit factors in between), and with one bead
    # a slice there is nothing to launch
    assert sent == [6, 0 if N == 1 else 6 if correction else 11]
    assert none == [0, 0]
    for k, (x, y) in enumerate(zip(a, b)):
        assert np.array_equal(x, y, equal_nan=True), k


def test_two_threads(gpu):
    want = {s: _walk(gpu, False, 0, 40, 64, True, s) for s in (1, 2)}
    got = {}
    ts = [threading.Thread(target=lambda s=s: got.update({s: _walk(gpu, True, 0, 40, 64, True, s)})) for s in (1, 2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for s in (1, 2):
        assert np.array_equal(got[s][1], want[s][1])
        assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(got[s][0], want[s][0]))


def _mixed_calls(gpu, packets, M, N, correction, seed):
    """Actions between short and long requests, one in three of them committed."""
    L = (N / 0.02198) ** (1.0 / 3.0)
    rng = np.random.default_rng(seed)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    ctx = _context(gpu, L, M, N, 0.004, L, 0, b, packets=packets)
    if correction:
        ctx.set_action_factors(*GSF)
    out = []
    for k in range(40):
        n = (5, 31, min(M, 90))[k % 3]
        sp = np.stack([rng.permutation(M)[:n], rng.integers(0, N, n)], axis=-1).astype(np.int32)
        new = rng.uniform(-0.5 * L, 0.5 * L, size=(n, 3))
        out += [np.asarray(ctx.potentialAction()), np.array(ctx.delta_action(sp, new, commit=k % 3 == 1))]
    return out, ctx.download_path(), [ctx.kernel_time(k)[1] for k in ("delta_packets", "action_packets")]


def test_turns_of_four_threads(gpu):
    """Contexts of four threads take turns on the queue and launch on their streams when
    they get none: the values are those of one context alone."""
    cases = {0: (40, 64, True), 1: (125, 16, False), 2: (100, 200, False), 3: (60, 33, True)}
    want = {s: _mixed_calls(gpu, False, *c, s) for s, c in cases.items()}
    alone = _mixed_calls(gpu, True, *cases[1], 1)
    assert alone[2] == [40, 39]   # the first action comes before there is a ring
    got = {}
    ts = [threading.Thread(target=lambda s=s, c=c: got.update({s: _mixed_calls(gpu, True, *c, s)}))
          for s, c in cases.items()]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for s in cases:
        assert np.array_equal(got[s][1], want[s][1])
        assert all(np.array_equal(x, y) for x, y in zip(got[s][0], want[s][0])), s
    assert sum(g[2][0] for g in got.values()) > 0
