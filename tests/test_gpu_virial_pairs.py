"""The virial pair sums over unordered pairs at the edges of their 64-bead tiles (one
to sixteen of them), beyond 1024 beads, for slices that need the T matrix and slices
that don't, for ragged slices, and with pairs exactly half a box apart (whose minimum
image has the same sign from either end), against the oracle.  Tolerances as in
test_gpu_virial: the bins and pair values are the same, only the summation order is not."""
import numpy as np
import pytest

from tests.test_gpu_virial import GSF, LB, PRIM, TOL, close, make

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


@pytest.mark.parametrize("N,M,mode,action", [(1, 4, 0, GSF), (2, 300, 2, GSF), (63, 6, 0, GSF), (64, 6, 2, GSF),
                                             (65, 6, 1, GSF), (128, 4, 0, LB), (129, 4, 2, PRIM), (181, 8, 0, GSF),
                                             (257, 4, 1, LB), (513, 4, 0, GSF), (1024, 2, 2, GSF), (1025, 2, 0, GSF)])
def test_tiles(orc, gpu, N, M, mode, action):
    ref, ctx, _ = make(orc, gpu, N, M, 0.01, mode, action, seed=N)
    for W in (1, 2, 7):
        assert close(ctx.virial_terms(W), ref.virial_terms(W), TOL[mode]), (N, mode, W)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_half_box(orc, gpu, mode):
    """x on a lattice of spacing L/4, y and z a little off one: pairs with |dx| = L/2."""
    L, M, N, tau, lam = 16.0, 6, 40, 0.01, 6.0596
    rng = np.random.default_rng(5)
    sites = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), axis=-1).reshape(-1, 3)
    b = np.stack([4.0 * sites[rng.permutation(64)[:N]] - 8.0 for _ in range(M)])
    b[..., 1:] += rng.uniform(0.1, 0.6, size=(M, N, 2))
    ref = orc.State(L, M, N, tau, lam, L)
    ref.set_beads(b)
    ref.set_action(1, GSF["vfactor"])
    ref.set_correction(GSF["gradvfactor"], GSF["period"])
    ctx = gpu.Context(L, M, N, tau, lam, L, v_mode=mode)
    ctx.upload_path(b)
    ctx.set_action_factors(GSF["vfactor"], GSF["gradvfactor"], GSF["period"])
    dx = b[:, :, None, 0] - b[:, None, :, 0]
    assert (np.abs(dx) == 0.5 * L).sum() > 100
    assert close(ctx.virial_terms(3), ref.virial_terms(3), TOL[mode])


@pytest.mark.parametrize("N", [70, 300])
def test_ragged(gpu, N):
    """Fewer beads on every slice than allocated: as a context allocated for just those."""
    M, n = 6, N - 37
    rng = np.random.default_rng(N)
    L = (N / 0.02198) ** (1.0 / 3.0)
    b = rng.uniform(-0.5 * L, 0.5 * L, size=(M, N, 3))
    out = []
    for alloc in (N, n):
        ctx = gpu.Context(L, M, alloc, 0.01, 6.0596, L, v_mode=2)
        if alloc == N:
            on = np.zeros((M, N), dtype=np.uint8)
            on[:, :n] = 1
            ctx.upload_path(b, bead_on=on, num_beads=np.full(M, n, dtype=np.int32))
        else:
            ctx.upload_path(np.ascontiguousarray(b[:, :n]))
        ctx.set_action_factors(GSF["vfactor"], GSF["gradvfactor"], GSF["period"])
        out.append(np.asarray(ctx.virial_terms(2)))
    assert close(out[0], out[1], 1e-11)
