"""Device runs of several uneven chains in one launch: every chain's host copy equals
its device path afterwards (the moved worldlines come back compactly, in blocks of
256 beads), and a chain gives the same decisions, deltas and worldlines alone or
beside others with other sizes and winding tables.  Exact equality throughout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KINDS = ["staging", "bisection", "com", "com", "staging"]


@pytest.fixture(scope="module")
def gpu():
    import pimc_amd
    return pimc_amd


def _chain(gpu, N, M, max_wind, seed):
    L = (N / 0.02198) ** (1.0 / 3.0)
    ctx = gpu.Context(L, M, N, 0.01, 6.0596, L)
    ctx.upload_path(gpu.gen_worldlines(seed, L, M, N, 6.0596, 0.01, 1))
    return ctx, gpu.Chain(ctx, 77 + seed, 6, 2, True, max_wind, 0.3)


SIZES = [(3, 12, 1), (64, 9, 2), (257, 7, 0), (300, 8, 1), (1, 10, 1)]


@pytest.mark.parametrize("moves", [1, 5, 40])
def test_uneven_chains(gpu, moves):
    kinds = (KINDS * 8)[:moves]
    pairs = [_chain(gpu, *s, k) for k, s in enumerate(SIZES)]
    for _ in range(2):   # the second run starts where the first ended
        acc, info, near = gpu.run_chains_device([c for _, c in pairs], kinds)
        for ctx, c in pairs:
            assert np.array_equal(c.positions(), ctx.download_path())
    for k, s in enumerate(SIZES):
        ctx, c = _chain(gpu, *s, k)
        c.run_device(kinds)
        a, i, n = c.run_device(kinds)
        assert np.array_equal(a, acc[k]) and np.array_equal(i, info[k]) and n == near[k]
        assert np.array_equal(c.positions(), pairs[k][1].positions())
        # a host-driven move goes on from there
        c.move("com")
        assert np.array_equal(c.positions(), ctx.download_path())


@pytest.mark.parametrize("how", ["update_beads", "delta_action", "upload_path", "another chain"])
def test_beads_changed_past_the_chain(gpu, how):
    """Beads changed through the context, or by another chain on it, between two device
    runs: after the second the chain's host copy is the device path, whichever worldlines
    that run moved."""
    rng = np.random.default_rng(3)
    N, M = 40, 12
    ctx, chain = _chain(gpu, N, M, 1, 6)
    other = gpu.Chain(ctx, 5, 6, 2, True, 1, 0.3)
    chain.run_device(KINDS)
    sp = np.stack([np.arange(M), rng.integers(0, N, M)], axis=-1).astype(np.int32)
    new = rng.uniform(-3.0, 3.0, size=(M, 3))
    if how == "update_beads":
        ctx.update_beads(sp, new)
    elif how == "delta_action":
        ctx.delta_action(sp, new, commit=True)
    elif how == "upload_path":
        ctx.upload_path(np.ascontiguousarray(ctx.download_path()[:, ::-1]))
    else:
        other.run_device(KINDS)
        other.move("staging")
    chain.run_device(["staging"])
    assert np.array_equal(chain.positions(), ctx.download_path())
    # and in step again: a host-driven move, then a run that moves few worldlines
    chain.move("com")
    chain.run_device(["bisection"])
    assert np.array_equal(chain.positions(), ctx.download_path())
