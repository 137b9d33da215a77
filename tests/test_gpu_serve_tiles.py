"""The server's step over samples whose node counts lie at the edges of its tiles (128, 256 or 512
nodes) and of the 256-node blocks of its arena: the plain solver's permeability, and the same bits
beside a batch mate large enough to change the order of the tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 127, 128, 129, 255, 256, 257, 511, 513, 1024]
LIMITS = dict(check_interval=50, min_steps=100, max_steps=100, tol=0.0)


def _sample(count):
    """The first count voxels of a short box, less a few of them, are pores."""
    solid = np.ones((8, 8, 17), np.int32)
    solid.flat[:count] = 0
    if count > 64:
        drop = np.random.default_rng(count).choice(count, 8, replace=False)
        solid.flat[drop] = 1
        solid.flat[count:count + 8] = 0
    assert np.count_nonzero(solid == 0) == count
    return solid


def _serve(pkg, samples, precision, block):
    with pkg.PermeabilityServer(capacity_nodes=400_000, precision=precision, block=block, **LIMITS) as srv:
        tickets = [srv.submit(s, 0.1, (1e-5, 2e-5, 0.0), 1) for s in samples]
        assert srv.wait_idle(60.0)
        done = {r["ticket"]: r for r in srv.poll()}
    assert all(done[t]["steps"] == 100 for t in tickets)
    return [done[t]["k"] for t in tickets]


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("block", [128, 256, 512])
def test_tile_edges(pkg, precision, block):
    print(precision, block, flush=True)
    samples = [_sample(c) for c in COUNTS]
    k = _serve(pkg, samples, precision, block)
    large = (np.random.default_rng(2).uniform(size=(64, 64, 48)) < 0.2).astype(np.int32)   # > 2^17 pores
    mixed = _serve(pkg, [large] + samples, precision, block)[1:]
    for count, s, a, b in zip(COUNTS, samples, k, mixed):
        np.testing.assert_array_equal(a, b)
        flow = pkg.SinglePhase(s, 0.1, (1e-5, 2e-5, 0.0), precision=precision)
        flow.step(100)
        plain = flow.Comput_Perm(1)[0][:2]
        # of the larger component: FP32 rounding of the velocities goes by the flow's speed, and the
        # x-planes of a sample cut off by a wall carry next to nothing
        assert np.abs(a[:2] - plain).max() <= 1e-6 * np.abs(plain).max(), count
