"""State reads across chunk and piece borders (readback.h): the same values whatever the outputs
asked for together, since each set of outputs splits the nodes into chunks and 2 MiB pieces at
other places, and from several threads at once.  Values are copied, never computed differently,
so every comparison is exact."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# node counts of one piece, of several pieces with a remainder, and of several chunks (a chunk is at
# most 8 MiB: 1,048,576 values of one output, 40,329 nodes of a whole colour-gradient state)
SHAPES = [(7, 5, 3), (31, 33, 35), (60, 51, 53), (128, 97, 89)]


def _solid(pkg, shape):
    return (np.random.default_rng(9).uniform(size=shape) < 0.1).astype(np.int32)


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("shape", SHAPES)
def test_outputs_agree_however_they_are_read(pkg, shape, precision):
    print("[gpu] read back", shape, precision, flush=True)
    solid = _solid(pkg, shape)
    pore = solid == 0
    s = pkg.SinglePhase(solid, 0.1, (1e-4, -2e-4, 3e-4), precision=precision)
    s.init(1.0, (0.01, 0.0, 0.0))
    s.set_power_law(0.05, 0.9)
    s.step(14)
    f, u, rho = s.state()
    fn, un, rhon = s.state_noalloc()         # by another path
    assert np.array_equal(f, fn) and np.array_equal(u, un) and np.array_equal(rho, rhon)
    assert np.array_equal(s.velocity(), u)
    ud, rhod = s.dense()
    assert np.array_equal(ud[pore], u) and np.array_equal(rhod[pore], rho)
    assert not ud[~pore].any() and (rhod[~pore] == 1.0).all()
    nu = s.viscosity()
    assert nu.shape == (s.count,) and np.isfinite(nu).all() and (nu > 0).all()

    psi = np.random.default_rng(10).uniform(-1.0, 1.0, shape)
    cg = pkg.ColorGradient(solid, 0.1, 0.05, 0.3, 0.01, (1e-4, 0, 0), precision=precision)
    cg.init(psi)
    rr, rb = cg.colour()
    assert np.abs(rr - (psi[pore] + 1) / 2).max() < 2e-9 and np.abs(rr + rb - 1).max() < 4e-9   # FP32: units of 2^-29
    cg.step(2)
    state = cg.state()
    assert all(np.isfinite(x).all() for x in state)
    rr, rb = cg.colour()
    assert np.array_equal(state[4], rr) and np.array_equal(state[5], rb)

    st = pkg.Solute(0.02, solid=solid, precision=precision)
    st.init(psi + 1.0)
    st.step(2)
    g, c = st.state()
    assert np.array_equal(st.concentration(), c)
    np.testing.assert_allclose(g.sum(1), c, rtol=1e-14, atol=0)


def test_reads_from_several_threads(pkg):
    """Four handles read at once, more than the two idle buffer sets that are kept."""
    solid = _solid(pkg, (60, 51, 53))
    handles = []
    for k in range(4):
        s = pkg.SinglePhase(solid, 0.1, (1e-4 * (k + 1), 0, 0), precision="fp64")
        s.init(1.0)
        s.step(3)
        handles.append((s, s.state_noalloc()))
    wrong = []

    def read(s, want):
        for _ in range(5):
            if not all(np.array_equal(a, b) for a, b in zip(s.state(), want)):
                wrong.append(s)

    threads = [threading.Thread(target=read, args=h) for h in handles]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
