"""The packed pull links (nbrpack.h) through the kernels that follow them, on boxes where the packing
is not the common case: axes of one, two and three voxels (every node's column wraps round in z,
or its neighbour columns are its own), solid and pore runs that end on a wave's last lane, and
planes of more pores than a 16-bit rank can span (waves that keep full words).

FP64 against the CPU oracle, which follows the reference's own index arithmetic.  A wrong link
moves a population of O(0.01) to another node; the tolerances are those of the other FP64 oracle
comparisons (populations 1e-13 relative after a few steps, colour gradient 1e-12)."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

SMALL = [(1, 1, 1), (1, 1, 2), (5, 1, 1), (1, 7, 3), (7, 5, 1), (6, 1, 9), (3, 2, 2), (2, 3, 64), (4, 4, 65), (9, 11, 13)]


def _case(shape, porosity, seed):
    rng = np.random.default_rng(seed)
    solid = (rng.uniform(size=shape) > porosity).astype(np.int32)
    solid[0, 0, 0] = 0
    return solid, rng


@pytest.mark.parametrize("porosity", [0.4, 0.8, 1.0])
@pytest.mark.parametrize("shape", SMALL)
def test_small_boxes_match_the_oracle(pkg, oracle_mod, shape, porosity):
    print("[gpu] links", shape, porosity, flush=True)
    solid, rng = _case(shape, porosity, 5)
    g, u0 = (1e-4, -2e-4, 3e-4), (0.01, -0.02, 0.015)
    s = pkg.SinglePhase(solid, 0.1, g, precision="fp64")
    s.init(1.0, u0)
    o = oracle_mod.SPOracle(solid, 0.1, g, u0)
    s.step(5)
    o.run(5)
    assert rel_err(s.state()[0], o.f[1:]) < 1e-13

    u, conc = rng.uniform(-0.05, 0.05, (s.count, 3)), rng.uniform(0.0, 1.0, shape)
    st = pkg.Solute(0.03, solid=solid, w0=0.25, precision="fp64")
    st.set_velocity(u)
    st.init(conc)
    so = oracle_mod.STOracle(solid, 0.03, u, conc, w0=0.25)
    st.step(5)
    so.run(5)
    assert np.abs(st.state()[0] - so.g[1:]).max() < 1e-14

    psi = rng.uniform(-1.0, 1.0, shape)
    cg = pkg.ColorGradient(solid, 0.1, 0.05, 0.3, 0.01, g, precision="fp64")
    cg.init(psi)
    co = oracle_mod.CGOracle(solid, psi, 0.1, 0.05, g, 0.01, 0.3)
    cg.step(3)
    co.run(3)
    f, _, _, psi_n, rho_r, rho_b = cg.state()
    assert rel_err(f, co.f[1:]) < 1e-12
    assert np.abs(rho_r - co.rho_r[1:]).max() < 1e-12 and np.abs(rho_b - co.rho_b[1:]).max() < 1e-12


@pytest.mark.parametrize("shape,porosity", [((3, 260, 260), 1.0), ((2, 300, 290), 0.8)])
def test_planes_wider_than_a_rank_match_the_oracle(pkg, oracle_mod, shape, porosity):
    print("[gpu] links, wide waves", shape, flush=True)
    solid, rng = _case(shape, porosity, 6)
    g, u0 = (1e-4, -2e-4, 3e-4), (0.01, -0.02, 0.015)
    s = pkg.SinglePhase(solid, 0.1, g, precision="fp64")
    s.init(1.0, u0)
    o = oracle_mod.SPOracle(solid, 0.1, g, u0, nthreads=8)
    u, conc = rng.uniform(-0.05, 0.05, (s.count, 3)), rng.uniform(0.0, 1.0, shape)
    st = pkg.Solute(0.03, solid=solid, w0=0.25, precision="fp64")
    st.set_velocity(u)
    st.init(conc)
    so = oracle_mod.STOracle(solid, 0.03, u, conc, w0=0.25, nthreads=8)
    for x in (s, st):
        x.step(3)
    for x in (o, so):
        x.run(3)
    assert rel_err(s.state()[0], o.f[1:]) < 1e-13
    assert np.abs(st.state()[0] - so.g[1:]).max() < 1e-14
