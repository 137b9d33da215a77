"""The ways a step kernel follows its links (LinkForm, nbrpack.h): ranks of 16 or 8 bits, 32-bit or 64-bit
offsets.

Boxes of 2^20 nodes and more on both sides of the rule for 8-bit ranks -- wide planes, where few
waves straddle a plane's wrap, and planes of eight columns, where too many do -- against the FP64
oracle, with the tolerances of the other links tests.  Then boxes just under and just over the
4 GiB a buffer that 32-bit offsets reach: steps taken one by one run the general kernel (the last
step of a call stores the velocity, and follows links in the general form), steps taken in one
call the chosen one, with the same arithmetic: the same bits."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

G, U0 = (1e-4, -2e-4, 3e-4), (0.01, -0.02, 0.015)


@pytest.mark.parametrize("shape,porosity", [((40, 170, 160), 0.97), ((37, 251, 229), 0.55), ((260, 8, 520), 0.98)])
def test_large_boxes_match_the_oracle(pkg, oracle_mod, shape, porosity):
    print("[gpu] link forms", shape, porosity, flush=True)
    rng = np.random.default_rng(11)
    solid = (rng.uniform(size=shape) > porosity).astype(np.int32)
    flow = pkg.SinglePhase(solid, 0.1, G, precision="fp64")
    assert flow.count >= 1 << 20
    flow.init(1.0, U0)
    fo = oracle_mod.SPOracle(solid, 0.1, G, U0, nthreads=8)
    flow.step(3)
    fo.run(3)
    conc = rng.uniform(0.0, 1.0, shape)
    st = pkg.Solute(0.03, flow=flow, w0=0.25, precision="fp64")
    st.init(conc)
    so = oracle_mod.STOracle(solid, 0.03, fo.u[1:].copy(), conc, w0=0.25, nthreads=8)
    st.step(3)
    for _ in range(3):
        so.u[1:] = fo.u[1:]
        so.run(1)
        fo.run(1)
    assert rel_err(flow.state()[0], fo.f[1:]) < 1e-13
    assert np.abs(st.state()[0] - so.g[1:]).max() < 1e-14


@pytest.mark.parametrize("shape", [(304, 304, 305), (305, 305, 305)])
def test_both_sides_of_four_gigabytes(pkg, shape):
    print("[gpu] link forms", shape, flush=True)
    solid = np.zeros(shape, np.int32)
    rng = np.random.default_rng(12)
    for c in rng.integers(0, 300, (40, 3)):
        solid[c[0]:c[0] + 4, c[1]:c[1] + 5, c[2]:c[2] + 6] = 1
    s = pkg.SinglePhase(solid, 0.1, G, precision="fp64")
    bytes_a_buffer = s.count * 19 * 8
    assert 0.99 * 2**32 < bytes_a_buffer < 1.01 * 2**32 and (bytes_a_buffer > 2**32) == (shape[0] == 305)
    s.init(1.0, U0)
    s.step(4)
    together = s.velocity()
    s.init(1.0, U0)
    for _ in range(4):
        s.step(1)
    assert np.array_equal(together, s.velocity())


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-6)])
@pytest.mark.parametrize("faces,law", [(True, 0.0), (False, 0.8)])
def test_faces_and_power_law_on_eight_bit_ranks(pkg, precision, tol, faces, law):
    """Steps in one call (the form the box allows) against steps one by one (the general form); the
    power law acts from the eleventh on.  The arithmetic is the same up to how it is contracted:
    the tolerances are the precisions' of the other comparisons."""
    print("[gpu] link forms", precision, faces, law, flush=True)
    solid = (np.random.default_rng(13).uniform(size=(40, 170, 160)) > 0.97).astype(np.int32)
    states = []
    for calls in ((14,), (1,) * 14):
        s = pkg.SinglePhase(solid, 0.1, (0.0, 0.0, 0.0) if faces else G, precision=precision)
        s.init(1.0, U0)
        if faces:
            s.set_boundaries(3, pre={"xp": 1.0 - 2e-4, "xn": 1.0 + 2e-4})
        if law:
            s.set_power_law(0.05, law)
        for n in calls:
            s.step(n)
        states.append(s.state()[0])
    assert rel_err(*states) < tol
