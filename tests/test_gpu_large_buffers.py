"""Buffers of more than 4 GiB against a box whose buffers are smaller: a geometry repeated twice along x
has the solution of one period in either half.  The half box follows its links with 32-bit offsets, the
whole one with 64-bit offsets, and nodes have other ids, places and workgroups: an offset that wraps
round at 4 GiB shows in the upper half.  Flow, coupled solute and colour gradient in FP64.  The arithmetic of a node is the same; the tolerance is that of the comparisons with the FP64
oracle."""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

G, U0 = (1e-4, -2e-4, 3e-4), (0.01, -0.02, 0.015)


def _period(shape, seed=12):
    rng = np.random.default_rng(seed)
    solid = np.zeros(shape, np.int32)
    for c in rng.integers(0, [n - 8 for n in shape], (60, 3)):
        solid[c[0]:c[0] + 4, c[1]:c[1] + 5, c[2]:c[2] + 6] = 1
    return solid


def _halves_agree(whole, half):
    n = len(half)
    assert len(whole) == 2 * n
    assert rel_err(whole[:n], half) < 1e-13 and rel_err(whole[n:], half) < 1e-13


def test_flow_and_solute(pkg):
    print("[gpu] large buffers, flow and solute", flush=True)
    half = _period((153, 305, 305))
    conc = np.random.default_rng(5).uniform(size=half.shape)
    reads = []
    for copies in (1, 2):
        flow = pkg.SinglePhase(np.concatenate([half] * copies), 0.1, G, precision="fp64")
        assert (flow.count * 19 * 8 > 2**32) == (copies == 2)
        flow.init(1.0, U0)
        flow.step(3)
        st = pkg.Solute(0.03, flow=flow, w0=0.25, precision="fp64")
        st.init(np.concatenate([conc] * copies))
        st.step(3)
        reads.append((flow.velocity(), st.concentration(), flow.diagnostics()["Q"] / copies))
        st.close()
        flow.close()
    (u1, c1, q1), (u2, c2, q2) = reads
    _halves_agree(u2, u1)
    _halves_agree(c2, c1)
    assert rel_err(q2, q1) < 1e-12


def test_colour_gradient(pkg):
    print("[gpu] large buffers, colour gradient", flush=True)
    half = _period((153, 305, 305), seed=13)
    psi = np.random.default_rng(6).uniform(-1, 1, half.shape)
    reads = []
    for copies in (1, 2):
        s = pkg.ColorGradient(np.concatenate([half] * copies), 0.1, 0.05, 0.3, 0.01, (1e-5, 0, 0), precision="fp64")
        assert (s.count * 19 * 8 > 2**32) == (copies == 2)
        s.init(np.concatenate([psi] * copies))
        s.step(3)
        reads.append(s.colour())
        s.close()
    for whole, part in zip(reads[1], reads[0]):
        _halves_agree(whole, part)
