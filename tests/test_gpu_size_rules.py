"""Launch settings that go by the size of a box (tune.h): the handle reports the rule's choice on
either side of each line, and the states are those of fixed settings, to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(edge, solid_share=0.0, seed=3):
    return (np.random.default_rng(seed).uniform(size=(edge,) * 3) < solid_share).astype(np.int32)


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("edge,small", [(5, True), (50, True), (51, False)])   # line at 131,072 nodes
def test_single_phase(pkg, edge, small):
    states = []
    for fixed in (False, True):
        s = pkg.SinglePhase(_box(edge), 0.1, (1e-5, 0, 0), precision="fp32")
        if fixed:
            s.set_launch(256, "hw")
        else:
            assert (s.launch()["block"], s.launch()["order"]) == ((128, "slab") if small else (256, "runs8"))
        s.init(1.0, (0.01, 0.0, 0.0))
        s.step(4)
        states.append(s.state())
    assert _same(*states)


@pytest.mark.parametrize("edge,small", [(5, True), (64, False)])               # line at 262,144 nodes
@pytest.mark.parametrize("coupled", [False, True])
def test_solute(pkg, edge, small, coupled):
    states = []
    for fixed in (False, True):
        flow = pkg.SinglePhase(_box(edge), 0.1, (1e-5, 0, 0), precision="fp32") if coupled else None
        st = pkg.Solute(0.02, solid=None if coupled else _box(edge), flow=flow, precision="fp32")
        if fixed:
            st.set_launch(256, "runs8")
        else:
            assert (st.launch()["block"], st.launch()["order"]) == ((128, "slab") if small else (256, "hw"))
        st.init(np.random.default_rng(4).uniform(size=(edge,) * 3))
        st.step(4)
        states.append(st.state())
    assert _same(*states)


# lines at 32,768 and 215,000 nodes; above the second the staged kernels are taken where most blocks
# read from their LDS runs: not in the cube, whose planes hold seven blocks, two of them on a wrap
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("shape,want", [((6, 6, 6), (128, 256, "gather")), ((32, 32, 32), (128, 256, "gather")),
                                        ((59, 59, 59), (256, 256, "gather")), ((61, 61, 61), (256, 256, "gather")),
                                        ((12, 150, 130), (512, 512, "staged"))])
def test_colour_gradient(pkg, precision, shape, want):
    solid = (np.random.default_rng(3).uniform(size=shape) < 0.02).astype(np.int32)
    states = []
    for fixed in (False, True):
        s = pkg.ColorGradient(solid, 0.1, 0.05, 0.3, 0.01, (1e-5, 0, 0), precision=precision)
        if fixed:
            s.set_launch("cg_collide", 256, "runs8", "gather")
            s.set_launch("cg_colour", 256, "slab", "gather")
        else:
            c, v = s.launch("cg_collide"), s.launch("cg_colour")
            assert (c["block"], v["block"], c["variant"], v["variant"], c["order"], v["order"]) == want + (want[2], "slab", "slab")
        s.init(np.random.default_rng(5).uniform(-1, 1, shape))
        s.step(4)
        states.append(s.state())
    assert _same(*states)
