"""Launch settings that go by the size of a box (tune.h): the handle reports the rule's choice on
either side of each line, and the states are those of fixed settings, to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(edge, solid_share=0.0, seed=3):
    return (np.random.default_rng(seed).uniform(size=(edge,) * 3) < solid_share).astype(np.int32)


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


# lines at 131,072 nodes and, for steps that fit the memory-side cache (FP64: 792,569 nodes), at 262,144
@pytest.mark.parametrize("precision,edge,want", [("fp32", 5, (128, "slab")), ("fp32", 50, (128, "slab")),
                                                 ("fp32", 51, (256, "runs8")), ("fp32", 63, (256, "runs8")),
                                                 ("fp32", 64, (256, "slab")), ("fp16", 66, (256, "slab")),
                                                 ("fp64", 92, (256, "slab")), ("fp64", 93, (256, "runs8"))])
def test_single_phase(pkg, precision, edge, want):
    states = []
    for fixed in (False, True):
        s = pkg.SinglePhase(_box(edge), 0.1, (1e-5, 0, 0), precision=precision)
        if fixed:
            s.set_launch(256, "hw")
        else:
            assert (s.launch()["block"], s.launch()["order"]) == want
        s.init(1.0, (0.01, 0.0, 0.0))
        s.step(4)
        states.append(s.state())
    assert _same(*states)


# line at 262,144 nodes, and where the steps stop to fit the memory-side cache (FP64: 588,505 nodes)
@pytest.mark.parametrize("precision,edge,want", [("fp32", 5, (128, "slab")), ("fp32", 63, (128, "slab")),
                                                 ("fp32", 64, (256, "slab")), ("fp64", 83, (256, "slab")),
                                                 ("fp64", 84, (256, "hw"))])
@pytest.mark.parametrize("coupled", [False, True])
def test_solute(pkg, precision, edge, want, coupled):
    states = []
    for fixed in (False, True):
        flow = pkg.SinglePhase(_box(edge), 0.1, (1e-5, 0, 0), precision=precision) if coupled else None
        st = pkg.Solute(0.02, solid=None if coupled else _box(edge), flow=flow, precision=precision)
        if fixed:
            st.set_launch(256, "runs8")
        else:
            assert (st.launch()["block"], st.launch()["order"]) == want
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
