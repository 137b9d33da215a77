"""Launch settings of a coupled flow + solute step, timed when the solute is created: the timing leaves a
flow in mid-run as it was, and times steps as a run makes them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _box(shape, seed=21):
    """Overlapping solid balls of radius 5, a fifth of the box solid."""
    rng = np.random.default_rng(seed)
    solid = np.zeros(shape, np.int32)
    o = np.stack(np.meshgrid(*[np.arange(-5, 6)] * 3, indexing="ij"), -1).reshape(-1, 3)
    o = o[(o ** 2).sum(1) <= 25]
    for c in rng.integers(0, shape, (int(0.22 * np.prod(shape) / len(o)), 3)):
        p = (c + o) % shape
        solid[p[:, 0], p[:, 1], p[:, 2]] = 1
    return solid


# steps that do not fit the memory-side cache (FP64 480 MB, FP32 500 MB) and one that does (FP16); with the
# flow at either buffer
@pytest.mark.parametrize("precision,shape,steps", [("fp64", (124, 116, 102), 4), ("fp64", (124, 116, 102), 5),
                                                   ("fp32", (150, 140, 130), 5), ("fp16", (124, 116, 102), 4)])
def test_timing_leaves_the_flow_and_times_a_run(pkg, precision, shape, steps):
    print("[gpu] coupled tuning", precision, shape, steps, flush=True)
    flow = pkg.SinglePhase(_box(shape), 0.1, (1e-4, 0, 0), precision=precision)
    assert flow.count >= 1 << 20
    flow.init(1.0, (0.01, 0.0, 0.0))
    flow.step(steps)
    before = flow.state()
    st = pkg.Solute(0.02, flow=flow, w0=0.25, precision="fp64" if precision == "fp64" else "fp32")
    assert all(np.array_equal(a, b) for a, b in zip(flow.state(), before))
    picked = st.launch()
    st.init(np.random.default_rng(4).uniform(size=shape))
    st.step(20)
    if picked["tuned"]:
        # a step's time varies by 2 % from run to run; timed from one buffer into the other over and over, it
        # came out 25 % short
        run = np.median([st.step_timed(60) / 60 * 1e3 for _ in range(5)])
        assert abs(picked["time_us"] / run - 1) < 0.15
