"""Graphs of odd and even step numbers where a tile covers a patch, replayed between
eager steps, kept states and retakes: the first step of an odd graph (and of an odd
eager advance beside one) writes the slab it reads, the others the other slab.  The
reference takes the same steps without a graph; FP32-bulk has the same bits in place
too, so everything is compared exactly."""
import numpy as np
import pytest

import forestclaw_amd as fa
from forestclaw_amd import problems as P
from helpers import setup_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", [0, 2])
@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
@pytest.mark.parametrize("name,mx,sync", [("swe", 8, True), ("swe", 16, True), ("swe", 32, False), ("adv", 16, False)])
def test_replays_among_eager_steps(gpu, name, mx, sync, precision, layout):
    if mx == 32 and layout == 0:
        pytest.skip("one layout is enough for the copied result")
    prob = P.dambreak_problem(2, 4, mx=mx) if name == "swe" else P.advection_problem(3, 3, mx=mx)
    (_, q0, _, sv), (_, _, _, ref) = (setup_problem(prob, precision=precision, time_sync=sync, tile=mx) for _ in range(2))
    for s in (sv, ref):
        s.set_ghost_layout(layout)
    dt = 0.5 * P.stable_dt(prob, P.build_forest(prob), q0)
    for steps in (1, 3, 4):
        sv.capture_graph(dt, steps)
        for k in range(5):
            print("case", name, mx, "precision", precision, "layout", layout, "steps", steps, "replay", k, flush=True)
            if k == 1:            # an odd eager advance
                sv.advance(dt, 1)
                ref.advance(dt, 1)
            elif k == 2:          # a step retaken
                sv.save_step()
                sv.advance(0.7 * dt, 1)
                sv.restore_step()
                sv.advance(0.5 * dt, 1)
                ref.advance(0.5 * dt, 1)
            elif k == 3:          # a state kept across a replay and given back
                sv.save_step()
                sv.replay_graph()
                sv.restore_step()
            sv.replay_graph()
            sv.sync()
            ref.advance(dt, steps)
            np.testing.assert_array_equal(sv.get_q(), ref.get_q())
