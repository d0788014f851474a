"""Registers that a synchronisation zeroed are written by the next update instead
of added to.  Calls of one coarse step begin without such knowledge, a call of
several has it from its second step on, and a captured graph replays it: all give
the same state and the same registers bit for bit (0 + x is x)."""
import numpy as np
import pytest

import forestclaw_amd as fa
from forestclaw_amd import problems as P
from test_gpu_subcycle_device import _setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
@pytest.mark.parametrize("name", ["dambreak", "shockbubble"])
def test_coarse_steps_together_and_one_by_one(gpu, precision, name):
    import torch
    prob = P.dambreak_problem(2, 5, mx=16) if name == "dambreak" else P.shockbubble_problem(1, 4, mx=8)

    def run(how):
        print("case", name, "precision", precision, how, flush=True)
        forest, _, _, sv, dt = _setup(prob, True, precision)
        if how == "together":
            sv.advance_subcycle(dt, 4)
        elif how == "one by one":
            for _ in range(4):
                sv.advance_subcycle(dt, 1)
        else:
            sv.capture_subcycle_graph(dt, 2)
            for _ in range(2):
                sv.replay_graph()
                sv.sync()
        slots = np.arange(sv.npatch, dtype=np.int32)
        out = torch.zeros((sv.npatch, sv.ghost_pack_elems()), device="cuda", dtype=torch.float64)
        sv.ghost_pack(slots, out.data_ptr())      # carries the registers
        return sv.get_q(), out.cpu().numpy()

    want = run("one by one")
    for how in ("together", "replayed"):
        got = run(how)
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
