"""hipclaw_waves names the waves per workgroup that the next update launches, any choice
of them gives the same bits, and the autotuner does not choose between trials that
launch the same kernels."""
import numpy as np
import pytest

import forestclaw_amd as fa
from forestclaw_amd import problems as P
from helpers import setup_problem

pytestmark = pytest.mark.gpu

STRIPS = 4     # strips' waves by default


def _setup(name, precision, minlevel, **kw):
    prob = (P.dambreak_problem(minlevel, minlevel, mx=16) if name == "swe"
            else P.shockbubble_problem(minlevel - 1, minlevel - 1, mx=16))
    return prob, setup_problem(prob, precision=precision, tile=16, **kw)


@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
@pytest.mark.parametrize("name", ["swe", "euler"])
def test_waves_by_default_and_by_choice(gpu, name, precision):
    prob, (forest, q0, _, sv) = _setup(name, precision, 5)
    assert forest.npatch == 1024
    assert sv.waves == STRIPS
    dt = 0.5 * P.stable_dt(prob, forest, q0)
    sv.advance(dt, 4)
    want = sv.get_q()
    for waves in (2, 3, 4):
        print("case", name, "precision", precision, "waves", waves, flush=True)
        sv.set_q(q0)
        sv.set_waves(waves)
        assert sv.waves == waves
        sv.advance(dt, 4)
        np.testing.assert_array_equal(sv.get_q(), want)
    sv.set_waves(0)
    assert sv.waves == STRIPS
    # a small launch: FP64 takes 16 x 16 tiles with four waves, FP32-bulk stays in strips
    _, (_, _, _, small) = _setup(name, precision, 2)
    assert small.waves == 4


@pytest.mark.parametrize("name,precision", [("swe", fa.FP64), ("swe", fa.FP32_BULK)])
def test_autotune_times_the_same_launches_once(gpu, name, precision):
    prob, (forest, q0, _, sv) = _setup(name, precision, 5)
    timings = sv.autotune(0.5 * P.stable_dt(prob, forest, q0), 2)
    assert set(timings) == {(t, w, l) for t, w in ((8, 0), (16, 2), (16, 3), (16, 4)) for l in (0, 1, 2)}
    assert (sv.tile, sv.waves, sv.ghost_layout) == min(timings, key=timings.get)
    # an 8 x 8 tile's strips are those of the 16 x 16 tile with four waves
    for layout in (0, 1, 2):
        assert timings[8, 0, layout] == timings[16, 4, layout]
    assert sv.tile == 16


@pytest.mark.parametrize("name", ["swe", "euler"])
def test_autotune_tries_the_tile_kernel_for_small_launches(gpu, name):
    """The trial of a 16 x 16 tile with four waves, the default, is the tile kernel where
    the default takes it; chosen waves are strips.  A step of tiles takes 0.83 (shallow
    water) and 0.78 (Euler) of the time of one of strips with three waves, strips with
    four 0.99."""
    prob, (forest, q0, _, sv) = _setup(name, fa.FP64, 4)
    assert forest.npatch == 256
    timings = sv.autotune(0.5 * P.stable_dt(prob, forest, q0), 16)
    print(name, timings, "tile", sv.tile, "waves", sv.waves, "layout", sv.ghost_layout, flush=True)
    assert timings[16, 4, 2] <= 0.92 * timings[16, 3, 2]
