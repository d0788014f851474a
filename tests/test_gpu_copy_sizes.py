"""The copy of a patch's state kept before an update: slabs of one chunk and of several,
with an even and an odd number of values, and the last chunk full or not.  Read back
as the time-interpolated state at alpha = 0, which is that copy on the message band;
copies only, so compared exactly."""
import ctypes as C

import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import random_aux, random_state
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,mx,my,npatch", [(fa.RP_ADVECTION, 9, 9, 3), (fa.RP_ADVECTION, 41, 61, 2),
                                                 (fa.RP_SHALLOW, 16, 16, 5), (fa.RP_SHALLOW, 33, 32, 3),
                                                 (fa.RP_SHALLOW, 64, 64, 2), (fa.RP_EULER, 28, 28, 4),
                                                 (fa.RP_EULER, 100, 90, 1)])
def test_the_state_before_the_update(gpu, solver, mx, my, npatch):
    rng = np.random.default_rng(mx)
    sv = fa.Solver(solver, mx, my, max_patches=npatch, subcycle=True)
    dx = np.full(npatch, 1.0 / mx)
    sv.set_geometry(dx, dx)
    q = random_state(solver, npatch, mx, my, rng)
    sv.set_q(q)
    if solver == fa.RP_ADVECTION:
        sv.set_aux(random_aux(npatch, mx, my, rng))
    slots = rng.permutation(npatch).astype(np.int32)

    hip = _Hip()

    def message(time_interp):
        shape = (npatch, sv.ghost_pack_elems())
        out = hip.put(np.zeros(shape))
        sv.ghost_pack(np.arange(npatch, dtype=np.int32), out.value, time_interp=time_interp)
        return hip.get(out, shape)

    # the values of a message that are interior cells: those a marked state changes
    mark = np.zeros_like(q)
    mark[:, :, 2:-2, 2:-2] = 1.0
    before = message(False)
    sv.set_q(mark)
    inside = message(False) == 1.0
    sv.set_q(q)
    sv.step_batch(slots, 0.01 / mx)
    assert (message(False) != before)[inside].any()
    fa._check(fa.lib().hipclaw_timeinterp(sv._h, C.c_void_p(slots.ctypes.data), npatch, C.c_double(0.0)), "hipclaw_timeinterp")
    got = message(True)
    # (the interpolation fills the band of mbc layers that the coarse side is read from)
    same = got[inside] == before[inside]
    filled = got[inside] != 0.0
    assert filled.any() and same[filled].all()
    hip.free()
