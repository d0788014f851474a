"""Slot lists of hipclaw_step_batch_noalloc below, at and beyond the part that goes up
with the cleared words, in any order: the same bits as hipclaw_step_batch gives, and
the patches that are not listed stay as they are."""
import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import random_state
from test_zz_no_alloc import _Hip, _noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nslots", [1, 15, 16, 17, 3071, 3072, 3073, 3100, 9000])
def test_lists_of_any_length(gpu, nslots):
    mx, npatch = 12, nslots + 3
    rng = np.random.default_rng(nslots)
    q = random_state(fa.RP_SHALLOW, npatch, mx, mx, rng)
    dx = rng.choice([1.0, 0.5], npatch) / mx
    slots = rng.permutation(npatch)[:nslots].astype(np.int32)
    sv = fa.Solver(fa.RP_SHALLOW, mx, mx, max_patches=npatch)
    sv.set_geometry(dx, dx)
    sv.set_q(q)
    want = sv.step_batch(slots, 0.05 / mx)
    ref = sv.get_q()
    hip = _Hip()
    try:
        for _ in range(2):       # the second call clears what the first left
            got, cfl = _noalloc(sv, hip, q, slots, dx, 0.05 / mx)
            assert cfl == want
            np.testing.assert_array_equal(got[slots][:, :, 2:-2, 2:-2], ref[slots][:, :, 2:-2, 2:-2])
            assert not got[np.setdiff1d(np.arange(npatch), slots)].any()
    finally:
        hip.free()
