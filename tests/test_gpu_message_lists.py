"""Ghost messages of short and long lists: every message is the same whichever
way its slot reaches the launch, and so is what unpacking leaves in the patches
(copies only, so everything is compared exactly)."""
import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx,my", [(8, 8), (9, 13), (20, 8)])
def test_lists_around_the_switch(gpu, mx, my):
    import torch
    npatch = 450
    sync = mx == my
    sv = fa.Solver(fa.RP_SHALLOW, mx, my, precision=fa.FP64, max_patches=npatch, tile=8, time_sync=sync)
    dx = 1.0 / np.arange(8, 8 + npatch)
    sv.set_geometry(dx, 0.5 * dx)
    sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
    q = random_state(fa.RP_SHALLOW, npatch, mx, my, np.random.default_rng(mx))
    sv.set_q(q)
    if sync:
        sv.advance(1e-5, 1)      # fills the registers
    before = sv.get_q()
    order = np.random.default_rng(1).permutation(npatch).astype(np.int32)

    def pack(slots):
        out = torch.full((len(slots), sv.ghost_pack_elems()), np.nan, device="cuda", dtype=torch.float64)
        sv.ghost_pack(slots, out.data_ptr())
        return out

    whole = pack(order)
    single = pack(order[:1])
    parts = torch.cat([pack(order[k:k + 150]) for k in range(0, npatch, 150)])
    np.testing.assert_array_equal(whole.cpu().numpy(), parts.cpu().numpy())
    np.testing.assert_array_equal(single.cpu().numpy(), parts[:1].cpu().numpy())
    assert not torch.isnan(whole).any()
    # patch k's message goes into the patch after it in the list, in both ways
    to = np.roll(order, -1)
    sv.ghost_unpack(to, whole.data_ptr())
    long = sv.get_q()
    sv.set_q(before)
    for k in range(0, npatch, 150):
        sv.ghost_unpack(to[k:k + 150].copy(), parts[k:k + 150].data_ptr())
    np.testing.assert_array_equal(sv.get_q(), long)
    mint = 4
    np.testing.assert_array_equal(long[to][:, :, :, :mint + 2], before[order][:, :, :, :mint + 2])
    inner = (slice(None), slice(None), slice(mint + 2, my + 2 - mint), slice(mint + 2, mx + 2 - mint))
    np.testing.assert_array_equal(long[inner], before[inner])
