"""The Courant number and the step times an advance collects on the device: over
any number of steps, after a replayed graph and after a batch.  The same steps
give the same bits, so every comparison is exact; times are those of a clock
that only counts up."""
import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import random_aux, random_state

pytestmark = pytest.mark.gpu


def _solver(solver, npatch=3, mx=16):
    rng = np.random.default_rng(solver)
    sv = fa.Solver(solver, mx, mx, precision=fa.FP64, max_patches=npatch, tile=8)
    dx = np.full(npatch, 1.0 / mx)
    sv.set_geometry(dx, dx)
    sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
    q = random_state(solver, npatch, mx, mx, rng)
    if solver == fa.RP_ADVECTION:
        sv.set_aux(random_aux(npatch, mx, mx, rng))
    sv.set_q(q)
    return sv, q


@pytest.mark.parametrize("nsteps", [0, 1, 2, 63, 64, 65, 129])
@pytest.mark.parametrize("solver", [fa.RP_ADVECTION, fa.RP_SHALLOW])
def test_largest_courant_number(gpu, solver, nsteps):
    sv, q = _solver(solver)
    dt = 1e-4
    single = [sv.advance(dt, 1) for _ in range(nsteps)]
    sv.set_q(q)
    assert sv.advance(dt, nsteps) == max(single, default=0.0)
    total, kernel = sv.timing(nsteps)
    if nsteps:
        assert 0.0 < kernel and kernel * nsteps <= total
    else:
        assert (total, kernel) == (0.0, 0.0)


def test_words_of_a_replay_and_a_batch_stay_out(gpu):
    sv, q = _solver(fa.RP_SHALLOW)
    want = sv.advance(1e-4, 2)
    sv.set_q(q)
    sv.capture_graph(1e-3, 2)      # ten times the Courant number
    sv.replay_graph()
    sv.sync()
    sv.set_q(q)
    assert sv.advance(1e-4, 2) == want
    times = sv.timing(2)
    assert sv.step_batch([0, 2], 1e-3) > want
    assert sv.timing(2) == times
    sv.set_q(q)
    assert sv.advance(1e-4, 2) == want
