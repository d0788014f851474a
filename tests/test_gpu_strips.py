"""The strip kernel at the edges of its layouts: patches that fill a wave, are
cut between waves or take several, counts that end inside a pattern, in-place
updates, and seams between strips of any height.

FP64: 1e-12 relative in max norm against the oracle (the arithmetic is the
reference's operation for operation).  FP32-bulk: 1e-4, and mass to 1e-13 of the
total (FP64 fluxes telescope: 50 steps' rounding of ~1e-16 each)."""
import ctypes as C

import numpy as np
import pytest

import forestclaw_amd as fa
from forestclaw_amd import problems as P
from helpers import claw_for, interior, random_aux, random_state, rel_max_err, setup_problem
from oracle_lib import step2_oracle

pytestmark = pytest.mark.gpu

# (mx, my, patches)
SHAPES = [(8, 8, 1), (8, 8, 11), (9, 13, 7), (16, 16, 4), (20, 9, 6), (33, 8, 3), (60, 8, 2), (61, 9, 2),
          (130, 8, 1), (500, 8, 1)]


@pytest.mark.parametrize("solver", [fa.RP_ADVECTION, fa.RP_SHALLOW, fa.RP_EULER])
@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d_%d" % s for s in SHAPES])
def test_step_of_any_layout(gpu, solver, shape):
    mx, my, npatch = shape
    rng = np.random.default_rng(mx + 10 * my + 100 * solver)
    q = random_state(solver, npatch, mx, my, rng)
    aux = random_aux(npatch, mx, my, rng) if solver == fa.RP_ADVECTION else None
    dx = np.full(npatch, 1.0 / max(mx, my))
    dt = 0.2 / max(mx, my)
    ref = [step2_oracle(claw_for(solver), q[p], None if aux is None else aux[p], dx[p], dx[p], dt)
           for p in range(npatch)]
    for precision, tol in ((fa.FP64, 1e-12), (fa.FP32_BULK, 1e-4)):
        print("case solver", solver, "shape", shape, "precision", precision, flush=True)
        sv = fa.Solver(solver, mx, my, precision=precision, max_patches=npatch, tile=8)
        sv.set_geometry(dx, dx)
        sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
        sv.set_q(q)
        if aux is not None:
            sv.set_aux(aux)
        cfl = sv.advance(dt, 1)
        qg = sv.get_q()
        for p in range(npatch):
            assert rel_max_err(interior(qg[p]), interior(ref[p][0])) <= tol, (precision, p)
        want = max(c for _, c in ref)
        assert abs(cfl - want) <= (1e-12 if precision == fa.FP64 else 1e-5) * want


@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
def test_in_place_equals_two_slabs(gpu, precision):
    """A 16 x 16 patch under one tile may be updated in place."""
    from test_zz_no_alloc import _Hip
    npatch, mx = 10, 16
    q = random_state(fa.RP_SHALLOW, npatch, mx, mx, np.random.default_rng(5))
    dx = np.full(npatch, 1.0 / mx)
    slots = np.arange(npatch, dtype=np.int32)
    sv = fa.Solver(fa.RP_SHALLOW, mx, mx, precision=precision, max_patches=npatch)
    hip = _Hip()
    try:
        out = []
        for inplace in (True, False):
            qi, dxp = hip.put(q), hip.put(dx)
            qo = qi if inplace else hip.put(q)
            cfl = C.c_double()
            assert fa.lib().hipclaw_step_batch_noalloc(C.byref(sv.cfg), npatch, qi, qo, None, dxp, dxp, slots,
                                                       npatch, 0.2 / mx, None, C.byref(cfl)) == 0
            out.append((hip.get(qo, q.shape), cfl.value))
        np.testing.assert_array_equal(out[0][0], out[1][0])
        assert out[0][1] == out[1][1]
    finally:
        hip.free()


@pytest.mark.parametrize("mx", [9, 18, 40])
@pytest.mark.parametrize("minlevel", [1, 3, 5])
def test_fp32_seams_conserve(gpu, mx, minlevel):
    """Periodic shallow water on 4, 64 and 1024 patches (strips of a row or two
    up to whole patches): a flux at the seam of two strips or two patches must
    have the same bits on both sides."""
    prob = P.dambreak_problem(minlevel, minlevel, mx=mx)
    prob.periodic = (True, True)
    forest, q0, aux, sv = setup_problem(prob, precision=fa.FP32_BULK)
    dt = P.stable_dt(prob, forest, q0)
    m0, _ = sv.mass()
    sv.advance(dt, 50)
    m1, _ = sv.mass()
    assert np.all(np.abs(m1 - m0) <= 1e-13 * abs(m0[0])), (m0, m1)


def test_odd_graph_where_a_tile_covers_a_patch(gpu):
    """Replays of a graph of three steps, and one after an eager step, equal the
    eager steps."""
    prob = P.dambreak_problem(2, 4, mx=16)
    forest, q0, aux, sv = setup_problem(prob, time_sync=True)
    _, _, _, ref = setup_problem(prob, time_sync=True)
    dt = P.stable_dt(prob, forest, q0)
    sv.capture_graph(dt, 3)
    for k in range(4):
        if k == 2:
            sv.advance(dt, 1)
            ref.advance(dt, 1)
        sv.replay_graph()
        sv.sync()
        ref.advance(dt, 3)
        sv.mass()
        np.testing.assert_array_equal(sv.get_q(), ref.get_q(), err_msg="replay %d" % k)
