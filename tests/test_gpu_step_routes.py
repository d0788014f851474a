"""A patch's update has the same bits from the tile kernel (small launches, and
small ones in place) as from the strip kernel (large ones): the same K patches
alone and repeated until the launch takes strips.  Everything is compared exactly
(zeros of either sign are equal, NaN equals NaN): FP64 divides and takes roots by
the IEEE operations in the tile kernel and by shared reciprocals in the strip
kernel, FP32-bulk names its fused operations in both."""
import ctypes as C

import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import random_aux, random_state
from test_gpu_step_ranges import _state
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu

K = 5
SOLVERS = [fa.RP_ADVECTION, fa.RP_SHALLOW, fa.RP_EULER]


def _methods(solver, other):
    mw = fa.SOLVER_SHAPES[solver][1]
    return dict(order=(2, 2), mthlim=[4] * mw) if not other else dict(order=(2, 1), mthlim=[2, 6, 0, 3][:mw])


def _batch(sv, hip, q, aux, dx, dt, inplace):
    """hipclaw_step_batch_noalloc over all patches of q."""
    n = q.shape[0]
    qi = hip.put(q)
    qo = qi if inplace else hip.put(q)
    cfl = C.c_double(-1.0)
    rc = fa.lib().hipclaw_step_batch_noalloc(C.byref(sv.cfg), n, qi, qo, hip.put(aux) if aux is not None else None,
                                             hip.put(dx), hip.put(dx), np.arange(n, dtype=np.int32), n, dt, None,
                                             C.byref(cfl))
    assert rc == 0, fa.lib().hipclaw_last_error()
    return hip.get(qo, q.shape), cfl.value


@pytest.mark.parametrize("other", [False, True], ids=["mc", "limiters"])
@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("mx,my,tile", [(8, 8, 8), (9, 13, 8), (20, 20, 8), (16, 16, 16), (40, 17, 16), (32, 32, 32)])
def test_batch_alone_and_among_many(gpu, solver, mx, my, tile, precision, other):
    if tile == 32 and (solver == fa.RP_EULER or (solver == fa.RP_ADVECTION and precision == fa.FP64)):
        pytest.skip("no 32 x 32 tile")
    rng = np.random.default_rng(mx + my + solver)
    q = random_state(solver, K, mx, my, rng)
    aux = random_aux(K, mx, my, rng) if solver == fa.RP_ADVECTION else None
    dx = rng.choice([1.0, 0.5], K) / mx
    many = 8192 // K if mx * my < 200 else 2048 // K
    sv = fa.Solver(solver, mx, my, precision=precision, max_patches=1, tile=tile, **_methods(solver, other))
    dt = 0.05 / mx
    hip = _Hip()
    try:
        want, cfl = _batch(sv, hip, np.tile(q, (many, 1, 1, 1)), None if aux is None else np.tile(aux, (many, 1, 1, 1)),
                           np.tile(dx, many), dt, False)
        for inplace in ((False, True) if mx == tile and my == tile else (False,)):
            print("case", solver, (mx, my, tile), "precision", precision, "in place", inplace, flush=True)
            got, c = _batch(sv, hip, q, aux, dx, dt, inplace)
            np.testing.assert_array_equal(got, want[:K])
            assert c == cfl
        np.testing.assert_array_equal(want[-K:, :, 2:-2, 2:-2], want[:K, :, 2:-2, 2:-2])
    finally:
        hip.free()


@pytest.mark.parametrize("kind", ["ordinary", "transonic", "supersonic", "at rest", "faint", "shallow", "deep", "mixed",
                                  "nan", "infinite", "edges"])
@pytest.mark.parametrize("solver", [fa.RP_SHALLOW, fa.RP_EULER])
def test_fp64_divisions_over_the_range(gpu, solver, kind):
    """The shared reciprocals and roots against IEEE divisions, beyond the range
    they are used in and at its edges."""
    rng = np.random.default_rng(23)
    q = _state(solver, kind, rng)
    inner = q[:, :, 6:14, 6:14]
    where = rng.random(inner[:, 0].shape) < 0.02
    if kind == "nan":
        inner[:, 1][where] = np.nan
    elif kind == "infinite":
        inner[:, 2][where] = np.inf
        inner[:, 1][rng.random(where.shape) < 0.01] = -np.inf
    elif kind == "edges":     # momenta and depths beside the exponents where the fast forms end
        low = -600 if solver == fa.RP_SHALLOW else -300
        for m, bounds in ((0, (-100, 100)), (1, (low, 200)), (2, (low, 200))):
            at = rng.random(where.shape) < 0.05
            e = rng.choice([b + d for b in bounds for d in (-2, -1, 0, 1, 2)], at.sum())
            inner[:, m][at] = np.ldexp(rng.uniform(0.5, 1.0, at.sum()), e)
    n, mx = q.shape[0], q.shape[3] - 4
    dt = 0.1 / mx / (4.0 * (2.0 ** 60 if solver == fa.RP_SHALLOW and kind in ("deep", "mixed") else 1.0))
    dx = np.full(n, 1.0 / mx)
    many = 2048 // n
    for lim in (4, 3):
        sv = fa.Solver(solver, mx, mx, max_patches=1, tile=16, mthlim=[lim] * fa.SOLVER_SHAPES[solver][1])
        hip = _Hip()
        try:
            want, cfl = _batch(sv, hip, np.tile(q, (many, 1, 1, 1)), None, np.tile(dx, many), dt, False)
            got, c = _batch(sv, hip, q, None, dx, dt, False)
            np.testing.assert_array_equal(got, want[:n])
            assert c == cfl
        finally:
            hip.free()


def _advanced(solver, precision, q, aux, dx, mx, sub, calls):
    n = q.shape[0]
    sv = fa.Solver(solver, mx, mx, precision=precision, max_patches=n, tile=8, time_sync=True, subcycle=sub)
    sv.set_geometry(dx, dx)
    sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
    sv.set_q(q)
    if aux is not None:
        sv.set_aux(aux)
    slots = np.arange(n, dtype=np.int32)
    for _ in range(calls):     # a subcycling state's registers add up
        cfl = sv.step_batch(slots, 0.03 / mx)
    return sv.get_q(), sv.get_registers(), cfl


@pytest.mark.parametrize("sub", [False, True], ids=["overwritten", "accumulated"])
@pytest.mark.parametrize("precision", [fa.FP64, fa.FP32_BULK])
@pytest.mark.parametrize("solver", SOLVERS)
@pytest.mark.parametrize("mx", [8, 20])
def test_registers_alone_and_among_many(gpu, solver, mx, precision, sub):
    rng = np.random.default_rng(mx + solver)
    q = random_state(solver, K, mx, mx, rng)
    aux = random_aux(K, mx, mx, rng) if solver == fa.RP_ADVECTION else None
    dx = rng.choice([1.0, 0.5], K) / mx
    many = 8192 // K if mx == 8 else 1024 // K     # (8 x 8 steps in place)
    print("case", solver, mx, "precision", precision, "subcycle", sub, flush=True)
    want = _advanced(solver, precision, np.tile(q, (many, 1, 1, 1)), None if aux is None else np.tile(aux, (many, 1, 1, 1)),
                     np.tile(dx, many), mx, sub, 2)
    got = _advanced(solver, precision, q, aux, dx, mx, sub, 2)
    np.testing.assert_array_equal(got[0], want[0][:K])
    np.testing.assert_array_equal(got[1], want[1][:K])
    assert got[2] == want[2]
