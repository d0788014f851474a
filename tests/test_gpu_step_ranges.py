"""FP64 steps of states whose values leave the range of the fast divisions, alone
and beside ordinary ones in the same wave, and of transonic and supersonic
states: the arithmetic is the reference's operation for operation, so the
tolerance is the one of every FP64 step against the oracle (1e-12 in max norm of
each patch and field, or equality where that is zero)."""
import numpy as np
import pytest

import forestclaw_amd as fa
from helpers import claw_for, interior
from oracle_lib import step2_oracle

pytestmark = pytest.mark.gpu

MX, NPATCH = 16, 6


def _state(solver, kind, rng):
    n = MX + 4
    shape = (NPATCH, n, n)
    depth = 1.0 + 0.3 * rng.random(shape)
    speed = np.sqrt(depth) if solver == fa.RP_SHALLOW else np.full(shape, 1.2)
    u = speed * rng.uniform(-0.4, 0.4, shape)
    v = speed * rng.uniform(-0.4, 0.4, shape)
    scale = np.ones(shape)
    if kind == "transonic":
        u, v = speed * rng.uniform(-1.3, 1.3, shape), speed * rng.uniform(-1.3, 1.3, shape)
    elif kind == "supersonic":
        u, v = speed * rng.choice([-3.0, 2.5, 3.0], shape), speed * rng.choice([-2.0, 3.0], shape)
    elif kind == "at rest":
        u[:], v[:], depth[:] = 0.0, -0.0, 1.0
        depth[1::2, 9, 9] = 1.5
    elif kind == "faint":          # momenta down to 1e-250 beside ordinary ones
        faint = 10.0 ** rng.uniform(-250, 0, shape)
        u, v = u * faint, v * faint[::-1]
    elif kind == "shallow":        # 2^-120 of an ordinary state, out of range
        scale[:] = 2.0 ** -120
    elif kind == "deep":
        scale[:] = 2.0 ** 120
    elif kind == "mixed":          # one such patch in a wave with ordinary ones
        scale[1] = 2.0 ** -120
        scale[4] = 2.0 ** 120
    rho = depth * scale
    q = np.empty((NPATCH, 3 if solver == fa.RP_SHALLOW else 4, n, n))
    q[:, 0], q[:, 1], q[:, 2] = rho, rho * u, rho * v
    if solver == fa.RP_EULER:
        q[:, 3] = scale / 0.4 + 0.5 * rho * (u * u + v * v)
    return q


@pytest.mark.parametrize("kind", ["ordinary", "transonic", "supersonic", "at rest", "faint", "shallow", "deep", "mixed"])
@pytest.mark.parametrize("solver", [fa.RP_SHALLOW, fa.RP_EULER])
def test_fp64_step_over_the_range(gpu, solver, kind):
    q = _state(solver, kind, np.random.default_rng(17))
    # the Courant number stays near 0.1: sound speeds go with the root of a depth
    dt = 0.1 / MX / (4.0 * (2.0 ** 60 if solver == fa.RP_SHALLOW and kind in ("deep", "mixed") else 1.0))
    dx = np.full(NPATCH, 1.0 / MX)
    sv = fa.Solver(solver, MX, MX, precision=fa.FP64, max_patches=NPATCH, tile=8)
    sv.set_geometry(dx, dx)
    sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
    sv.set_q(q)
    cfl = sv.advance(dt, 1)
    got = interior(sv.get_q())
    most = 0.0
    for p in range(NPATCH):
        want, c = step2_oracle(claw_for(solver), q[p], None, dx[p], dx[p], dt)
        want = interior(want)
        most = max(most, c)
        for m in range(q.shape[1]):
            tol = 1e-12 * np.abs(want[m]).max()
            assert np.abs(got[p, m] - want[m]).max() <= tol, (p, m)
    assert abs(cfl - most) <= 1e-12 * most
