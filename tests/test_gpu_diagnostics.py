"""Mass sums and gradient tags against numpy: patch counts below, at and above the
workgroups that share the sum, patches smaller and larger than a workgroup's
pass, and thresholds that cells meet exactly.

Sums: math.fsum is exact and a double-double sum of n terms is within n^2 2^-106,
far below the last place, so hi must be its rounding within one unit.  Tags are
yes or no and must be equal."""
import math

import numpy as np
import pytest

import forestclaw_amd as fa

pytestmark = pytest.mark.gpu


def _solver(npatch, mx, my, rng):
    sv = fa.Solver(fa.RP_SHALLOW, mx, my, precision=fa.FP64, max_patches=npatch, tile=8)
    dx, dy = rng.choice([0.25, 0.1, 0.03], npatch), rng.choice([0.5, 0.07], npatch)
    sv.set_geometry(dx, dy)
    sv.set_ghost_program(np.zeros((0, 8), np.int32), np.zeros(7, np.int32))
    q = rng.normal(0, 1, (npatch, 3, my + 4, mx + 4)) * 10.0 ** rng.integers(-6, 6, (npatch, 3, my + 4, mx + 4))
    sv.set_q(q)
    return sv, q, dx, dy


@pytest.mark.parametrize("npatch,mx,my", [(1, 8, 8), (3, 33, 9), (5, 40, 50), (2047, 8, 8), (2048, 8, 9), (2049, 9, 8),
                                          (5000, 8, 8)])
def test_mass_is_the_exact_sum(gpu, npatch, mx, my):
    sv, q, dx, dy = _solver(npatch, mx, my, np.random.default_rng(npatch))
    terms = q[:, :, 2:-2, 2:-2] * (dx * dy)[:, None, None, None]
    hi, lo = sv.mass()
    for m in range(3):
        want = math.fsum(terms[:, m].ravel())
        assert abs(hi[m] - want) <= math.ulp(want)
        assert abs(lo[m]) <= math.ulp(hi[m])


@pytest.mark.parametrize("npatch,mx,my", [(1, 8, 8), (37, 33, 9), (20, 40, 50)])
def test_tags_at_the_threshold(gpu, npatch, mx, my):
    sv, q, dx, dy = _solver(npatch, mx, my, np.random.default_rng(7 * mx))
    q[:, 0] = np.random.default_rng(3).random(q[:, 0].shape)
    q[npatch // 2, 0] = 1.5          # a patch without gradients
    sv.set_q(q)
    f = q[:, 0]
    gx = (f[:, 2:-2, 3:-1] - f[:, 2:-2, 1:-3]) / (2 * dx)[:, None, None]
    gy = (f[:, 3:-1, 2:-2] - f[:, 1:-3, 2:-2]) / (2 * dy)[:, None, None]
    most = np.sqrt(gx * gx + gy * gy + 0.0).reshape(npatch, -1).max(axis=1)
    top = float(np.sort(most)[-1])
    near = [np.nextafter(top, 0.0), top, np.nextafter(top, np.inf), float(np.median(most)), 1e-200, 1e200]
    for thr in near:
        er, ec = sv.tag(0, thr, thr)
        np.testing.assert_array_equal(er, most > thr)
        np.testing.assert_array_equal(ec, (most > thr) | (thr <= 0))   # (a coarsen threshold <= 0 always counts)
    er, ec = sv.tag(0, -1.0, 0.0)
    assert er.all() and ec.all()
