"""A forest that outgrows its state: the new slab replaces both old ones, whichever
holds the state, with a kept state and a captured graph at the time of the regrid.
The reference's room is large enough from the start, so nothing there is moved;
everything is compared exactly."""
import numpy as np
import pytest

import forestclaw_amd as fa
from forestclaw_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["dambreak", "advection"])
@pytest.mark.parametrize("tile", [8, 16])
@pytest.mark.parametrize("steps", [2, 3])
def test_growth_from_either_slab(gpu, name, tile, steps):
    mk = P.dambreak_problem if name == "dambreak" else P.advection_problem

    def run(room):
        prob = mk(2, 3, mx=16)
        forest = P.build_forest(prob)
        q0, aux = P.initial_data(prob, forest)
        n = forest.npatch
        sv = fa.Solver(prob.solver, 16, 16, mthbc=prob.mthbc, tile=tile, max_patches=n * room,
                       time_sync=name == "dambreak")
        sv.set_forest(forest, prob.extent)
        sv.set_q(q0)
        if aux is not None:
            sv.set_aux(aux)
        sv.ghost_fill()
        dt = 0.1 * P.stable_dt(prob, forest, q0)
        out = []
        for cycle in range(2):
            sv.capture_graph(dt, 2)
            sv.replay_graph()
            sv.advance(dt, steps)
            sv.save_step()
            sv.advance(dt, 1)
            refine = np.ones(forest.npatch, np.int32)     # everywhere: four times the patches
            kind, src = forest.adapt(refine, np.zeros_like(refine), 2, 4 + cycle)
            sv.regrid(forest, kind, src, prob.extent)
            if aux is not None:
                sv.set_aux(P.initial_data(prob, forest)[1])
            with pytest.raises(fa.HipclawError):
                sv.restore_step()
            with pytest.raises(fa.HipclawError):
                sv.replay_graph()
            sv.ghost_fill()
            sv.advance(dt, 3)
            out += [sv.get_q(), sv.mass()[0]]
        return out

    for a, b in zip(run(1), run(40)):
        np.testing.assert_array_equal(a, b)
