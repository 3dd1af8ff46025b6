"""GPU: graph replays of several steps equal eager steps bit for bit.

The first captured run records one step, later runs of eight or more steps a graph
of eight; the counts below use the small graph alone, the large one alone, and both,
with synchronisation and time reads between the replays, and a change of the step
form, which drops both graphs: the runs behind it capture both again.  The slab form
records its second stream's fork, join and slab events eight times in one capture.
"""
import numpy as np
import pytest

import exahype_amd as E
from exahype_amd import problems as P

pytestmark = pytest.mark.gpu

RUNS = (3, 8, 7, 19, 16, 1, 11, 9)


@pytest.mark.parametrize("dim,order,bc,fp32", [(2, 3, "periodic", False), (2, 4, "wall", False),
                                               (3, 2, "dirichlet", False), (3, 5, "periodic", True)])
def test_graph_runs_equal_eager_runs(dim, order, bc, fp32):
    print(f"[graph steps] dim={dim} order={order} bc={bc} fp32={fp32}", flush=True)
    n = 5 if dim == 2 else 3
    luh = P.density_wave_2d(n, order) if dim == 2 else P.density_wave_3d(n, order, seed=3)
    meshes = []
    for _ in range(2):
        ctx = E.Context(dim, order, precision=E.PREC_FP32 if fp32 else E.PREC_FP64, picard_max=1 if fp32 else 0)
        if fp32:
            ctx.set_initial_guess(E.GUESS_CERK)
        m = E.Mesh(ctx, n, 1.0 / n)
        m.set_solution(luh)
        if bc != "periodic":
            m.set_boundary([E.BC_WALL if bc == "wall" else E.BC_DIRICHLET_ENTROPY_WAVE] * (2 * dim))
        m.init_dt(0.0)
        meshes.append(m)
    eager, graph = meshes
    for i, steps in enumerate(RUNS):
        eager.run(steps)
        graph.run(steps, use_graph=True)
        assert eager.time() == graph.time(), steps
        np.testing.assert_array_equal(eager.get_solution(), graph.get_solution())
        if i == 3:
            for m in meshes:
                m.set_fused(False)


@pytest.mark.parametrize("slabs", [3, 5])
def test_graph_runs_of_the_slab_form(slabs):
    print(f"[graph steps] slabs={slabs}", flush=True)
    n = 5
    meshes = []
    for s in (0, slabs):
        ctx = E.Context(3, 5, precision=E.PREC_FP32, picard_max=1)
        ctx.set_initial_guess(E.GUESS_CERK)
        m = E.Mesh(ctx, n, 1.0 / n)
        m.set_solution(P.density_wave_3d(n, 5, seed=3))
        m.init_dt(0.0)
        if s:
            m.set_overlap(s)
        meshes.append(m)
    eager, graph = meshes
    for steps in (1, 8, 19, 3, 9):
        eager.run(steps)
        graph.run(steps, use_graph=True)
        assert eager.time() == graph.time(), steps
        np.testing.assert_array_equal(eager.get_solution(), graph.get_solution())
        np.testing.assert_array_equal(eager.picard(), graph.picard())
