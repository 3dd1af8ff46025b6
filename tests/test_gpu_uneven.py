"""GPU: edges of the uneven-work kernels against the oracle.

* face prolongation and restriction of the two-level mesh at every compiled 3D
  order (one refined cell: six coarse faces, 54 subfaces), two steps;
* an ensemble of more instances than a corrector workgroup has cells, of one to
  four cells per side, so that workgroups hold cells of several instances and
  their stable-dt minima are merged cell by cell; again after the autotuner,
  whose trials must leave no minima behind.

<= 1e-12 relative L2 (the FP64 parity bar); dt to 1e-13, as a minimum of values
that differ by rounding.
"""
import numpy as np
import pytest

import exahype_amd as E
from exahype_amd import problems as P
import oracle as O

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(np.ravel(b))


@pytest.mark.parametrize("order", [1, 2, 3, 4, 5])
def test_two_level_faces_at_every_order(order):
    print(f"[uneven] two-level order={order}", flush=True)
    n = 3
    refined = np.zeros(n ** 3, dtype=np.uint8)
    refined[13] = 1
    mesh = E.Amr(E.Context(3, order), n, refined)
    level, coords = mesh.leaves()
    luh = P.amr_density_wave(order, n, level, coords)
    ref = luh.copy()
    dt_ref = O.AmrOracle(3, order).amr_run(ref, n, refined, 2)
    mesh.set_solution(luh)
    mesh.init_dt(0.0)
    mesh.run(2)
    assert rel_l2(mesh.get_solution(), ref) <= 1e-12
    assert abs(mesh.time()[1] - dt_ref) <= 1e-13 * dt_ref


@pytest.mark.parametrize("dim,order", [(2, 1), (2, 4), (2, 6), (3, 2)])
def test_ensemble_workgroups_with_several_instances(dim, order):
    print(f"[uneven] ensemble dim={dim} order={order}", flush=True)
    sizes = [1, 2, 1, 1, 3, 1, 2, 4] * (5 if dim == 2 else 2)
    ens = E.Ensemble(E.Context(dim, order), sizes)
    orc = O.Oracle(dim, order)
    states, refs = [], []
    for i, n in enumerate(sizes):
        if dim == 2:
            pts = P.node_points(n, order, 2)
            rho = 1.0 + 0.1 * np.sin(2 * np.pi * (pts[..., 0] + pts[..., 1]) + i)
            one = np.ones_like(rho)
            luh = P.euler_state(rho, one, (0.3 + 0.1 * i) * one, 0 * one, one)
        else:
            luh = P.density_wave_3d(n, order, seed=i)
        states.append(np.ascontiguousarray(luh, dtype=np.float64).ravel())
        ref = states[-1].copy()
        dt, _ = orc.run_uniform(ref, n, 1.0 / n, 2)
        refs.append((ref, dt))
    for tuned in (False, True):
        for i, luh in enumerate(states):
            ens.set_solution(i, luh)
        ens.init_dt(0.0)
        if tuned:
            ens.autotune()
        ens.run(2, use_graph=tuned)
        for i, (ref, dt) in enumerate(refs):
            assert rel_l2(ens.get_solution(i), ref) <= 1e-12, (tuned, i)
            assert abs(ens.time(i)[1] - dt) <= 1e-13 * dt, (tuned, i)
