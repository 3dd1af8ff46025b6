"""GPU: edges of the uneven-work kernels against the oracle.

* face prolongation and restriction of the two-level mesh at every compiled 3D
  order (one refined cell: six coarse faces, 54 subfaces), two steps;
* an ensemble of more instances than a corrector workgroup has cells, of one to
  four cells per side, so that workgroups hold cells of several instances and
  their stable-dt minima are merged cell by cell; again after the autotuner,
  whose trials must leave no minima behind.

* a list of more 3D order 4 faces than two share a wavefront, against the same
  faces in two lists that are shorter, bit for bit (a face's sums are the same).

<= 1e-12 relative L2 (the FP64 parity bar); dt to 1e-13, as a minimum of values
that differ by rounding.
"""
import numpy as np
import pytest
import torch

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


def test_long_and_short_face_lists():
    print("[uneven] face lists", flush=True)
    ctx = E.Context(3, 4)
    n, s = 3334, torch.cuda.current_stream().cuda_stream
    i = torch.arange(n, dtype=torch.int32)
    faces = torch.cat([torch.stack([i, (i + 7) % n, torch.full_like(i, d), torch.zeros_like(i)], 1)
                       for d in range(3)]).contiguous().cuda()  # 10,002
    g = torch.Generator().manual_seed(3)
    qb = 1.0 + torch.rand(n, 6, 25, 5, generator=g, dtype=torch.float64)
    qb[..., 4] += 8.0
    fb = torch.rand(n, 6, 25, 5, generator=g, dtype=torch.float64)
    qb, long, short = qb.cuda(), fb.cuda(), fb.cuda()
    ctx.batch_riemann(s, len(faces), faces.data_ptr(), qb.data_ptr(), long.data_ptr())
    for part in (faces[:5001], faces[5001:]):
        ctx.batch_riemann(s, len(part), part.data_ptr(), qb.data_ptr(), short.data_ptr())
    torch.cuda.synchronize()
    assert torch.equal(long, short) and not torch.equal(long, fb.cuda())
    ctx.close()
