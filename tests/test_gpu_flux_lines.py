"""GPU: the FP32 predictors of 3D order 5, whose spatial contractions after the sweeps
run over lines of the per-point arrays, through exa_batch_predictor against the
FP64 oracle with the same guess and iteration count.

Each variable of a cell gets its own seeded variation in each direction, so that a
line taken along another direction, of another variable or at another place is an
error of the size of the variation (0.03 to 0.1), far over the bounds.

Bounds (relative L2): inputs, fluxes and sums carry 2^-24 = 6e-8 each.  The
extrapolated state sums a B-point line with |phi(0)| <= 2 of values that the
iteration moved by dt/h |dudx| B terms (order one at the CFL step): 64 roundings
cover it, 4e-6; the flux multiplies by speeds up to 4, 1.6e-5; lduh is a difference
of fluxes whose sum is some 1/30 of its terms, 5e-4.
"""
import numpy as np
import pytest
import torch

import exahype_amd as E
from exahype_amd import problems as P
import oracle as O

pytestmark = pytest.mark.gpu

ORDER, B = 5, 6


def states(count, seed):
    rng = np.random.default_rng(seed)
    xi = np.polynomial.legendre.leggauss(B)[0] * 0.5 + 0.5
    grids = np.meshgrid(xi, xi, xi, indexing="ij")
    out = np.zeros((count, B ** 3, 5))
    for i in range(count):
        f = [sum(rng.uniform(0.03, 0.1) * np.sin(2 * np.pi * g + rng.uniform(0, 6)) for g in grids).ravel()
             for _ in range(5)]
        rho, p = 1.0 + f[0], 1.0 + f[4]
        vel = [0.4 + f[1], -0.3 + f[2], 0.2 + f[3]]
        out[i, :, 0] = rho
        for d in range(3):
            out[i, :, 1 + d] = rho * vel[d]
        out[i, :, 4] = p / 0.4 + 0.5 * rho * sum(v * v for v in vel)
    return out


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def batch(ctx, luh, h, dt):
    n, faces = len(luh), 6 * B * B * 5
    t = {"luh": torch.as_tensor(luh, device="cuda"), "h": torch.full((n,), h, dtype=torch.float64, device="cuda"),
         "dt": torch.full((1,), dt, dtype=torch.float64, device="cuda"),
         "lduh": torch.full((n, B ** 3, 5), np.nan, dtype=torch.float64, device="cuda"),
         "qb": torch.full((n, faces), np.nan, dtype=torch.float64, device="cuda"),
         "fb": torch.full((n, faces), np.nan, dtype=torch.float64, device="cuda"),
         "pic": torch.full((n,), -1, dtype=torch.int32, device="cuda")}
    p = {k: v.data_ptr() for k, v in t.items()}
    ctx.batch_predictor(torch.cuda.current_stream().cuda_stream, n, p["luh"], p["h"], p["dt"], p["lduh"], p["qb"],
                        p["fb"], p["pic"])
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in t.items()}


# (Picard iterations, CERK guess, predictor variant): the one-iteration kernels, the
# fixed-count kernels, the tile kernel
@pytest.mark.parametrize("picard,cerk,variant", [(1, True, 0), (1, False, 0), (3, True, 0), (3, False, 0),
                                                 (3, False, 4)])
def test_every_line_of_a_cell(picard, cerk, variant):
    print(f"[flux lines] picard={picard} cerk={cerk} variant={variant}", flush=True)
    ctx = E.Context(3, ORDER, precision=E.PREC_FP32, picard_max=picard)
    if cerk:
        ctx.set_initial_guess(E.GUESS_CERK)
    ctx.set_predictor_variant(variant)
    ctx.set_picard_guard(0.0)  # every cell at the fixed count
    orc = O.Oracle(3, ORDER, max_picard=picard, dialect="cerk" if cerk else None)
    h = 0.1
    luh = states(3, 10 * picard + cerk)
    dt = 0.4 * min(orc.stable_dt(u.ravel().copy(), [h] * 3) for u in luh)
    want = [orc.fused(u.ravel().copy(), [h] * 3, dt) for u in luh]
    got = batch(ctx, luh, h, dt)
    for key, ref, tol in (("lduh", "lduh", 5e-4), ("qb", "lQhbnd", 4e-6), ("fb", "lFhbnd", 1.6e-5)):
        for i, w in enumerate(want):
            assert rel_l2(got[key][i].ravel(), np.ravel(w[ref])) <= tol, (key, i)
    alone = batch(ctx, luh[2:], h, dt)
    for key in ("lduh", "qb", "fb"):
        np.testing.assert_array_equal(alone[key][0], got[key][2])
    ctx.close()


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_rounding_of_one_step(seed):
    """One CERK iteration in FP32 against the same rule in FP64 on 18^3 cells: the node form, which sums all
    products of a line, was 2.519e-8 to 2.521e-8 off; half a percent more is another order of summation."""
    print(f"[flux lines] rounding seed={seed}", flush=True)
    n, got = 18, []
    luh = P.density_wave_3d(n, ORDER, seed=seed)
    for precision in (E.PREC_FP32, E.PREC_FP64):
        ctx = E.Context(3, ORDER, precision=precision, picard_max=1)
        ctx.set_initial_guess(E.GUESS_CERK)
        if precision == E.PREC_FP32:
            ctx.set_picard_guard(0.0)
        mesh = E.Mesh(ctx, n, 1.0 / n)
        mesh.set_solution(luh)
        mesh.init_dt(0.0)
        mesh.run(1)
        mesh.sync()
        got.append(mesh.get_solution())
        mesh.close()
        ctx.close()
    assert rel_l2(*got) <= 2.533e-8
