"""GPU: the column / line predictor at the edges of its workgroups, through
exa_batch_predictor against the oracle cell by cell.

The kernel packs several small cells into a workgroup and takes the derivative
lines of all of them as one list of tasks, so the batch sizes are the ones around
a workgroup's cell count: one cell, one less, exactly, one more, and two
workgroups and a cell.  Cells of one workgroup differ in roughness, so that they
stop after different Picard counts and frozen cells share rounds with running ones.

FP64: <= 1e-12 relative L2 per array (the FP64 parity bar) and identical counts.
FP32 (three fixed iterations): inputs, fluxes and sums carry 2^-24 = 6e-8 each.
The extrapolated state sums a B-point line with |phi(0)| <= 2 of values that the
iteration moved by dt/h |dudx| B terms (order one at the CFL step): 64 roundings
cover it, 4e-6; the flux multiplies by speeds up to 4, 1.6e-5; lduh is a difference
of fluxes whose sum is some 1/30 of its terms, 5e-4.
"""
import numpy as np
import pytest
import torch

import exahype_amd as E
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (2, 6), (3, 1), (3, 2), (3, 3), (3, 4), (3, 5)]


def cells_per_workgroup(dim, order, form):
    """The kernel's packing: the smallest workgroup of 64, 128 or 256 lanes that is 93 % full; 256 lanes at
    order 1, 64 in 3D at order 2 in FP64."""
    ns = (order + 1) ** dim
    if order == 1:
        return 256 // ns
    if (dim, order) == (3, 2) and form != "fp32":
        return 64 // ns
    for t in (64, 128, 256):
        if t // ns * ns * 100 >= 93 * t:
            return t // ns
    return 256 // ns


def states(dim, order, count, seed):
    """One smooth Euler state per cell; amplitudes from 1e-9 (two iterations) to 0.1."""
    rng = np.random.default_rng(seed)
    B = order + 1
    xi = np.polynomial.legendre.leggauss(B)[0] * 0.5 + 0.5
    grids = np.meshgrid(*([xi] * dim), indexing="ij")
    out = np.zeros((count, B ** dim, 5))
    for i in range(count):
        amp = 10.0 ** rng.uniform(-9, -1)
        f = [amp * sum(rng.uniform(-1, 1) * np.sin(2 * np.pi * g + rng.uniform(0, 6)) for g in grids).ravel()
             for _ in range(5)]
        rho, p = 1.0 + f[0], 1.0 + f[4]
        vel = [0.4 + f[1], -0.3 + f[2], (0.2 + f[3]) if dim == 3 else 0.0 * rho]
        out[i, :, 0] = rho
        for d in range(3):
            out[i, :, 1 + d] = rho * vel[d]
        out[i, :, 4] = p / 0.4 + 0.5 * rho * sum(v * v for v in vel)
    return out


def rel_l2(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def batch(ctx, luh, h, dt, dim, order):
    n, B = len(luh), order + 1
    nf = B ** (dim - 1)
    t = {"luh": torch.as_tensor(luh, device="cuda"), "h": torch.full((n,), h, dtype=torch.float64, device="cuda"),
         "dt": torch.full((1,), dt, dtype=torch.float64, device="cuda"),
         "lduh": torch.full((n, B ** dim, 5), np.nan, dtype=torch.float64, device="cuda"),
         "qb": torch.full((n, 2 * dim * nf * 5), np.nan, dtype=torch.float64, device="cuda"),
         "fb": torch.full((n, 2 * dim * nf * 5), np.nan, dtype=torch.float64, device="cuda"),
         "pic": torch.full((n,), -1, dtype=torch.int32, device="cuda")}
    p = {k: v.data_ptr() for k, v in t.items()}
    ctx.batch_predictor(torch.cuda.current_stream().cuda_stream, n, p["luh"], p["h"], p["dt"], p["lduh"], p["qb"],
                        p["fb"], p["pic"])
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in t.items()}


@pytest.mark.parametrize("form", ["fp64", "fp64-cerk", "fp32"])
@pytest.mark.parametrize("dim,order", CASES)
def test_batches_around_a_workgroup(dim, order, form):
    cpb = cells_per_workgroup(dim, order, form)
    print(f"[columns] dim={dim} order={order} form={form} cells per workgroup={cpb}", flush=True)
    ctx = E.Context(dim, order, precision=E.PREC_FP32 if form == "fp32" else E.PREC_FP64,
                    picard_max=3 if form == "fp32" else 0)
    if form == "fp64-cerk":
        ctx.set_dialect(E.DIALECT_OPTIMISED_CERK)
    ctx.set_predictor_variant(1)  # 3D order 5 in FP32 too: not the x-line kernel
    orc = O.Oracle(dim, order, dialect="optimised-cerk") if form == "fp64-cerk" else O.Oracle(
        dim, order, max_picard=3 if form == "fp32" else None)
    h = 0.1
    sizes = sorted({1, max(cpb - 1, 1), cpb, cpb + 1, 2 * cpb + 1})
    luh = states(dim, order, sizes[-1], 10 * dim + order)
    dt = 0.4 * min(orc.stable_dt(u.ravel().copy(), [h] * dim) for u in luh)
    want = [orc.fused(u.ravel().copy(), [h] * dim, dt) for u in luh]
    tol = dict(lduh=5e-4, qb=4e-6, fb=1.6e-5) if form == "fp32" else dict(lduh=1e-12, qb=1e-12, fb=1e-12)
    for n in sizes:
        got = batch(ctx, luh[:n], h, dt, dim, order)
        if form != "fp32":
            assert got["pic"].tolist() == [w["iters"] for w in want[:n]]
        for key, ref in (("lduh", "lduh"), ("qb", "lQhbnd"), ("fb", "lFhbnd")):
            ref = np.concatenate([np.ravel(w[ref]) for w in want[:n]])
            assert rel_l2(got[key].ravel(), ref) <= tol[key], (n, key)
        # the cells of a batch do not depend on their neighbours in it
        alone = batch(ctx, luh[n - 1:n], h, dt, dim, order)
        for key in ("lduh", "qb", "fb", "pic"):
            np.testing.assert_array_equal(alone[key][0], got[key][n - 1])
    ctx.close()


@pytest.mark.parametrize("pde,form", [("euler", "trivial"), ("euler", "cerk"), ("advection", "trivial"),
                                      ("advection", "cerk")])
def test_two_and_three_waves_of_order4(pde, form):
    """3D order 4 in FP64: one batch beyond the cells that two waves per SIMD hold against its halves
    within, cell by cell the same operations: bit for bit."""
    print(f"[columns] waves pde={pde} form={form}", flush=True)
    adv = [1.0, 0.5, 0.25]
    ctx = E.Context(3, 4, 5, 0, E.PDE_EULER if pde == "euler" else E.PDE_ADVECTION, picard_max=2)
    if pde != "euler":
        ctx.set_advection(np.array(adv))
    if form == "cerk":
        ctx.set_initial_guess(E.GUESS_CERK)
    luh = np.tile(states(3, 4, 50, 11), (27, 1, 1))[:1301]
    whole = batch(ctx, luh, 0.1, 1e-3, 3, 4)
    halves = [batch(ctx, part, 0.1, 1e-3, 3, 4) for part in (luh[:651], luh[651:])]
    for key in ("lduh", "qb", "fb"):
        np.testing.assert_array_equal(whole[key], np.concatenate([h[key] for h in halves]))
    orc = O.Oracle(3, 4, pde=O.PDE_EULER if pde == "euler" else O.PDE_ADVECTION, adv=adv, max_picard=2,
                   dialect="cerk" if form == "cerk" else None)
    for c in (0, 1300):
        want = orc.fused(luh[c].ravel().copy(), [0.1] * 3, 1e-3)
        for key, ref in (("lduh", "lduh"), ("qb", "lQhbnd"), ("fb", "lFhbnd")):
            assert rel_l2(whole[key][c].ravel(), np.ravel(want[ref])) <= 1e-12, (key, c)
    ctx.close()
