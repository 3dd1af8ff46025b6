"""GPU: the fused transposed step of the acoustic mesh at every compiled order,
against the oracle's FP64 adjoint.

The mesh sizes leave the last workgroup with empty cell slots, two receivers sit
in one cell and one in the source's (their residuals are added inside the step),
and the checkpoint intervals cover a segment of one step, a shorter last segment
and one segment for the whole run.  Bar: 1e-10 relative L2 of the gradient, as of
the other gradient tests; J and the forward state 1e-12.
"""
import ctypes

import numpy as np
import pytest

import exahype_amd as E
import oracle as O
from exahype_amd import problems as P

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / np.linalg.norm(np.ravel(b))


@pytest.mark.parametrize("every", [1, 3, 50])
@pytest.mark.parametrize("order,n", [(1, 3), (2, 5), (3, 3), (4, 3), (5, 2)])
def test_gradient_at_every_order(order, n, every):
    print(f"[adjoint step] order={order} n={n} every={every}", flush=True)
    rng = np.random.default_rng(100 * order + n)
    h, steps = 1.0 / n, 5
    c = 1.0 + 0.2 * rng.uniform(-1, 1, n ** 3)
    rho = 1.0 + 0.1 * rng.uniform(-1, 1, n ** 3)
    u = 0.1 * rng.normal(size=(n ** 3, (order + 1) ** 3, 4))
    luh = P.acoustic_state(n, order, c, rho, u)
    ctx = E.Context(3, order, 4, 2, E.PDE_ACOUSTIC)
    ac = E.Acoustic(ctx, n, h)
    ac.set_solution(luh)
    ac.set_dt(0.0)
    dt = ac.time()[2]
    src = ((0.4 * h, 0.6 * h, 0.3 * h), 1.0, 5.0, 0.05)
    rec = np.array([[0.2, 0.3, 0.4], [0.9, 0.8, 0.1], [0.55, 0.15, 0.75]]) * 0.999
    rec = np.concatenate([rec, rec[1:2] * 0.99, np.array([[0.3 * h, 0.3 * h, 0.3 * h]])])
    obs = rng.normal(0.0, 0.1, (steps, len(rec)))
    orc = O.LinearOracle(3, order)
    J_ref, g_ref = orc.misfit_grad(luh, n, h, dt, steps, src, rec, obs)
    ac.set_source(*src)
    ac.set_receivers(rec)
    J, g = ac.misfit_gradient(steps, obs, checkpoint_every=every)
    assert abs(J - J_ref) <= 1e-12 * abs(J_ref)
    assert rel_l2(g, g_ref) <= 1e-10
    ref = luh.copy()
    orc.run(ref, n, h, dt, steps, src, rec)
    assert rel_l2(ac.get_solution(), ref) <= 1e-12


@pytest.mark.parametrize("order,n", [(1, 1), (2, 1), (2, 2), (3, 2), (4, 1), (4, 2), (5, 1)])
def test_fused_steps_on_the_smallest_meshes(order, n):
    """Corrector and next predictor in one kernel where a cell is its own neighbour, or both
    neighbours of a direction are one cell; receivers in the same cell. <= 1e-12 (the parity bar)."""
    print(f"[fused steps] order={order} n={n}", flush=True)
    rng = np.random.default_rng(7 * order + n)
    h, steps = 1.0 / n, 4
    c, rho = 1.0 + 0.2 * rng.uniform(-1, 1, n ** 3), 1.0 + 0.1 * rng.uniform(-1, 1, n ** 3)
    luh = P.acoustic_state(n, order, c, rho, 0.1 * rng.normal(size=(n ** 3, (order + 1) ** 3, 4)))
    src = ((0.4 * h, 0.6 * h, 0.3 * h), 1.0, 5.0, 0.05)
    rec = rng.uniform(0.05, 0.95, size=(6, 3))
    ac = E.Acoustic(E.Context(3, order, 4, 2, E.PDE_ACOUSTIC), n, h)
    ac.set_solution(luh)
    ac.set_dt(0.0)
    dt = ac.time()[2]
    ac.set_source(*src)
    ac.set_receivers(rec)
    got = np.concatenate([ac.run(steps - 1), ac.run(1)])  # fused steps, then a single plain one
    ref = luh.copy()
    want, _ = O.LinearOracle(3, order).run(ref, n, h, dt, steps, src, rec)
    assert rel_l2(got, want) <= 1e-12
    assert rel_l2(ac.get_solution(), ref) <= 1e-12


@pytest.mark.parametrize("order,n", [(2, 49), (3, 41), (4, 13)])
def test_line_predictor_in_large_workgroups(order, n):
    """Sizes at which the line predictor takes 256 lanes, the last workgroup partly empty, against the node
    form: single steps (predictor and corrector apart), the faces of a gradient, and a captured run."""
    print(f"[large workgroups] order={order} n={n}", flush=True)
    rng = np.random.default_rng(order)
    c, rho = 1.0 + 0.2 * rng.uniform(-1, 1, n ** 3), 1.0 + 0.1 * rng.uniform(-1, 1, n ** 3)
    luh = P.acoustic_state(n, order, c, rho, 0.1 * rng.normal(size=(n ** 3, (order + 1) ** 3, 4)))
    ac = E.Acoustic(E.Context(3, order, 4, 2, E.PDE_ACOUSTIC), n, 1.0 / n)
    ac.set_dt(0.0)
    ac.set_source((0.4, 0.6, 0.3), 1.0, 5.0, 0.05)
    ac.set_receivers(rng.uniform(0.05, 0.95, size=(6, 3)))
    obs = rng.normal(0.0, 0.1, (2, 6))
    got = []
    for variant in (0, 1):
        ac.set_predictor(variant)
        ac.set_solution(luh)
        ac.set_step(0)
        ac.run(1)
        ac.run(1)
        u = ac.get_solution()
        J, g = ac.misfit_gradient(2, obs, checkpoint_every=1)
        ac.run(2, use_graph=True)
        got.append((u, g, ac.get_solution()))
    ac.close()
    for line, node, tol in zip(*got, (1e-12, 1e-10, 1e-12)):
        assert rel_l2(line, node) <= tol


def shot(order=4, n=5, receivers=3, seed=0):
    rng = np.random.default_rng(seed)
    c, rho = 1.0 + 0.2 * rng.uniform(-1, 1, n ** 3), 1.0 + 0.1 * rng.uniform(-1, 1, n ** 3)
    luh = P.acoustic_state(n, order, c, rho, 0.1 * rng.normal(size=(n ** 3, (order + 1) ** 3, 4)))
    ac = E.Acoustic(E.Context(3, order, 4, 2, E.PDE_ACOUSTIC), n, 1.0 / n)
    ac.set_solution(luh)
    ac.set_dt(0.0)
    ac.set_source((0.4, 0.6, 0.3), 1.0, 5.0, 0.05)
    place(ac, receivers)
    return ac, luh


def place(ac, receivers):
    ac.set_receivers(np.random.default_rng(receivers).uniform(0.05, 0.95, size=(receivers, 3)))


def one_gradient(ac, luh, steps, receivers, every):
    ac.set_solution(luh)
    ac.set_step(0)
    obs = np.random.default_rng(steps + receivers).normal(0.0, 0.1, (steps, receivers))
    J, g = ac.misfit_gradient(steps, obs, checkpoint_every=every)
    return J, g, ac.get_solution()


def test_gradients_on_buffers_of_earlier_calls():
    """One object through other intervals, step counts and receivers, runs in between, against fresh
    objects: bit for bit."""
    ac, luh = shot()
    for steps, receivers, every in ((9, 3, 1), (9, 3, 50), (7, 5, 3), (12, 2, 4), (3, 5, 2), (12, 2, 12)):
        print(f"[kept buffers] steps={steps} receivers={receivers} every={every}", flush=True)
        place(ac, receivers)
        got = one_gradient(ac, luh, steps, receivers, every)
        ac.run(3)
        fresh, _ = shot(receivers=receivers)
        want = one_gradient(fresh, luh, steps, receivers, every)
        fresh.close()
        assert got[0] == want[0]
        np.testing.assert_array_equal(got[1], want[1])
        np.testing.assert_array_equal(got[2], want[2])
    ac.close()


def test_gradient_without_memory_for_the_faces():
    """A segment's faces larger than a quarter of what is free (most of the memory is held by the test):
    they are formed step by step, and the gradient is the one with the faces kept, bit for bit."""
    n, order, every, steps = 13, 4, 130, 131
    faces = n ** 3 * 6 * (order + 1) ** 2 * 4 * 8 * every
    ac, luh = shot(order, n)
    want = one_gradient(ac, luh, steps, 3, every)
    ac.close()
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    held = ctypes.c_void_p()

    def free():
        f, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(total)) == 0
        return f.value

    hold = free() - (4 << 30)
    print(f"[no faces] holding {hold >> 20} MiB", flush=True)
    assert hip.hipMalloc(ctypes.byref(held), ctypes.c_size_t(hold)) == 0
    try:
        ac, luh = shot(order, n)
        assert faces > free() // 4
        got = one_gradient(ac, luh, steps, 3, every)
        ac.close()
    finally:
        assert hip.hipFree(held) == 0
    assert got[0] == want[0]
    np.testing.assert_array_equal(got[1], want[1])
    np.testing.assert_array_equal(got[2], want[2])
