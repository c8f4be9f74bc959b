"""A new velocity's first pass forms the state trajectory's predictor plan and the
bounds of both directions: what is computed from it must not depend on when the
characteristic scheme or the time integrator was chosen, nor on which direction
comes first, and a velocity whose extremes differ takes its own route each way."""
import numpy as np
import pytest

from claire_amd import ADJOINT, STATE, Claire, synth

pytestmark = pytest.mark.gpu
SHAPE, NT = (48, 32, 64), 4


def _fresh(v, **kw):
    c = Claire(SHAPE, nt=NT, regnorm="h1sn", beta=(1e-2, 0.0, 0.0), **kw)
    try:
        c.set_velocity(v)
        return c.trajectory(STATE), c.trajectory(ADJOINT)
    finally:
        c.close()


def test_scheme_chosen_after_the_velocity():
    v = synth.bandlimited_velocity(SHAPE, kmax=4, cfl=2.0, nt=NT, seed=1)
    w = synth.bandlimited_velocity(SHAPE, kmax=4, cfl=5.0, nt=NT, seed=2)
    want = {(k, order): _fresh(u, rk_order=order) for k, u in (("v", v), ("w", w)) for order in (2, 4)}
    c = Claire(SHAPE, nt=NT, regnorm="h1sn", beta=(1e-2, 0.0, 0.0), pde_solver="rk2")
    try:
        c.set_velocity(v)  # the explicit integrator forms no trajectory
        c.set_pde_solver("sl")
        for k, order in (("v", 2), ("v", 4), ("v", 2), ("w", 2), ("w", 4)):
            if k == "w" and order == 2:
                c.set_velocity(w)
            c.set_rk_order(order)
            print(f"[gpu case] velocity {k} order {order}", flush=True)
            got = c.trajectory(ADJOINT), c.trajectory(STATE)
            assert np.array_equal(got[0], want[k, order][1])
            assert np.array_equal(got[1], want[k, order][0])
    finally:
        c.close()


@pytest.mark.parametrize("order", [2, 4])
def test_one_sided_velocity(order):
    """Up to 5.5 cells per step one way and 0.5 the other: one direction beyond
    the LDS window, the other well inside for part of its stages."""
    from oracle import oracle_py

    x1, x2, x3 = synth.coords(SHAPE, np.float64)
    v = np.zeros((3,) + SHAPE)
    for a, n in enumerate(SHAPE):
        h = synth.TWO_PI / n
        v[a] = NT * h * (2.5 + 3.0 * np.sin(x1 + a) * np.cos(x2) * np.cos(x3 + a))
    v = v.astype(np.float32)
    print(f"[gpu case] one-sided velocity order {order}", flush=True)
    with oracle_py.rk_order(order):
        for got, sigma in zip(_fresh(v, rk_order=order), (+1, -1)):
            # a few FP32 roundings of points of order 1
            assert np.abs(got - oracle_py.trajectory(v, NT, sigma, prec="f32")).max() < 1e-6
