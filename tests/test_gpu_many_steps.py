"""More time steps than one launch takes fields of: on 8^3 the gradients of 22001
states are 66003 fields, beyond the 65535 of a launch."""
import numpy as np
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu

SHAPE, BETA = (8, 8, 8), (1e-2, 0.0, 0.0)


def _solve(nt, mT, mR, vt):
    c = Claire(SHAPE, nt=nt, regnorm="h1sn", beta=BETA)
    try:
        c.set_template_image(mT)
        c.set_reference_image(mR)
        c.set_velocity(np.zeros((3,) + SHAPE, np.float32))
        return c.solve_adjoint()[1], c.hessian_matvec(vt), c.grad(mT)
    finally:
        c.close()


def test_gradients_of_a_long_series():
    print("\n[gpu case] 22000 time steps at 8^3", flush=True)
    nt = 22000
    mT, mR = (synth.gaussian_blobs(SHAPE, count=3, seed=s) for s in (1, 2))
    vt = synth.bandlimited_velocity(SHAPE, kmax=2, cfl=1.0, nt=4, seed=3)
    b, H, g = _solve(nt, mT, mR, vt)
    hd = float(np.prod([synth.TWO_PI / n for n in SHAPE]))
    want = hd * (mR - mT)[None] * g  # the body force of v = 0
    assert np.abs(b - want).max() <= 1e-5 * np.abs(want).max()
    # the matvec sums nt terms in FP32
    few = _solve(4, mT, mR, vt)[1]
    assert np.abs(H - few).max() <= nt * 2.0 ** -24 * np.abs(few).max()
