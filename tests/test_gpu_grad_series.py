"""The gradients of the state's time series go through passes of several fields
per launch.  A constant velocity of one cell per time step shifts the fields, so
the adjoint's body force is a sum of shifted products that single-field gradients
give directly: for series in one group, in uneven groups and one field at a
time."""
import numpy as np
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,nt", [((16, 32, 48), 3), ((192, 150, 192), 4), ((256, 192, 256), 2)],
                         ids=["one-group", "uneven-groups", "single-fields"])
def test_body_force_of_a_shift(shape, nt):
    print(f"\n[gpu case] gradient series {shape} nt={nt}", flush=True)
    mT = synth.gaussian_blobs(shape, count=6, seed=3)
    mR = synth.gaussian_blobs(shape, count=6, seed=4)
    v = np.zeros((3,) + shape, np.float32)
    v[0] = nt * synth.TWO_PI / shape[0]
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=(1e-2, 0.0, 0.0))
    try:
        g = c.grad(mT)
        c.set_template_image(mT)
        c.set_reference_image(mR)
        c.set_velocity(v)
        _, b = c.solve_adjoint()
    finally:
        c.close()
    lam0 = mR - np.roll(mT, nt, axis=0)
    hd, ht = float(np.prod([synth.TWO_PI / n for n in shape])), 1.0 / nt
    for a in range(3):
        want = np.zeros(shape)
        for j in range(nt + 1):
            w = 0.5 * ht if j in (0, nt) else ht
            want += hd * w * np.roll(lam0, -j, axis=0) * np.roll(g[a], nt - j, axis=0)
        # foot points are off their nodes by FP32 roundings of x/2π, about 2^-24·N
        # cells, over nt steps, where the fields vary by up to their size per cell
        assert np.abs(b[a] - want).max() <= 4 * nt * 2.0 ** -24 * max(shape) * np.abs(want).max()
