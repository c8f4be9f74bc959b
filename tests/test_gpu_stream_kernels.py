"""The streaming kernels of the Hessian matvec on grids below and above the size from
which they take two runs per wave, for time steps that do not divide into groups: a
matvec of several nt against the FP32 oracle, to the bound that the matvec's parity
tests use."""
import numpy as np
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu
BETA = (1e-2, 0.0, 0.0)


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle_py

    return oracle_py


@pytest.mark.parametrize("nt", [1, 3, 5, 6])
@pytest.mark.parametrize("shape", [(16, 8, 48), (64, 64, 128)], ids=["small", "large"])
def test_matvec(shape, nt, oracle):
    print(f"\n[gpu case] streaming kernels {shape} nt={nt}", flush=True)
    v = synth.bandlimited_velocity(shape, kmax=2, cfl=1.0, nt=nt, seed=1)
    vt = synth.bandlimited_velocity(shape, kmax=2, cfl=1.0, nt=nt, seed=2)
    m = synth.gaussian_blobs(shape, count=6, seed=3)
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=BETA)
    try:
        c.set_template_image(m)
        c.set_velocity(v)
        c.solve_state()
        got = c.hessian_matvec(vt)
    finally:
        c.close()
    series = oracle.solve_state(v, m, nt)
    want = oracle.hessian_matvec(v, series, vt, nt, "h1sn", BETA)
    f32 = oracle.hessian_matvec(v, oracle.solve_state(v, m, nt, prec="f32"), vt, nt, "h1sn", BETA, prec="f32")
    err = lambda x: np.linalg.norm(x - want) / np.linalg.norm(want)
    assert err(got) <= 2 * err(f32) + 1e-6
