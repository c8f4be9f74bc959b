"""The gradients of the state series are gathered several fields per launch: a Hessian
matvec whose series goes in uneven groups (15 and 3 fields of 2^22 points) against the
oracle, to the bound of the matvec's parity tests."""
import numpy as np
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu
BETA = (1e-2, 0.0, 0.0)


@pytest.mark.parametrize("shape,nt", [((64, 256, 256), 6)], ids=["uneven-groups"])
def test_matvec(shape, nt):
    from oracle import oracle_py as oracle

    print(f"\n[gpu case] gather series {shape} nt={nt}", flush=True)
    v = synth.bandlimited_velocity(shape, kmax=3, cfl=1.5, nt=nt, seed=1)
    vt = synth.bandlimited_velocity(shape, kmax=3, cfl=1.0, nt=nt, seed=2)
    m = synth.gaussian_blobs(shape, count=6, seed=3)
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=BETA)
    try:
        c.set_template_image(m)
        c.set_velocity(v)
        series = c.solve_state()
        got = c.hessian_matvec(vt)
    finally:
        c.close()
    want = oracle.hessian_matvec(v, series, vt, nt, "h1sn", BETA)
    f32 = oracle.hessian_matvec(v, series, vt, nt, "h1sn", BETA, prec="f32")
    err = lambda x: np.linalg.norm(x - want) / np.linalg.norm(want)
    assert err(got) <= max(1e-5, 2 * err(f32))
