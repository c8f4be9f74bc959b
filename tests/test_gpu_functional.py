"""Regularization functionals on grids whose x1, x2 and x3 passes take every
radix plan, including the one whose block is no multiple of a wave (150) and the
shortest (8): against the FP64 oracle.  Each of the forward transform's values
carries a few FP32 roundings (relative 1e-6 of the field's norm at most), the
sums are FP64."""
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(8, 16, 32), (150, 48, 16), (96, 8, 150), (192, 16, 48), (16, 150, 8)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("norm", ["h1", "h1sn", "h2", "h2sn"])
def test_functional_all_radix_plans(shape, norm):
    from oracle import oracle_py

    beta = (1e-2, 1e-1, 0.0)
    print(f"\n[gpu case] functional shape={shape} norm={norm}", flush=True)
    v = synth.bandlimited_velocity(shape, kmax=2, cfl=1.0, nt=4, seed=3)
    c = Claire(shape, nt=4, regnorm=norm, beta=beta)
    try:
        got = c.reg_functional(v)
        want = oracle_py.reg_functional(v, norm, beta)
        assert abs(got - want) <= 2e-6 * abs(want)
    finally:
        c.close()
