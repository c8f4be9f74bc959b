"""Every FFT length on each axis, with small and wide blocks, blocks of rows and
columns that the grid does not fill, and x1 planes on and off 128-byte alignment:
gradient, divergence and the multiplier of the inverse regularization operator
against FP64 transforms of numpy.
FP32 roundings of a transform of N points grow like 2^-24·log2(N) of the result's
norm; forward and backward over three axes of up to 512 points that is below
2^-24·54 = 3.2e-6."""
import numpy as np
import pytest

from claire_amd import Claire

pytestmark = pytest.mark.gpu
BETA = (0.4, 0.0, 0.0)


def _k(shape, zero_nyquist=True):
    ks = []
    for a, n in enumerate(shape):
        k = (np.fft.rfftfreq(n) if a == 2 else np.fft.fftfreq(n)) * n
        k[n // 2] = 0.0 if zero_nyquist else n / 2
        ks.append(k.reshape([-1 if i == a else 1 for i in range(3)]))
    return ks


@pytest.mark.parametrize("shape", [(8, 16, 48), (48, 8, 16), (16, 48, 8), (96, 150, 32), (150, 192, 96), (192, 96, 150),
                                   (32, 64, 192), (64, 512, 64), (512, 32, 128), (512, 256, 256), (128, 128, 512), (256, 256, 256)],
                         ids=lambda s: "x".join(map(str, s)))
def test_operators(shape):
    print(f"\n[gpu case] FFT lengths {shape}", flush=True)
    v = np.random.default_rng(5).standard_normal((3,) + shape).astype(np.float32)
    c = Claire(shape, nt=4, regnorm="h1sn", beta=BETA)
    try:
        g, d, p = c.grad(v[0]), c.div(v), c.apply_inv_reg(v)
    finally:
        c.close()
    k = _k(shape)
    vh = np.fft.rfftn(v.astype(np.float64), axes=(1, 2, 3))
    back = lambda x: np.fft.irfftn(x, s=shape, axes=(0, 1, 2))
    lap = sum(x * x for x in k)
    m = 1.0 / np.where(lap == 0, BETA[0], BETA[0] * lap)
    for got, want in [(d, back(sum(1j * k[a] * vh[a] for a in range(3))))] + \
            [(g[a], back(1j * k[a] * vh[0])) for a in range(3)] + [(p[a], back(m * vh[a])) for a in range(3)]:
        assert np.linalg.norm(got - want) <= 3.2e-6 * np.linalg.norm(want)
