"""Gathers whose points leave the two-cell window around themselves: windows
centred per block, points outside them read from global memory, blocks of
scattered points that stage nothing, and the list of outside points running over.
Against the FP32 oracle, the two computing the same FP32 products up to the order
of a few roundings per value."""
import numpy as np
import pytest

from claire_amd import ADJOINT, STATE, Claire, synth

pytestmark = pytest.mark.gpu
SHAPE = (64, 128, 128)  # 2^20 points: raw points take the staged kernel


@pytest.fixture(scope="module")
def oracle():
    from oracle import oracle_py

    return oracle_py


def _points(kind, rng):
    i = np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in SHAPE], indexing="ij"), -1)
    n = np.asarray(SHAPE, dtype=np.float64)
    if kind == "smooth":
        u = np.stack([3.0 * np.sin(2 * np.pi * i[..., (a + 1) % 3] / n[(a + 1) % 3] + a) for a in range(3)], -1)
    elif kind == "shift":  # beyond any fixed window, and across the periodic seam
        u = np.broadcast_to([20.3, -41.7, 61.2], i.shape)
    elif kind == "scattered":
        u = (rng.random(i.shape) - 0.5) * 4 * n
    else:  # most points at home, 40% anywhere: more than a block's list holds
        u = np.where(rng.random(i.shape[:3] + (1,)) < 0.4, (rng.random(i.shape) - 0.5) * n, 0.3)
    return ((i + u) / n).astype(np.float32)


@pytest.mark.parametrize("chunk", [0, 7, 64], ids=["tuned", "chunk-7", "longest-chunk"])
@pytest.mark.parametrize("kind", ["smooth", "shift", "scattered", "mixed"])
def test_interpolation_at_points(kind, chunk, oracle, monkeypatch):
    print(f"\n[gpu case] points {kind} chunk={chunk}", flush=True)
    monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", str(chunk))
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    X = _points(kind, np.random.default_rng(2))
    c = Claire(SHAPE, nt=4)
    try:
        got = c.interp_points(f, X)
    finally:
        c.close()
    want = oracle.interp(f, X, prec="f32")
    assert np.abs(got - want).max() <= 2e-6 * np.abs(f).max()


def test_points_that_are_not_finite(oracle):
    print("\n[gpu case] points not finite", flush=True)
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    X = _points("smooth", None)
    bad = np.zeros(SHAPE, dtype=bool)
    bad[3, 5, 7] = bad[40, 100, 127] = bad[63, 0, 0] = True
    X[3, 5, 7, 1] = np.nan
    X[40, 100, 127, 0] = np.nan
    X[63, 0, 0, 2] = np.nan
    c = Claire(SHAPE, nt=4)
    try:
        got = c.interp_points(f, X)
    finally:
        c.close()
    assert np.isnan(got[bad]).all()
    X[bad] = 0.25
    want = oracle.interp(f, X, prec="f32")
    assert np.abs(got - want)[~bad].max() <= 2e-6 * np.abs(f).max()


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("cfl", [4.5, 9.0])
def test_large_displacements_along_a_trajectory(cfl, order, oracle):
    shape, nt = (96, 64, 96), 4
    print(f"\n[gpu case] trajectory cfl={cfl} order={order}", flush=True)
    v = synth.bandlimited_velocity(shape, kmax=6, cfl=cfl, nt=nt, seed=7)
    f = synth.gaussian_blobs(shape, count=12, seed=8)
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=(1e-2, 0.0, 0.0), rk_order=order)
    try:
        c.set_velocity(v)
        with oracle.rk_order(order):
            for flag, sigma in ((STATE, 1), (ADJOINT, -1)):
                X = c.trajectory(flag)
                assert np.abs(X - oracle.trajectory(v, nt, sigma, prec="f32")).max() < 1e-6
                got = c.interp_scalar(f, flag), c.interp_vector(v, flag)
                assert np.abs(got[0] - oracle.interp(f, X, prec="f32")).max() <= 2e-6 * np.abs(f).max()
                for a in range(3):
                    assert np.abs(got[1][a] - oracle.interp(v[a], X, prec="f32")).max() <= 2e-6 * np.abs(v).max()
    finally:
        c.close()
