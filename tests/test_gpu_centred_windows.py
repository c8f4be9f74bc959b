"""Gathers through windows centred per block: which points lie in a window depends on
the block's planes, so every chunk length, the raw points and the trajectory must
agree bit for bit; and points outside the window, by groups and one by one, at the
most a block can have of them."""
import numpy as np
import pytest

from claire_amd import STATE, Claire, synth

pytestmark = pytest.mark.gpu
SHAPE, NT = (64, 128, 128), 4  # 2^20 points: raw points take the staged kernel


def _grid():
    return np.stack(np.meshgrid(*[np.arange(n, dtype=np.float64) for n in SHAPE], indexing="ij"), -1)


def _velocity(u):
    """Velocity whose points move by -u cells in a time step."""
    h = np.array([2.0 * np.pi / n for n in SHAPE]).reshape(3, 1, 1, 1)
    return (np.moveaxis(np.broadcast_to(u, SHAPE + (3,)), -1, 0) * h * NT).astype(np.float32)


def _smooth(cells):
    i = _grid()
    return np.stack([cells * np.sin(2 * np.pi * (a + 1) * i[..., (a + 1) % 3] / SHAPE[(a + 1) % 3] + a)
                     for a in range(3)], -1)


def _outside(kind):
    """Points far from their block's others, none of them on the planes that a block
    of 64 or 32 planes samples (a quarter and three quarters of the way)."""
    rng = np.random.default_rng(3)
    x1, x2, x3 = np.meshgrid(*[np.arange(n) for n in SHAPE], indexing="ij")
    if kind == "groups":  # whole waves of two rows
        out = (x2 // 2) % 2 == 0
    elif kind == "points":  # 31 of a wave's 64: as many as are listed one by one
        out = (x3 % 32 < 16) & ~((x2 % 2 == 0) & (x3 % 32 == 0))
    else:
        out = rng.random(SHAPE) < 0.4
    return out & ~np.isin(x1 % 32, (8, 24, 16))


@pytest.mark.parametrize("cells", [3.4, 7.0], ids=["bound-4", "bound-8"])
@pytest.mark.parametrize("fields", [1, 3])
def test_bitwise_over_chunk_lengths(fields, cells, monkeypatch):
    print(f"\n[gpu case] centred windows, {fields} fields, {cells} cells", flush=True)
    v = _velocity(_smooth(cells))
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    c = Claire(SHAPE, nt=NT)
    try:
        def along():
            return c.interp_scalar(f, STATE) if fields == 1 else c.interp_vector(v, STATE)

        monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", "32")
        c.set_velocity(v)
        X, want = c.trajectory(STATE), along()
        src = [f] if fields == 1 else list(v)
        for chunk in (1, 7, 32, 64, 0):
            monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", str(chunk))
            assert np.array_equal(along(), want), chunk
            for s, w in zip(src, [want] if fields == 1 else list(want)):
                assert np.array_equal(c.interp_points(s, X), w), chunk
        for chunk in (1, 64):  # and the foot points themselves
            monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", str(chunk))
            c.set_velocity(v)
            assert np.array_equal(c.trajectory(STATE), X), chunk
    finally:
        c.close()


@pytest.mark.parametrize("kind", ["groups", "points", "mixed"])
@pytest.mark.parametrize("raw", [True, False], ids=["raw-points", "trajectory"])
def test_points_outside_the_window(raw, kind, oracle, monkeypatch):
    print(f"\n[gpu case] outside the window: {kind} raw={raw}", flush=True)
    monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", "32" if raw else "64")
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    out = _outside(kind)
    u = np.where(out[..., None], np.array([9.3, -13.4, 17.2]), 0.0)
    c = Claire(SHAPE, nt=NT)
    try:
        if raw:
            X = ((_grid() - u) / np.array(SHAPE)).astype(np.float32)
            got = c.interp_points(f, X)
        else:
            c.set_velocity(_velocity(u))
            X = c.trajectory(STATE)
            got = c.interp_scalar(f, STATE)
    finally:
        c.close()
    assert np.abs(got - oracle.interp(f, X, prec="f32")).max() <= 2e-6 * np.abs(f).max()


def test_points_at_infinity(oracle):
    print("\n[gpu case] points at infinity", flush=True)
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    X = ((_grid() - _smooth(3.0)) / np.array(SHAPE)).astype(np.float32)
    bad = np.zeros(SHAPE, dtype=bool)
    for k, (at, axis) in enumerate([((3, 5, 7), 1), ((40, 100, 127), 0), ((63, 0, 0), 2), ((0, 64, 33), 0)]):
        bad[at] = True
        X[at + (axis,)] = np.inf if k % 2 else -np.inf
    c = Claire(SHAPE, nt=NT)
    try:
        got = c.interp_points(f, X)
    finally:
        c.close()
    assert not np.isfinite(got[bad]).any()
    X[bad] = 0.25
    want = oracle.interp(f, X, prec="f32")
    assert np.abs(got - want)[~bad].max() <= 2e-6 * np.abs(f).max()


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("cells", [2.8, 3.9, 8.0])
def test_displacements_of_noise(cells, order, oracle):
    """Points too far apart for centred windows take the kernels without them, which
    round as the others do."""
    print(f"\n[gpu case] noise of {cells} cells, rk{order}", flush=True)
    rng = np.random.default_rng(5)
    v = _velocity((rng.random(SHAPE + (3,)) - 0.5) * 2 * cells)
    f = synth.gaussian_blobs(SHAPE, count=12, seed=1)
    c = Claire(SHAPE, nt=NT, rk_order=order)
    try:
        c.set_velocity(v)
        X = c.trajectory(STATE)
        got = c.interp_scalar(f, STATE), c.interp_vector(v, STATE)
        points = c.interp_points(f, X)
    finally:
        c.close()
    # 12 roundings a side of sums that are at most 1.25^3 of the largest value
    assert np.abs(got[0] - oracle.interp(f, X, prec="f32")).max() <= 4e-6 * np.abs(f).max()
    assert np.array_equal(points, got[0])
    for a in range(3):
        assert np.abs(got[1][a] - oracle.interp(v[a], X, prec="f32")).max() <= 4e-6 * np.abs(v).max()


@pytest.mark.parametrize("cells", [3.5, 6.0])
def test_bits_do_not_depend_on_the_kernel(cells):
    """Few points (fixed windows or the direct kernel) against three fields at once
    (centred windows) and raw points (direct kernel)."""
    print(f"\n[gpu case] kernels agree at {cells} cells", flush=True)
    shape = (48, 64, 64)
    f = synth.gaussian_blobs(shape, count=12, seed=1) + 1.0
    c = Claire(shape, nt=NT)
    try:
        v = synth.bandlimited_velocity(shape, kmax=3, cfl=1.0, nt=NT, seed=2)
        h = np.array([2.0 * np.pi / n for n in shape], np.float32).reshape(3, 1, 1, 1)
        c.set_velocity(v * np.float32(cells * NT) / np.abs(v / h).max())
        want = c.interp_points(f, c.trajectory(STATE))
        assert np.array_equal(c.interp_scalar(f, STATE), want)
        for got in c.interp_vector(np.stack([f, f, f]), STATE):
            assert np.array_equal(got, want)
    finally:
        c.close()
