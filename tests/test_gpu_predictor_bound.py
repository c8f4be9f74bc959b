"""The displacement bound of the Euler predictor, which one kernel finds, against
the predictor's plan, which another writes: a point a rounding away from a cell
boundary must be on the same side for both.  Every plane below holds a velocity
whose adjoint predictor lies there, two cells away; a bound that is one cell short
makes the staged gather read a neighbouring plane (an error of 1e-2)."""
import numpy as np
import pytest

from claire_amd import ADJOINT, STATE, Claire

pytestmark = pytest.mark.gpu


def _cells(t, n):
    """First stencil node relative to the point, of points t (float32, in x)."""
    q = (t.astype(np.float64) / (2.0 * np.pi)).astype(np.float32)
    q = np.where(q <= -np.float32(1.0 / n), q + np.float32(1), q)
    q = np.where(q >= 1, q - np.float32(1), q)
    u = (q.astype(np.float64) * n + 3.0).astype(np.float32)
    return (np.floor(u).astype(int) - 4 - np.arange(n) + n // 2) % n - n // 2


def _boundary_velocities(n, nt):
    """Per index the velocity whose predictor x + v/nt is a cell further when the
    sum is rounded once than when the product and the sum are (0: none)."""
    h = np.float32(2.0 * np.pi / n)
    i = np.arange(n, dtype=np.float32)
    out = np.zeros(n, dtype=np.float32)
    v = np.float32(-2.0 * float(h) * nt)
    for _ in range(16):
        v = np.nextafter(v, np.float32(0), dtype=np.float32)
    for _ in range(32):
        s = np.float32(v / np.float32(nt))
        once = (h.astype(np.float64) * i + np.float64(s)).astype(np.float32)
        twice = (h * i).astype(np.float32) + s
        out = np.where((_cells(once, n) == -4) & (_cells(twice, n) == -3), v, out)
        v = np.nextafter(v, np.float32(-np.inf), dtype=np.float32)
    return out


@pytest.mark.parametrize("shape", [(16, 16, 16), (128, 64, 64)], ids=["one-value-layout", "pair-layout"])
def test_predictor_on_a_cell_boundary(shape, oracle, monkeypatch):
    print(f"\n[gpu case] predictor bound {shape}", flush=True)
    monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", "1")  # every plane opens a block
    nt = 2
    rng = np.random.default_rng(4)
    h = np.array([2.0 * np.pi / n for n in shape], dtype=np.float32).reshape(3, 1, 1, 1)
    v = (rng.random((3,) + shape) - 0.5).astype(np.float32) * h * nt
    at = _boundary_velocities(shape[0], nt)
    assert (at != 0).sum() >= 2
    v[0, at != 0] = at[at != 0][:, None, None]
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=(1e-2, 0.0, 0.0))
    try:
        c.set_velocity(v)
        for flag, sigma in ((STATE, 1), (ADJOINT, -1)):
            X = c.trajectory(flag)
            assert np.abs(X - oracle.trajectory(v, nt, sigma, prec="f32")).max() < 1e-6
    finally:
        c.close()
