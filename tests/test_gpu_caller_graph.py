"""Calls that a caller captures into a graph of its own.  After a forward solve the
adjoint solve and gathers along the adjoint trajectory can be captured, and a replay
at a new velocity moves along that velocity's trajectories."""
import ctypes

import numpy as np
import pytest

import claire_amd
from claire_amd import ADJOINT, STATE, Claire, DeviceArray, synth

pytestmark = pytest.mark.gpu
NT = 4


def _relerr(a, b):
    return float(np.linalg.norm((a - b).astype(np.float64)) / np.linalg.norm(b.astype(np.float64)))


class _Problem:
    def __init__(self, shape, rk_order, stream):
        self.shape = shape
        im = [synth.gaussian_blobs(shape, count=6, seed=s) for s in (3, 4)]
        self.v = [DeviceArray.from_host(synth.bandlimited_velocity(shape, kmax=4, cfl=c, nt=NT, seed=s))
                  for c, s in ((1.5, 1), (1.2, 2))]
        self.f = DeviceArray.from_host(im[0])
        self.c = Claire(shape, nt=NT, regnorm="h1sn", beta=(1e-2, 1e-4, 0.0), rk_order=rk_order, stream=stream)
        self.c.set_template_image(im[0])
        self.c.set_reference_image(im[1])

    def call(self, name, *args):
        claire_amd._check(getattr(claire_amd.lib(), name)(self.c.ctx, *args))

    def forward(self, k):
        self.call("clr_set_velocity", ctypes.c_void_p(self.v[k].ptr))
        self.call("clr_solve_state", None)


class _Graphs:
    """A stream and graphs of the HIP runtime that the library is linked to."""

    def __init__(self):
        claire_amd.lib()
        with open("/proc/self/maps") as f:
            self.hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
        self.stream = ctypes.c_void_p()
        self._ok(self.hip.hipStreamCreateWithFlags(ctypes.byref(self.stream), 1))  # non-blocking

    def _ok(self, rc):
        assert rc == 0, f"HIP error {rc}"

    def sync(self):
        self._ok(self.hip.hipStreamSynchronize(self.stream))

    def capture(self, body):
        self.sync()
        graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
        self._ok(self.hip.hipStreamBeginCapture(self.stream, 1))  # thread-local mode
        try:
            body()
        finally:
            rc = self.hip.hipStreamEndCapture(self.stream, ctypes.byref(graph))
        self._ok(rc)
        self._ok(self.hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)))
        return ex

    def replay(self, ex):
        self._ok(self.hip.hipGraphLaunch(ex, self.stream))
        self.sync()


@pytest.fixture
def graphs():
    g = _Graphs()
    yield g
    g.hip.hipGetLastError()


@pytest.mark.parametrize("rk_order", [2, 4])
@pytest.mark.parametrize("shape", [(32, 32, 32), (64, 96, 128)], ids=["small", "large"])
@pytest.mark.parametrize("what", ["gradient", "matvec"])
def test_call_after_a_forward_solve(what, shape, rk_order, graphs):
    print(f"\n[gpu case] captured {what} {shape} rk{rk_order}", flush=True)
    p = _Problem(shape, rk_order, graphs.stream.value)
    try:
        out = DeviceArray((3,) + shape)
        if what == "gradient":
            run = lambda: p.call("clr_evaluate_gradient", None, ctypes.c_void_p(out.ptr))
        else:
            run = lambda: p.call("clr_hessian_matvec", ctypes.c_void_p(out.ptr), ctypes.c_void_p(p.v[1].ptr), 1)
        p.forward(0)
        g = graphs.capture(run)
        got = []
        for _ in range(3):
            out.upload(np.zeros((3,) + shape, np.float32))
            graphs.replay(g)
            got.append(out.download())
            p.c.dot(got[-1], got[-1])
        p.forward(0)
        run()
        graphs.sync()
        eager = out.download()
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
        assert _relerr(got[0], eager) < 1e-5
    finally:
        p.c.close()


@pytest.mark.parametrize("rk_order", [2, 4])
def test_replay_at_a_new_velocity(rk_order, graphs):
    print(f"\n[gpu case] replay at a new velocity rk{rk_order}", flush=True)
    shape = (32, 32, 32)
    p, q = _Problem(shape, rk_order, graphs.stream.value), _Problem(shape, rk_order, None)
    try:
        out = DeviceArray(shape)
        along = lambda r: r.call("clr_interp_scalar", ADJOINT, ctypes.c_void_p(r.f.ptr), ctypes.c_void_p(out.ptr))
        p.forward(0)
        along(p)
        g = graphs.capture(lambda: along(p))
        for k in (1, 0, 1):
            q.forward(k)
            along(q)
            want = out.download()
            p.forward(k)
            graphs.replay(g)
            assert np.array_equal(out.download(), want)
    finally:
        p.c.close()
        q.c.close()


@pytest.mark.parametrize("rk_order", [2, 4])
@pytest.mark.parametrize("cells", [1.5, 3.5, 7.0, 25.0])
def test_foot_points_do_not_depend_on_the_kernel(cells, rk_order, graphs):
    """In a capture the direct kernels form the trajectories, else those that suit
    the displacement: fixed windows, centred ones or the direct kernels."""
    print(f"\n[gpu case] foot points of {cells} cells rk{rk_order}", flush=True)
    shape = (64, 96, 96)  # three fields have more than 2^19 points
    h = np.array([2.0 * np.pi / n for n in shape], np.float32).reshape(3, 1, 1, 1)
    v = synth.bandlimited_velocity(shape, kmax=4, cfl=1.0, nt=NT, seed=5)
    v *= np.float32(cells * NT) / np.abs(v / h).max()
    d, X = DeviceArray.from_host(v), DeviceArray(shape + (3,))
    c = Claire(shape, nt=NT, rk_order=rk_order, stream=graphs.stream.value)
    try:
        for flag in (STATE, ADJOINT):
            call = lambda: claire_amd._check(claire_amd.lib().clr_trajectory(c.ctx, flag, ctypes.c_void_p(X.ptr)))
            c.set_velocity_device(d)
            g = graphs.capture(call)
            graphs.replay(g)
            direct = X.download()
            c.set_velocity_device(d)
            call()
            graphs.sync()
            assert np.array_equal(X.download(), direct)
    finally:
        c.close()
