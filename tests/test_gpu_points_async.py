"""Interpolation at points is queued: its first call on a grid, like any other,
returns while earlier work of the stream still runs."""
import ctypes

import numpy as np
import pytest

import claire_amd
from claire_amd import Claire, DeviceArray, synth

pytestmark = pytest.mark.gpu
NOT_READY = 600  # hipErrorNotReady


def test_first_call_does_not_wait():
    lib = claire_amd.lib()
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    shape = (96, 150, 96)  # above 2^20 points, and a grid that no other test interpolates on
    f = synth.gaussian_blobs(shape, count=6, seed=1)
    i = np.stack(np.meshgrid(*[np.arange(n) / n for n in shape], indexing="ij"), -1)
    fd, X, out = DeviceArray.from_host(f), DeviceArray.from_host(i + 0.02 * np.sin(2 * np.pi * i)), DeviceArray(shape)
    big = (256, 256, 256)
    c, busy = Claire(shape, nt=1), Claire(big, nt=1)
    g, a = DeviceArray((3,) + big), DeviceArray(big)
    vp = ctypes.c_void_p
    ev = vp()
    assert hip.hipEventCreate(ctypes.byref(ev)) == 0
    try:
        for _ in range(400):  # about 60 ms
            assert lib.clr_grad(busy.ctx, vp(a.ptr), vp(g.ptr)) == 0
        assert hip.hipEventRecord(ev, None) == 0
        assert lib.clr_interp_points(c.ctx, vp(fd.ptr), vp(X.ptr), vp(out.ptr)) == 0
        state = hip.hipEventQuery(ev)
        hip.hipGetLastError()  # "not ready" counts as an error
        c.sync()
        assert state == NOT_READY
        assert np.array_equal(out.download(), c.interp_points(f, X.download()))
    finally:
        hip.hipEventDestroy(ev)
        c.close()
        busy.close()
