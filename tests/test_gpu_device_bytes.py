"""clr_device_bytes against the fields that a problem keeps, and against the memory
that the GPU has less while it lives (which says nothing below: the runtime serves
small allocations from memory that it already holds)."""
import ctypes

import numpy as np
import pytest

import claire_amd
from claire_amd import ADJOINT, STATE, Claire, DeviceArray, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(), dict(rk_order=4, precision="mixed"), dict(pde_solver="rk2", pde="continuity")],
                         ids=["default", "rk4-mixed", "rk2-continuity"])
def test_device_bytes(kw):
    print(f"\n[gpu case] device bytes {kw}", flush=True)
    shape, nt = (128, 128, 192), 4
    claire_amd.lib()
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    im = synth.gaussian_blobs(shape, count=4, seed=1)
    v = DeviceArray.from_host(synth.bandlimited_velocity(shape, kmax=3, cfl=0.4, nt=nt, seed=2))
    mT, mR = DeviceArray.from_host(im), DeviceArray.from_host(np.roll(im, 2, 0))
    out = DeviceArray((3,) + shape)
    p = lambda d: ctypes.c_void_p(d.ptr)
    lib, chk = claire_amd.lib(), claire_amd._check
    before = free()
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=(1e-2, 1e-4, 0.0), **kw)
    try:
        J = ctypes.c_double()
        chk(lib.clr_set_template_image(c.ctx, p(mT)))
        chk(lib.clr_set_reference_image(c.ctx, p(mR)))
        chk(lib.clr_evaluate_objective(c.ctx, p(v), ctypes.byref(J), None, None))
        chk(lib.clr_evaluate_gradient(c.ctx, None, p(out)))
        chk(lib.clr_hessian_matvec(c.ctx, p(out), p(v), 1))
        for flag in (STATE, ADJOINT):
            chk(lib.clr_interp_vector(c.ctx, flag, p(out), p(out)))
        held = c.device_bytes()
        used = before - free()
    finally:
        c.close()
    nl = float(np.prod(shape))
    sl = kw.get("pde_solver") != "rk2"
    # five vector fields, v~ at the foot points, reference, two adjoints, two
    # incremental states, div v, adjoint coefficient; the series of the state, its
    # gradients here and at the foot points, decrements, adjoint
    fields = 15 + 3 + 7 + (nt + 1) + 3 * (nt + 1) + 3 * nt + nt + (nt + 1)
    fields += 12 + 3 + 6 * (kw.get("rk_order") == 4)  # foot points, plans, interpolation in place, RK4 sums
    fields += 0 if sl else 1 + 6  # continuity coefficient, RK2 work
    spectra = 3 + 3 * 5  # the operators', and the gradients of all five states at once
    want = 4 * fields * nl + 8 * spectra * shape[0] * shape[1] * (shape[2] // 2 + 1)
    if kw.get("precision") == "mixed" and sl:  # 16 bits a value, 32 for each block of them
        want += (2 * nt + 1) * 3 * nl * 2
        assert 0 < held - want < 0.01 * want
    else:
        assert 0 <= held - want < 1e6  # partial sums
    assert used <= held + 100e6  # the granularity of about 40 allocations
