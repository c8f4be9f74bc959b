"""Gather blocks of one to three planes, which small grids use to reach every
compute unit: the chunk length only splits the planes among blocks, so every
length must reproduce the launch of one block per tile bit for bit."""
import numpy as np
import pytest

from claire_amd import ADJOINT, STATE, Claire, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (32, 48, 96)], ids=["16", "32x48x96"])
@pytest.mark.parametrize("cfl", [1.5, 4.5], ids=["pair-layout", "bound-4"])
def test_short_chunks_bitwise(shape, cfl, monkeypatch):
    v = synth.bandlimited_velocity(shape, kmax=4, cfl=cfl, nt=4, seed=5)
    f = synth.gaussian_blobs(shape, count=6, seed=6)

    def outputs():
        c = Claire(shape, nt=4, regnorm="h1sn", beta=(1e-2, 1e-4, 0.0))
        try:
            c.set_velocity(v)  # the trajectory stages run in the same chunks
            return [c.interp_scalar(f, STATE), c.interp_scalar(f, ADJOINT), c.interp_vector(v, STATE)]
        finally:
            c.close()

    monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", str(shape[0]))
    want = outputs()
    for chunk in (1, 2, 3, 0):  # 0: the tuned length
        print(f"[gpu case] shape={shape} cfl={cfl} chunk={chunk}", flush=True)
        monkeypatch.setenv("CLAIRE_AMD_GATHER_CHUNK", str(chunk))
        for a, b in zip(outputs(), want):
            assert np.array_equal(a, b), (chunk, float(np.abs(a - b).max()))
