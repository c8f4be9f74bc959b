"""The state series keeps the template as its first field: it stays there over solves
of new velocities (zero and not), and a new template replaces it."""
import numpy as np
import pytest

from claire_amd import Claire, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pde,solver", [("transport", "sl"), ("transport", "rk2"), ("continuity", "sl")])
def test_first_field_of_the_state(pde, solver):
    shape, nt = (16, 24 * 2, 32), 3
    print(f"\n[gpu case] template in the state {pde} {solver}", flush=True)
    v = synth.bandlimited_velocity(shape, kmax=2, cfl=0.5, nt=nt, seed=1)
    images = [synth.gaussian_blobs(shape, count=4, seed=s) for s in (2, 3)]
    c = Claire(shape, nt=nt, regnorm="h1sn", beta=(1e-2, 0.0, 0.0))
    try:
        c.set_pde_type(pde)
        c.set_pde_solver(solver)
        first = []
        for image in images + images[:1]:
            c.set_template_image(image)
            for w in (v, np.zeros_like(v), v):
                c.set_velocity(w)
                m = c.solve_state()
                assert (m[0] == image).all()
                assert (m[nt] == image).all() == (not w.any())
            first.append(m)
    finally:
        c.close()
    assert (first[0] == first[2]).all() and (first[0] != first[1]).any()
