"""The trajectory stages take the pair-layout gather from 2^19 points on and the
one-value layout below: both must give the same foot points bit for bit, so that
the switch moves nothing.  The one-value layout is forced in a process of its
own (the switch is read once per process)."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import hashlib, json, sys
sys.path.insert(0, sys.argv[1])
from claire_amd import ADJOINT, STATE, Claire, synth
out = {}
for shape in ((96, 96, 96), (64, 96, 96), (150, 48, 128)):
    v = synth.bandlimited_velocity(shape, kmax=6, cfl=1.8, nt=4, seed=9)
    for order in (2, 4):
        c = Claire(shape, nt=4, regnorm="h1sn", beta=(1e-2, 0.0, 0.0), rk_order=order)
        c.set_velocity(v)
        out[str((shape, order))] = [hashlib.sha256(c.trajectory(f).tobytes()).hexdigest() for f in (STATE, ADJOINT)]
        c.close()
print("HASHES " + json.dumps(out))
"""


def _hashes(pair):
    env = dict(os.environ, CLAIRE_AMD_GATHER_PAIR=pair)
    r = subprocess.run([sys.executable, "-c", SCRIPT, ROOT], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    line = [x for x in r.stdout.splitlines() if x.startswith("HASHES ")][-1]
    return json.loads(line[len("HASHES "):])


def test_stages_equal_in_both_layouts():
    print("\n[gpu case] trajectory stages, pair and one-value layout", flush=True)
    a, b = _hashes("1"), _hashes("0")
    assert a and a == b
