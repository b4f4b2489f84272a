"""A step that fails leaves nothing behind that fails the next one."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

SCRIPT = """
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
sys.path.insert(0, sys.argv[1] + "/tests")
from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import solver
be = solver.product_backend()
be.set_dt_coefs(0.2, 0.5, 0.95)
net = solver.CurvatureNet(be)
a, b = (solver.Case(be, 64, 64, 1.0, 1.0, 35.0, 1.0, 1e-2, 1e-2, 10.0) for _ in range(2))
initial_state(a, 7, velocity=0.05, ly=1.0, r=0.2)
copy_state(a, b)
net.use(True)
try:
    a.integrate()
    raise SystemExit("a step without a network succeeded")
except solver.SolverError as e:
    assert "no trained network" in str(e), e
net.set_params((0.05 * np.random.default_rng(3).uniform(-1, 1, net.num_params)).astype(np.float32))
for _ in range(5):
    assert a.integrate() == b.integrate()
for n in ("vof", "ux", "uy", "p", "psi0", "den1", "txy"):
    assert np.array_equal(a.get(n), b.get(n)), n
print("ok", flush=True)
"""


def test_step_after_a_refused_one():
    """Without a trained network the learned step is refused; with one set, the
    same case steps as another that was never refused (5 steps, bit for bit).  In
    a child process, where no network is set yet."""
    root = str(Path(__file__).resolve().parents[1])
    r = subprocess.run([sys.executable, "-c", SCRIPT, root], env=dict(os.environ), capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
