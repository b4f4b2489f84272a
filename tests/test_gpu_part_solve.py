"""The partitioned tridiagonal solve in one launch (a case alone) against the
two launches that an ensemble's members take: the same fields bit for bit."""
import ctypes as C

import numpy as np
import pytest

from harness import initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0")

# (nx, ny, longest chunk): fewer modes than a workgroup's four, three chunks and
# the four, five, eight, nine and 32 at which the modes per workgroup change or
# end, chunks of 2, 4, 8, 16 and 32 rows, and 33 chunks, past the rule
SHAPES = [(2, 6, 32), (4, 96, 32), (8, 40, 32), (32, 64, 32), (16, 128, 32), (64, 256, 32), (16, 72, 32),
          (32, 128, 4), (32, 1024, 32), (16, 1056, 32)]


@pytest.mark.parametrize("nx,ny,chunk", SHAPES)
def test_one_launch_matches_two_bitwise(product, nx, ny, chunk):
    """4 steps: eager, captured and replayed."""
    print(f"{nx} x {ny} chunk {chunk}", flush=True)
    ly = ny / nx
    spec = dict(nx=nx, ny=ny, lx=1.0, ly=ly, Re=35.0, Fr=1.0, denr=1e-2, visr=1e-2, We=10.0)
    product.lib.sbfs_set_tdm.argtypes = [C.c_int, C.c_int]
    assert product.lib.sbfs_set_tdm(1, chunk) == 0
    e = solver.Ensemble(product, [spec])
    c = solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0)
    try:
        for g in (c, e.cases[0]):
            initial_state(g, 5, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.2)
        for _ in range(4):
            assert c.integrate() == e.step()[0]
        for n in FIELDS:
            got = c.get(n)
            assert np.isfinite(got).all() and np.array_equal(got, e.cases[0].get(n)), n
    finally:
        c.close()
        e.close()
        assert product.lib.sbfs_set_tdm(1, 32) == 0
