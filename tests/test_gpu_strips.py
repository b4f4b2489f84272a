"""The FP64 marching kernel's two bodies (strips that touch a wall and strips
that do not) against the staged path: the same fields bit for bit."""
import os

import numpy as np
import pytest

from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0", "den1", "txy")

# strips of 58 columns: none away from a wall, exactly one, three, several
# and a ragged last one; a bubble wider than a strip lies over both bodies
SHAPES = [(64, 40), (128, 33), (256, 96), (512, 21)]


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_inner_and_wall_strips_match_staged_bitwise(product, nx, ny):
    """5 steps: eager, captured and replayed."""
    print(f"{nx} x {ny}", flush=True)
    saved = os.environ.get("SBFS_MARCH_TILE")
    ly = ny / nx
    cases = [solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0) for _ in range(2)]
    try:
        os.environ["SBFS_MARCH_TILE"] = "0"
        initial_state(cases[0], 7, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.3 * min(1.0, ly))
        copy_state(cases[0], cases[1])
        for _ in range(5):
            dts = []
            for c, staged in zip(cases, (0, 1)):
                assert product.lib.sbfs_set_path(staged) == 0
                dts.append(c.integrate())
            assert dts[0] == dts[1]
        for n in FIELDS:
            assert np.array_equal(cases[0].get(n), cases[1].get(n)), n
    finally:
        assert product.lib.sbfs_set_path(1) == 0
        if saved is None:
            os.environ.pop("SBFS_MARCH_TILE", None)
        else:
            os.environ["SBFS_MARCH_TILE"] = saved
        for c in cases:
            c.close()
