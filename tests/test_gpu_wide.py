"""The mixed marching kernels' 64-bit row addresses (fields of 4 GiB or more)
against the 32-bit ones: the same fields bit for bit."""
import os

import numpy as np
import pytest

from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0", "den1", "txy")


@pytest.mark.parametrize("nx,ny", [(64, 12), (128, 100), (512, 33)])
def test_wide_rows_match_bitwise(product, nx, ny):
    """5 steps (eager, captured and replayed) on one strip, two and several."""
    print(f"{nx} x {ny}", flush=True)
    names = ("SBFS_MARCH_TILE", "SBFS_MARCH_WIDE")
    saved = {k: os.environ.get(k) for k in names}
    ly = ny / nx
    cases = [solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0) for _ in range(2)]
    assert product.lib.sbfs_set_precision(1) == 0
    try:
        os.environ["SBFS_MARCH_TILE"] = "0"
        initial_state(cases[0], 5, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.2 * min(1.0, ly))
        copy_state(cases[0], cases[1])
        for _ in range(5):
            dts = []
            for c, wide in zip(cases, ("0", "1")):
                os.environ["SBFS_MARCH_WIDE"] = wide
                dts.append(c.integrate())
            assert dts[0] == dts[1]
        for n in FIELDS:
            assert np.array_equal(cases[0].get(n), cases[1].get(n)), n
    finally:
        for k, v in saved.items():
            os.environ.pop(k, None) if v is None else os.environ.__setitem__(k, v)
        assert product.lib.sbfs_set_precision(0) == 0
        for c in cases:
            c.close()
