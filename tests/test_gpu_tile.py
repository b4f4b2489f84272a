"""The small grids' stage kernel (one row per wavefront) against the marching
one: the same fields bit for bit."""
import os

import numpy as np
import pytest

from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0", "den1", "txy")

# one strip and less, just past one and two strips; fewer rows than a tile and
# than its halo, one row in the last tile, whole tiles
SHAPES = [(2, 4), (32, 5), (64, 11), (64, 12), (128, 33), (128, 100), (256, 47)]


@pytest.mark.parametrize("form", ["fp64", "mixed", "learned"])
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_tiles_match_marching_kernel_bitwise(product, nx, ny, form):
    """6 steps (eager, captured and replayed) with the marching kernel, short
    tiles and tall tiles."""
    print(f"{nx} x {ny} {form}", flush=True)
    net = solver.CurvatureNet(product)
    if form == "learned":
        rng = np.random.default_rng(3)
        net.set_params((0.05 * rng.uniform(-1, 1, net.num_params)).astype(np.float32))
    saved = os.environ.get("SBFS_MARCH_TILE")
    ly = ny / nx
    cases = [solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0) for _ in range(3)]
    assert product.lib.sbfs_set_precision(0 if form == "fp64" else 1) == 0
    net.use(form == "learned")
    try:
        initial_state(cases[0], 5, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.2)
        for c in cases[1:]:
            copy_state(cases[0], c)
        for _ in range(6):
            dts = []
            for c, h in zip(cases, ("0", "3", "11")):
                os.environ["SBFS_MARCH_TILE"] = h
                dts.append(c.integrate())
            assert dts[1:] == dts[:1] * 2
        for n in FIELDS:
            want = cases[0].get(n)
            for c in cases[1:]:
                assert np.array_equal(c.get(n), want), n
    finally:
        if saved is None:
            os.environ.pop("SBFS_MARCH_TILE", None)
        else:
            os.environ["SBFS_MARCH_TILE"] = saved
        net.use(False)
        assert product.lib.sbfs_set_precision(0) == 0
        for c in cases:
            c.close()
