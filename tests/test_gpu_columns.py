"""The sequential tridiagonal solve with whole columns in LDS: the reference's
operations in the reference's order, so its result is the oracle's bit for bit."""
import ctypes as C

import numpy as np
import pytest

from harness import copy_state, initial_state, new_pair
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

# the shortest column; the edges of the sweeps' 8-row batches and of the 24-row
# loop over them; the longest column of 4, 2 and 1 modes per workgroup and the
# first past each (the last one is solved in global memory); fewer modes than a
# workgroup takes
SHAPES = [(4, 4), (8, 5), (16, 11), (16, 12), (2, 27), (32, 28), (64, 35), (8, 51), (256, 511), (16, 2528), (8, 2529),
          (16, 5088), (2, 5089), (8, 10208), (4, 10209)]


@pytest.mark.parametrize("nx,ny", SHAPES)
def test_columns_match_oracle_bitwise(oracle_mod, product, nx, ny):
    print(f"{nx} x {ny}", flush=True)
    product.lib.sbfs_set_tdm.argtypes = [C.c_int, C.c_int]
    oracle_mod.set_poisson(dct=oracle_mod.DCT_FFT, tdm=oracle_mod.TDM_SEQUENTIAL)
    o, g = new_pair(oracle_mod, product, nx, ny, lx=1.0, ly=ny / nx)
    try:
        initial_state(o, 3, velocity=0.1, ly=ny / nx, cy=0.5 * ny / nx, r=0.2)
        o.compute_density(0)
        o.compute_density(1)
        copy_state(o, g)
        assert product.lib.sbfs_set_tdm(0, 32) == 0
        for c in (o, g):
            c.compute_potential(3e-4, 5e-4)
        assert np.array_equal(g.get("psi1"), o.get("psi1"))
    finally:
        assert product.lib.sbfs_set_tdm(1, 32) == 0
        o.close()
        g.close()


def test_ensemble_of_odd_columns_matches_cases_alone(product):
    """Odd columns (solved in LDS), whole chunks and both lengths past the LDS
    in one ensemble: each member's fields and dt after 5 steps (eager, captured
    and replayed) are those of the case stepped alone, bit for bit."""
    shapes = [(32, 23), (64, 127), (32, 64), (8, 2529), (4, 10209), (2, 5089)]
    specs = [dict(nx=nx, ny=ny, lx=1.0, ly=ny / nx, Re=35.0, Fr=1.0, denr=1e-2, visr=1e-2, We=10.0) for nx, ny in shapes]
    e = solver.Ensemble(product, specs)
    alone = [solver.Case(product, s["nx"], s["ny"], 1.0, s["ly"], 35.0, 1.0, 1e-2, 1e-2, 10.0) for s in specs]
    try:
        for k, (m, c) in enumerate(zip(e.cases, alone)):
            initial_state(c, k, velocity=0.05, ly=specs[k]["ly"], cy=0.5 * specs[k]["ly"], r=0.2)
            copy_state(c, m)
        for _ in range(5):
            dts = e.step()
            assert [c.integrate() for c in alone] == list(dts)
        for k, (m, c) in enumerate(zip(e.cases, alone)):
            for n in ("vof", "ux", "uy", "p", "psi0"):
                assert np.array_equal(m.get(n), c.get(n)), (shapes[k], n)
    finally:
        e.close()
        for c in alone:
            c.close()
