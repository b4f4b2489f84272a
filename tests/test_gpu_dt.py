"""decide_dt's one-launch reduction at the edges of its grid."""
import numpy as np
import pytest

from simplebubblyflowsolver_amd import abi, solver

pytestmark = pytest.mark.gpu


# one workgroup and less; a row, a column past one; 4-row and (over 2048
# workgroups) 16-row batches with a ragged end; several thousand partial minima
@pytest.mark.parametrize("nx,ny", [(2, 4), (64, 5), (256, 17), (257, 16), (1000, 2050), (4096, 601), (513, 4097)])
def test_dt_is_the_smallest_advective_limit(product, nx, ny):
    """dt = 0.2 min h / (|u| + 1e-8) over the interior faces, bit for bit, where
    the other limits are out of reach; twice in a row (the counter returns to
    0), with the smallest in the last row, then in the first column."""
    print(f"{nx} x {ny}", flush=True)
    c = solver.Case(product, nx, ny, 1.0, ny / nx, 1e12, 1.0, 1.0, 1.0, 1e12)
    try:
        rng = np.random.default_rng(nx + ny)
        for fast in ((ny - 1, nx - 1), (0, 0)):
            ux, uy = rng.uniform(-1, 1, c.shape("ux")), rng.uniform(-1, 1, c.shape("uy"))
            abi.interior("uy", uy, nx, ny)[fast] = -3.0
            c.set("ux", ux)
            c.set("uy", uy)
            hx = c.metric("hxxf")[1:nx]
            lim = [1.0, (c.domain.hy / (np.abs(abi.interior("uy", uy, nx, ny)) + 1e-8)).min()]
            if nx > 1:
                lim.append((hx / (np.abs(ux[1:ny + 1, 1:nx]) + 1e-8)).min())
            want = np.float64(min(lim)) * np.float64(0.2)
            assert c.decide_dt() == want
    finally:
        c.close()
