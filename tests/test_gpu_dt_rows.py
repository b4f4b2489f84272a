"""decide_dt's reduction with more than 4 rows per workgroup: their number is 4,
doubled up to 64 while the workgroups (256 columns each) are more than 2048."""
import os

import numpy as np
import pytest

from simplebubblyflowsolver_amd import abi, solver

pytestmark = pytest.mark.gpu

# 16 rows with 3 in the last workgroup, 32 with 20, 64 with 49, 64 at the cap
# (2188 workgroups) with 33 and (67188, more than 65535 in y) with 32
SHAPES = [(257, 8195), (4096, 2100), (2, 70001), (2, 140001), (2, 4300000)]


@pytest.mark.parametrize("stream", ["0", "1"])
@pytest.mark.parametrize("nx,ny", SHAPES)
def test_dt_is_the_smallest_advective_limit(product, nx, ny, stream):
    """dt = 0.2 min h / (|u| + 1e-8) over the interior faces, bit for bit, with
    ordinary and with streaming loads, and the largest velocity in the last row,
    then in the first column, then in the row that ends a full workgroup."""
    print(f"{nx} x {ny}, stream {stream}", flush=True)
    saved = os.environ.get("SBFS_STREAM")
    os.environ["SBFS_STREAM"] = stream
    c = solver.Case(product, nx, ny, 1.0, ny / nx, 1e12, 1.0, 1.0, 1.0, 1e12)
    try:
        rng = np.random.default_rng(nx + ny)
        ux, uy = rng.uniform(-1, 1, c.shape("ux")), rng.uniform(-1, 1, c.shape("uy"))
        c.set("ux", ux)
        hx = c.metric("hxxf")[1:nx]
        limx = (hx / (np.abs(ux[1:ny + 1, 1:nx]) + 1e-8)).min()
        inner = abi.interior("uy", uy, nx, ny)
        for fast in ((ny - 1, nx - 1), (0, 0), (ny // 64 * 64 - 1, 0)):
            was, inner[fast] = inner[fast], -3.0
            c.set("uy", uy)
            want = np.float64(min(1.0, limx, (c.domain.hy / (np.abs(inner) + 1e-8)).min())) * np.float64(0.2)
            assert c.decide_dt() == want
            inner[fast] = was
    finally:
        c.close()
        if saved is None:
            os.environ.pop("SBFS_STREAM", None)
        else:
            os.environ["SBFS_STREAM"] = saved
