"""The diagnostics' sums over columns of rows against numpy on the same fields."""
import numpy as np
import pytest

from harness import initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu


# fewer rows than a thread's four, a ragged last group of rows, fewer and more
# columns than a workgroup's 256, and more rows than 1024 workgroups take by fours
@pytest.mark.parametrize("nx,ny", [(2, 4), (64, 7), (256, 33), (512, 18), (1024, 1030)])
def test_sums_match_numpy(product, nx, ny):
    print(f"{nx} x {ny}", flush=True)
    ly = ny / nx
    c = solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0)
    try:
        initial_state(c, 3, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.2)
        d = c.diagnostics()
        vof, ux, uy = c.get("vof"), c.get("ux"), c.get("uy")
        h = 1.0 / nx
        rows = vof[1 : ny + 2]  # rows 0..ny, columns 0..nx+1
        v = rows[1:, 1:-1]
        uxr, uyr = ux[1 : ny + 1], uy[1 : ny + 2, 1:-1]
        x = (np.arange(nx) + 0.5) * h
        u = 0.5 * uxr[:, :-1] + 0.5 * uxr[:, 1:]
        dv = np.abs(np.diff(rows[1:], axis=1)).sum() + np.abs(np.diff(rows[:, 1:-1], axis=0)).sum()
        div = np.abs((np.diff(uxr, axis=1) + np.diff(uyr, axis=0)) / h).max()
        # a sum of n terms in any order errs by at most n eps times the sum of
        # the terms' sizes, a quotient of two by twice that
        tol = 2 * (2 * nx * ny + 8) * np.finfo(float).eps
        assert d["vofmin"] == v.min() and d["vofmax"] == v.max()
        assert abs(d["vofmean"] - v.mean()) <= tol * v.mean()
        assert abs(d["centroid"] - (v * x).sum() / v.sum()) <= tol
        assert abs(d["rise_velocity"] - (v * u).sum() / v.sum()) <= tol * np.abs(u).max()
        assert abs(d["area"] / d["volume"] * h - dv / v.sum()) <= 2 * tol * dv / v.sum()
        assert abs(d["divmax"] - div) <= 16 * np.finfo(float).eps * 4 * max(np.abs(ux).max(), np.abs(uy).max()) / h
    finally:
        c.close()
