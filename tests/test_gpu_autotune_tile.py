"""sbfs_ensemble_autotune where the stage kernel has no bands (small ensembles):
no trial runs and the band stays; with the marching kernel it times its bands."""
import os

import numpy as np
import pytest

from simplebubblyflowsolver_amd import configs, solver

pytestmark = pytest.mark.gpu


def specs_of(ws):
    return [dict(nx=w.nx, ny=w.ny, lx=w.lx, ly=w.ly, Re=w.Re, Fr=w.Fr, denr=w.denr, visr=w.visr, We=w.We)
            for w in ws]


@pytest.mark.parametrize("steps", [0, 2])
@pytest.mark.parametrize("tile", ["3", "11", None, "0"])
def test_trials_only_where_bands_matter(product, tile, steps):
    """Three small cases, freshly created and after two steps; 24 rows are not
    among the autotuner's candidates."""
    ws = configs.ensemble(3, seed=11)
    for w, (nx, ny) in zip(ws, ((32, 64), (64, 70), (128, 100))):
        w.nx, w.ny = nx, ny
    saved = os.environ.get("SBFS_MARCH_TILE")
    try:
        os.environ.pop("SBFS_MARCH_TILE", None)
        if tile is not None:
            os.environ["SBFS_MARCH_TILE"] = tile
        e = solver.Ensemble(product, specs_of(ws))
        try:
            e.set_band(24)
            for c, w in zip(e.cases, ws):
                c.load_initial_condition(w.vof())
            for _ in range(steps):
                e.step()
            before = [{n: c.get(n) for n in ("ux", "uy", "p", "psi0", "vof")} for c in e.cases]
            assert product.lib.sbfs_profile_start() == 0
            band = e.autotune()
            assert product.lib.sbfs_profile_stop() == 0
            kernels = product.lib.sbfs_profile_count()
            print(f"tile {tile}, {steps} steps: band {band}, {kernels} kernels timed", flush=True)
            if tile == "0":
                assert band in (8, 16, 32, 64, 128) and kernels > 0
            else:
                assert band == 24 and kernels == 0
            for k, c in enumerate(e.cases):
                for n, v in before[k].items():
                    assert np.array_equal(c.get(n), v), (k, n)
            for _ in range(2):
                e.step()
        finally:
            e.close()
    finally:
        os.environ.pop("SBFS_MARCH_TILE", None)
        if saved is not None:
            os.environ["SBFS_MARCH_TILE"] = saved
