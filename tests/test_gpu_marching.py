"""The marching stage kernel on grids that take the small grids' one by
themselves (SBFS_MARCH_TILE=0): its dispatch order, its unfolded stages and its
ensemble form, each bit for bit."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import configs, solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0", "den1", "txy")
SWITCHES = ("SBFS_MARCH_TILE", "SBFS_MARCH_ORDER", "SBFS_MARCH_BAND")


@pytest.fixture
def switches():
    saved = {k: os.environ.pop(k, None) for k in SWITCHES}
    yield os.environ
    for k, v in saved.items():
        os.environ.pop(k, None)
        if v is not None:
            os.environ[k] = v


# units of the ordered case: 9 strips x 147 bands (10 rounds of 128 dispatch
# slots and 43 units), 5 x 25 (not quite one), 2 x 64 (exactly one), 1 x 4
@pytest.mark.parametrize("mixed", [0, 1])
@pytest.mark.parametrize("nx,ny,bands", [(512, 1024, ("11", "7")), (256, 300, ("9", "12")), (64, 256, ("5", "4")),
                                         (32, 40, ("40", "13"))])
def test_dispatch_order_and_bands(product, switches, nx, ny, bands, mixed):
    """5 steps in the grid's order with one band height, and heaviest first with
    another."""
    print(f"{nx} x {ny}, bands {bands}, mixed {mixed}", flush=True)
    ly = ny / nx
    cases = [solver.Case(product, nx, ny, 1.0, ly, 35.0, 1.0, 1e-2, 1e-2, 10.0) for _ in range(2)]
    assert product.lib.sbfs_set_precision(mixed) == 0
    switches["SBFS_MARCH_TILE"] = "0"
    try:
        if nx == 512:
            cases[0].load_initial_condition(configs.bubble_swarm(nx, ny, 16, steps=5, seed=3).vof())
        else:
            initial_state(cases[0], 7, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.3 * min(1.0, ly))
        copy_state(cases[0], cases[1])
        for _ in range(5):
            dts = []
            for g, order, band in zip(cases, ("0", "1"), bands):
                switches["SBFS_MARCH_ORDER"] = order
                switches["SBFS_MARCH_BAND"] = band
                dts.append(g.integrate())
            assert dts[0] == dts[1]
        for n in FIELDS:
            assert np.array_equal(cases[0].get(n), cases[1].get(n)), n
    finally:
        assert product.lib.sbfs_set_precision(0) == 0
        for g in cases:
            g.close()


@pytest.mark.parametrize("precision,tdm,band", [(0, 1, 32), (0, 1, 7), (0, 0, 32), (1, 1, 7)])
def test_ensemble_matches_cases_alone(product, switches, precision, tdm, band):
    """Six uneven cases stepped together by the marching kernels, against each of
    them alone with the stage kernel of its size: 6 steps."""
    ws = configs.ensemble(6, seed=11)
    ws[0].nx, ws[0].ny = 32, 64
    specs = [dict(nx=w.nx, ny=w.ny, lx=w.lx, ly=w.ly, Re=w.Re, Fr=w.Fr, denr=w.denr, visr=w.visr, We=w.We)
             for w in ws]
    assert product.lib.sbfs_set_precision(precision) == 0
    assert product.lib.sbfs_set_tdm(tdm, 32) == 0
    try:
        switches["SBFS_MARCH_TILE"] = "0"
        e = solver.Ensemble(product, specs)
        try:
            e.set_band(band)
            for c, w in zip(e.cases, ws):
                c.load_initial_condition(w.vof())
            dts = np.array([e.step() for _ in range(6)])
            got = [{n: c.get(n) for n in FIELDS} for c in e.cases]
        finally:
            e.close()
        del switches["SBFS_MARCH_TILE"]
        for k, w in enumerate(ws):
            g = solver.Case(product, w.nx, w.ny, w.lx, w.ly, w.Re, w.Fr, w.denr, w.visr, w.We)
            try:
                g.load_initial_condition(w.vof())
                assert [g.integrate() for _ in range(6)] == list(dts[:, k]), k
                for n in FIELDS:
                    assert np.array_equal(got[k][n], g.get(n)), (k, n)
            finally:
                g.close()
    finally:
        product.lib.sbfs_set_precision(0)
        product.lib.sbfs_set_tdm(1, 32)


UNFOLDED = """
import os
import sys
import numpy as np
sys.path.insert(0, sys.argv[1])
sys.path.insert(0, sys.argv[1] + "/tests")
from harness import copy_state, initial_state
from simplebubblyflowsolver_amd import solver
be = solver.product_backend()
be.set_dt_coefs(0.2, 0.5, 0.95)
for nx, ny, mixed in ((64, 128, 0), (256, 96, 0), (64, 128, 1), (256, 96, 1)):
    assert be.lib.sbfs_set_precision(mixed) == 0
    ly = ny / nx
    a, b, c = (solver.Case(be, nx, ny, 1.0, ly, 35.0, 1.0, 1e-3, 1e-2, 10.0) for _ in range(3))
    initial_state(a, 7, velocity=0.05, ly=ly, cy=0.5 * ly, r=0.3 * min(1.0, ly))
    copy_state(a, b)
    copy_state(a, c)
    for _ in range(8):
        os.environ["SBFS_MARCH_TILE"] = "0"
        dta = a.integrate()
        os.environ["SBFS_MARCH_TILE"] = "3"
        assert b.integrate() == dta
        if not mixed:
            assert be.lib.sbfs_set_path(0) == 0
            assert c.integrate() == dta
            assert be.lib.sbfs_set_path(1) == 0
    for n in ("vof", "ux", "uy", "p", "psi0", "den1", "txy"):
        x = a.get(n)
        assert np.array_equal(x, b.get(n)), (nx, mixed, n)
        assert mixed or np.array_equal(x, c.get(n)), (nx, mixed, n)
    for g in (a, b, c):
        g.close()
    print(f"{nx} x {ny}, mixed {mixed}: unfolded marching and tile kernels agree", flush=True)
"""


def test_unfolded_marching_kernel():
    """With SBFS_MARCH_FOLD=0, which is read once per process, every stage of the
    marching kernel is the unfolded one: 8 steps equal to the tile kernel's and,
    in FP64, to the staged path's."""
    env = dict(os.environ, SBFS_MARCH_FOLD="0")
    root = str(Path(__file__).resolve().parents[1])
    r = subprocess.run([sys.executable, "-c", UNFOLDED, root], env=env, capture_output=True, text=True, timeout=100)
    print(r.stdout.strip())
    assert r.returncode == 0, r.stdout + r.stderr
