"""Several cases of one process stepped in turn: each domain keeps its own
scratch, tables and captured steps."""
import numpy as np
import pytest

from harness import initial_state
from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu

FIELDS = ("vof", "ux", "uy", "p", "psi0", "den1", "txy")


def new_case(product, nx, ny, seed, Re):
    c = solver.Case(product, nx, ny, 1.0, ny / nx, Re, 1.0, 1e-2, 1e-2, 10.0)
    initial_state(c, seed, velocity=0.05, ly=ny / nx, cy=0.5 * ny / nx, r=0.2)
    return c


@pytest.mark.parametrize("form", ["fp64", "mixed", "learned"])
def test_cases_in_turn_match_cases_alone(product, form):
    """Two cases of one size and one of another advance in turn for 7 steps
    (eager, captured and replayed); after 4 one is closed and another of its
    size opened, which takes over the scratch given back.  Every case's dt history
    and fields equal those of the same case stepped alone, bit for bit."""
    net = solver.CurvatureNet(product)
    if form == "learned":
        rng = np.random.default_rng(3)
        net.set_params((0.05 * rng.uniform(-1, 1, net.num_params)).astype(np.float32))
    specs = [(64, 128, 1, 35.0), (64, 128, 2, 50.0), (32, 70, 3, 35.0), (64, 128, 4, 20.0)]
    steps = [7, 4, 7, 3]
    assert product.lib.sbfs_set_precision(0 if form == "fp64" else 1) == 0
    net.use(form == "learned")
    try:
        alone = []
        for spec, n in zip(specs, steps):
            c = new_case(product, *spec)
            alone.append(([c.integrate() for _ in range(n)], {f: c.get(f) for f in FIELDS}))
            c.close()
        cases = [new_case(product, *s) for s in specs[:3]]
        dts = [[] for _ in specs]
        done = {}
        for n in range(7):
            if n == 4:
                done[1] = {f: cases[1].get(f) for f in FIELDS}
                cases[1].close()
                cases[1] = new_case(product, *specs[3])
            for k, c in enumerate(cases):
                dts[3 if n >= 4 and k == 1 else k].append(c.integrate())
        for k, c in ((0, cases[0]), (3, cases[1]), (2, cases[2])):
            done[k] = {f: c.get(f) for f in FIELDS}
            c.close()
        for k in range(4):
            assert dts[k] == alone[k][0], k
            for f in FIELDS:
                assert np.array_equal(done[k][f], alone[k][1][f]), (k, f)
    finally:
        net.use(False)
        assert product.lib.sbfs_set_precision(0) == 0
