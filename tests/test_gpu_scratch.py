"""The scratch that closed domains leave behind: bounded, and none of a large
case stays once a case of another size runs."""
import numpy as np
import pytest
import torch

from simplebubblyflowsolver_amd import solver

pytestmark = pytest.mark.gpu


def free_bytes(product):
    assert product.synchronize() == 0
    return torch.cuda.mem_get_info()[0]


def step_once(product, nx, ny):
    c = solver.Case(product, nx, ny, 1.0, ny / nx, 35.0, 1.0, 1e-2, 1e-2, 10.0)
    c.load_initial_condition(np.zeros((ny, nx + 2)))
    c.integrate()
    return c


def test_a_large_case_gives_its_scratch_back(product):
    """A 2048 x 16384 case (1.6 GB of scratch) is stepped and closed; while a
    64 x 128 case is open and stepped, at most 0.3 GB more than before is taken."""
    step_once(product, 64, 128).close()
    before = free_bytes(product)
    step_once(product, 2048, 16384).close()
    c = step_once(product, 64, 128)
    try:
        held = before - free_bytes(product)
        print(f"held {held / 1e9:.2f} GB", flush=True)
        assert held < 0.3e9
    finally:
        c.close()
