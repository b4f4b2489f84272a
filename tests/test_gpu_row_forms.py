"""The row transforms' two forms (4 and 16 points per lane) against the
oracle: the same bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (columns, rows): the lengths that the short form starts and ends with and
# those between that change its rows per wavefront or its wavefronts per row,
# with a ragged last unit, and both sides of its row limit at 2048 columns
SHAPES = [(4, 3), (8, 65), (32, 17), (64, 9), (256, 3), (512, 2), (1024, 3), (2048, 1024), (2048, 1025)]


@pytest.mark.parametrize("n,rows", SHAPES)
def test_row_forms_match_oracle_bitwise(oracle_mod, product, n, rows):
    print(f"{rows} rows of {n}", flush=True)
    x = np.random.default_rng(n + rows).normal(size=(rows, n))
    f = product.lib.sbfs_dct_rows
    f.argtypes = [C.c_int, C.c_size_t, C.c_size_t, C.c_void_p, C.c_void_p]
    for inverse, ref in ((0, oracle_mod.dct2), (1, oracle_mod.dct3)):
        out = np.empty_like(x)
        assert f(inverse, n, rows, x.ctypes.data, out.ctypes.data) == 0
        # (the first, the last and a few rows between)
        for r in sorted({0, 1, rows // 2, rows - 2, rows - 1}):
            assert np.array_equal(out[r : r + 1], ref(x[r : r + 1].copy(), oracle_mod.DCT_FFT)), (inverse, r)
