"""Rows about the length at which the sorting product changes from one merge round to
radix passes (128 products), over widths of one, two and three passes."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncols", [200, 256, 257, 65536, 3000000])
def test_short_rows_sorted(controls, ncols):
    """Rows of 65 to 200 products, with all, some and none of them alike."""
    rng = np.random.default_rng(ncols)
    inner, length = 400, 13
    start = rng.integers(0, ncols - length, inner)
    start[:60] = start[0]
    c = start[:, None] + np.sort(np.argsort(rng.random((inner, length)), axis=1), axis=1)
    c[::3, -1] = ncols - 1
    key = np.unique(np.arange(inner)[:, None] * ncols + c)
    B = oracle.pairs_to_dcsr((key // ncols).astype(np.uint32), (key % ncols).astype(np.uint32), inner, ncols)
    lens = np.concatenate([np.arange(5, 17), [9, 10, 10, 10]]).repeat(8)
    pick = [rng.choice(60 if k % 3 == 0 else inner, n, replace=False) for k, n in enumerate(lens)]
    A = oracle.pairs_to_dcsr(np.repeat(np.arange(lens.size), lens).astype(np.uint32),
                             np.concatenate([np.sort(p) for p in pick]).astype(np.uint32), lens.size, inner)
    a, b = upload(controls, A, lens.size, inner), upload(controls, B, inner, ncols)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication(controls, a, b), oracle.spgemm(A, B))
