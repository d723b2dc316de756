"""Rows of the sorting product that are expanded and sorted in global memory
(more than 8192 products): product counts about the tiles of 4096 values,
column ranges of every number of passes, all products equal, all different,
and few or many such rows.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _dcsr(rows, cols, nrows, ncols):
    key = np.unique((rows.astype(np.uint64) << np.uint64(32)) | cols.astype(np.uint64))
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), nrows, ncols)


def _check(controls, A, B, nrows, inner, ncols):
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication(controls, a, b), oracle.spgemm(A, B), "sorted")


@pytest.mark.parametrize("products", [8192, 8193, 12287, 12288, 12289, 16385, 100001])
@pytest.mark.parametrize("ncols", [1, 2, 200, 256, 257, 65536, 65537, 1 << 24, (1 << 24) + 1, (1 << 32) - 1])
def test_long_row(controls, products, ncols):
    """One row of exactly that many products, over B rows of the widest length
    that fits, beside short ones."""
    rng = np.random.default_rng(products + ncols % 1000)
    per = int(min(ncols, 64))
    inner = products // per + 2
    full, rest = products // per, products % per
    br = [np.full(per, k) for k in range(full)] + [np.full(rest, full)]
    bc = [rng.choice(ncols, per, replace=False) if ncols < 1 << 20 else np.unique(rng.integers(0, ncols, 4 * per))[:per]
          for _ in range(full)]
    bc.append(bc[0][:rest])
    B = _dcsr(np.concatenate(br), np.concatenate(bc), inner, ncols)
    assert B.nnz == products
    ar = np.concatenate([np.full(inner, 3), np.arange(10, 40)])
    ac = np.concatenate([np.arange(inner), rng.integers(0, inner, 30)])
    _check(controls, _dcsr(ar, ac, 50, inner), B, 50, inner, ncols)


@pytest.mark.parametrize("kind", ["same", "apart", "mixed"])
@pytest.mark.parametrize("rows", [1, 1025])
def test_long_rows(controls, kind, rows):
    """Rows of 9000 products: the same 90 columns, or no column twice."""
    rng = np.random.default_rng(rows)
    inner, per = 100, 90
    ncols = {"same": 90, "apart": 9000, "mixed": 5000}[kind]
    cols = {"same": np.tile(np.arange(90), inner), "apart": rng.permutation(9000)}.get(
        kind, np.concatenate([rng.choice(ncols, per, replace=False) for _ in range(inner)]))
    B = _dcsr(np.repeat(np.arange(inner), per), cols, inner, ncols)
    ar = np.concatenate([np.repeat(np.arange(rows), inner), rows + np.arange(50)])
    ac = np.concatenate([np.tile(np.arange(inner), rows), rng.integers(0, inner, 50)])
    _check(controls, _dcsr(ar, ac, rows + 50, inner), B, rows + 50, inner, ncols)
