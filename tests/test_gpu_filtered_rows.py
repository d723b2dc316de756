"""Products whose B stores few of A's columns (under one row id in 16), where
the row kernels run over A without the nonzeros that have no B row: sizes of A
about the tiles it is filtered by, some or all of its
nonzeros left, one column window and several, each mode,
and row blocks.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _dcsr(rows, cols, nrows, ncols):
    key = np.unique((rows.astype(np.uint64) << np.uint64(32)) | cols.astype(np.uint64))
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), nrows, ncols)


def _b(rng, stored, inner, ncols, lens=(1, 3, 40, 500)):
    n = np.minimum(rng.choice(lens, stored.size), ncols)
    c = np.concatenate([rng.choice(ncols, k, replace=False) if k < ncols else np.arange(ncols) for k in n])
    return _dcsr(np.repeat(stored, n), c, inner, ncols)


def _check(controls, A, B, nrows, inner, ncols):
    ref = oracle.spgemm(A, B)
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    for mode, name in ((cb.SPGEMM_PLAIN, "plain"), (cb.SPGEMM_BOUND, "bound")):
        assert_dcsr_equal(controls, cb.dcsr.spgemm(controls, a, b, mode=mode)[0], ref, name)
        got = [np.zeros(0, np.uint32)]
        plan = cb.dcsr.plan(controls, a, b, mode=mode, block_bound=max(ncols, ref.nnz // 3 + 1))
        plan.run_all(lambda k, c, st: got.append(c.to_host(controls)[2]) if c.nnz else None)
        plan.close()
        assert np.array_equal(np.concatenate(got), ref.cols), name
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication(controls, a, b), ref, "sorted")


@pytest.mark.parametrize("nnz", [65535, 65536, 65537, 67583, 67584, 69633])
@pytest.mark.parametrize("hit", ["none", "some", "all"])
def test_filtered(controls, nnz, hit):
    """A's nonzeros: none but one row's, about a tenth or all have a B row."""
    rng = np.random.default_rng(nnz)
    nrows, inner, ncols = 3000, 90000, 1100000
    stored = np.sort(rng.choice(inner, 900, replace=False))
    other = np.setdiff1d(np.arange(inner), stored)
    r = np.arange(nnz) * nrows // nnz
    per = np.bincount(r, minlength=nrows)
    cols = []
    for i, n in enumerate(per):
        k = {"none": 0 if i != 1234 else n, "all": n}.get(hit, int(rng.binomial(n, 0.1)))
        cols.append(np.sort(np.concatenate([rng.choice(stored, k, replace=False),
                                            rng.choice(other, n - k, replace=False)])))
    A = _dcsr(r, np.concatenate(cols), nrows, inner)
    assert A.nnz == nnz
    _check(controls, A, _b(rng, stored, inner, ncols, (70, 900)), nrows, inner, ncols)


# split tables of 3 entries a row: the last id count without the filter and the
# first with it; 4 a row; and one window, which needs no table
@pytest.mark.parametrize("inner,ncols", [(87381, 1100000), (87382, 1100000), (87382, 1048576), (87382, 600000),
                                         (70000, 2200000), (90000, 400000), (90000, 1)])
@pytest.mark.parametrize("long_rows", [0, 3])
def test_filtered_windows(controls, inner, ncols, long_rows):
    """Column windows of every kind; a few A rows that span many tiles."""
    rng = np.random.default_rng(ncols + long_rows)
    nrows = 500
    stored = np.sort(rng.choice(inner, 400, replace=False))
    stored[0], stored[-1] = 0, inner - 1
    r = [np.repeat(np.arange(nrows), 160)]
    c = [rng.integers(0, inner, nrows * 160)]
    c[0][::7] = rng.choice(stored, c[0][::7].size)
    for k in range(long_rows):
        r.append(np.full(inner, 100 * k + 7))
        c.append(np.arange(inner))
    A = _dcsr(np.concatenate(r), np.concatenate(c), nrows, inner)
    _check(controls, A, _b(rng, stored, inner, ncols, (2, 70, 3000)), nrows, inner, ncols)


@pytest.mark.parametrize("ncols", [600000, 1100000])
def test_filtered_and_packed(controls, ncols):
    """2^24 products over B rows that share column groups."""
    rng = np.random.default_rng(ncols)
    nrows, inner = 700, 90000
    stored = np.sort(rng.choice(inner, 30, replace=False))
    rows = np.repeat(stored, 9000)
    cols = np.repeat(rng.integers(0, ncols - 9000, 30), 9000) + np.tile(np.arange(9000), 30)
    B = _dcsr(rows, cols, inner, ncols)
    r = np.concatenate([np.repeat(np.arange(nrows), 120), np.repeat(np.arange(nrows), 12)])
    c = np.concatenate([rng.integers(0, inner, nrows * 120), rng.choice(stored, nrows * 12)])
    _check(controls, _dcsr(r, c, nrows, inner), B, nrows, inner, ncols)
