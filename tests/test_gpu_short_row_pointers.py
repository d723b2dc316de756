"""A CSR matrix whose row pointers cover fewer entries than it has columns (the
rest is unused, as in csr addition) and what is made of it: its rows come out
as they are.  Whole numbers: equality with the oracle."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _matrix(controls, nrows, ncols, lens, unused, rng):
    cols = np.concatenate([np.sort(rng.choice(ncols, k, replace=False)) for k in lens]).astype(np.uint32)
    rpt = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    tail = rng.integers(0, ncols, unused).astype(np.uint32)
    csr = cb.csr_from_cpu(controls, rpt, np.concatenate([cols, tail]), nrows, ncols)
    row = np.repeat(np.arange(nrows, dtype=np.uint32), lens)
    return cb.csr_to_dcsr(controls, csr), oracle.pairs_to_dcsr(row, cols, nrows, ncols), row


@pytest.mark.parametrize("unused", [1, 2047, 2048, 9000])
@pytest.mark.parametrize("count", [1, 2048, 5000])
def test_rows_of_entries(controls, count, unused):
    rng = np.random.default_rng(count + unused)
    lens = np.bincount(rng.integers(0, 300, count), minlength=300)
    a, ref, row = _matrix(controls, 300, 6000, lens, unused, rng)
    assert a.nnz == count + unused
    for f in (cb.dcsr_to_coo_shallow, cb.dcsr_to_coo_deep):
        r, c = f(controls, a).to_host(controls)
        assert np.array_equal(r[:count], row) and np.array_equal(c[:count], ref.cols)


@pytest.mark.parametrize("unused", [1, 3000, 9000])
def test_product(controls, unused):
    # 800 * 60 * 400 = 19 million products: B is packed
    rng = np.random.default_rng(unused)
    inner, ncols, nrows = 150, 700, 800
    b, B, _ = _matrix(controls, inner, ncols, np.full(inner, 400), unused, rng)
    A = oracle.pairs_to_dcsr(np.repeat(np.arange(nrows, dtype=np.uint32), 60),
                             np.concatenate([np.sort(rng.choice(inner, 60, replace=False))
                                             for _ in range(nrows)]).astype(np.uint32), nrows, inner)
    a, want = upload(controls, A, nrows, inner), oracle.spgemm(A, B)
    for mode in (cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND):
        assert_dcsr_equal(controls, cb.dcsr.spgemm(controls, a, b, mode=mode)[0], want)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication(controls, a, b), want)
