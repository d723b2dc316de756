"""Pairs that need no sort: one, or all of them alike."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 4097])
@pytest.mark.parametrize("r,c", [(0, 0), (5, 70000), (0, 1)])
def test_pairs_alike(controls, n, r, c):
    rows, cols = np.full(n, r, np.uint32), np.full(n, c, np.uint32)
    m = cb.matrix_coo.from_host(controls, rows, cols, r + 1, c + 1, sorted=False, noDuplicates=False)
    assert [x.tolist() for x in m.to_host(controls)] == [[r], [c]]
    m = cb.matrix_coo.from_host(controls, rows, cols, r + 1, c + 1, sorted=False, noDuplicates=True)
    assert np.array_equal(m.to_host(controls)[0], rows) and np.array_equal(m.to_host(controls)[1], cols)
    br, bc = cb.Buffer.from_array(controls, rows), cb.Buffer.from_array(controls, cols)
    cb.coo.sort_arrays(controls, br, bc, n)
    assert np.array_equal(br.read(controls, n), rows) and np.array_equal(bc.read(controls, n), cols)


@pytest.mark.parametrize("n", [1, 3000])
def test_transpose_of_one_column(controls, n):
    A = oracle.pairs_to_dcsr(np.arange(n, dtype=np.uint32) * 2, np.zeros(n, np.uint32), 2 * n, 1)
    a = upload(controls, A, 2 * n, 1)
    assert_dcsr_equal(controls, cb.dcsr.transpose(controls, a), oracle.transpose(oracle.Dcsr(A.rpt, A.rows, A.cols, 2 * n, 1)))
