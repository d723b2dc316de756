"""Timed one-pass products whose bitmap rows are kept: the kernel that writes
them is in the statistics, with its columns."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
ONEPASS_EMIT = 2 * 4 + 3


@pytest.mark.parametrize("nrows", [200, 400])  # 0.96 and 1.9 million columns: below and above a small tail
def test_kept_rows_are_timed(controls, nrows):
    rng = np.random.default_rng(nrows)
    ncols, inner = 5000, 40
    key = np.unique(np.repeat(np.arange(inner), 900) * ncols + rng.integers(0, ncols, inner * 900))
    B = oracle.pairs_to_dcsr((key // ncols).astype(np.uint32), (key % ncols).astype(np.uint32), inner, ncols)
    A = oracle.pairs_to_dcsr(np.repeat(np.arange(nrows), 20).astype(np.uint32),
                             np.concatenate([np.sort(rng.choice(inner, 20, replace=False))
                                             for _ in range(nrows)]).astype(np.uint32), nrows, inner)
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    got, st = cb.dcsr.spgemm(controls, a, b, mode=cb.SPGEMM_BOUND, timing=True)
    assert_dcsr_equal(controls, got, oracle.spgemm(A, B))
    assert st["launches"][ONEPASS_EMIT] == 1 and st["ms_kernel"][ONEPASS_EMIT] > 0
    # every row has 16 to 18 thousand products in a window of 157 words
    assert st["bin_out_nnz"][13] == st["nnz"] == sum(st["bin_out_nnz"])
