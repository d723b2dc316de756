"""One-pass products of many short rows (their compaction takes 64 rows to a
wave from 65536 rows on): row sizes about a wave and about a workgroup's rows,
empty rows between, the last wave short, bitmap rows beside them, and rows that
are run again because the predictor sized them too small.  Whole numbers:
equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _dcsr(rows, cols, nrows, ncols):
    key = np.unique((rows.astype(np.uint64) << np.uint64(32)) | cols.astype(np.uint64))
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), nrows, ncols)


@pytest.mark.parametrize("nrows", [65535, 65536, 65537, 65600, 70001])
@pytest.mark.parametrize("mode", [cb.SPGEMM_BOUND, cb.SPGEMM_LEARNED])
def test_short_rows(controls, nrows, mode):
    rng = np.random.default_rng(nrows)
    sizes = np.array([1, 2, 3, 30, 62, 63, 64, 65, 127, 700, 2047, 2048, 2049, 5000])
    inner, ncols = 200, 6000
    lens = np.concatenate([sizes, rng.choice([1, 2, 5], inner - sizes.size)])
    B = _dcsr(np.repeat(np.arange(inner), lens),
              np.concatenate([rng.choice(ncols, n, replace=False) for n in lens]), inner, ncols)
    # columns of A from 200 on have no B row: some rows stay empty
    a_rows = np.concatenate([np.arange(nrows), rng.integers(0, nrows, nrows // 2), np.arange(100)])
    a_cols = np.concatenate([rng.integers(sizes.size, inner + 60, nrows),
                             rng.integers(sizes.size, inner + 60, nrows // 2), np.arange(100) % sizes.size])
    A = _dcsr(a_rows, a_cols, nrows, inner + 60)
    B = oracle.pairs_to_dcsr(np.repeat(B.rows, np.diff(B.rpt)).astype(np.uint32), B.cols, inner + 60, ncols)
    ref = oracle.spgemm(A, B)
    assert ref.nnz < 64 * nrows
    if mode == cb.SPGEMM_LEARNED:
        cb.predictor_reset(controls, seed=5)
        m = _dcsr(np.arange(3000) // 3, rng.integers(0, 1000, 3000), 1000, 1000)
        t = upload(controls, m, 1000, 1000)
        cb.predictor_harvest(controls, t, t)
        cb.predictor_train(controls, epochs=2, batch=256, lr=1e-3, seed=1)
    a, b = upload(controls, A, nrows, inner + 60), upload(controls, B, inner + 60, ncols)
    got, st = cb.dcsr.spgemm(controls, a, b, mode=mode)
    assert_dcsr_equal(controls, got, ref, "one pass")
