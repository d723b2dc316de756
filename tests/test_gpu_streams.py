"""Products about the amount of work up to which a pass runs on one stream
(products and four per A nonzero): rows of every class, one class only, and
row blocks.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
WORK, LEN = 3 << 19, 12  # every B row has 12 columns: 16 of work per A nonzero


def _dcsr(rows, cols, nrows, ncols):
    key = np.unique((rows.astype(np.uint64) << np.uint64(32)) | cols.astype(np.uint64))
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), nrows, ncols)


@pytest.mark.parametrize("nnz", [WORK // 16 - 1, WORK // 16, WORK // 16 + 1])
@pytest.mark.parametrize("kind", ["mixed", "tiny", "bitmap"])
def test_one_stream(controls, nnz, kind):
    rng = np.random.default_rng(nnz)
    inner, ncols = 4000, 5000
    B = _dcsr(np.repeat(np.arange(inner), LEN), (rng.integers(0, ncols, inner)[:, None] +
                                                 np.arange(LEN) * 7).ravel() % ncols, inner, ncols)
    lens = {"tiny": [5], "bitmap": [1500], "mixed": [1, 3, 8, 20, 60, 150, 400, 1500]}[kind]
    n, r = 0, []
    while n < nnz:
        r.append(min(int(rng.choice(lens)), nnz - n))
        n += r[-1]
    A = _dcsr(np.repeat(np.arange(len(r)), r), np.concatenate([rng.choice(inner, k, replace=False) for k in r]),
              len(r), inner)
    assert A.nnz == nnz and B.nnz == LEN * inner
    ref = oracle.spgemm(A, B)
    a, b = upload(controls, A, len(r), inner), upload(controls, B, inner, ncols)
    for mode, name in ((cb.SPGEMM_PLAIN, "plain"), (cb.SPGEMM_BOUND, "bound")):
        got, _ = cb.dcsr.spgemm(controls, a, b, mode=mode)
        assert_dcsr_equal(controls, got, ref, name)
        cols = []
        plan = cb.dcsr.plan(controls, a, b, mode=mode, block_bound=ref.nnz // 3 + ncols)
        plan.run_all(lambda k, c, st: cols.append(c.to_host(controls)[2]))
        plan.close()
        assert np.array_equal(np.concatenate(cols), ref.cols), name
