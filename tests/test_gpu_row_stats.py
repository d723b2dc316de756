"""Row statistics, binning and size scans of a product at the edges of their
tiles (1024 and 2048 nonzeros, 1024 and 2048 rows): the product and its count
against the oracle for matrices whose rows end at, cross and span tiles, taken
whole and in row blocks, plain and sized by the bound; and the predictor, whose
features come from the same pass, against its network in numpy."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
N = 9000


def _matrix(lens, seed):
    rng = np.random.default_rng(seed)
    rows = np.sort(rng.choice(N, len(lens), replace=False))
    key = np.concatenate([(np.uint64(r) << np.uint64(32)) | np.sort(rng.choice(N, k, replace=False)).astype(np.uint64)
                          for r, k in zip(rows, lens)])
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), N, N)


LENS = [[1], [1023], [1024], [1025], [2048, 1], [1, 2047, 2], [700] * 3 + [5000, 1], [1] * 2049, [3] * 4097,
        [1] * 1023 + [2100] + [2] * 1024]


@pytest.mark.parametrize("lens", LENS, ids=lambda v: f"{len(v)}rows{sum(v)}")
def test_products(controls, lens):
    A, B = _matrix(lens, 1), _matrix([2, 1, 40, 3] * 700, 2)
    a, b = upload(controls, A, N, N), upload(controls, B, N, N)
    ref = oracle.spgemm(A, B)
    blen = np.zeros(N, np.int64)
    blen[B.rows] = np.diff(B.rpt.astype(np.int64))
    products = int(blen[A.cols].sum())
    for mode in (cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND):
        got, st = cb.dcsr.spgemm(controls, a, b, mode=mode)
        assert st["products"] == products
        assert_dcsr_equal(controls, got, ref, "whole")
        cols = []
        for r0 in range(0, A.nzr, max(1, A.nzr // 3)):
            got, _ = cb.dcsr.spgemm(controls, a, b, mode=mode, row_begin=r0,
                                    row_end=min(A.nzr, r0 + max(1, A.nzr // 3)))
            if got.nnz:
                cols.append(got.to_host(controls)[2])
        assert np.array_equal(np.concatenate(cols) if cols else np.zeros(0, np.uint32), ref.cols)


@pytest.mark.parametrize("lens", LENS, ids=lambda v: f"{len(v)}rows{sum(v)}")
def test_features(controls, lens):
    A, B = _matrix(lens, 3), _matrix([2, 1, 40, 3] * 700, 4)
    a, b = upload(controls, A, N, N), upload(controls, B, N, N)
    beg, end = np.zeros(N, np.int64), np.zeros(N, np.int64)
    beg[B.rows], end[B.rows] = B.rpt[:-1], B.rpt[1:]
    x = np.zeros((A.nzr, 5), np.float32)
    for i in range(A.nzr):
        k = A.cols[A.rpt[i]:A.rpt[i + 1]]
        n = k.size
        k = k[end[k] > beg[k]]
        ln = end[k] - beg[k]
        span = int(B.cols[end[k] - 1].max()) - int(B.cols[beg[k]].min()) + 1 if k.size else 0
        v = [ln.sum(), n, ln.min() if k.size else 0, ln.max() if k.size else 0, span]
        x[i] = np.log2(1.0 + np.array(v, np.float32)).astype(np.float32) / np.float32(32)
    p = np.zeros(cb.MLP_PARAMS, np.float32)
    p[:] = np.random.default_rng(5).normal(0, 0.2, cb.MLP_PARAMS)
    cb.predictor_set_params(controls, p)
    y = cb.mlp_forward(controls, p, x)
    want = np.where(x[:, 0] > 0, np.exp2(np.clip(y.astype(np.float64), 0, 1) * 32) - 1, 0)
    # one rounding of a feature (2^-24 of at most 1) moves y by less than 2^-20
    # with these weights, and y * 32 in the exponent by less than 2^-15
    assert np.allclose(cb.predictor_predict(controls, a, b), want, rtol=1e-4, atol=1e-4)
