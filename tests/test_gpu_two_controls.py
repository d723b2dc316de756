"""Two threads, each with its own Controls of one GPU, at the calls whose
temporaries are released while their kernels run: results as from one thread
alone (whole numbers: equality)."""
import threading

import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
ROUNDS = 60


def _dcsr(key, n):
    return oracle.pairs_to_dcsr((key // n).astype(np.uint32), (key % n).astype(np.uint32), n, n)


def _keys(rng, n, nnz):
    return np.unique(rng.integers(0, n * n, nnz))


def _work(seed, n, nnz, start, errors):
    try:
        ctl = cb.create_controls()
        rng = np.random.default_rng(seed)
        ka, kb = _keys(rng, n, nnz), _keys(rng, n, nnz // 3)
        A, B, union = _dcsr(ka, n), _dcsr(kb, n), _dcsr(np.union1d(ka, kb), n)
        rows = (ka // n).astype(np.uint32)
        product = oracle.spgemm(A, B)
        a, b = upload(ctl, A, n, n), upload(ctl, B, n, n)
        step = [upload(ctl, A, n, n), upload(ctl, B, n, n)]
        triples = [(0, 0, 1), (1, 1, 0)]
        cb.closure_step(ctl, step, triples, mode=cb.CLOSURE_PER_TRIPLE)
        want = [m.to_host(ctl) for m in step]
        start.wait()
        for k in range(ROUNDS):
            coo = (cb.dcsr_to_coo_shallow, cb.dcsr_to_coo_deep)[k % 2](ctl, a)
            r, c = coo.to_host(ctl)
            assert np.array_equal(r, rows) and np.array_equal(c, A.cols), f"{seed}: coo, round {k}"
            assert_dcsr_equal(ctl, cb.dcsr.addition(ctl, a, b), union, f"{seed}: union, round {k}")
            assert_dcsr_equal(ctl, cb.dcsr.matrix_multiplication_hash(ctl, a, b), product, f"{seed}: product {k}")
            assert_dcsr_equal(ctl, cb.dcsr.matrix_multiplication(ctl, a, b), product, f"{seed}: sorted {k}")
            mats = [a, b]
            cb.closure_step(ctl, mats, triples, mode=cb.CLOSURE_BATCHED)
            for m, w in zip(mats, want):
                assert all(np.array_equal(x, y) for x, y in zip(m.to_host(ctl), w)), f"{seed}: closure, round {k}"
        ctl.close()
    except BaseException as e:
        errors.append(e)
        start.abort()


def test_two_controls():
    start, errors = threading.Barrier(2), []
    ts = [threading.Thread(target=_work, args=(seed, n, nnz, start, errors))
          for seed, n, nnz in ((1, 700, 9000), (2, 2500, 60000))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
