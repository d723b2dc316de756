"""Plans released after their Controls was destroyed, and on another thread while
their Controls multiplies (results are whole numbers: equality)."""
import threading

import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _square(n, nnz, seed):
    key = np.unique(np.random.default_rng(seed).integers(0, n * n, nnz))
    A = oracle.pairs_to_dcsr((key // n).astype(np.uint32), (key % n).astype(np.uint32), n, n)
    return A, oracle.spgemm(A, A)


@pytest.mark.parametrize("mode", [cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND])
def test_after_the_controls(mode):
    n = 600
    A, C = _square(n, 9000, 1)
    ctl = cb.create_controls()
    a = upload(ctl, A, n, n)
    plans = [cb.dcsr.plan(ctl, a, a, mode=mode, block_bound=C.nnz // 3) for _ in range(2)]
    blocks = [blk for blk, _ in plans[0]]
    assert sum(b.nnz for b in blocks) == C.nnz
    ctl.close()
    for p in plans:
        p.close()
    other = cb.create_controls()
    assert_dcsr_equal(other, cb.dcsr.matrix_multiplication_hash(other, a, a), C)
    other.close()


def test_on_another_thread():
    n = 1500
    A, C = _square(n, 40000, 2)
    ctl = cb.create_controls()
    a = upload(ctl, A, n, n)
    for k in range(20):
        plan = cb.dcsr.plan(ctl, a, a, mode=(cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND)[k % 2], block_bound=C.nnz)
        t = threading.Thread(target=plan.close)
        t.start()
        got = cb.dcsr.matrix_multiplication_hash(ctl, a, a)
        t.join()
        assert_dcsr_equal(ctl, got, C, f"round {k}")
    ctl.close()
