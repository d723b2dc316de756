"""Calls that fit the device's memory only without the scratch that saves time
(kept bitmaps, packed B, unions in batches): they give it up and succeed.
Digests against the same call with room."""
import numpy as np
import pytest

import clbool_amd as cb
from helpers import hold_memory

pytestmark = pytest.mark.gpu
MIB = 1 << 20
N, INNER, ROWS, A_LEN, B_LEN = 1 << 16, 4096, 1 << 15, 128, 16


def _operands(ctl):
    """ROWS rows of 2048 products each over N columns: bitmaps of 8 KiB a row,
    256 MiB in all, as much as the result's columns."""
    rng = np.random.default_rng(5)

    def dcsr(nrows, ncols, length):
        step = ncols // length  # one column in every stretch of step
        cols = (np.arange(length) * step + rng.integers(0, step, (nrows, length))).astype(np.uint32)
        return cb.matrix_dcsr_from_cpu(ctl, (np.arange(nrows + 1) * length).astype(np.uint32),
                                       np.arange(nrows, dtype=np.uint32), cols.ravel(), nrows, ncols)
    return dcsr(ROWS, INNER, A_LEN), dcsr(INNER, N, B_LEN)


def _product(ctl, a, b, mode):
    return [cb.dcsr.digest(ctl, cb.dcsr.spgemm(ctl, a, b, mode=mode)[0])]


def _run_all(ctl, a, b, mode):
    plan, out = cb.dcsr.plan(ctl, a, b, mode=mode), []
    plan.run_all(lambda k, m, st: out.append(cb.dcsr.digest(ctl, m)))
    plan.close()
    return out


def _run(ctl, a, b, mode):
    plan = cb.dcsr.plan(ctl, a, b, mode=mode)
    out = [cb.dcsr.digest(ctl, m) for m, _ in (plan.run(k) for k in range(plan.nblocks))]
    plan.close()
    return out


# the result takes 252 MiB and the bitmaps 256; the one pass has slots of 256 besides
CALLS = [(call, mode) for call in (_product, _run_all, _run) for mode in (cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND)]
LEAVE = {cb.SPGEMM_PLAIN: 430 * MIB, cb.SPGEMM_BOUND: 690 * MIB}


def _graph(ctl):
    """Six matrices of two million nonzeros and two small ones to multiply."""
    rng = np.random.default_rng(6)
    n = 1 << 16

    def matrix(nnz):
        k = np.unique(rng.integers(0, n * n, nnz))
        rows, cnt = np.unique(k // n, return_counts=True)
        return cb.matrix_dcsr_from_cpu(ctl, np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32),
                                       rows.astype(np.uint32), (k % n).astype(np.uint32), n, n)
    return [matrix(1 << 21) for _ in range(6)] + [matrix(30000) for _ in range(2)]


def _step(ctl, mats):
    out = list(mats)
    cb.closure_step(ctl, out, [(x, 6, 7) for x in range(6)], mode=cb.CLOSURE_BATCHED)
    return [cb.dcsr.digest(ctl, m) for m in out[:6]]


@pytest.fixture(scope="module")
def crowded():
    """Controls, operands and results with room; then all memory but 4 GiB is held."""
    ctl = cb.create_controls()
    ab, mats = _operands(ctl), _graph(ctl)
    want = {(call, mode): call(ctl, *ab, mode) for call, mode in CALLS}
    want["step"] = _step(ctl, mats)
    held = hold_memory(ctl, 4 << 30)
    yield ctl, ab, mats, want
    del held, ab, mats
    ctl.trim()
    ctl.close()


@pytest.mark.parametrize("call,mode", CALLS)
def test_product(crowded, call, mode):
    ctl, ab, _, want = crowded
    held = hold_memory(ctl, LEAVE[mode])
    got = call(ctl, *ab, mode)
    del held
    ctl.trim()
    assert got == want[call, mode]


def test_unions(crowded):
    """96 MiB of keys and the new matrices together, 16 one by one."""
    ctl, _, mats, want = crowded
    held = hold_memory(ctl, 110 * MIB)
    got = _step(ctl, mats)
    del held
    ctl.trim()
    assert got == want["step"]
