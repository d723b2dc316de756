"""Products whose kept bitmaps are limited by the memory at hand, with a little more
of it at every call: they use the block of the call before instead of new memory,
and give the same result."""
import numpy as np
import pytest

import clbool_amd as cb
from helpers import hold_memory

pytestmark = pytest.mark.gpu
GIB = 1 << 30
N, ROWS, A_LEN, INNER, B_LEN = 1 << 20, 1 << 14, 16, 64, 1 << 10


def _operands(ctl):
    """ROWS rows of A_LEN * B_LEN products over N columns: bitmaps of 128 KiB a
    row, 2 GiB in all, and a result of 1 GiB (row k of B has every INNER-th
    column, so that nothing is met twice)."""
    rng = np.random.default_rng(7)
    a_cols = (np.arange(A_LEN) * (INNER // A_LEN) + rng.integers(0, INNER // A_LEN, (ROWS, A_LEN))).astype(np.uint32)
    b_cols = (np.arange(B_LEN) * (N // B_LEN) + np.arange(INNER)[:, None]).astype(np.uint32)

    def dcsr(cols, ncols):
        n, length = cols.shape
        return cb.matrix_dcsr_from_cpu(ctl, (np.arange(n + 1) * length).astype(np.uint32),
                                       np.arange(n, dtype=np.uint32), cols.ravel(), n, ncols)
    return dcsr(a_cols, INNER), dcsr(b_cols, N)


def _planned(ctl, a, b):
    out = []
    plan = cb.dcsr.plan(ctl, a, b, mode=cb.SPGEMM_PLAIN)
    plan.run_all(lambda k, m, st: out.append((cb.dcsr.digest(ctl, m), st["bin_rows"][13])))
    plan.close()
    return out


def _called(ctl, a, b):
    m, st = cb.dcsr.spgemm(ctl, a, b, mode=cb.SPGEMM_PLAIN)
    return [(cb.dcsr.digest(ctl, m), st["bin_rows"][13])]


@pytest.mark.parametrize("call", [_called, _planned])
def test_no_new_memory(call):
    ctl = cb.create_controls()
    a, b = _operands(ctl)
    want = call(ctl, a, b)
    assert sum(kept for _, kept in want) == ROWS  # with room, all of them
    held = hold_memory(ctl, 6 * GIB)
    try:
        seen, mallocs = [], []
        for k in range(5):
            del held[-4:]  # 64 MiB more
            seen.append(call(ctl, a, b))
            mallocs.append(ctl.pool_stats()["mallocs"])
        assert all([d for d, _ in s] == [d for d, _ in want] for s in seen)
        assert all(ROWS // 2 < s[0][1] < ROWS for s in seen), seen  # some of them are kept
        assert mallocs[1:] == mallocs[1:2] * 4, mallocs
    finally:
        del held
        ctl.trim()
        ctl.close()
