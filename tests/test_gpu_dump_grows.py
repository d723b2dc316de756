"""One-pass products that dump more rows from call to call, until HIP has no room for
another block: the dump takes the largest block there is, nothing is handed back
to HIP, and results are the same."""
import numpy as np
import pytest

import clbool_amd as cb
from helpers import hold_memory

pytestmark = pytest.mark.gpu
GIB = 1 << 30
N, A_LEN, INNER, B_LEN = 1 << 20, 16, 64, 1 << 10
# rows of 128 KiB in the dump, 64 KiB in the temporary slots and 64 KiB of columns
ROWS = [6144, 8192, 10240, 12288, 14336, 16384, 17408]


def _dcsr(ctl, cols, ncols):
    n, length = cols.shape
    return cb.matrix_dcsr_from_cpu(ctl, (np.arange(n + 1) * length).astype(np.uint32), np.arange(n, dtype=np.uint32),
                                   np.ascontiguousarray(cols).ravel(), n, ncols)


def _call(ctl, a, b):
    m, st = cb.dcsr.spgemm(ctl, a, b, mode=cb.SPGEMM_BOUND, timing=True)
    return cb.dcsr.digest(ctl, m), st["dense_rows"]


def test_nothing_is_handed_back():
    ctl = cb.create_controls()
    rng = np.random.default_rng(8)
    b = _dcsr(ctl, (np.arange(B_LEN) * (N // B_LEN) + np.arange(INNER)[:, None]).astype(np.uint32), N)
    step = INNER // A_LEN
    a = [_dcsr(ctl, (np.arange(A_LEN) * step + rng.integers(0, step, (n, A_LEN))).astype(np.uint32), INNER)
         for n in ROWS]
    want = [_call(ctl, x, b) for x in a]
    assert [d for _, d in want] == ROWS  # with room, every row is dumped
    held = hold_memory(ctl, 9 * GIB)
    try:
        drops = ctl.pool_stats()["drops"]
        got = [_call(ctl, x, b) for x in a]
        assert [d for d, _ in got] == [d for d, _ in want]
        assert all(2 * d >= n for (_, d), n in zip(got, ROWS)) and got[-1][1] < ROWS[-1], got
        assert ctl.pool_stats()["drops"] == drops
    finally:
        del held
        ctl.trim()
        ctl.close()
