"""When a plan packs B.  Short rows don't ask for it.  A plan made while bitmap_persistent is set, which packs nothing, and run
without it: its blocks pack B by themselves, over the plan's split table.
Whole numbers: equality with the oracle."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,dump,ncols", [(cb.SPGEMM_BOUND, 0, (1 << 20) - 3), (cb.SPGEMM_BOUND, 0, (1 << 21) + 5),
                                             (cb.SPGEMM_PLAIN, 65535, (1 << 21) + 5)])
def test_block_packs_b(controls, mode, dump, ncols):
    # 360 * 100 * 512 = 18.4 million products, over 2^24, 14 for each of B's 1.3 million nonzeros
    rng = np.random.default_rng(ncols)
    inner, nrows, take, runs = 2500, 360, 100, 32
    first = np.sort(rng.choice(ncols // 16, (inner, runs)), axis=1)  # runs of 16 columns; equal ones merge
    cols = (first[:, :, None] * 16 + np.arange(16)).reshape(inner, -1)
    key = np.unique(np.arange(inner)[:, None] * (1 << 32) + cols)
    B = oracle.pairs_to_dcsr((key >> 32).astype(np.uint32), (key & 0xFFFFFFFF).astype(np.uint32), inner, ncols)
    A = oracle.pairs_to_dcsr(np.repeat(np.arange(nrows), take).astype(np.uint32),
                             np.concatenate([np.sort(rng.choice(inner, take, replace=False))
                                             for _ in range(nrows)]).astype(np.uint32), nrows, inner)
    ref = oracle.spgemm(A, B)
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    old, t = controls.tuning(), controls.tuning()
    try:
        t.bitmap_persistent, t.dump_bits_per_chunk = 1, dump
        controls.set_tuning(t)
        plan = cb.dcsr.plan(controls, a, b, mode=mode)
        t.bitmap_persistent = 0
        controls.set_tuning(t)
        got = []
        plan.run_all(lambda k, m, st: got.append(m.to_host(controls)[2]))
        plan.close()
    finally:
        controls.set_tuning(old)
    assert np.array_equal(np.concatenate(got), ref.cols)


@pytest.mark.parametrize("mode", [cb.SPGEMM_PLAIN, cb.SPGEMM_BOUND])
def test_plan_of_short_rows_packs_nothing(controls, mode):
    """16.8 million products, 10 for each of B's nonzeros, none of them in a
    bitmap row: the plan holds no more than one that may not pack."""
    length, inner, nrows, ncols = 28, 60000, 600000, 1 << 16
    rng = np.random.default_rng(3)
    cols = (rng.integers(0, ncols - length, inner)[:, None] + np.arange(length)).astype(np.uint32)
    b = cb.matrix_dcsr_from_cpu(controls, (np.arange(inner + 1) * length).astype(np.uint32),
                                np.arange(inner, dtype=np.uint32), cols.ravel(), inner, ncols)
    a = cb.matrix_dcsr_from_cpu(controls, np.arange(nrows + 1, dtype=np.uint32), np.arange(nrows, dtype=np.uint32),
                                rng.integers(0, inner, nrows).astype(np.uint32), nrows, inner)

    def held(plan):  # bytes in use while the plan is there
        st = controls.pool_stats()
        return st["malloc_bytes"] - st["cached_bytes"]

    old, t = controls.tuning(), controls.tuning()
    used = {}
    try:
        for persistent in (1, 0, 1, 0):
            t.bitmap_persistent = persistent
            controls.set_tuning(t)
            base = held(None)
            plan = cb.dcsr.plan(controls, a, b, mode=mode)
            controls.sync()
            used[persistent] = held(plan) - base
            plan.close()
    finally:
        controls.set_tuning(old)
    # packed B takes 1.1 MB; blocks may be a quarter larger than asked for
    assert abs(used[0] - used[1]) < 256 << 10, used
