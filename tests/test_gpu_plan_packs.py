"""A plan made while bitmap_persistent is set, which packs nothing, and run
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
