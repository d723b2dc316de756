"""A row block that does not fit the device's memory, after small blocks whose
tails still run: the call fails, leaves nothing in flight, and the same plan
gives the whole result once there is room."""
import numpy as np
import pytest

import clbool_amd as cb
from helpers import hold_memory

pytestmark = pytest.mark.gpu
WIDE, LONG, SMALL = 1 << 20, 64, 10  # B: LONG rows of WIDE columns, side by side, and short rows


@pytest.mark.parametrize("mode", [cb.SPGEMM_BOUND])
def test_failed_block(mode):
    ctl = cb.create_controls()
    ncols, shorts, srows = WIDE * LONG, 50, 100
    lens = np.concatenate([np.full(LONG, WIDE), np.full(shorts, SMALL)])
    bcols = np.concatenate([np.arange(ncols, dtype=np.uint32), np.tile(np.arange(SMALL) * 1000, shorts).astype(np.uint32)])
    b = cb.matrix_dcsr_from_cpu(ctl, np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32),
                                np.arange(LONG + shorts, dtype=np.uint32), bcols, LONG + shorts, ncols)
    # rows of one short B row, and a last one of all the long rows
    alen = np.concatenate([np.ones(srows, np.int64), [LONG]])
    acols = np.concatenate([LONG + np.arange(srows) % shorts, np.arange(LONG)]).astype(np.uint32)
    a = cb.matrix_dcsr_from_cpu(ctl, np.concatenate([[0], np.cumsum(alen)]).astype(np.uint32),
                                np.arange(srows + 1, dtype=np.uint32), acols, srows + 1, LONG + shorts)
    want = np.concatenate([np.tile(np.arange(SMALL) * 1000, srows), np.arange(ncols)])
    plan = cb.dcsr.plan(ctl, a, b, mode=mode, block_bound=srows * SMALL // 2)
    assert plan.nblocks == 3
    held = hold_memory(ctl, 200 << 20)  # less than the last row's slot of 256 MiB
    got = []
    with pytest.raises(cb.ClboolError, match="device allocation"):
        plan.run_all(lambda k, m, s: got.append(m.to_host(ctl)[2]))
    held.clear()
    ctl.trim()
    got.clear()
    plan.run_all(lambda k, m, s: got.append(m.to_host(ctl)[2]))
    plan.close()
    assert np.array_equal(np.concatenate(got), want)
    ctl.close()
