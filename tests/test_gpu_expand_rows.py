"""Row ids of the nonzeros, by rows and by tiles: rows about the length a wave takes
and its multiples, stored rows without entries, and the number of rows at which
the route changes."""
import numpy as np
import pytest

import clbool_amd as cb

pytestmark = pytest.mark.gpu
LONG = 4096
EDGE = (1 << 16) + (1 << 16) // 64  # rows of one nonzero up to which they go by rows


@pytest.mark.parametrize("lens", [
    [1], [LONG - 1], [LONG], [LONG + 1], [2 * LONG], [2 * LONG + 1],
    [LONG, 1, 0, 0, 2 * LONG + 1, LONG - 1], [0, 0, 5000, 0], [3 * LONG + 1, 3, 3], [5, 20 * LONG, 5, 0],
    [7] * 600 + [9 * LONG + 17] + [0] * 300 + [7] * 600, [1] * (EDGE - 8), [1] * (EDGE + 100),
    [0] * 70000 + [LONG + 2], [300000] + [2] * 70000,
], ids=lambda v: f"{len(v)}rows{sum(v)}")
def test_row_ids(controls, lens):
    lens = np.array(lens)
    rows = (np.arange(lens.size) * 3 + 1).astype(np.uint32)
    rpt = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    cols = np.concatenate([np.arange(n) for n in lens[lens > 0]]).astype(np.uint32)
    nrows, ncols = int(rows[-1]) + 1, int(lens.max()) + 1
    a = cb.matrix_dcsr_from_cpu(controls, rpt, rows, cols, nrows, ncols)
    want = np.repeat(rows, lens)
    for to_coo in (cb.dcsr_to_coo_shallow, cb.dcsr_to_coo_deep):
        r, c = to_coo(controls, a).to_host(controls)
        assert np.array_equal(r, want) and np.array_equal(c, cols)
    trpt, trows, tcols = cb.dcsr.transpose(controls, a).to_host(controls)
    order = np.lexsort((want, cols))
    assert np.array_equal(tcols, want[order]) and np.array_equal(np.repeat(trows, np.diff(trpt.astype(np.int64))),
                                                                cols[order])
