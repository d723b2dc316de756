"""With gather_combine set, rows with most of the products run the combining gather
like all bitmap rows: one bitmap launch a pass, where the heavy rows otherwise
have one of their own."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from clbool_amd import autotune as at
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
SYM_BITMAP = 4 * 0 + 2


@pytest.mark.parametrize("combine", [0, 1])
def test_heavy_rows(controls, combine):
    rng = np.random.default_rng(3)
    n, hubs = 40000, 3
    # the hubs hold 20000 of the rows: 2.4 million products each, the others
    # some 14 thousand
    r = np.concatenate([np.repeat(np.arange(hubs), 20000), rng.integers(hubs, n, n * 120)])
    c = np.concatenate([rng.integers(hubs, n, hubs * 20000), rng.integers(hubs, n, n * 120)])
    key = np.unique(r.astype(np.int64) * n + c)
    r, c = (key // n).astype(np.uint32), (key % n).astype(np.uint32)
    B = oracle.pairs_to_dcsr(r, c, n, n)
    few = r < 40  # rows of A
    A = oracle.pairs_to_dcsr(r[few], c[few], n, n)
    a, b = upload(controls, A, n, n), upload(controls, B, n, n)
    before = at.tuning_dict(controls.tuning())
    try:
        at.apply(controls, {**before, "gather_combine": combine})
        got, st = cb.dcsr.spgemm(controls, a, b, mode=cb.SPGEMM_PLAIN, timing=True)
    finally:
        at.apply(controls, before)
    assert_dcsr_equal(controls, got, oracle.spgemm(A, B))
    assert st["launches"][SYM_BITMAP] == (1 if combine else 2)
