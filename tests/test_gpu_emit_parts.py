"""Dumped rows expanded by one and by several workgroups each: few and many rows,
one and several windows (3: a number of parts that no power of two reaches), and
slices kept as words and as pairs."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from clbool_amd import autotune as at
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncols", [1 << 19, 1 << 20, (1 << 21) + 5, 3 << 20, (1 << 22) - 1])
@pytest.mark.parametrize("nrows", [1, 5, 130, 1100])
def test_parts(controls, ncols, nrows):
    rng = np.random.default_rng(ncols + nrows)
    inner, a_len, b_len = 64, 12, 2000
    starts = rng.integers(0, ncols - 40000, inner)
    starts[::2] = 0  # half of B's rows are spread over all columns, half stay close together
    width = np.where(np.arange(inner) % 2, 40000, ncols)
    c = starts[:, None] + (rng.random((inner, b_len)) * width[:, None]).astype(np.int64)
    c[:, 0], c[::2, 1] = starts, ncols - 1
    key = np.unique(np.arange(inner)[:, None] * ncols + c)
    B = oracle.pairs_to_dcsr((key // ncols).astype(np.uint32), (key % ncols).astype(np.uint32), inner, ncols)
    pick = np.argsort(rng.random((nrows, inner)), axis=1)[:, :a_len]
    pick[::3] = pick[::3] // 2 * 2  # rows of the spread ones only
    key = np.unique(np.arange(nrows)[:, None] * inner + pick)
    A = oracle.pairs_to_dcsr((key // inner).astype(np.uint32), (key % inner).astype(np.uint32), nrows, inner)
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    ref = oracle.spgemm(A, B)
    before = at.tuning_dict(controls.tuning())
    try:
        for bits in (0, 14):
            at.apply(controls, {**before, "dump_bits_per_chunk": 1, "bitmap_min_products": 4096,
                                "onepass_bitmap_min": 4096, "hash_max_slots": 4096, "bitmap_window_bits": bits})
            for mode in (cb.SPGEMM_BOUND, cb.SPGEMM_PLAIN):
                got, st = cb.dcsr.spgemm(controls, a, b, mode=mode, timing=True)
                assert_dcsr_equal(controls, got, ref, f"mode {mode}, bits {bits}")
                assert st["dense_rows"] > nrows // 2
    finally:
        at.apply(controls, before)
