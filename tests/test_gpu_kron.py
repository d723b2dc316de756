"""Kronecker products by tiles of 1024 B nonzeros and groups of A rows: sizes
about a tile, rows over many tiles, and A rows enough for groups of several.
Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu


def _matrix(rng, lens, ncols):
    """Rows of the given lengths, every third row id without entries."""
    lens = np.asarray(lens)
    ids = np.arange(lens.size) * 3 // 2
    cols = np.concatenate([np.sort(rng.choice(ncols, n, replace=False)) for n in lens])
    return np.repeat(ids, lens).astype(np.uint32), cols.astype(np.uint32), int(ids[-1]) + 2


@pytest.mark.parametrize("la,lb", [
    ([1], [1]), ([1], [2, 1]), ([1], [1023]), ([1], [1024]), ([1], [1025]), ([1, 1], [2049]), ([3], [1, 1366]),
    ([2, 5, 1, 7], [1, 2, 3, 4, 5, 600, 1, 1]),
    ([200], [9000]),                             # one row over many tiles
    ([1], [1] * 9001),                           # a row per nonzero of a tile
    ([1, 2] * 600, [1, 2, 1]),
    ([1, 2] * 6001, [1, 2, 1]),                  # groups, the last one short
    ([1, 3, 2] * 1367, [1025, 3]),
    ([40, 1, 1, 300], [1] * 700 + [5000] + [2] * 700),
])
def test_kron_tiles(controls, la, lb):
    rng = np.random.default_rng(len(la) * 131 + len(lb))
    ca, cbn = max(la) + 3, max(lb) + 5
    ar, ac, na = _matrix(rng, la, ca)
    br, bc, nb = _matrix(rng, lb, cbn)
    A, B = oracle.pairs_to_dcsr(ar, ac, na, ca), oracle.pairs_to_dcsr(br, bc, nb, cbn)
    out = cb.dcsr.kronecker_product(controls, upload(controls, A, na, ca), upload(controls, B, nb, cbn))
    # the product from its definition: every pair of entries
    r = (ar.astype(np.uint64)[:, None] * nb + br).ravel()
    c = (ac.astype(np.uint64)[:, None] * cbn + bc).ravel()
    key = np.sort((r << np.uint64(32)) | c)
    ref = oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), na * nb, ca * cbn)
    assert_dcsr_equal(controls, out, ref, "kron")
