"""Bitmap rows that are kept by the symbolic or the one pass and expanded
later, and the packed gather of B, against the oracle: column counts at the
edges of every window size, rows from empty to full (so that rounds are
expanded by rank and bit by bit), rows of one heavy workgroup, and B rows that
share words or never do.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from clbool_amd import generators as gen
from helpers import assert_dcsr_equal, upload

pytestmark = pytest.mark.gpu
NROWS = 400


def _dcsr(rows, cols, nrows, ncols):
    key = np.unique((rows.astype(np.uint64) << np.uint64(32)) | cols.astype(np.uint64))
    return oracle.pairs_to_dcsr((key >> np.uint64(32)).astype(np.uint32), key.astype(np.uint32), nrows, ncols)


def _operands(ncols, kind, seed=3):
    """A of NROWS rows over 40 B rows, with over 2^20 products in all but the
    narrowest; the first A rows read all of B."""
    rng = np.random.default_rng(seed)
    inner, nrows = 40, NROWS
    br, bc = [], []
    for k in range(inner):
        n = int(min(ncols, rng.choice([1, 40, 300, 2000, 9000])))
        if kind == "runs":  # neighbours: many columns per word, some words full
            start = int(rng.integers(0, max(1, ncols - n)))
            c = np.arange(start, min(ncols, start + n))
        else:  # one column per word
            c = rng.integers(0, (ncols + 31) // 32, n) * 32
            c = c[c < ncols]
        br.append(np.full(c.size, k))
        bc.append(c)
    ar, ac = [], []
    for r in range(nrows):
        n = inner if r < 30 else int(rng.integers(0, 12))
        ac.append(rng.choice(inner, n, replace=False))
        ar.append(np.full(n, r))
    return (_dcsr(np.concatenate(ar), np.concatenate(ac), nrows, inner),
            _dcsr(np.concatenate(br), np.concatenate(bc), inner, ncols))


@pytest.mark.parametrize("ncols", [1, 31, 2047, 2048, 2049, 4097, 8191, 16385, 32769, 65535, 131073, 262145, 524289,
                                   1048576, 1048577, 3000001])
@pytest.mark.parametrize("kind", ["runs", "apart"])
def test_kept_rows(controls, ncols, kind):
    A, B = _operands(ncols, kind)
    ref = oracle.spgemm(A, B)
    a, b = upload(controls, A, NROWS, 40), upload(controls, B, 40, ncols)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication_hash(controls, a, b), ref, "plain")
    got, _ = cb.dcsr.spgemm(controls, a, b, mode=cb.SPGEMM_BOUND)
    assert_dcsr_equal(controls, got, ref, "bound")
    blocks = []
    plan = cb.dcsr.plan(controls, a, b, mode=cb.SPGEMM_PLAIN, block_bound=max(ncols, ref.nnz // 3 + 1))
    plan.run_all(lambda k, m, st: blocks.append(m.to_host(controls)[2] if m.nnz else np.zeros(0, np.uint32)))
    plan.close()
    assert np.array_equal(np.concatenate(blocks), ref.cols)


@pytest.mark.parametrize("hubs", [1, 5])
def test_heavy_rows(controls, hubs):
    """A few rows with most of the products run on the widest workgroups."""
    rng = np.random.default_rng(hubs)
    n = 20000
    r = np.concatenate([np.repeat(np.arange(hubs), 3000), rng.integers(0, n, 60000)])
    c = np.concatenate([rng.integers(0, n, hubs * 3000), rng.integers(0, n, 60000)])
    A = _dcsr(r, c, n, n)
    ref = oracle.spgemm(A, A)
    a = upload(controls, A, n, n)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication_hash(controls, a, a), ref, "plain")
    assert_dcsr_equal(controls, cb.dcsr.spgemm(controls, a, a, mode=cb.SPGEMM_BOUND)[0], ref, "bound")


@pytest.mark.parametrize("ncols", [4097, 16385, 65537, 1048575, 1048577, 1100000])
def test_packed(controls, ncols):
    """Enough products for B to be packed: B rows of about every second column
    of a range, with group 65535 and 0 modulo 65536 where there are so many."""
    rng = np.random.default_rng(ncols)
    inner, nrows = 40, 600
    br, bc = [], []
    for k in range(inner):
        n = int(min(ncols, rng.integers(3000, 9000)))
        start = int(rng.integers(0, ncols - n + 1)) if k % 4 else ncols - n
        c = start + np.flatnonzero(rng.random(n) < 0.6)
        br.append(np.full(c.size, k))
        bc.append(c)
    A = _dcsr(np.repeat(np.arange(nrows), 20), rng.integers(0, inner, nrows * 20), nrows, inner)
    B = _dcsr(np.concatenate(br), np.concatenate(bc), inner, ncols)
    ref = oracle.spgemm(A, B)
    a, b = upload(controls, A, nrows, inner), upload(controls, B, inner, ncols)
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication_hash(controls, a, b), ref, "plain")
    assert_dcsr_equal(controls, cb.dcsr.spgemm(controls, a, b, mode=cb.SPGEMM_BOUND)[0], ref, "bound")


@pytest.mark.parametrize("ncols", [4097, 1100000])
@pytest.mark.parametrize("lens", [(9000,), (2048,), (512, 1536, 4096, 2047, 2049)])
def test_packed_with_empty_stored_rows(controls, ncols, lens):
    """Stored rows of B without entries, before, between and after the others,
    where rows end at the packing's tiles of 2048 columns and where they don't,
    against the product without them."""
    rng = np.random.default_rng(ncols + len(lens))
    full = 40
    n = np.minimum(np.resize(lens, full), ncols)
    ids = np.arange(full) * 4 + 3  # ids 4k .. 4k + 2 may be stored without entries
    cols = np.concatenate([np.sort(rng.choice(min(ncols, 3 * k), k, replace=False)) for k in n])
    inner, nrows = 4 * full + 8, 800
    stored = np.sort(np.concatenate([ids, [0, 1, 2, 40, 41, 81, 82], [inner - 3, inner - 1]]))
    length = dict(zip(ids, n))
    rpt = np.concatenate([[0], np.cumsum([length.get(k, 0) for k in stored])]).astype(np.uint32)
    A = _dcsr(np.repeat(np.arange(nrows), 60), rng.integers(0, inner, nrows * 60), nrows, inner)
    B = _dcsr(np.repeat(ids, n), cols, inner, ncols)
    ref = oracle.spgemm(A, B)
    a = upload(controls, A, nrows, inner)
    b = cb.matrix_dcsr_from_cpu(controls, rpt, stored.astype(np.uint32), cols.astype(np.uint32), inner, ncols)
    assert_dcsr_equal(controls, cb.dcsr.spgemm(controls, a, b, mode=cb.SPGEMM_BOUND)[0], ref, "bound")
    assert_dcsr_equal(controls, cb.dcsr.matrix_multiplication_hash(controls, a, b), ref, "plain")
