"""Passes over the nonzeros that know each one's row (dcsr_to_coo, the keys of
the additions) and the row compression of coo_to_dcsr, against numpy: totals
around the tiles of 2048 and 4096 entries, rows of one entry, one row of all
of them, and CSR matrices with more empty rows inside a tile than its copy of
the row pointer holds.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
import oracle
from helpers import assert_dcsr_equal

pytestmark = pytest.mark.gpu


def _lens(kind, total):
    if kind == "ones":
        return np.ones(total, np.int64)
    if kind == "one row":
        return np.array([total])
    rng = np.random.default_rng(total)
    lens = []
    while sum(lens) < total:
        lens.append(int(min(total - sum(lens), rng.choice([1, 2, 7, 64, 700, 3000]))))
    return np.array(lens)


@pytest.mark.parametrize("total", [1, 255, 2047, 2048, 2049, 4095, 4096, 4097, 70001])
@pytest.mark.parametrize("kind", ["ones", "one row", "mixed"])
def test_rows_out_and_back(controls, kind, total):
    lens = _lens(kind, total)
    rows = (np.arange(lens.size) * 3 + 1).astype(np.uint32)
    cols = np.concatenate([np.arange(k) for k in lens]).astype(np.uint32)
    rpt = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    n = max(int(rows[-1]) + 1, total)
    a = cb.matrix_dcsr_from_cpu(controls, rpt, rows, cols, n)
    coo = cb.dcsr_to_coo_shallow(controls, a)
    assert np.array_equal(coo.to_host(controls)[0], np.repeat(rows, lens))
    back = cb.coo_to_dcsr_shallow(controls, coo)
    for got, want in zip(back.to_host(controls), (rpt, rows, cols)):
        assert np.array_equal(got, want)
    same = cb.dcsr.addition(controls, a, back)
    for got, want in zip(same.to_host(controls), (rpt, rows, cols)):
        assert np.array_equal(got, want)


@pytest.mark.parametrize("gap", [1, 2303, 2304, 2305, 50000])
def test_csr_addition_over_empty_rows(controls, gap):
    n = 3 * gap + 7
    ar, ac = np.array([0, gap, gap, 2 * gap, n - 1], np.uint32), np.array([5, 0, 3, 1, 6], np.uint32)
    br, bc = np.array([gap, gap + 1, 2 * gap + 1], np.uint32), np.array([3, 2, 0], np.uint32)

    def up(r, c):
        rpt = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.uint32)
        return cb.csr_from_cpu(controls, rpt, c, n, n)

    got_rpt, got_cols = cb.csr.matrix_addition(controls, up(ar, ac), up(br, bc)).to_host(controls)
    key = np.unique(np.concatenate([(ar.astype(np.uint64) << np.uint64(32)) | ac,
                                    (br.astype(np.uint64) << np.uint64(32)) | bc]))
    want = np.concatenate([[0], np.cumsum(np.bincount((key >> np.uint64(32)).astype(np.int64), minlength=n))])
    assert np.array_equal(got_rpt, want) and np.array_equal(got_cols, key.astype(np.uint32))


@pytest.mark.parametrize("na", [1, 255, 2047, 2048, 2049, 6145])
@pytest.mark.parametrize("nb", [1, 257, 2048, 4097])
def test_two_matrices_in_one_launch(controls, na, nb):
    """Additions expand both operands by the same launches: sizes about a tile,
    and one row a nonzero or rows of several."""
    rng = np.random.default_rng(na * 7 + nb)
    n = 9000
    keys = []
    for m, per in ((na, 1), (nb, 3)):
        rows = (np.arange(m) // per).astype(np.uint64) * np.uint64(per)
        cols = np.arange(m, dtype=np.uint64) % np.uint64(per) + rng.integers(0, n - per, m).astype(np.uint64) // 3 * 3
        keys.append(np.unique((rows << np.uint64(32)) | cols))
    pair = [((k >> np.uint64(32)).astype(np.uint32), k.astype(np.uint32)) for k in keys]
    u = np.union1d(*keys)
    ur, uc = (u >> np.uint64(32)).astype(np.uint32), u.astype(np.uint32)
    D = [oracle.pairs_to_dcsr(r, c, n, n) for r, c in pair]
    d = [cb.matrix_dcsr_from_cpu(controls, m.rpt, m.rows, m.cols, n) for m in D]
    assert_dcsr_equal(controls, cb.dcsr.addition(controls, *d), oracle.pairs_to_dcsr(ur, uc, n, n), "dcsr")
    s = [cb.csr_from_cpu(controls, *oracle.csr_from_pairs(r, c, n), n, n) for r, c in pair]
    rpt, cols = cb.csr.matrix_addition(controls, *s).to_host(controls)
    er, ec = oracle.csr_from_pairs(ur, uc, n)
    assert np.array_equal(rpt, er) and np.array_equal(cols, ec)
