"""The unions that end a batched closure step, against sets of pairs: matrices
with no, one and several products, with empty and unchanged matrices between
them, products cut into row blocks, and sizes around the merge tile of 2048
keys.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
from clbool_amd import generators as gen

pytestmark = pytest.mark.gpu


def _mat(n, nnz, seed):
    if not nnz:
        return np.zeros((n, n), bool)
    m = np.zeros((n, n), bool)
    r, c = gen.uniform_pairs(nnz, n, n, seed)
    m[r, c] = True
    return m


def _up(ctl, m):
    r, c = np.nonzero(m)
    if not r.size:
        return cb.matrix_dcsr(m.shape[0], m.shape[1])
    return cb.matrix_dcsr_from_cpu(ctl, *gen.to_dcsr(r, c), *m.shape)


@pytest.mark.parametrize("n,sizes,bound", [(7, [0, 5, 0, 3, 49, 1], 0), (64, [900, 0, 2047, 1, 2048, 300], 0),
                                           (64, [900, 40, 2047, 1, 2048, 300], 128),
                                           (300, [3000, 500, 1, 0, 9000, 2500], 900)])
@pytest.mark.parametrize("triples", [[(1, 0, 4)], [(0, 1, 3), (0, 4, 4), (0, 5, 3), (2, 4, 0), (5, 2, 2)],
                                     [(4, 4, 4), (3, 5, 5), (3, 0, 2), (1, 3, 5), (4, 1, 0), (0, 0, 0)]])
def test_batched_step(controls, n, sizes, bound, triples):
    dense = [_mat(n, k, i + 1) for i, k in enumerate(sizes)]
    mats = [_up(controls, m) for m in dense]
    st = cb.closure_step(controls, mats, triples, mode=cb.CLOSURE_BATCHED, spgemm_mode=cb.SPGEMM_PLAIN,
                         block_bound=bound)
    want = [m.copy() for m in dense]
    for x, y, z in triples:
        want[x] |= (dense[y].astype(np.int64) @ dense[z].astype(np.int64)) > 0
    assert st["changed"] == sum(int(a.sum() != b.sum()) for a, b in zip(want, dense))
    for got, w in zip(mats, want):
        r, c = np.nonzero(w)
        assert got.nnz == r.size
        if r.size:
            for a, b in zip(got.to_host(controls), gen.to_dcsr(r, c)):
                assert np.array_equal(a, b)
