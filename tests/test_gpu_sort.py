"""The pair sort (coo::sort_arrays, the COO constructor, dcsr::transpose)
against numpy: sizes around the tile of 4096 pairs, one to many tiles, and
row and column widths from zero bits to 32 each, so that digits straddle the
two halves and the number of passes is odd and even.  Whole numbers: equality."""
import numpy as np
import pytest

import clbool_amd as cb
from clbool_amd import generators as gen

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 4095, 4096, 4097, 12293, 300007]
WIDTHS = [(0, 0), (1, 0), (0, 7), (3, 6), (9, 8), (13, 20), (32, 32)]


def _pairs(n, rb, cb_, seed):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, 1 << rb, n, dtype=np.uint64).astype(np.uint32)
    c = rng.integers(0, 1 << cb_, n, dtype=np.uint64).astype(np.uint32)
    return r, c


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("widths", WIDTHS)
def test_sort_arrays(controls, n, widths):
    r, c = _pairs(n, *widths, seed=n)
    br, bc = cb.Buffer.from_array(controls, r), cb.Buffer.from_array(controls, c)
    cb.coo.sort_arrays(controls, br, bc, n)
    o = np.lexsort((c, r))
    assert np.array_equal(br.read(controls, n), r[o])
    assert np.array_equal(bc.read(controls, n), c[o])


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("widths", WIDTHS[:-1])
def test_construct_drops_duplicates(controls, n, widths):
    r, c = _pairs(n, *widths, seed=n + 1)
    m = cb.matrix_coo.from_host(controls, r, c, 1 << 20, 1 << 20, sorted=False, noDuplicates=False)
    key = np.unique((r.astype(np.uint64) << np.uint64(32)) | c)
    gr, gc = m.to_host(controls)
    assert np.array_equal(gr, (key >> np.uint64(32)).astype(np.uint32))
    assert np.array_equal(gc, key.astype(np.uint32))


@pytest.mark.parametrize("nrows,ncols,nnz", [(1, 1, 1), (1, 5000, 4097), (5000, 1, 4097), (257, 255, 20000),
                                             (70000, 1 << 20, 200003)])
def test_transpose(controls, nrows, ncols, nnz):
    nnz = min(nnz, nrows * ncols)
    r, c = gen.uniform_pairs(nnz, nrows, ncols, 5)
    a = cb.matrix_dcsr_from_cpu(controls, *gen.to_dcsr(r, c), nrows, ncols)
    t = cb.dcsr.transpose(controls, a)
    o = np.lexsort((r, c))
    for got, want in zip(t.to_host(controls), gen.to_dcsr(c[o], r[o])):
        assert np.array_equal(got, want)
