"""Closure unions and products that find no room at first, with HIP's last few
megabytes in different amounts: what the first attempt took must not be in the way
of the second.  Digests against the same calls with room."""
import numpy as np
import pytest

import clbool_amd as cb
from helpers import hold_memory

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def _matrix(ctl, rng, n, nnz):
    k = np.unique(rng.integers(0, n * n, nnz))
    rows, cnt = np.unique(k // n, return_counts=True)
    return cb.matrix_dcsr_from_cpu(ctl, np.concatenate([[0], np.cumsum(cnt)]).astype(np.uint32), rows.astype(np.uint32),
                                   (k % n).astype(np.uint32), n, n)


def _step(ctl, mats):
    out = list(mats)
    cb.closure_step(ctl, out, [(x, 6, 7) for x in range(6)], mode=cb.CLOSURE_BATCHED)
    return [cb.dcsr.digest(ctl, m) for m in out[:6]]


@pytest.fixture(scope="module")
def crowded():
    """Controls, six matrices of two million nonzeros and two small ones, the step's
    results with room; then all memory but 4 GiB is held."""
    ctl = cb.create_controls()
    rng = np.random.default_rng(6)
    mats = [_matrix(ctl, rng, 1 << 16, nnz) for nnz in [1 << 21] * 6 + [30000] * 2]
    want = _step(ctl, mats)
    held = hold_memory(ctl, 4 << 30)
    yield ctl, mats, want
    del held, mats
    ctl.trim()
    ctl.close()


@pytest.mark.parametrize("less", range(0, 16, 2))
def test_unions(crowded, less):
    """96 MiB of keys and the new matrices together, 16 one by one."""
    ctl, mats, want = crowded
    held = hold_memory(ctl, 112 * MIB)
    held += [cb.Buffer.create(ctl, 2 * MIB) for _ in range(less // 2)]
    got = _step(ctl, mats)
    del held
    ctl.trim()
    assert got == want
