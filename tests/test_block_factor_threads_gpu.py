"""The block factorisation with every thread count it is launched with (64 to 1024, 4 to
64 rows of a level at once), rows of up to 16, 32 and 64 entries, alone and among shorter
ones, staged and in place:
each row's arithmetic is the same, so the factors are equal bit for bit and FP64's is
the oracle's (1e-12, as in test_ilu_shapes_gpu.py).  And the two precisions built in turn on
one matrix, against a matrix of its own each."""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import device
from oracle import oracle as O
from test_ilu_shapes_gpu import SHAPES, _band, _csr, _hubs

pytestmark = pytest.mark.gpu

WHICH = ["diagonal", "tridiagonal", "row of 9 L entries", "row of 17 L entries", "rows of 63 entries", "box",
         "grid of 64-wide levels", "blocks of rows of up to 16, 32 and 64", "most of up to 64"]
# the first blocks have short rows, later ones a few of 25 to 51 entries (block-local for 64 rows too)
MIXED = {"blocks of rows of up to 16, 32 and 64": sp.block_diag([_band(320, 2), _hubs(64, 24, 1, 24), _band(64, 1),
                                                                 _hubs(64, 50, 1, 50), _band(1600, 3)]),
         "most of up to 64": sp.block_diag([_band(64, 2), *[_band(128, 20)] * 4])}


def _build(which, ptype, rows, overlap=0, A=None):
    import torch
    from fvmpor_amd.lib import CsrMatrix
    ia, ja, a = _csr({**SHAPES, **MIXED}[which], 5)
    if A is None:
        A = CsrMatrix(ia, ja)
        A.precon_block_rows(rows)
        A.precon_overlap(overlap)
        A.set_values(torch.tensor(a, device=device()))
    assert A.precon_build(ptype) == 0
    x = torch.tensor(np.random.default_rng(6).normal(size=len(ia) - 1), device=device())
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    A.precon_apply(x, y)
    torch.cuda.synchronize()
    return A, A.precon_values(len(ja)) if overlap == 0 else None, y.cpu().numpy()


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("which", WHICH)
@pytest.mark.parametrize("rows", [64, 1024])
def test_every_thread_count_gives_the_same_factor(which, rows, fp32, monkeypatch):
    from fvmpor_amd.lib import PRECON_BJILU0, PRECON_BJILU0_F32
    ptype = PRECON_BJILU0_F32 if fp32 else PRECON_BJILU0
    _, lu, y = _build(which, ptype, rows)
    if not fp32:
        ia, ja, a = _csr({**SHAPES, **MIXED}[which], 5)
        n = len(ia) - 1
        row = np.repeat(np.arange(n), np.diff(ia))
        keep = row // rows == ja // rows
        B = sp.csr_matrix((a[keep], (row[keep], ja[keep])), shape=(n, n)).sorted_indices()
        ref, _ = O.ilu0(B.indptr, B.indices, B.data)
        np.testing.assert_allclose(lu[keep], ref, rtol=1e-12, atol=1e-14)
    for mode in ("1", "0"):
        monkeypatch.setenv("FVP_BJ_FACTOR_MODE", mode)
        for threads in (64, 128, 256, 512, 1024):
            monkeypatch.setenv("FVP_BJ_FACTOR_THREADS", str(threads))
            _, lu_t, y_t = _build(which, ptype, rows)
            np.testing.assert_array_equal(lu_t, lu)
            np.testing.assert_array_equal(y_t, y)


@pytest.mark.parametrize("overlap", [0, 1])
@pytest.mark.parametrize("which", ["tridiagonal", "row of 9 L entries", "box", *MIXED])
def test_both_precisions_on_one_matrix(which, overlap):
    from fvmpor_amd.lib import PRECON_BJILU0, PRECON_BJILU0_F32
    own = {t: _build(which, t, 256, overlap)[2] for t in (PRECON_BJILU0, PRECON_BJILU0_F32)}
    for first in (PRECON_BJILU0, PRECON_BJILU0_F32):
        A = None
        for t in (first, PRECON_BJILU0 + PRECON_BJILU0_F32 - first, first):
            A, _, y = _build(which, t, 256, overlap, A)
            np.testing.assert_array_equal(y, own[t])
