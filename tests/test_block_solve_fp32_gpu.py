"""The block solve with FP32 factors, rows of one lane (up to four or six entries a
triangle), of two, and of several slots, and blocks of 20480 rows, against the FP64 solution
with the same factors: at most ten roundings of 2^-24 a row, growth by the dominant diagonal
below 2, five rows deep (1e-5)."""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import device
from oracle import oracle as O
from test_ilu_shapes_gpu import SHAPES, _band, _csr

pytestmark = pytest.mark.gpu


def _fp32(ia, ja, a, rows, overlap=0):
    import torch
    from fvmpor_amd.lib import PRECON_BJILU0_F32, CsrMatrix
    n = len(ia) - 1
    A = CsrMatrix(ia, ja)
    A.precon_block_rows(rows)
    A.precon_overlap(overlap)
    A.set_values(torch.tensor(a, device=device()))
    assert A.precon_build(PRECON_BJILU0_F32) == 0
    x = torch.tensor(np.random.default_rng(6).normal(size=n), device=device())
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    A.precon_apply(x, y)
    torch.cuda.synchronize()
    return A, x.cpu().numpy(), y.cpu().numpy()


def _solve(ia, ja, lu, rows, x):
    """With the factors lu (U's diagonal inverted) of the blocks of `rows` rows, in FP64"""
    n = len(ia) - 1
    y = x.copy()
    row = np.repeat(np.arange(n), np.diff(ia))
    keep = row // rows == ja // rows
    M = sp.csr_matrix((lu[keep], (row[keep], ja[keep])), shape=(n, n)).sorted_indices()
    d = M.diagonal()
    L, U = sp.tril(M, -1).tocsr(), sp.triu(M, 1).tocsr()
    for r in range(n):
        y[r] -= L.data[L.indptr[r]:L.indptr[r + 1]] @ y[L.indices[L.indptr[r]:L.indptr[r + 1]]]
    for r in reversed(range(n)):
        y[r] -= U.data[U.indptr[r]:U.indptr[r + 1]] @ y[U.indices[U.indptr[r]:U.indptr[r + 1]]]
        y[r] *= d[r]
    return y


@pytest.mark.parametrize("rows", [64, 512])
@pytest.mark.parametrize("which", ["band of 4", "band of 5", "band of 6", "band of 7", "row of 8 L entries",
                                   "row of 9 L entries",
                                   "row of 17 L entries", "rows of 63 entries", "a chain and rows of 20 entries",
                                   "box"])
def test_solution_with_the_fp32_factors(which, rows):
    ia, ja, a = _csr(_band(300, int(which[-1])) if which.startswith("band") else SHAPES[which], 5)
    A, x, y = _fp32(ia, ja, a, rows)
    ref = _solve(ia, ja, A.precon_values(len(ja)), rows, x)
    np.testing.assert_allclose(y, ref, rtol=0, atol=1e-5 * np.abs(ref).max())


def test_a_block_of_20480_rows():
    # block 0: 4096 rows and, one layer out, four neighbours of each; and a row of 5
    # entries a triangle
    m = 4096
    hub = np.repeat(np.arange(m), 4)
    P = sp.coo_matrix((np.ones(4 * m + 5), (np.r_[hub, np.full(5, 9)], np.r_[m + np.arange(4 * m), np.arange(5)])),
                      shape=(5 * m, 5 * m))
    ia, ja, a = _csr(P, 5)
    A, x, y = _fp32(ia, ja, a, m, overlap=1)
    ref = _solve(ia, ja, O.ilu0(ia, ja, a)[0], 5 * m, x)  # the whole matrix is in the block
    np.testing.assert_allclose(y[:m], ref[:m], rtol=0, atol=1e-5 * np.abs(ref).max())
