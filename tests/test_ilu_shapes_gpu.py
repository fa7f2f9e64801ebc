"""ILU(0) at the shapes where its factor and solve kernels change form: rows of
1 to 64 entries (the register rows hold 16, 32 or 64), more than eight and more
than sixteen L entries, triangle windows of 4 to 32 entries, levels of one row
and levels wider than a workgroup, and matrices past the one-workgroup limits.
The oracle's ILU(0) is the reference.  Tolerances: factors and solutions of
diagonally dominant matrices carry at most a few hundred roundings per row, so
1e-12 of the entry and 1e-11 of the solution in FP64 (1e-4 in FP32)."""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import device
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _csr(P, seed):
    """Diagonally dominant values on the symmetric pattern of P plus the diagonal."""
    P = sp.csr_matrix((P + P.T + sp.eye(P.shape[0])) != 0).sorted_indices()
    rng = np.random.default_rng(seed)
    a = rng.uniform(-1, 1, P.nnz)
    ia, ja = P.indptr.astype(np.int32), P.indices.astype(np.int32)
    rows = np.repeat(np.arange(P.shape[0]), np.diff(ia))
    a[rows == ja] = 1.3 * np.diff(ia)
    return ia, ja, a


def _band(n, width):
    return sp.diags([np.ones(n - k) for k in range(1, width + 1)], list(range(1, width + 1)), shape=(n, n))


def _grid(nx, ny, nz=1, diagonals=True):
    i = np.arange(nx * ny * nz).reshape(nz, ny, nx)
    pairs = []
    for dz, dy, dx in [(0, 0, 1), (0, 1, 0), (0, 1, 1), (1, 0, 0), (1, 1, 0), (1, 0, 1), (1, 1, 1)]:
        if not diagonals and dz + dy + dx > 1:
            continue
        a = i[:nz - dz, :ny - dy, :nx - dx].ravel()
        pairs.append(np.stack([a, i[dz:, dy:, dx:].ravel()]))
    r, c = np.concatenate(pairs, axis=1)
    return sp.coo_matrix((np.ones(len(r)), (r, c)), shape=(i.size, i.size))


def _hubs(n, first, count, width, extra=0):
    """Rows first, first + 1, ... that couple to `width` rows before `first` each (all of one level, or a chain
    with extra = 1): more entries of one level than a solve window holds."""
    r = np.repeat(np.arange(first, first + count), width)
    c = np.concatenate([np.arange(k % 3, k % 3 + width) for k in range(count)])
    P = sp.coo_matrix((np.ones(len(r)), (r, c)), shape=(n, n))
    return P + _band(n, 1) if extra else P


SHAPES = {
    "one row": sp.coo_matrix((1, 1)),
    "diagonal": sp.coo_matrix((700, 700)),                 # a single level wider than a workgroup's pieces
    "tridiagonal": _band(300, 1),                          # one row per level
    "row of 8 L entries": _band(130, 8),
    "row of 9 L entries": _band(130, 9),
    "row of 17 L entries": _band(90, 17),
    "rows of 63 entries": _band(140, 31),                  # four registers, 31 L entries
    "rows with 30 entries of one level": _hubs(150, 40, 20, 30),
    "a chain and rows of 20 entries": _hubs(700, 60, 7, 20, extra=1),  # windows of 4, a few rows of several
    "wide grid": _grid(97, 3, diagonals=False),
    "grid of 64-wide levels": _grid(65, 130),
    "box": _grid(13, 11, 9),
    "wide box": _grid(40, 30, 16, diagonals=False),        # 19200 rows: past the LDS of the one-workgroup solve
    "two rows in 20000": sp.coo_matrix(([1.0], ([3], [19000])), shape=(20000, 20000)),
}


@pytest.mark.parametrize("which", list(SHAPES))
def test_global_ilu0(which):
    import torch
    from fvmpor_amd.lib import CsrMatrix, PRECON_ILU0
    ia, ja, a = _csr(SHAPES[which], 3)
    n = len(ia) - 1
    A = CsrMatrix(ia, ja)
    for seed in (0, 1):  # the second build reuses the tables with other values
        a = a * np.random.default_rng(seed).uniform(0.9, 1.1, len(a))
        A.set_values(torch.tensor(a, device=device()))
        assert A.precon_build(PRECON_ILU0) == 0
        lu, dp = O.ilu0(ia, ja, a)
        np.testing.assert_allclose(A.precon_values(len(ja)), lu, rtol=1e-12, atol=1e-14)
        x = np.random.default_rng(4 + seed).normal(size=n)
        y = torch.empty(n, dtype=torch.float64, device=device())
        xd = torch.tensor(x, device=device())
        torch.cuda.synchronize()
        A.precon_apply(xd, y)
        torch.cuda.synchronize()
        np.testing.assert_allclose(y.cpu().numpy(), O.ilu0_apply(ia, ja, lu, dp, x), rtol=1e-11, atol=1e-13)


@pytest.mark.parametrize("which", ["diagonal", "tridiagonal", "row of 17 L entries", "rows of 63 entries", "box"])
@pytest.mark.parametrize("fp32", [False, True])
def test_block_ilu0(which, fp32):
    import torch
    from fvmpor_amd.lib import CsrMatrix, PRECON_BJILU0, PRECON_BJILU0_F32
    ia, ja, a = _csr(SHAPES[which], 5)
    n = len(ia) - 1
    A = CsrMatrix(ia, ja)
    A.precon_block_rows(64)
    A.set_values(torch.tensor(a, device=device()))
    assert A.precon_build(PRECON_BJILU0_F32 if fp32 else PRECON_BJILU0) == 0
    M = sp.csr_matrix((a, ja, ia), shape=(n, n)).tocoo()
    keep = M.row // 64 == M.col // 64
    B = sp.csr_matrix((M.data[keep], (M.row[keep], M.col[keep])), shape=(n, n)).sorted_indices()
    lu, dp = O.ilu0(B.indptr, B.indices, B.data)
    x = np.random.default_rng(6).normal(size=n)
    y = torch.empty(n, dtype=torch.float64, device=device())
    xd = torch.tensor(x, device=device())
    torch.cuda.synchronize()
    A.precon_apply(xd, y)
    torch.cuda.synchronize()
    ref = O.ilu0_apply(B.indptr, B.indices, lu, dp, x)
    if fp32:
        assert np.abs(y.cpu().numpy() - ref).max() <= 1e-4 * np.abs(ref).max()
    else:
        np.testing.assert_allclose(y.cpu().numpy(), ref, rtol=1e-11, atol=1e-13)


def test_zero_pivot_inside_the_one_workgroup_factor():
    import torch
    from fvmpor_amd.lib import CsrMatrix, ERR_PIVOT, PRECON_ILU0
    ia, ja, a = _csr(_band(40, 1), 7)
    row = 20
    for k in range(ia[row], ia[row + 1]):
        a[k] = 0.0  # the whole row: its pivot stays zero
    A = CsrMatrix(ia, ja)
    A.set_values(torch.tensor(a, device=device()))
    assert A.precon_build(PRECON_ILU0) == ERR_PIVOT
