"""The Gram-Schmidt kernels of GMRES at the sizes where they change: one row to
more workgroups than half the partials' room, odd lengths (row pairs), 1 to 40
columns (row pairs up to 16, single rows up to 32, chunks beyond), with and
without the second pass, with the diagonal preconditioner.  One cycle without
convergence must leave the residual of the minimum over the Krylov space, which
is computed here in numpy with a basis orthogonalised twice.  The minimum of the
residual moves by no more than a small multiple of m eps ||b|| under rounding in
the basis (GMRES is backward stable); 1e-12 ||b|| is allowed for 40 columns."""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import device

pytestmark = pytest.mark.gpu


def _system(n, seed):
    rng = np.random.default_rng(seed)
    d = rng.uniform(2.05, 2.6, n)
    S = sp.diags([-1.2 * np.ones(n - 1), d, -0.8 * np.ones(n - 1)], [-1, 0, 1]) if n > 1 else sp.diags([d], [0])
    S = S.tocsr()
    S.sort_indices()
    return S, rng.normal(size=n)


def _min_residual(S, scale, b, m):
    Q = [b / np.linalg.norm(b)]
    W = []
    for j in range(m):
        w = S @ (scale * Q[-1])
        W.append(w.copy())
        for _ in range(2):
            for q in Q:
                w -= (q @ w) * q
        Q.append(w / np.linalg.norm(w))
    y = np.linalg.lstsq(np.array(Q) @ np.array(W).T, np.array(Q) @ b, rcond=None)[0]
    return np.linalg.norm(b - np.array(W).T @ y)


@pytest.mark.parametrize("n,m,ptype,reorth,noalloc", [
    (17, 3, 0, 1, False), (63, 8, 2, 1, False), (1023, 16, 2, 1, False), (1025, 17, 2, 2, False),
    (4141, 32, 0, 0, False), (2051, 33, 2, 1, False), (2050, 40, 0, 2, False), (2049, 40, 2, 0, False),
    (70001, 17, 2, 1, True), (131072, 5, 2, 1, False), (131075, 20, 2, 1, False), (262147, 9, 0, 1, False),
    (300001, 24, 2, 0, False)])
def test_one_cycle_is_the_minimum_over_the_krylov_space(n, m, ptype, reorth, noalloc):
    import torch
    from fvmpor_amd.lib import CsrMatrix
    S, b = _system(n, n)
    ref = _min_residual(S, 1.0 / S.diagonal() if ptype == 2 else np.ones(n), b, m)
    A = CsrMatrix(S.indptr.astype(np.int32), S.indices.astype(np.int32))
    A.set_values(torch.tensor(S.data, device=device()))
    assert A.precon_build(ptype) == 0
    bd = torch.tensor(b, device=device())
    x = torch.zeros(n, dtype=torch.float64, device=device())
    torch.cuda.synchronize()
    rc, st = (A.gmres_noalloc if noalloc else A.gmres)(bd, x, m=m, max_restarts=0, tol=1e-15, reorth=reorth)
    assert rc != 0 and not st["converged"] and st["iterations"] == m, st
    bn = np.linalg.norm(b)
    r = np.linalg.norm(b - S @ x.cpu().numpy())
    print(n, m, r / bn, ref / bn)
    assert abs(r - ref) <= 1e-12 * bn
    assert abs(st["residual"] - ref) <= 1e-12 * bn


@pytest.mark.parametrize("n3,reorth", [(1, 1), (700, 1), (50001, 1), (50001, 2), (100001, 1)])
def test_a_krylov_space_of_three_dimensions(n3, reorth):
    """The same 3 x 3 block down the diagonal: the third step's vector lies in
    the span of the basis, so that only rounding is left of it and the norm of
    the second update is taken directly."""
    import torch
    from fvmpor_amd.lib import CsrMatrix
    rng = np.random.default_rng(5)
    B = np.array([[3.0, 1.0, 0.5], [-0.5, 4.0, 1.0], [0.25, -1.0, 5.0]])
    S = sp.block_diag([B] * n3, format="csr") if n3 < 1000 else sp.kron(sp.identity(n3), B, format="csr")
    S.sort_indices()
    xt = rng.normal(size=3 * n3)
    A = CsrMatrix(S.indptr.astype(np.int32), S.indices.astype(np.int32))
    A.set_values(torch.tensor(S.data, device=device()))
    assert A.precon_build(0) == 0
    x = torch.zeros(3 * n3, dtype=torch.float64, device=device())
    torch.cuda.synchronize()
    rc, st = A.gmres(torch.tensor(S @ xt, device=device()), x, m=10, max_restarts=0, tol=1e-13, reorth=reorth)
    assert rc == 0 and st["converged"] and st["iterations"] == 3, st
    assert np.abs(x.cpu().numpy() - xt).max() <= 1e-12 * np.abs(xt).max()
