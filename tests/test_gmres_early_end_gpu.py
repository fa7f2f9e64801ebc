"""Where a GMRES cycle ends early: at the last steps whose kernels leave once the
estimate meets the tolerance and the first that run on regardless (32 columns), with
and without the diagonal preconditioner, in the static workspace too; and restarts,
after a full cycle and after one whose estimate met the tolerance though the residual
had not.  The steps and the solution are those of the minimum over the Krylov space,
computed in numpy.  Under rounding the residual moves by a small multiple of
m eps ||b||, 1e-12 ||b|| is allowed as in test_gmres_shapes_gpu.py, and the solution by
that times ||S^-1|| <= 1 / 0.05 (diagonal dominance)."""
import numpy as np
import pytest
import scipy.sparse as sp

from conftest import device
from test_gmres_shapes_gpu import _system

pytestmark = pytest.mark.gpu


def _cycle(S, scale, r, m, stop):
    """Residual norm and correction of GMRES after each step, up to m or the first norm below stop."""
    Q, W, out = [r / np.linalg.norm(r)], [], []
    for _ in range(m):
        w = S @ (scale * Q[-1])
        W.append(w.copy())
        for _ in range(2):
            for q in Q:
                w -= (q @ w) * q
        Q.append(w / np.linalg.norm(w))
        y = np.linalg.lstsq(np.array(Q) @ np.array(W).T, np.array(Q) @ r, rcond=None)[0]
        out.append((np.linalg.norm(r - np.array(W).T @ y), scale * (np.array(Q[:-1]).T @ y)))
        if out[-1][0] < stop:
            break
    return out


def _solve(S, b, ptype, noalloc=False, **kw):
    import torch
    from fvmpor_amd.lib import CsrMatrix
    A = CsrMatrix(S.indptr.astype(np.int32), S.indices.astype(np.int32))
    A.set_values(torch.tensor(S.data, device=device()))
    assert A.precon_build(ptype) == 0
    x = torch.zeros(S.shape[0], dtype=torch.float64, device=device())
    torch.cuda.synchronize()
    rc, st = (A.gmres_noalloc if noalloc else A.gmres)(torch.tensor(b, device=device()), x, **kw)
    return rc, st, x.cpu().numpy()


@pytest.mark.parametrize("ptype", [0, 2])
@pytest.mark.parametrize("steps,m,reorth,noalloc", [(30, 40, 1, False), (31, 40, 1, False), (32, 40, 1, False),
                                                    (32, 40, 0, False), (33, 40, 1, False), (34, 40, 2, False),
                                                    (32, 32, 1, False), (32, 33, 1, False), (32, 40, 1, True)])
def test_ends_at_the_step_that_meets_the_tolerance(steps, m, reorth, noalloc, ptype):
    S, b = _system(2049, 7)
    bn = np.linalg.norm(b)
    hist = _cycle(S, 1.0 / S.diagonal() if ptype == 2 else np.ones(len(b)), b, steps, 0.0)
    tol = np.sqrt(hist[-1][0] * hist[-2][0]) / bn  # a factor 0.7 a step: met at the last one
    rc, st, x = _solve(S, b, ptype, noalloc, m=m, max_restarts=0, tol=tol, reorth=reorth)
    assert rc == 0 and st["converged"] and st["iterations"] == steps and st["restarts"] == 0, st
    assert abs(st["residual"] - hist[-1][0]) <= 1e-12 * bn
    assert np.linalg.norm(x - hist[-1][1]) <= 1e-12 * bn / 0.05


@pytest.mark.parametrize("ptype", [0, 2])
@pytest.mark.parametrize("m", [12, 33])
def test_restarts_after_full_cycles(m, ptype):
    S, b = _system(2049, 7)
    bn, scale = np.linalg.norm(b), 1.0 / S.diagonal() if ptype == 2 else np.ones(2049)
    tol, x_ref, r, steps, cycles = 3e-7, np.zeros(2049), b, 0, 0
    while np.linalg.norm(r) >= tol * bn:
        hist = _cycle(S, scale, r, m, tol * bn)
        x_ref = x_ref + hist[-1][1]
        r = b - S @ x_ref
        steps += len(hist)
        cycles += 1
    assert cycles > 1
    rc, st, x = _solve(S, b, ptype, m=m, max_restarts=10, tol=tol, reorth=1)
    assert rc == 0 and st["iterations"] == steps and st["restarts"] == cycles - 1, (st, steps, cycles)
    assert np.linalg.norm(x - x_ref) <= 1e-12 * bn / 0.05


@pytest.mark.parametrize("n3", [700, 50001])
def test_restarts_after_an_estimate_that_was_met(n3):
    """The same 3 x 3 block of eigenvalues 1, 1e-2, 1e-5 down the diagonal: each cycle's
    estimate falls to rounding after three steps, the true residual to eps ||A|| ||x|| only
    (1e-11 of ||b||), so every restart begins a cycle that ends early again."""
    rng = np.random.default_rng(5)
    V = np.array([[1.0, 0.3, -0.2], [0.1, 1.0, 0.4], [-0.3, 0.2, 1.0]])
    B = V @ np.diag([1.0, 1e-2, 1e-5]) @ np.linalg.inv(V)
    S = sp.kron(sp.identity(n3), B, format="csr")
    S.sort_indices()
    b = rng.normal(size=3 * n3)
    rc, st, x = _solve(S, b, 0, m=10, max_restarts=4, tol=1e-14, reorth=1)
    assert rc > 0 and not st["converged"] and st["restarts"] == 4, st
    assert 3 + 4 <= st["iterations"] < 50, st
    assert np.linalg.norm(b - S @ x) <= 1e-9 * np.linalg.norm(b)
