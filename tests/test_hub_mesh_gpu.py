"""A hub of so many elements that they export more than 65 535 contributions from a
tile of 128 nodes, but fewer from one of 512 (33 000 triangles around node 0: 65 746
against 64 978).  Its windows do not fit the LDS, so the context takes the gathering
kernel in tiles of 512.  At the residual's bar, 1e-12 of the flux scale, against the
formulas in extended precision: the triangles' angle at the hub is 2e-4, where the CPU
oracle's face geometry is itself 7e-9 off them."""
import numpy as np
import pytest

from conftest import device
from oracle.oracle import OracleProblem
from test_jacobian_shapes_gpu import _fans
from test_residual_gpu import TOL, _rel, _state

pytestmark = pytest.mark.gpu


def _extended(prob, psi, psip, w_front):
    """The residual of a 2D problem of one zone without boundary fluxes, in extended precision."""
    L = np.longdouble
    x, c, h = prob.mesh.xyz[:, :2].astype(L), prob.mesh.conn, psi.astype(L)
    kx, ky, _, phi, alpha, n, sr, ss = prob.zones[0].astype(L)
    m = 1 - 1 / n
    dry = np.where(h < 0, h, L(-1))
    a = (-alpha * dry) ** n
    se = (1 + a) ** -m
    kr = np.where(h < 0, np.sqrt(se) * ((1 - 1 / (1 + a)) ** m - 1) ** 2, L(1))
    sw = np.where(h < 0, sr + (1 - sr) * se, L(1))
    ds = np.where(h < 0, -(1 - sr) * (n - 1) * a / (1 + a) * se / dry, L(0))
    e1, e2 = x[c[:, 1]] - x[c[:, 0]], x[c[:, 2]] - x[c[:, 0]]
    det = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0]
    g1, g2 = (np.stack(v, 1) / det[:, None] for v in ((e2[:, 1], -e2[:, 0]), (-e1[:, 1], e1[:, 0])))
    grad = [-(g1 + g2), g1, g2]
    q = sum(h[c[:, k]][:, None] * grad[k] for k in range(3))
    q[:, 1] += 1
    q *= -np.array([kx, ky]) * prob.ekmul.astype(L)[:, None]
    part = abs(det) / 6
    flow = [(g * q).sum(1) * part for g in grad]
    V, acc = np.zeros(len(h), L), np.zeros(len(h), L)
    np.add.at(V, c.ravel(), np.repeat(part, 3))
    # edges by (lower, higher) node; the front is the first node of the first element's local edge
    ends = np.stack([c[:, [0, 1]], c[:, [1, 2]], c[:, [2, 0]]], 1).reshape(-1, 2).astype(np.int64)
    _, first, edge = np.unique(ends.min(1) * len(h) + ends.max(1), return_index=True, return_inverse=True)
    up = np.where((w_front[edge] == 1) == (ends[first, 0][edge] == ends[:, 0]), ends[:, 0], ends[:, 1])
    up = up.reshape(-1, 3)
    for j, (i, k) in enumerate(((0, 1), (1, 2), (2, 0))):
        M = L(prob.rho0) * kr[up[:, j]] * (flow[k] - flow[i])
        np.add.at(acc, c[:, i], -M)
        np.add.at(acc, c[:, k], M)
    return acc / V - psip.astype(L) * L(prob.rho0) * (phi * ds + ss * sw)


def test_a_hub_past_the_small_tiles_exports():
    import torch
    from fvmpor_amd.lib import Context, FvpError
    prob = _fans((33000,), (0,))
    dev = device()
    ctx = Context(prob)
    psi, psip = _state(prob, 3)
    op = OracleProblem(prob)
    tp, tpp = torch.tensor(psi, device=dev), torch.tensor(psip, device=dev)
    F = torch.empty_like(tp)
    torch.cuda.synchronize()
    ctx.begin_step(0.0, tp, tpp)
    wf, _ = ctx.get_upwind()
    op.set_weights(wf)
    op.residual(0.0, psi, psip)
    Fx = _extended(prob, psi, psip, wf).astype(np.float64)
    for tile in (None, 128):
        if tile:
            with pytest.raises(FvpError, match="exports more than 65535"):
                ctx.set_residual_launch(0, tile, True)  # refused; the context keeps its tiles
        F.zero_()
        torch.cuda.synchronize()
        ctx.residual(0.0, tp, tpp, F)
        ctx.synchronize()
        assert _rel(F.cpu().numpy(), Fx, op.flux_scale()) <= TOL
