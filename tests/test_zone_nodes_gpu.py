"""The soil law's pass over nodes that touch several zones, which its first
workgroups take from a list: none, some around a workgroup's 256, and most of the
nodes; with the averaged weights, at a step's start and beyond 65 535 nodes, where
that pass runs by itself.  Against the oracle at the residual's bar, 1e-12 of the flux
scale (sums of about 30 terms of that scale per node, each a few ulp); J v at the
difference quotient's noise, 1e-6, as in test_residual_gpu.py."""
import dataclasses

import numpy as np
import pytest

from conftest import device
from oracle.oracle import OracleProblem
from test_residual_gpu import TOL, _rel, _state
from test_residual_windows_gpu import _zoned

pytestmark = pytest.mark.gpu


def _several(conn, zone, n):
    """How many nodes touch several of the zones 0 and 1."""
    on = np.zeros((2, n), dtype=bool)
    for z in (0, 1):
        on[z, conn[zone == z].reshape(-1)] = True
    return int((on[0] & on[1]).sum())


def _problem(count):
    """The slice with two zones and count nodes, or one or two more, that touch both; "large": beyond 65 535 nodes, three zones."""
    from fvmpor_amd.problems import slice2d_bc_problem, slice2d_problem
    if count == "large":
        return _zoned(slice2d_bc_problem(nx=331, ny=201), 3)
    prob = _zoned(slice2d_problem(nx=37, ny=15), 2)
    zone = np.zeros(prob.mesh.n_elements, dtype=np.int32)
    got = 0
    for e in np.random.default_rng(count).permutation(len(zone)):
        if got >= count:
            break
        zone[e] = 1
        got = _several(prob.mesh.conn, zone, prob.mesh.n_nodes)
    assert count <= got <= count + 2
    return dataclasses.replace(prob, ezone=zone)


@pytest.mark.parametrize("count", [0, 1, 253, 254, 255, 256, 257, 500, "large"])
def test_residual_and_jv(count):
    import torch
    from fvmpor_amd.lib import Context
    prob = _problem(count)
    dev = device()
    ctx = Context(prob)
    psi, psip = _state(prob, 3)
    op = OracleProblem(prob)
    tp, tpp = torch.tensor(psi, device=dev), torch.tensor(psip, device=dev)
    F, Jv = torch.empty_like(tp), torch.empty_like(tp)
    v = np.random.default_rng(9).normal(size=len(psi))
    tv = torch.tensor(v, device=dev)
    torch.cuda.synchronize()
    wf, _ = ctx.get_upwind()  # averaged weights to begin with
    op.set_weights(wf)
    ctx.residual(0.0, tp, tpp, F)
    ctx.synchronize()
    assert _rel(F.cpu().numpy(), op.residual(0.0, psi, psip), op.flux_scale()) <= TOL
    ctx.begin_step(0.0, tp, tpp)
    wf, _ = ctx.get_upwind()
    op.set_weights(wf)
    Fc = op.residual(0.0, psi, psip)
    sig = np.sqrt(2.0 ** -52) * np.linalg.norm(psi) / np.linalg.norm(v)
    Jc = (op.residual(0.0, psi + sig * v, psip + 2.5 * (sig * v)) - Fc) / sig
    for tile in (None, 512):
        if tile:
            ctx.set_residual_launch(0, tile, True)
        ctx.residual(0.0, tp, tpp, F)
        ctx.jv(0.0, tp, tpp, F, 2.5, tv, Jv)
        ctx.synchronize()
        assert _rel(F.cpu().numpy(), Fc, op.flux_scale()) <= TOL, tile
        assert np.abs(Jv.cpu().numpy() - Jc).max() <= 1e-6 * np.abs(Jc).max(), tile


@pytest.mark.parametrize("count", [0, 255, 257, 500])
def test_jacobian_forms_agree(count):
    """The element-local Jacobian, whose node pass has the same list, against the coloured form: the bar of
    test_jacobian_shapes_gpu.py, 1e-4 of a row's largest entry (the quotients' rounding noise)."""
    import torch
    from fvmpor_amd.lib import Context, JACOBIAN_COLOURED, JACOBIAN_ELEMENT, PRECON_JACOBI, PRECON_BJILU0_F32
    prob = _problem(count)
    ctx = Context(prob)
    psi, psip = _state(prob, 3)
    y, yp = (torch.tensor(a, device=device()) for a in (psi, psip))
    F0, ewt = torch.empty_like(y), 1.0 / (1e-6 * y.abs() + 1e-6)
    torch.cuda.synchronize()
    ctx.begin_step(0.0, y, yp)
    ctx.residual(0.0, y, yp, F0)
    n, conn = prob.mesh.n_nodes, prob.mesh.conn.astype(np.int64)
    key = np.unique(np.concatenate([conn[:, a] * n + conn[:, b] for a in range(3) for b in range(3)]))
    J = ctx.jacobian()
    vals = []
    for mode, precon in ((JACOBIAN_COLOURED, PRECON_JACOBI), (JACOBIAN_ELEMENT, PRECON_JACOBI),
                         (JACOBIAN_ELEMENT, PRECON_BJILU0_F32)):
        ctx.set_jacobian_mode(mode)
        assert ctx.precon_setup(0.0, 12.0, 0.05, y, yp, F0, ewt, precon) == 0
        vals.append(J.get_values(len(key)))
    rows, rowmax = key // n, np.zeros(n)
    np.maximum.at(rowmax, rows, np.abs(vals[0]))
    for v in vals[1:]:
        assert (np.abs(v - vals[0]) / rowmax[rows]).max() < 1e-4
