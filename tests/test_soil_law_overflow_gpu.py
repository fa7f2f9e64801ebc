"""A node so dry that (alpha |h|)^n overflows: its saturation and relative permeability
are S_r and 0, as the oracle's, so that the residual of its neighbours stays finite.
Its own capacity (inf / inf in the law's own order) is NaN in both.  The neighbours
see fluxes of the dry head's size and the other nodes see none, so each group is held
to the residual's bar, 1e-12, of its own largest value."""
import numpy as np
import pytest

from conftest import device
from oracle.oracle import OracleProblem
from test_residual_gpu import _state
from test_residual_windows_gpu import _zoned

pytestmark = pytest.mark.gpu


def _problem(which):
    from fvmpor_amd.problems import box3d_problem, slice2d_bc_problem, slice2d_problem
    if which == "slice":
        return slice2d_problem(nx=37, ny=15)
    if which == "box zones":
        return _zoned(box3d_problem(nx=9, ny=8, nz=7), 3)
    return _zoned(slice2d_bc_problem(nx=331, ny=201), 2)  # beyond 65 535 nodes the soil law is a pass of its own


@pytest.mark.parametrize("which", ["slice", "box zones", "slice over 65 535"])
def test_neighbours_stay_finite(which):
    import torch
    from fvmpor_amd.lib import Context
    prob = _problem(which)
    dev = device()
    ctx = Context(prob)
    psi, psip = _state(prob, 3)
    n = len(psi)
    dry = np.array([n // 3, n // 2 + 5])
    wet = psi.copy()
    psi[dry] = -1e298
    near = np.zeros(n, dtype=bool)
    near[prob.mesh.conn[np.isin(prob.mesh.conn, dry).any(axis=1)].ravel()] = True
    op = OracleProblem(prob)
    tp, tw, tpp = (torch.tensor(a, device=dev) for a in (psi, wet, psip))
    F = torch.empty_like(tp)
    torch.cuda.synchronize()
    for upwind in (False, True):
        if upwind:
            ctx.begin_step(0.0, tw, tpp)
        wf, _ = ctx.get_upwind()
        op.set_weights(wf)
        Fc = op.residual(0.0, psi, psip)
        for tile in (128, 512) if upwind else (128,):
            ctx.set_residual_launch(0, tile, True)
            ctx.residual(0.0, tp, tpp, F)
            ctx.synchronize()
            Fg = F.cpu().numpy()
            assert np.array_equal(np.isnan(Fg), np.isnan(Fc)), (upwind, tile)
            for group in (near, ~near):
                ok = group & ~np.isnan(Fc)
                assert np.abs(Fg[ok] - Fc[ok]).max() <= 1e-12 * np.abs(Fc[ok]).max(), (upwind, tile)
        assert np.isnan(Fc).sum() == len(dry)
