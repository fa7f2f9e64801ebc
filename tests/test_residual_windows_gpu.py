"""The element-owner residual from LDS windows where it changes course: nodes of
one to eight zones (up to four fit a window's records, more take the gathering
kernel), meshes of one tile and of a partly filled last tile, the van Genuchten
pass inside and before the element kernel (65 535 nodes), both workgroup sizes,
and results in place of an input.  Against the oracle at the residual's bar, 1e-12
of the flux scale (sums of about 30 terms of that scale per node, each a few ulp);
J v at the difference quotient's noise, 1e-6, as in test_residual_gpu.py."""
import dataclasses

import numpy as np
import pytest

from conftest import device
from oracle.oracle import OracleProblem
from test_residual_gpu import TOL, _rel, _state

pytestmark = pytest.mark.gpu


def _zoned(prob, nz, seed=3):
    """The problem with nz zones, each element's drawn at random."""
    rng = np.random.default_rng(seed)
    zones = np.repeat(prob.zones[:1], nz, axis=0)
    zones[:, :3] *= rng.uniform(0.5, 2.0, (nz, 3))
    zones[:, 4] *= rng.uniform(0.8, 1.2, nz)
    zones[:, 5] = 1.0 + (zones[:, 5] - 1.0) * rng.uniform(0.8, 1.2, nz)
    return dataclasses.replace(prob, zones=zones, ezone=rng.integers(0, nz, prob.mesh.n_elements).astype(np.int32))


def _problem(which):
    from fvmpor_amd.problems import box3d_problem, slice2d_bc_problem, slice2d_problem
    name, _, n = which.partition(":")
    if name == "triangle pair":
        return slice2d_problem(nx=2, ny=2)
    if name == "slice":
        return slice2d_problem(nx=37, ny=15)
    if name == "slice zones":
        return _zoned(slice2d_problem(nx=37, ny=15), int(n))
    if name == "box zones":
        return _zoned(box3d_problem(nx=9, ny=8, nz=7), int(n))
    if name == "slice over 65 535":
        return slice2d_bc_problem(nx=331, ny=201)
    raise ValueError(which)


@pytest.mark.parametrize("which", ["triangle pair", "slice", "slice zones:2", "slice zones:5", "box zones:2",
                                   "box zones:4", "box zones:5", "box zones:8", "slice over 65 535"])
def test_residual_and_jv(which):
    import torch
    from fvmpor_amd.lib import Context
    prob = _problem(which)
    dev = device()
    ctx = Context(prob)
    psi, psip = _state(prob, 3)
    op = OracleProblem(prob)
    tp, tpp = torch.tensor(psi, device=dev), torch.tensor(psip, device=dev)
    torch.cuda.synchronize()
    ctx.begin_step(0.0, tp, tpp)
    wf, _ = ctx.get_upwind()
    op.set_weights(wf)
    Fc = op.residual(0.0, psi, psip)
    scale = op.flux_scale()
    v = np.random.default_rng(9).normal(size=len(psi))
    cj = 2.5
    sig = np.sqrt(2.0 ** -52) * np.linalg.norm(psi) / np.linalg.norm(v)
    Jc = (op.residual(0.0, psi + sig * v, psip + cj * (sig * v)) - Fc) / sig
    tv = torch.tensor(v, device=dev)
    F, Jv, cap = torch.empty_like(tp), torch.empty_like(tp), torch.empty_like(tp)
    torch.cuda.synchronize()
    for tile in (None, 64, 128, 256):
        if tile:
            ctx.set_residual_launch(0, tile, tile != 128)
        ctx.residual(0.0, tp, tpp, F)
        ctx.jv(0.0, tp, tpp, F, cj, tv, Jv)
        ctx.synchronize()
        assert _rel(F.cpu().numpy(), Fc, scale) <= TOL, tile
        assert np.abs(Jv.cpu().numpy() - Jc).max() <= 1e-6 * np.abs(Jc).max(), tile
        # in place of the direction and of the state: the same to the sums' rounding
        w, x = tv.clone(), tp.clone()
        torch.cuda.synchronize()
        ctx.jv(0.0, tp, tpp, F, cj, w, w)
        ctx.residual(0.0, x, tpp, x)
        ctx.synchronize()
        assert np.abs(w.cpu().numpy() - Jc).max() <= 1e-6 * np.abs(Jc).max(), tile
        assert _rel(x.cpu().numpy(), Fc, scale) <= TOL, tile


@pytest.mark.parametrize("soil", ["clay", "loam", "sandy_loam", "sand"])
def test_capacity_over_the_range_of_heads(soil):
    """The soil law from saturation to a dry head of 1e5 m, and at the edges of
    ln and e^x: against the same law in extended precision.  Its relative error
    is that of the exponents, |n ln(alpha |h|)| <= 40 times 2^-53 and a few like
    it, below 2e-14; 1e-13 is allowed."""
    import torch
    from fvmpor_amd.lib import Context
    from fvmpor_amd.problems import SOIL_CLASSES, slice2d_problem
    base = slice2d_problem(nx=41, ny=26)
    alpha, nv, tr, ts = SOIL_CLASSES[soil]
    zone = np.array([[1.0, 1.0, 1.0, ts, alpha, nv, tr / ts, 1e-5]])
    prob = dataclasses.replace(base, zones=zone)
    ctx = Context(prob)
    n = prob.mesh.n_nodes
    psi = -np.logspace(-12, 5, n)
    psi[:8] = [0.0, -0.0, 1.0, -5e-324, -1e-300, -1e-100, -1.0 / alpha, -1e-17]
    dev = device()
    tp, cap = torch.tensor(psi, device=dev), torch.zeros(n, dtype=torch.float64, device=dev)
    F = torch.zeros_like(cap)
    torch.cuda.synchronize()
    ctx.residual(0.0, tp, torch.zeros_like(cap), F)
    ctx.capacity(cap)
    torch.cuda.synchronize()
    h = np.where(psi < 0, psi, -1.0).astype(np.longdouble)
    a, nl, sr = np.longdouble(alpha), np.longdouble(nv), np.longdouble(tr / ts)
    m = 1 - 1 / nl
    d = (a * -h) ** nl
    se = (1 + d) ** -m
    ds = -(1 - sr) * (nl - 1) * (d / (1 + d)) * se / h
    sw = np.where(psi < 0, sr + (1 - sr) * se, 1)
    want = (ts * np.where(psi < 0, ds, 0) + np.longdouble(1e-5) * sw) * 1000
    # the node's zone weight sums the shares of its elements: 1 to rounding
    err = np.abs(cap.cpu().numpy() - want) / np.abs(want)
    print(soil, err.max())
    assert err.max() < 1e-13
