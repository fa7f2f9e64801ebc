"""The launch shape that a context is made with, on a mesh that only it suits: 2 200
hubs of 129 triangles each on five shared rims, one soil zone to a rim.  Tiles of 128
nodes export 33 024 contributions; those of 256 and more pass 65 535 and are refused,
and every tile touches five zones, one more than the window variant takes."""
import numpy as np
import pytest

from conftest import device

pytestmark = pytest.mark.gpu


def _hubs():
    from fvmpor_amd import meshgen, problems
    hubs, rims, k = 2200, 5, 129
    a = 2 * np.pi * np.arange(k) / k
    xyz = np.zeros((hubs + rims * k, 3))
    rng = np.random.default_rng(1)
    for r in range(rims):
        xyz[hubs + r * k:hubs + (r + 1) * k, 0] = 3.0 * r + np.cos(a)
        xyz[hubs + r * k:hubs + (r + 1) * k, 1] = np.sin(a)
    own = np.arange(hubs) % rims
    xyz[:hubs, 0] = 3.0 * own + rng.uniform(-0.3, 0.3, hubs)
    xyz[:hubs, 1] = rng.uniform(-0.3, 0.3, hubs)
    first = hubs + k * np.repeat(own, k)
    step = np.tile(np.arange(k), hubs)
    conn = np.stack([np.repeat(np.arange(hubs), k), first + step, first + (step + 1) % k], 1).astype(np.int32)
    n = len(xyz)
    mesh = meshgen.Mesh(2, xyz, conn, np.zeros(conn.shape, dtype=np.int32), np.zeros(n + 1, dtype=np.int32),
                        np.zeros(0, dtype=np.int32), np.zeros(len(conn), dtype=np.int32))
    alpha, m, tr, ts = problems.SOIL_CLASSES["loam"]
    zones = np.tile([1.0, 1.0, 1.0, ts, alpha, m, tr / ts, 1e-5], (rims, 1))
    zones[:, :3] *= np.linspace(0.5, 2.0, rims)[:, None]
    return problems.Problem("hubs", mesh, zones, np.repeat(own, k).astype(np.int32), np.ones(len(conn)),
                            np.array([0], dtype=np.int32), np.zeros((1, 6)), 1000.0, -0.8 - 0.1 * xyz[:, 0], 1.0, "day")


def _context():
    import torch
    from fvmpor_amd.lib import Context
    prob = _hubs()
    ctx = Context(prob)
    rng = np.random.default_rng(2)
    n = prob.mesh.n_nodes
    psi = torch.tensor(prob.psi0 + rng.uniform(-0.2, 0.2, n), device=device())
    psip = torch.tensor(rng.normal(scale=0.1, size=n), device=device())
    torch.cuda.synchronize()
    ctx.begin_step(0.0, psi, psip)
    F = torch.empty_like(psi)

    def residual():
        ctx.residual(0.0, psi, psip, F)
        ctx.synchronize()
        return F.cpu().numpy().copy()

    return ctx, psi, psip, residual


def test_the_autotuner_times_it():
    ctx, psi, psip, residual = _context()
    before = residual()
    pick = ctx.autotune(0.0, psi, psip)
    assert pick["variant"] == 0 and pick["tile_nodes"] == 128 and 0.0 < pick["residual_us"] < 1e6, pick
    # a node sums 129 elements or 880, in any order: their rounding is below 1e-13 of the largest sum
    assert np.abs(residual() - before).max() <= 1e-12 * np.abs(before).max()


def test_a_launch_without_a_tile_size_is_it():
    ctx, psi, psip, residual = _context()
    before = residual()
    for tile in (64, None):
        if tile:
            ctx.set_residual_launch(0, tile)
        else:
            ctx.set_residual_launch()
        assert np.abs(residual() - before).max() <= 1e-12 * np.abs(before).max()
