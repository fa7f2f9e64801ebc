"""The element-local Jacobian's row sums where their form changes: workgroups of
64 rows, of fewer (two hubs whose elements do not fit the LDS together) and
without staging (one hub of more elements than the LDS holds), in both
arithmetics, against the coloured form on the same state and increments.  Both
are difference quotients with increments of sqrt(eps) size, so they agree to
the quotients' rounding noise; 1e-4 of a row's largest entry is the bar that the
two forms have on the other meshes."""
import numpy as np
import pytest

from conftest import device

pytestmark = pytest.mark.gpu


def _fans(counts, start):
    """One closed fan of triangles per count, hubs at the given node numbers, rims numbered around them."""
    from fvmpor_amd import meshgen, problems
    n = sum(counts) + len(counts)
    free = [i for i in range(n) if i not in start]
    xyz = np.zeros((n, 3))
    conn, rim = [], np.zeros(n, dtype=bool)
    for f, (c, hub) in enumerate(zip(counts, start)):
        ids, free = np.array(free[:c]), free[c:]
        a = 2 * np.pi * np.arange(c) / c
        xyz[hub, :2] = [3.0 * f, 0.0]
        xyz[ids, 0] = 3.0 * f + np.cos(a)
        xyz[ids, 1] = 0.3 * np.sin(a)
        rim[ids] = True
        conn += [[hub, ids[k], ids[(k + 1) % c]] for k in range(c)]
    conn = np.array(conn, dtype=np.int32)
    conn = np.ascontiguousarray(conn[np.argsort(conn.min(axis=1), kind="stable")])
    tags = np.zeros(conn.shape, dtype=np.int32)
    for f, nodes in enumerate(meshgen.TRI_FACES):
        tags[:, f] = rim[conn[:, list(nodes)]].all(axis=1)
    ptr = np.concatenate([[0], np.cumsum(rim)]).astype(np.int32)
    mesh = meshgen.Mesh(2, xyz, conn, tags, ptr, np.ones(rim.sum(), dtype=np.int32),
                        np.zeros(len(conn), dtype=np.int32))
    alpha, m, tr, ts = problems.SOIL_CLASSES["loam"]
    rng = np.random.default_rng(3)
    return problems.Problem("fans", mesh, np.array([[1.0, 1.0, 1.0, ts, alpha, m, tr / ts, 1e-5]]),
                            np.zeros(len(conn), dtype=np.int32), np.exp(0.3 * rng.standard_normal(len(conn))),
                            np.array([0, 3], dtype=np.int32), np.zeros((2, 6)), 1000.0,
                            -0.6 - 0.2 * xyz[:, 0], 1.0, "day")


@pytest.mark.parametrize("counts,start", [((70,), (0,)), ((1200, 1200), (0, 33)), ((2300,), (5,))])
def test_row_sums_of_every_form(counts, start):
    import torch
    from fvmpor_amd.lib import (Context, JACOBIAN_COLOURED, JACOBIAN_ELEMENT, PRECON_JACOBI, PRECON_BJILU0_F32)
    prob = _fans(counts, start)
    ctx = Context(prob)
    n = prob.mesh.n_nodes
    rng = np.random.default_rng(11)
    dev = lambda a: torch.tensor(a, dtype=torch.float64, device=device())
    y = dev(prob.psi0 + rng.uniform(-0.2, 0.2, n))
    yp = dev(rng.normal(scale=0.05, size=n))
    ctx.begin_step(0.0, y, yp)
    F0 = torch.empty_like(y)
    ctx.residual(0.0, y, yp, F0)
    ewt = 1.0 / (1e-6 * y.abs() + 1e-6)
    torch.cuda.synchronize()
    conn = prob.mesh.conn.astype(np.int64)
    key = np.unique(np.concatenate([conn[:, a] * n + conn[:, b] for a in range(3) for b in range(3)]))
    ia = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    J = ctx.jacobian()
    J.precon_block_rows(64)  # the block preconditioners hold rows of at most 64 entries within a block
    vals = {}
    for mode, precon in ((JACOBIAN_COLOURED, PRECON_JACOBI), (JACOBIAN_ELEMENT, PRECON_JACOBI),
                         (JACOBIAN_ELEMENT, PRECON_JACOBI), (JACOBIAN_ELEMENT, PRECON_BJILU0_F32)):
        ctx.set_jacobian_mode(mode)
        assert ctx.precon_setup(0.0, 12.0, 0.05, y, yp, F0, ewt, precon) == 0
        vals.setdefault((mode, precon), []).append(J.get_values(len(key)))
    col = vals[JACOBIAN_COLOURED, PRECON_JACOBI][0]
    f64 = vals[JACOBIAN_ELEMENT, PRECON_JACOBI]
    f32 = vals[JACOBIAN_ELEMENT, PRECON_BJILU0_F32][0]
    rowmax = np.repeat(np.maximum.reduceat(np.abs(col), ia[:-1]), np.diff(ia))
    e64, e32 = (np.abs(f64[0] - col) / rowmax).max(), (np.abs(f32 - col) / rowmax).max()
    print(counts, e64, e32)
    assert e64 < 1e-4 and e32 < 1e-4
    assert np.array_equal(f64[0], f64[1])
