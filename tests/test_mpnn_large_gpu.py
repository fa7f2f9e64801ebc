"""A network past 33 554 430 nodes, where row offsets take 64 bits: 32 768 copies of a
graph of 1 025 nodes (2^25 is no multiple of that, so a row taken modulo 2^25 is another
node's).  A node's sums run in its list's order, so the outputs are the small
network's bit for bit; 2 e / N is scaled by a power of two, so are the gradients' terms,
whose sums over the rows differ by FP32 rounding (4 100 additions in a chain of at most
2^-24 each, times what the terms cancel, below 32): 8e-3 of a tensor's norm."""
import numpy as np
import pytest

from conftest import device
from oracle import mpnn_ref as R
from test_mpnn_gpu import _params, _rel
from test_mpnn_shapes_gpu import _graph

pytestmark = pytest.mark.gpu


def test_copies_of_a_small_graph():
    import torch
    from fvmpor_amd.lib import Mpnn, mpnn_pack, mpnn_unpack
    dev = device()
    n, copies = 1025, 32768
    assert n * copies + 1 > 1 << 25
    ia, ja = _graph(n, [2, 1, 3], 11)
    at = np.arange(copies, dtype=np.int32)[:, None]
    IA = np.concatenate([np.zeros(1, dtype=np.int32), (ia[None, 1:] + at * np.int32(len(ja))).ravel()])
    JA = (ja[None, :] + at * np.int32(n)).ravel()
    params = mpnn_pack(_params(1, 5), 1)
    rng = np.random.default_rng(12)
    x = torch.tensor(rng.normal(size=(n, R.F_IN)).astype(np.float32), device=dev)
    t = torch.tensor(rng.normal(size=n).astype(np.float32), device=dev)
    res = []
    for a, j, k in ((ia, ja, 1), (IA, JA, copies)):
        net = Mpnn(a, j, layers=1)
        net.set_params(params)
        xs, ts, y = x.repeat(k, 1), t.repeat(k), torch.empty(n * k, dtype=torch.float32, device=dev)
        torch.cuda.synchronize()
        net.forward(xs, y)
        net.synchronize()
        loss = net.loss_grad(xs, ts)
        res.append((y.reshape(k, n), loss, mpnn_unpack(net.get_grads(), 1)))
        net.close()
    assert torch.equal(res[1][0], res[0][0].expand(copies, n))
    assert abs(res[1][1] - res[0][1]) <= 1e-12 * res[0][1]
    for k, g in res[0][2].items():
        assert _rel(res[1][2][k], g) <= 8e-3, k
