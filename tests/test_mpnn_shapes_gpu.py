"""The network's kernels at the sizes where they change course: node counts around
a wavefront's 32 and a workgroup's 128 nodes, neighbour lists that are empty, end
inside and at the edges of the groups of eight, and run past the two groups
fetched ahead, one layer and eight, several tiles per workgroup, and features at an
address that is only float-aligned.  One layer on whole numbers has to match the
reference bit for bit; gradients as in test_mpnn_gpu.py (2e-2 per tensor: one-unit
flips of BF16 roundings)."""
import numpy as np
import pytest

from conftest import device
from oracle import mpnn_ref as R
from test_mpnn_gpu import _params, _rel

pytestmark = pytest.mark.gpu


def _graph(n, degrees, seed):
    """A symmetric graph of n nodes whose first nodes have the given degrees (as far as n allows)."""
    rng = np.random.default_rng(seed)
    sets = [set() for _ in range(n)]
    for i in range(n - 1):
        want = degrees[i % len(degrees)]
        far = rng.permutation(np.arange(i + 1, min(n, i + 90)))
        for j in far[:max(0, want - len(sets[i]))]:
            sets[i].add(int(j))
            sets[j].add(i)
    ia = np.concatenate([[0], np.cumsum([len(s) for s in sets])]).astype(np.int32)
    return ia, np.array([j for s in sets for j in sorted(s)], dtype=np.int32)


CASES = [(1, [0], 3), (2, [1], 1), (31, [0, 1], 2), (33, [8, 9, 10], 3), (127, [14, 15, 16, 17], 3),
         (129, [24, 25, 40], 8), (1000, [0, 3, 7, 12, 13], 1), (140001, [4, 14, 6], 2)]


def _whole_number_params(seed):
    """One layer of few, small whole weights: every sum is exact in FP32 (24 bits hold them in
    any order) and no mean comes near a BF16 rounding boundary by less than FP32 resolves, so
    device and reference have the same bits."""
    rng = np.random.default_rng(seed)

    def sparse(shape, per):
        w = np.zeros(shape)
        for c in range(shape[1]):
            w[rng.choice(shape[0], per, replace=False), c] = rng.choice([-1.0, 1.0], per)
        return w

    p = {"We": np.abs(sparse((R.F_IN, R.HIDDEN), 3)), "be": rng.integers(-2, 3, R.HIDDEN).astype(float)}
    p.update({"W1_0": sparse((R.HIDDEN, R.HIDDEN), 4), "W2_0": sparse((R.HIDDEN, R.HIDDEN), 4),
              "b_0": rng.integers(-2, 3, R.HIDDEN).astype(float)})
    p.update({"Wd": sparse((R.HIDDEN, 1), 4), "bd": np.array([3.0])})
    return p


@pytest.mark.parametrize("n,degrees", [c[:2] for c in CASES])
def test_one_layer_is_exact_on_whole_numbers(n, degrees):
    import torch
    from fvmpor_amd.lib import Mpnn, mpnn_pack
    dev = device()
    ia, ja = _graph(n, degrees, n)
    X = np.random.default_rng(n).integers(0, 4, (n, R.F_IN)).astype(np.float32)
    p = _whole_number_params(n)
    m = Mpnn(ia, ja, layers=1)
    m.set_params(mpnn_pack(p, 1))
    flat = torch.empty(n * R.F_IN + 1, dtype=torch.float32, device=dev)
    xd = flat[1:]  # float-aligned only
    xd.copy_(torch.tensor(X.ravel(), device=dev))
    y = torch.empty(n, dtype=torch.float32, device=dev)
    torch.cuda.synchronize()
    m.forward(xd, y)
    m.synchronize()
    yr, _ = R.forward(p, X.astype(np.float64), ia, ja, 1)
    np.testing.assert_array_equal(y.cpu().numpy(), yr.astype(np.float32))


@pytest.mark.parametrize("n,degrees,layers", CASES)
def test_gradients(n, degrees, layers):
    import torch
    from fvmpor_amd.lib import Mpnn, mpnn_pack, mpnn_unpack
    dev = device()
    ia, ja = _graph(n, degrees, n)
    rng = np.random.default_rng(n)
    X = rng.normal(size=(n, R.F_IN)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    p = _params(layers, 5)
    m = Mpnn(ia, ja, layers=layers)
    m.set_params(mpnn_pack(p, layers))
    xd, td = torch.tensor(X, device=dev), torch.tensor(t, device=dev)
    torch.cuda.synchronize()
    loss = m.loss_grad(xd, td)
    g = m.get_grads()
    yr, cache = R.forward(p, X.astype(np.float64), ia, ja, layers)
    gr = R.backward(p, cache, yr, t.astype(np.float64), ia, ja, layers)
    gd = mpnn_unpack(g, layers)
    for k in gr:
        # a gradient that cancels to nothing has no relative error
        if np.linalg.norm(gr[k]) > 1e-6:
            assert _rel(gd[k], gr[k]) <= 2e-2, k
    # fixed-order sums: the same inputs give the same bits
    assert m.loss_grad(xd, td) == loss and np.array_equal(m.get_grads(), g)
