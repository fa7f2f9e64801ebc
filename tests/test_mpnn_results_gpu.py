"""What the network hands to the host without a copy of the runtime's: the loss and
the gradients of the pass before, over repeated passes, both of several networks
that share a stream, and zeros before the first pass."""
import numpy as np
import pytest

from conftest import device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,layers", [(1, 1), (130, 3), (5000, 8)])
def test_results_follow_their_own_pass(n, layers):
    import torch
    from fvmpor_amd.lib import Mpnn
    dev = device()
    i = np.arange(n)                                        # a ring
    ja = np.stack([(i - 1) % n, (i + 1) % n], 1) if n > 2 else np.zeros((n, 0))
    ja = np.sort(ja.astype(np.int32), axis=1)
    ia = np.arange(n + 1, dtype=np.int32) * ja.shape[1]
    stream = torch.cuda.Stream()
    nets = [Mpnn(ia, ja.reshape(-1), layers=layers, seed=s) for s in (1, 2)]
    g = torch.Generator(device=dev).manual_seed(3)
    x, t = torch.randn(n, 16, device=dev, generator=g), torch.randn(n, device=dev, generator=g)
    y = torch.empty(n, device=dev)
    torch.cuda.synchronize()
    for net in nets:
        net.set_stream(stream.cuda_stream)
        assert not net.get_grads().any()
    first = [(net.loss_grad(x, t), net.get_grads()) for net in nets]
    assert first[0][0] != first[1][0] and first[0][1].any() and first[1][1].any()
    for _ in range(20):                                     # every value is its own pass's, bit for bit
        for net, (loss, grad) in zip(nets, first):
            assert net.loss_grad(x, t) == loss
        for net, (loss, grad) in zip(nets, first):
            assert np.array_equal(net.get_grads(), grad)
    for net, (loss, _) in zip(nets, first):                 # the loss is the mean squared error of the output
        net.forward(x, y)
        net.synchronize()
        d = y.double().cpu().numpy() - t.double().cpu().numpy()
        assert abs(loss - (d * d).mean()) <= 1e-6 * (d * d).mean()
        before = net.get_params()
        net.adam(1e-3)                                      # Adam's first step: the moments began at zero
        grad = net.get_grads()
        step = before - net.get_params()
        moved = np.abs(grad) > 1e-4
        assert np.allclose(step[moved], 1e-3 * np.sign(grad[moved]), rtol=2e-2)
