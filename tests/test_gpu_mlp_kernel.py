"""The network in one kernel against the same network layer by layer through
the matrix-core product: identical bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _layered(net, x):
    """The forward pass that training keeps its activations from."""
    return net.forward(x, keep=True)


@pytest.mark.parametrize('n', [1, 15, 16, 17, 47, 48, 49, 191, 192, 193, 385, 4096, 70_001])
def test_rows_equal_the_layered_pass(n):
    import torch
    from xtrack_amd.surrogate import MLP
    net = MLP(seed=n)
    for b in net.b:
        b.normal_(generator=torch.Generator(device='cuda').manual_seed(n))
    x = torch.randn((n, 16), generator=torch.Generator().manual_seed(n)).cuda()
    assert torch.equal(net.forward(x), _layered(net, x))
    # a view that starts off a 16-byte boundary, and transposed storage
    buf = torch.empty(16 * n + 1, device='cuda')
    buf[1:] = x.reshape(-1)
    assert torch.equal(net.forward(buf[1:].view(n, 16)), _layered(net, x))
    assert torch.equal(net.forward(x.t().contiguous().t()), _layered(net, x))


@pytest.mark.parametrize('n', [1, 100, 65_536, 65_537])
def test_prediction_with_normalisation(n):
    import torch
    from xtrack_amd.surrogate import MLP
    net = MLP(seed=3)
    g = torch.Generator().manual_seed(n)
    x = (torch.randn((n, 16), generator=g) * torch.logspace(-3, 2, 16)).cuda()
    net.x_mean = torch.randn(16, generator=g).cuda()
    net.x_std = (torch.rand(16, generator=g) + 0.1).cuda()
    net.y_mean, net.y_std = 6.25, 1.7
    want = _layered(net, (x - net.x_mean) / net.x_std) * net.y_std + net.y_mean
    assert torch.equal(net.predict(x), want)


def test_infinities_and_nan():
    import torch
    from xtrack_amd.surrogate import MLP
    net = MLP(seed=4)
    x = torch.randn((64, 16), generator=torch.Generator().manual_seed(1)).cuda()
    x[3, 2], x[7, 15], x[20, 0] = float('inf'), float('-inf'), float('nan')
    a, b = net.forward(x), _layered(net, x)
    assert np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)


def test_other_networks_keep_the_layered_pass():
    import torch
    from xtrack_amd._native import NativeError
    from xtrack_amd.surrogate import MLP
    x = torch.randn((33, 16), generator=torch.Generator().manual_seed(2)).cuda()
    net = MLP(sizes=(16, 64, 1), seed=5)
    assert torch.equal(net.forward(x), _layered(net, x))
    with pytest.raises(NativeError):      # as the products refuse it
        MLP(seed=5).forward(x[:0])
