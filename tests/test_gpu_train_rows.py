"""The training step at row counts where the column sums are cut, against
the same step product by product and 64-bit sums."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('sizes', [(16, 256, 256, 256, 1), (5, 33, 17, 1)], ids=str)
@pytest.mark.parametrize('n', [1023, 1025, 2049, 16_384, 65_537])
def test_gradients_of_large_batches(sizes, n):
    import torch
    from xtrack_amd.surrogate import MLP
    net = MLP(sizes=sizes, seed=n)
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, sizes[0]), generator=g).cuda()
    dout = (torch.randn(n, generator=g) / n).cuda()
    out = net.forward(x, keep=True)
    gw, gb = net.backward(dout)
    want = net._forward_layers(x, True)
    ww, wb = net._backward_layers(dout)
    assert torch.equal(out, want)
    for a, b in zip(gw, ww):
        assert torch.equal(a, b)
    for a, b in zip(gb, wb):
        # the layered sums of n FP32 terms: within n 2^-24 of the terms' sum
        scale = float(b.abs().max()) + float(dout.abs().sum())
        assert torch.allclose(a, b, rtol=0, atol=n * 2.0 ** -23 * scale)
    # the output layer's bias gradient is the sum of dout, rounded once from
    # a 64-bit sum: within one unit of its last place
    exact = float(dout.double().sum())
    assert abs(float(gb[-1]) - exact) <= 2.0 ** -23 * abs(exact) + 1e-12
