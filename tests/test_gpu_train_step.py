"""The library's training step against the same step product by product:
products and their gradients bit for bit, column sums and Adam within the
rounding of their sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _net(sizes, seed):
    import torch
    from xtrack_amd.surrogate import MLP
    net = MLP(sizes=sizes, seed=seed)
    g = torch.Generator(device='cuda').manual_seed(seed)
    for b in net.b:
        b.normal_(std=0.1, generator=g)
    return net


@pytest.mark.parametrize('sizes', [(16, 256, 256, 256, 1), (16, 64, 48, 32, 1), (7, 33, 1),
                                   (5, 1)], ids=str)
@pytest.mark.parametrize('n', [1, 17, 255, 1024, 4097])
def test_gradients_equal_the_layered_step(sizes, n):
    import torch
    net = _net(sizes, n)
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, sizes[0]), generator=g).cuda()
    dout = (torch.randn(n, generator=g) / n).cuda()
    out = net.forward(x, keep=True)
    gw, gb = net.backward(dout)
    assert len(net._cache) == 3
    want = net._forward_layers(x, True)
    ww, wb = net._backward_layers(dout)
    assert torch.equal(out, want)
    for a, b in zip(gw, ww):
        assert torch.equal(a, b)
    for a, b in zip(gb, wb):
        # two sums of n FP32 terms: each within n 2^-24 of the terms' sum
        scale = float(b.abs().max()) + float(dout.abs().sum())
        assert torch.allclose(a, b, rtol=0, atol=max(n, 16) * 2.0 ** -23 * scale)


def test_other_networks_take_the_layered_step():
    import torch
    x = torch.randn((9, 16), generator=torch.Generator().manual_seed(1)).cuda()
    deep = _net((16,) * 10 + (1,), 2)
    deep.forward(x, keep=True)
    assert len(deep._cache) == 2
    gw, gb = deep.backward(torch.ones(9, device='cuda'))
    assert len(gw) == len(gb) == 10
    wide = _net((16, 32, 3), 3)
    assert wide.forward(x).shape == (9,)


@pytest.mark.parametrize('steps', [1, 2, 7])
def test_adam_equals_its_definition(steps):
    import torch
    net = _net((16, 64, 48, 1), 4)
    ref = [p.double().cpu().numpy() for p in net.W + net.b]
    m, v = [0 * r for r in ref], [0 * r for r in ref]
    g = torch.Generator().manual_seed(steps)
    for t in range(1, steps + 1):
        gw = [torch.randn(w.shape, generator=g).cuda() for w in net.W]
        gb = [torch.randn(b.shape, generator=g).cuda() for b in net.b]
        net.adam_step(gw, gb, lr=1e-2)
        for k, gr in enumerate(gw + gb):
            d = gr.double().cpu().numpy()
            m[k] = 0.9 * m[k] + 0.1 * d
            v[k] = 0.999 * v[k] + 0.001 * d * d
            ref[k] = ref[k] - 1e-2 * (m[k] / (1 - 0.9 ** t)) / (np.sqrt(v[k] / (1 - 0.999 ** t))
                                                               + 1e-8)
    for p, r in zip(net.W + net.b, ref):
        # a step moves a weight by about lr; 1 - 0.999^t in FP32 is good to
        # 2^-24 / (0.001 t) = 6e-5, half of it in the square root
        assert np.abs(p.double().cpu().numpy() - r).max() < steps * (1e-2 * 1e-4 + 5e-7)
