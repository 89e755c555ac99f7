"""Which library calls the network's methods make: the library's entry points
are recorded and CPU tensors stand for device tensors, so that the choice
between the library's steps and the layered pass is seen without a GPU."""
import pytest
import torch

from xtrack_amd import surrogate


class _Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 4096 if name == 'xtm_mlp_workspace_bytes' else 0
        return call

    def names(self):
        out = [n for n, _ in self.calls if n != 'xtm_mlp_workspace_bytes']
        self.calls.clear()
        return out


@pytest.fixture
def lib(monkeypatch):
    rec = _Recorder()
    monkeypatch.setattr(surrogate._native, 'load', lambda: rec)
    monkeypatch.setattr(surrogate, '_stream', lambda dev: None)
    monkeypatch.setattr(torch.Tensor, 'is_cuda', property(lambda t: True))
    return rec


def _net(sizes=surrogate.SIZES):
    return surrogate.MLP(device='cpu', sizes=sizes)


def test_layers_beyond_the_limits_of_the_step(lib):
    net = _net((4, 2 ** 20 + 1, 1))
    net.forward(torch.zeros(1, 4), keep=True)
    assert lib.names() == ['xtm_gemm_bf16'] * 2
    _net((4, 32, 1)).forward(torch.zeros(1, 4), keep=True)
    assert lib.names() == ['xtm_mlp_train_forward']


@pytest.mark.parametrize('shape', [(2, 16, 3), (16,), (3, 16, 16)], ids=str)
@pytest.mark.parametrize('keep', [False, True])
def test_inputs_that_are_not_rows_are_refused(lib, shape, keep):
    for sizes in (surrogate.SIZES, (16, 32, 1)):
        with pytest.raises(ValueError, match='2-D'):
            _net(sizes).forward(torch.zeros(shape), keep=keep)
    assert not lib.names()


def test_prediction_with_scalar_and_tensor_normalisation(lib):
    """Means and deviations that broadcast as tensor operations do, numbers
    and device scalars among them."""
    x = torch.zeros(5, 16)
    net = _net()
    net.x_mean, net.x_std = torch.zeros(16), torch.ones(16)
    net.predict(x)
    assert lib.names() == ['xtm_mlp_forward']
    for mean, std in ((0.0, 1.0), (torch.zeros(()), torch.ones(())), (torch.zeros(16), 2.0)):
        net.x_mean, net.x_std = mean, std
        assert net.predict(x).shape == (5,)
        (name, args), = [c for c in lib.calls if c[0] == 'xtm_mlp_forward']
        assert args[1] is None and args[8] == 0      # normalised before and after
        lib.names()
    net.x_mean, net.x_std = torch.zeros(16), torch.ones(16)
    net.y_mean, net.y_std = torch.zeros(()), torch.ones(())
    assert net.predict(x).shape == (5,)
    (name, args), = [c for c in lib.calls if c[0] == 'xtm_mlp_forward']
    assert args[8] == 0


@pytest.mark.parametrize('change', ['strides', 'dtype', 'shape'])
def test_weights_changed_between_the_passes(lib, change):
    """The backward pass looks at the weights that it is given."""
    net = _net((16, 32, 32, 1))
    x, dout = torch.zeros(7, 16), torch.ones(7)
    net.forward(x, keep=True)
    net.backward(dout)
    assert lib.names() == ['xtm_mlp_train_forward', 'xtm_mlp_train_backward']
    net.forward(x, keep=True)
    lib.names()
    w = net.W[1]
    net.W[1] = {'strides': lambda: w.t().contiguous().t(), 'dtype': lambda: w.double(),
                'shape': lambda: w[:, :8].contiguous()}[change]()
    if change == 'shape':
        with pytest.raises(ValueError, match='inner dimensions'):
            net.backward(dout)
        return
    gw, gb = net.backward(dout)
    assert lib.names() == ['xtm_gemm_bf16'] * 5
    assert [tuple(g.shape) for g in gw] == [(16, 32), (32, 32), (32, 1)]
    assert [tuple(g.shape) for g in gb] == [(32,), (32,), (1,)]


def test_adam_with_a_tensor_learning_rate(lib):
    """A learning rate on the device (changed between graph replays) is not
    read by the host."""
    net = _net((4, 8, 1))
    g = [torch.ones_like(w) for w in net.W], [torch.ones_like(b) for b in net.b]
    net.adam_step(*g, lr=1e-3)
    assert lib.names() == ['xtm_adam_step']
    before = [p.clone() for p in net.W + net.b]
    net.adam_step(*g, lr=torch.tensor(0.25))
    assert not lib.names()
    # the first recorded step changed no moment: m = 0.1, v = 0.001, t = 2
    step = 0.25 * (0.1 / (1 - 0.9 ** 2)) / ((0.001 / (1 - 0.999 ** 2)) ** 0.5 + 1e-8)
    for p, q in zip(net.W + net.b, before):
        assert torch.allclose(q - p, torch.full_like(p, step), rtol=1e-4, atol=1e-6)
