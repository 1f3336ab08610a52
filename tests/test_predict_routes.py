"""Which calls the one-call inference of contraction layers takes, on the CPU: the library call is replaced by a recorder, so a
call that reaches it has been routed, and one that does not runs the layer path (replaced as well)."""

import pytest
import torch

from hgq2_amd import _lib, core, ops
from hgq2_amd.config import LayerConfigScope
from hgq2_amd.core import Layer, Sequential
from hgq2_amd.layers import QDense, QEinsumDense
from hgq2_amd.layers.core import _stack, dense, einsum_dense
from hgq2_amd.quantizer.internal import FixedPointQuantizerKBI, FixedPointQuantizerKIF


@pytest.fixture
def routed(monkeypatch):
    """Descriptions (K, N, activation) of the layers that library calls were asked for, call by call."""
    calls = []

    def predict(x, descs, n, rows, n_out):
        calls.append([(d.K, d.N, d.act) for d in descs[:n]])
        return torch.zeros((rows, n_out))

    def layer_path(x, iq, qkernel, qbias, act, training, oq=None, out_shape=None):
        K, N = qkernel.shape
        x = x if iq is None else iq(x, training=training)
        y = x.reshape(-1, K)[:, :1] * 0.0 + torch.zeros(N)
        return y, act == 'relu', None, False

    monkeypatch.setattr(_stack, '_plain_input', lambda x: type(x) is torch.Tensor and x.numel() > 0)
    monkeypatch.setattr(ops, 'dense_stack_predict', predict)
    for module in (dense, einsum_dense):
        monkeypatch.setattr(module, 'dense_contraction', layer_path)
    monkeypatch.setattr(core, '_default_device', torch.device('cpu'))
    # a quantizer hands its input on
    for kind in (FixedPointQuantizerKBI, FixedPointQuantizerKIF):
        monkeypatch.setattr(kind, 'call', lambda self, inputs, training=None: inputs)
    return calls


def _dense(units, k_in, **kw):
    with LayerConfigScope(enable_ebops=False):
        layer = QDense(units, **kw)
    layer.build((None, k_in))
    layer.built = True
    return layer


def _einsum(equation, output_shape, input_shape, iq=True, **kw):
    with LayerConfigScope(enable_ebops=False, enable_iq=iq):
        layer = QEinsumDense(equation, output_shape, **kw)
    layer.build(input_shape)
    layer.built = True
    return layer


def linear(t):
    return 2.0 * t + 1.0


def _kinds():
    return [('dense', lambda **kw: _dense(3, 4, **kw), (5, 4)),
            ('einsum', lambda **kw: _einsum('bpf,fh->bph', (2, 3), (None, 2, 4), **kw), (5, 2, 4))]


@pytest.mark.parametrize('kind', [0, 1])
def test_activations_that_are_not_the_kernels_own_are_applied(kind, routed):
    _, make, shape = _kinds()[kind]
    x = torch.ones(shape)
    changed = make()
    changed.activation = torch.sigmoid
    for layer, want in ((make(activation=linear), 1.0), (changed, 0.5), (make(activation='tanh'), 0.0)):
        for net in (layer, Sequential([layer])):
            with torch.no_grad():
                y = net(x, training=False)
            assert torch.equal(y, torch.full_like(y, want)) and not routed
    for act, code in ((None, _lib.ACT_NONE), ('linear', _lib.ACT_NONE), ('relu', _lib.ACT_RELU), (torch.relu, _lib.ACT_RELU)):
        with torch.no_grad():
            make(activation=act)(x, training=False)
        assert routed.pop()[0][2] == code and not routed


class _Split(Layer):
    def call(self, x, training=None):
        return [x, x + 1.0] if self.name == 'list' else (x, x + 1.0)


class _Join(Layer):
    def call(self, xs, training=None):
        return xs[0] + xs[1]


@pytest.mark.parametrize('kind', ['list', 'tuple'])
def test_lists_and_tuples_pass_between_the_layers_of_a_sequence(kind, routed):
    net = Sequential([_Split(name=kind), _Join(), _dense(3, 4), _Split(name=kind)])
    x = torch.ones((5, 4))
    with torch.no_grad():
        a, b = net(x, training=False)
        assert len(routed) == 1 and torch.equal(b - a, torch.ones((5, 3)))
        assert torch.equal(Sequential([_Join()])([x, x], training=False), 2 * x)
    assert torch.equal(Sequential([_Split(name=kind), _Join()])(x, training=False), 2 * x + 1)


def test_inputs_that_are_no_whole_number_of_rows_stay_refused(routed):
    layer = _einsum('bpf,fh->bph', (2, 3), (None, 2, 4), iq=False)
    for shape in ((2, 9), (2, 3, 3), (2, 11), (1, 7)):
        for grad in (True, False):
            with torch.set_grad_enabled(grad), pytest.raises(RuntimeError):
                layer(torch.ones(shape), training=False)
    with torch.no_grad():
        layer(torch.ones((2, 2, 4)), training=False)
    assert routed == [[(4, 3, _lib.ACT_NONE)]]


def test_a_single_value_without_axes(routed):
    layer = _dense(3, 1)
    for grad in (True, False):
        with torch.set_grad_enabled(grad):
            assert layer(torch.tensor(2.0), training=False).shape == (3,)
    assert not routed


@pytest.mark.parametrize('place', ['_iq', '_kq', '_bq', '_oq'])
@pytest.mark.parametrize('inner', [False, True])
def test_replaced_quantizer_calls_run(place, inner, routed):
    with LayerConfigScope(enable_oq=True):
        layer = _dense(3, 4)
    q, seen = getattr(layer, place), []
    target = q.quantizer if inner else q
    target.call = lambda x, training=None: seen.append(place) or x
    x = torch.ones((5, 4))
    for net in (layer, Sequential([layer])):
        with torch.no_grad():
            net(x, training=False)
    assert seen == [place, place] and not routed
