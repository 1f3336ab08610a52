"""The one-call inference of consecutive QDense layers against the layer-by-layer path.

Quantized operands: sums of fixed-point products that fit 24 bits come out the same in any order, so outputs are equal bit
for bit; the un-quantized case (no input quantizer) allows the rounding of two fp32 summation orders."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from hgq2_amd import _lib, core, ops  # noqa: E402
from hgq2_amd.config import LayerConfigScope, QuantizerConfigScope  # noqa: E402
from hgq2_amd.core import Sequential  # noqa: E402
from hgq2_amd.layers import QDense, QEinsumDense  # noqa: E402
from hgq2_amd.layers.core import _stack  # noqa: E402
from hgq2_amd.utils.minmax_trace import trace_minmax  # noqa: E402


def _net(dims, datalane='kif', over='WRAP', weights='SAT_SYM', rnd='RND', iq=True, bias=True, **kw):
    with QuantizerConfigScope(place='all', default_q_type='kbi', overflow_mode=weights, round_mode=rnd), \
            QuantizerConfigScope(place='datalane', default_q_type=datalane, overflow_mode=over, round_mode=rnd, **kw), \
            LayerConfigScope(enable_ebops=False, enable_iq=iq):
        net = Sequential([QDense(d, activation='relu' if n % 2 == 0 else None, use_bias=bias) for n, d in enumerate(dims[1:])])
    core.set_default_device('cuda')
    return net


def _layerwise(net, x, monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(_stack, '_plain_input', lambda x: False)
        with torch.no_grad():
            return net(x)


def _spread(net, g):
    """Bit-widths and weights that differ from entry to entry; some words empty."""
    for name, p in net.named_parameters():
        if name.endswith(('_var_b', '_var_f')):
            p.data += torch.randint(-3, 2, p.shape, generator=g).float().to(p.device)
        elif name.endswith(('kernel', 'bias')):
            p.data.copy_(torch.randn(p.shape, generator=g).to(p.device) * 0.3)


@pytest.mark.parametrize('dims,rows', [((16, 64, 32, 32, 5), 1), ((1, 1), 3), ((17, 33, 64, 2), 63), ((64,) * 8, 65), ((3, 5, 31, 32, 33, 16), 130),
                                       ((30, 20), 40000), ((6, 33, 64, 5), 70001), ((64,) * 9, 70), ((8, 65, 10), 1), ((100, 130, 31, 77), 257), ((256, 512, 128, 10), 1031),
                                       ((65, 3, 64), 20)])
@pytest.mark.parametrize('kw', [dict(), dict(datalane='kbi', over='SAT', weights='SAT', rnd='RND_CONV'), dict(over='SAT_SYM', rnd='TRN', bias=False),
                                dict(homogeneous_axis=(0, 1), heterogeneous_axis=None)])
def test_equals_the_layers_one_by_one(dims, rows, kw, monkeypatch):
    g = torch.Generator().manual_seed(rows + len(dims))
    net = _net(dims, **kw)
    x = torch.randn((max(rows, 200), dims[0]), generator=g).cuda()
    net(x)
    _spread(net, g)
    trace_minmax(net, x)
    taken, inner = [], ops.dense_stack_predict
    monkeypatch.setattr(ops, 'dense_stack_predict', lambda *a: taken.append(a[2]) or inner(*a))
    with torch.no_grad():
        got = net(x[:rows])
    want = _layerwise(net, x[:rows], monkeypatch)
    assert taken and got.shape == want.shape and torch.equal(got, want)
    with torch.no_grad():  # the variables are read again on every call
        net.layers[0]._kernel.mul_(0.5)
        assert torch.equal(net(x[:rows].t().contiguous().t()), _layerwise(net, x[:rows], monkeypatch))


@pytest.mark.parametrize('K,N', [(17, 33), (100, 70)])
@pytest.mark.parametrize('rnd', ['RND', 'RND_CONV'])
def test_wrapping_weight_quantizers(K, N, rnd, monkeypatch):
    # each weight's own integer bits put its last place elsewhere: the sums no longer fit 24 bits and their order shows
    g = torch.Generator().manual_seed(K)
    net = _net((K, N), weights='WRAP', rnd=rnd)
    x = torch.randn((300, K), generator=g).cuda()
    net(x)
    _spread(net, g)
    trace_minmax(net, x)
    taken, inner = [], ops.dense_stack_predict
    monkeypatch.setattr(ops, 'dense_stack_predict', lambda *a: taken.append(a[2]) or inner(*a))
    with torch.no_grad():
        got = net(x)
    want = _layerwise(net, x, monkeypatch)
    magnitude = x.abs().max() * net.layers[0]._kernel.abs().sum(0).max() + 1.0
    assert taken and (got - want).abs().max() <= 2 * (K + 8) * 2.0**-24 * magnitude


def test_non_finite_samples_stay_in_their_rows(monkeypatch):
    net = _net((6, 40, 50, 30, 4), over='SAT')
    x = torch.randn((300, 6), generator=torch.Generator().manual_seed(1)).cuda()
    net(x)
    x[7, 2], x[70, 1], x[200, 5] = float('nan'), float('inf'), float('-inf')
    with torch.no_grad():
        got = net(x)
    want = _layerwise(net, x, monkeypatch)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))


def test_without_input_quantizers(monkeypatch):
    for dims in ((12, 24, 36), (12, 240, 36)):
        net = _net(dims, iq=False)
        x = torch.randn((99, 12), generator=torch.Generator().manual_seed(2)).cuda()
        net(x)
        with torch.no_grad():
            got = net(x)
        want = _layerwise(net, x, monkeypatch)
        assert (got - want).abs().max() <= 2 * (dims[1] + 8) * 2.0**-24 * (1 + want.abs().max()) * dims[1]


def test_takes_no_part_in_training_tracing_or_gradients(monkeypatch):
    net = _net((5, 6, 7))
    x = torch.randn((9, 5)).cuda()
    net(x)
    monkeypatch.setattr(ops, 'dense_stack_predict', lambda *a: pytest.fail('the layers have to run'))
    net(x)
    with torch.no_grad():
        net(x, training=True)
    trace_minmax(net, x)
    with torch.no_grad():
        net(x.double().float().requires_grad_(), training=True)


def test_replays_in_a_graph():
    net = _net((10, 20, 80, 5))
    x = torch.randn((50, 10), generator=torch.Generator().manual_seed(3)).cuda()
    net(x)
    side = torch.cuda.Stream()
    with torch.no_grad(), torch.cuda.stream(side):
        net(x)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = net(x)
    for s in range(3):
        x.copy_(torch.randn((50, 10), generator=torch.Generator().manual_seed(10 + s)))
        graph.replay()
        torch.cuda.synchronize()
        with torch.no_grad():
            assert torch.equal(y, net(x))


# tables over positions (as many rows as positions, or one), narrow and wide widths, with and without an output quantizer
@pytest.mark.parametrize('T,K,N,H', [(1, 5, 3, 2), (50, 48, 3, 16), (7, 64, 1, 64), (33, 70, 5, 20), (64, 96, 8, 32), (10, 17, 2, 33)])
@pytest.mark.parametrize('oq', [True, False])
@pytest.mark.parametrize('shared', [None, (0, 1)])
def test_projections_over_positions(T, K, N, H, oq, shared, monkeypatch):
    g = torch.Generator().manual_seed(T + K)
    kw = dict(homogeneous_axis=shared, heterogeneous_axis=None) if shared else {}
    with QuantizerConfigScope(place='all', default_q_type='kbi', overflow_mode='SAT_SYM'), \
            QuantizerConfigScope(place='datalane', default_q_type='kif', overflow_mode='WRAP', **kw), LayerConfigScope(enable_ebops=False):
        net = QEinsumDense('btf,fnh->btnh', output_shape=(T, N, H), bias_axes='nh', enable_oq=oq)
    core.set_default_device('cuda')
    x = torch.randn((37, T, K), generator=g).cuda()
    net(x)
    _spread(net, g)
    trace_minmax(net, x)
    taken, inner = [], ops.dense_stack_predict
    monkeypatch.setattr(ops, 'dense_stack_predict', lambda *a: taken.append(a[2]) or inner(*a))
    with torch.no_grad():
        got = net(x)
    want = _layerwise(net, x, monkeypatch)
    assert taken and torch.equal(got, want)
    with torch.no_grad():
        assert torch.equal(net(x[:1]), _layerwise(net, x[:1], monkeypatch))
        assert net(x[:0]).shape == (0, T, N, H)
        many = x.repeat(40000 // (37 * T) + 2, 1, 1)  # beyond the rows one launch takes
        assert torch.equal(net(many), _layerwise(net, many, monkeypatch))


# widths of the one-launch form and of the tiled products; samples of one bf16 part beside kernels of two (zero parts among them)
@pytest.mark.parametrize('dims', [(7, 20), (8, 20), (33, 64), (5, 40, 3), (64, 5), (7, 80), (100, 30)])
def test_infinities_as_in_a_sum_of_products(dims):
    g = torch.Generator().manual_seed(len(dims) + dims[0])
    net = _net(dims, iq=False, bias=False)
    x = torch.round(4 * torch.randn((70, dims[0]), generator=g)) / 4
    net(x.cuda())
    for layer in net.layers:
        layer._kernel.data.copy_(torch.randn(layer._kernel.shape, generator=g) * 0.3)
        layer.kq.quantizer._b.data.fill_(12.0)
    x[3, 2], x[40, 1], x[69, 0], x[10, 3] = float('inf'), float('-inf'), float('nan'), float('inf')
    want = x.double()
    for layer in net.layers:
        want = want @ layer.qkernel.detach().double().cpu()
        if layer._act_name == 'relu':
            want = torch.where(want > 0, want, torch.zeros_like(want))
    with torch.no_grad():
        got = net(x.cuda())
    got = got.cpu()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want))
    assert len(dims) > 2 or torch.isposinf(want).any()


@pytest.mark.parametrize('K,N', [(8, 5), (48, 64)])
def test_the_choice_of_matrix_instruction_holds(K, N):
    # samples of three parts against kernels of one: three rounded sums per product on the bf16 instruction, one on the fp32 one
    g = torch.Generator().manual_seed(K)
    net = _net((K, N), iq=False, bias=False)
    x = torch.randn((500, K), generator=g).cuda()
    net(x)
    lib = _lib.load()
    with torch.no_grad():
        on = net(x)
        before = lib.hgq_dense_use_bf16_parts(0)
        try:
            off = net(x)
        finally:
            lib.hgq_dense_use_bf16_parts(before)
        w = net.layers[0].qkernel.double()
        exact, magnitude = (x.double() @ w).relu(), x.abs().double() @ w.abs()
    for y in (on, off):  # any order of summation, the parts at most nine sums per product
        assert ((y - exact).abs() <= 2 * (K + 8) * 2.0**-24 * magnitude + 1e-30).all()
    assert not torch.equal(off, on)


# long contractions onto few columns or few rows: a wavefront per row, a split along k with and without a quantizer behind it,
# first, middle and last layer, output quantizer by column and by position
@pytest.mark.parametrize('dims,rows', [((3872, 10), 1), ((3872, 10), 1024), ((1025, 16), 7), ((1024, 17), 130), ((513, 3), 20000), ((700, 20, 5), 65),
                                       ((70, 1100, 33), 3), ((1030, 70, 1500, 40, 2), 200), ((2048, 512), 64), ((511, 9), 31), ((1023, 65), 12)])
def test_long_contractions(dims, rows, monkeypatch):
    g = torch.Generator().manual_seed(rows)
    net = _net(dims)
    x = torch.randn((max(rows, 200), dims[0]), generator=g).cuda()
    net(x)
    _spread(net, g)
    trace_minmax(net, x)
    taken, inner = [], ops.dense_stack_predict
    monkeypatch.setattr(ops, 'dense_stack_predict', lambda *a: taken.append(a[2]) or inner(*a))
    with torch.no_grad():
        got = net(x[:rows])
    assert taken and torch.equal(got, _layerwise(net, x[:rows], monkeypatch))


@pytest.mark.parametrize('shared', [None, (0, 1)])
@pytest.mark.parametrize('T,K,N', [(1, 2000, 8), (3, 1500, 40)])
def test_long_contractions_with_an_output_quantizer(T, K, N, shared, monkeypatch):
    kw = dict(homogeneous_axis=shared, heterogeneous_axis=None) if shared else {}
    g = torch.Generator().manual_seed(K)
    with QuantizerConfigScope(place='all', default_q_type='kbi', overflow_mode='SAT_SYM'), \
            QuantizerConfigScope(place='datalane', default_q_type='kif', overflow_mode='WRAP', **kw), LayerConfigScope(enable_ebops=False):
        net = QEinsumDense('btf,fh->bth', output_shape=(T, N), bias_axes='h', enable_oq=True)
    core.set_default_device('cuda')
    x = torch.randn((37, T, K), generator=g).cuda()
    net(x)
    _spread(net, g)
    trace_minmax(net, x)
    with torch.no_grad():
        got = net(x)
    assert torch.equal(got, _layerwise(net, x, monkeypatch))


def test_long_contractions_are_split_along_k():
    """The workspace shows the form: partial sums along k where a product has few tiles and many steps, none elsewhere."""
    lib = _lib.load()
    one = torch.ones(1, device='cuda')
    u8 = torch.ones(1, dtype=torch.uint8, device='cuda')

    def floats(rows, K, N):
        d = (_lib.StackLayer * 1)()
        d[0].w, d[0].K, d[0].N = one.data_ptr(), K, N
        d[0].kq.k, d[0].kq.i, d[0].kq.fb, d[0].kq.size, d[0].kq.inner = u8.data_ptr(), one.data_ptr(), one.data_ptr(), 1, 1
        return lib.hgq_dense_stack_workspace(d, 1, rows)

    def image(K, N):
        return (K * N + 3) // 4 * 4 + (N + 3) // 4 * 4

    for rows, K, N in ((64, 2048, 512), (1, 4096, 100), (300, 600, 20)):
        assert floats(rows, K, N) >= image(K, N) + 2 * rows * N
    for rows, K, N in ((1024, 512, 512), (64, 600, 64), (50000, 2048, 512)):
        assert floats(rows, K, N) == image(K, N)


def test_the_answer_for_a_workspace_holds_when_the_matrix_instruction_changes():
    net = _net((100, 70), bias=False)
    x = torch.randn((40, 100), generator=torch.Generator().manual_seed(8)).cuda()
    net(x)
    lib = _lib.load()
    descs = (_lib.StackLayer * 1)()
    assert _stack._layer(net.layers[0], 40, 100, x.device, descs[0], True)
    with torch.no_grad():
        want = net(x)
    floats = lib.hgq_dense_stack_workspace(descs, 1, 40)
    assert floats > 0
    y, ws = torch.empty_like(want), torch.empty(floats, device='cuda')
    before = lib.hgq_dense_use_bf16_parts(0)
    try:
        assert lib.hgq_dense_stack_workspace(descs, 1, 40) == -1
        rc = lib.hgq_dense_stack_predict(descs, 1, x.data_ptr(), y.data_ptr(), 40, ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    assert rc == 0 and torch.equal(y, want)
