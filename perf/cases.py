"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a network (or a bare quantizer) at given sizes and one use of it:

* ``train``   - one call of the step that ``hgq2_amd.train.train_step_for`` returns: forward, loss with its EBOPs terms,
  backward, SGD update.  The inputs are resident in device memory, as in an epoch over a data set that fits there.
* ``loop``    - the same step written out by the user with the layer API (own loss expression, ``SGD``), launched eagerly.
* ``predict`` - ``model(x)`` without gradients on a model whose integer bits were calibrated by ``trace_minmax``.
* ``quantize`` - the stateless quantizer callable with its surrogate backward.
"""

from __future__ import annotations

import math

import torch

from hgq2_amd import ops
from hgq2_amd.quantizer.fixed_point_ops import get_fixed_quantizer
from hgq2_amd.train import SGD, model_loss, train_step_for
from hgq2_amd.utils import models
from hgq2_amd.utils.minmax_trace import trace_minmax

LR = 0.01
CALIBRATION = 1024  # samples a model sees in `trace_minmax` before it predicts


def listed():
    return [
        # one event through a trained network: a trigger emulation, a notebook; nothing but latency
        dict(name='dense_predict_one', net='dense', use='predict', dims='16-64-32-32-5', batch=1),
        # a small tabular set in a training loop of the user's own, with odd widths and a last, ragged batch
        dict(name='dense_loop_1000', net='dense', use='loop', dims='21-47-19-3', batch=1000),
        # the benchmark's training step: jet features, large batches
        dict(name='dense_train_16384', net='dense', use='train', dims='16-64-32-32-5', batch=16384),
        # layers beyond 64 units: an autoencoder-sized classifier
        dict(name='wide_train_4096', net='dense', use='train', dims='256-512-256-128-10', batch=4096),
        # scoring a whole test set with it, the batch not a multiple of anything
        dict(name='wide_predict_50000', net='dense', use='predict', dims='256-512-256-128-10', batch=50000),
        # the benchmark's per-particle network at its full size
        dict(name='particle_train_4096', net='particle', use='train', particles=64, features=16, hidden='64-32', classes=5, batch=4096),
        # a jet tagger with 30 particles of 7 features: neither count is a power of two
        dict(name='particle_train_ragged', net='particle', use='train', particles=30, features=7, hidden='64-32', classes=5, batch=1531),
        # the benchmark's image network at its full size
        dict(name='conv_train_1024', net='conv', use='train', height=28, width=28, channels=1, filters=32, classes=10, batch=1024),
        # small colour images, more filters than one wavefront is wide, a ragged batch
        dict(name='conv_train_colour', net='conv', use='train', height=24, width=24, channels=3, filters=40, classes=10, batch=300),
        # the benchmark's attention block, trained in a loop of the user's own with batches that keep the device ahead of it
        dict(name='attention_loop_16384', net='attention', use='loop', positions=64, features=64, heads=4, head=16, batch=16384),
        # inference of an attention block over 50 positions
        dict(name='attention_predict_ragged', net='attention', use='predict', positions=50, features=48, heads=3, head=16, batch=500),
        # the bare quantizer, every element with bit-widths of its own: the benchmark's bandwidth case, four times its size
        dict(name='quantize_16Mi', net='quantizer', use='quantize', n=16 * 2**20, rounding='RND', overflow='SAT'),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _drawn(rng):
    net = rng.choice(('dense', 'dense', 'wide', 'particle', 'conv', 'attention', 'quantizer'))
    if net == 'quantizer':
        return dict(net=net, use='quantize', n=_log(rng, 1024, 16 * 2**20), rounding=rng.choice(('RND', 'TRN', 'RND_CONV')),
                    overflow=rng.choice(('WRAP', 'SAT', 'SAT_SYM')))
    use = rng.choice(('train', 'train', 'predict'))
    if net == 'dense':
        widths = [rng.randint(4, 64) for _ in range(rng.randint(2, 4))] + [rng.randint(2, 10)]
        use = rng.choice(('train', 'loop', 'predict'))
        return dict(net=net, use=use, dims='-'.join(map(str, widths)), batch=_log(rng, 1 if use == 'predict' else 32, 65536))
    if net == 'wide':
        widths = [rng.randint(32, 512) for _ in range(rng.randint(2, 4))] + [rng.randint(2, 100)]
        return dict(net='dense', use=use, dims='-'.join(map(str, widths)), batch=_log(rng, 1 if use == 'predict' else 64, 50000))
    if net == 'particle':
        return dict(net=net, use=use, particles=rng.randint(8, 128), features=rng.randint(3, 32),
                    hidden=f'{rng.randint(8, 64)}-{rng.randint(8, 64)}', classes=rng.randint(2, 10), batch=_log(rng, 64, 8192))
    if net == 'conv':
        return dict(net=net, use=use, height=rng.randint(12, 32), width=rng.randint(12, 32), channels=rng.choice((1, 3)),
                    filters=rng.randint(4, 48), classes=10, batch=_log(rng, 16, 1024))
    use = rng.choice(('loop', 'loop', 'predict'))
    return dict(net=net, use=use, positions=rng.randint(8, 64), features=rng.randint(8, 96), heads=rng.randint(1, 8),
                head=rng.choice((8, 16, 32)), batch=_log(rng, 16, 16384))


def draw(rng):
    most = {k: max(work(c)[k] for c in listed()) for k in ('bytes', 'flops')}
    while True:
        case = _drawn(rng)
        w = work(case)
        if all(w[k] <= most[k] for k in most) and not (case['net'] == 'conv' and math.prod(_conv_maps(case)[2]) * case['filters'] > 4096) \
                and not (case['net'] == 'particle' and case['batch'] * case['particles'] > 262144):
            return case


def _conv_maps(case):
    """Height and width behind the first convolution, the pooling and the second convolution of ``models.conv_stack``."""
    a = (case['height'] - 2, case['width'] - 2)
    b = (a[0] // 2, a[1] // 2)
    return a, b, (b[0] - 2, b[1] - 2)


def _dims(text):
    return tuple(int(d) for d in text.split('-'))


def _model(case, dev):
    if case['net'] == 'dense':
        return models.qdense_mlp(_dims(case['dims']), device=dev)
    if case['net'] == 'particle':
        return models.particle_mlp(case['particles'], case['features'], _dims(case['hidden']), case['classes'], device=dev)
    if case['net'] == 'conv':
        return models.conv_stack(case['filters'], case['classes'], device=dev)
    return models.mha_block(case['heads'], case['head'], device=dev)


def _data(case, seed, dev):
    """Samples around one centre per class (pixels in [0, 1] for images), and what they are trained towards."""
    g = torch.Generator(device=dev).manual_seed(seed)
    rows = case['batch']
    if case['net'] == 'dense':
        shape, classes = _dims(case['dims'])[:1], _dims(case['dims'])[-1]
    elif case['net'] == 'particle':
        shape, classes = (case['particles'], case['features']), case['classes']
    elif case['net'] == 'conv':
        shape, classes = (case['height'], case['width'], case['channels']), case['classes']
    else:
        shape, classes = (case['positions'], case['features']), 0
    if case['net'] == 'conv':
        x = torch.rand((rows,) + shape, generator=g, device=dev)
        y = torch.randint(0, classes, (rows,), generator=g, device=dev)
        return x, y
    x = torch.randn((rows,) + shape, generator=g, device=dev)
    if not classes:
        return x, torch.randn((rows,) + shape, generator=g, device=dev)
    y = torch.randint(0, classes, (rows,), generator=g, device=dev)
    centres = 0.5 * torch.randn((classes, shape[-1]), generator=g, device=dev)
    x += centres[y].view((rows,) + (1,) * (len(shape) - 1) + shape[-1:])
    return x, y


def _variables(model):
    """What a step changes: every trainable variable, and the integer bits that follow the data."""
    return [p for name, p in model.named_parameters() if p.requires_grad or name.endswith('_var_i')]


def prepare(case, seed):
    dev = torch.device('cuda:0')
    if case['net'] == 'quantizer':
        g = torch.Generator(device=dev).manual_seed(seed)
        n = case['n']
        x = (2.0 * torch.randn(n, generator=g, device=dev)).requires_grad_()
        k = torch.ones(n, device=dev)
        i = torch.randint(0, 5, (n,), generator=g, device=dev).float().requires_grad_()
        f = torch.randint(0, 9, (n,), generator=g, device=dev).float().requires_grad_()
        dy = torch.randn(n, generator=g, device=dev)
        return dict(use='quantize', q=get_fixed_quantizer(case['rounding'], case['overflow']), x=x, k=k, i=i, f=f, dy=dy)
    torch.manual_seed(seed)  # the initial weights
    x, y = _data(case, seed, dev)
    model = _model(case, dev)
    state = dict(use=case['use'], model=model, x=x, y=y)
    if case['use'] == 'predict':
        calibration = x if case['batch'] >= CALIBRATION else _data(dict(case, batch=CALIBRATION), seed + 1, dev)[0]
        model(calibration[:CALIBRATION])
        trace_minmax(model, calibration[:CALIBRATION])
    elif case['use'] == 'train':
        state['step'] = train_step_for(model, x, y, lr=LR)
        state['variables'] = _variables(model)
    else:
        model(x, training=True)
        state['loss'] = ops.mse if case['net'] == 'attention' else ops.sparse_ce
        state['optimizer'] = SGD(model.parameters(), lr=LR, fold_regularizers=True)
        state['variables'] = _variables(model)
    return state


def run(state):
    use = state['use']
    if use == 'quantize':
        y = state['q'](state['x'], state['k'], state['i'], state['f'], True)
        return (y,) + torch.autograd.grad(y, (state['x'], state['i'], state['f']), state['dy'])
    if use == 'predict':
        with torch.no_grad():
            return state['model'](state['x'])
    if use == 'train':
        loss = state['step'](state['x'], state['y'])
        return [loss] + state['variables']
    model, opt = state['model'], state['optimizer']
    opt.zero_grad()
    out = model(state['x'], training=True)
    loss = model_loss(model, state['loss'](out, state['y']), True)
    opt.backward(loss)
    opt.step()
    return [loss, out] + state['variables']


def _layers(case):
    """``[(rows, K, N, contractions of the forward pass)]``, the values of a sample in and out, the values of the variables."""
    rows = case['batch']
    if case['net'] == 'dense':
        dims = _dims(case['dims'])
        layers = [(rows, k, n, 1) for k, n in zip(dims, dims[1:])]
        lanes = sum(dims[:-1])
        size = dims[0], dims[-1]
    elif case['net'] == 'particle':
        dims = (case['features'],) + _dims(case['hidden'])
        p = case['particles']
        # the batch statistics take the un-quantized kernel, the output the quantized one: two contractions
        layers = [(rows * p, k, n, 2 if case['use'] == 'train' else 1) for k, n in zip(dims, dims[1:])] + [(rows, dims[-1], case['classes'], 1)]
        lanes = p * sum(dims[:-1]) + dims[-1]
        size = p * case['features'], case['classes']
    elif case['net'] == 'conv':
        a, b, c = _conv_maps(case)
        f, flat = case['filters'], math.prod(c) * case['filters']
        layers = [(rows * math.prod(a), 9 * case['channels'], f, 1), (rows * math.prod(c), 9 * f, f, 1), (rows, flat, case['classes'], 1)]
        lanes = case['height'] * case['width'] * case['channels'] + math.prod(b) * f + flat
        size = case['height'] * case['width'] * case['channels'], case['classes']
    else:
        t, f, n, h = case['positions'], case['features'], case['heads'], case['head']
        layers = [(rows * t, f, n * h, 1)] * 3 + [(rows * t, n * h, f, 1), (rows * n * t, h, t, 1), (rows * n * t, t, h, 1)]
        lanes = 3 * t * f + 4 * t * n * h + n * t * t
        size = t * f, t * f
    weights = sum(k * n + n for _, k, n, _ in layers)
    return layers, size, 3 * weights + 2 * lanes


def work(case):
    if case['net'] == 'quantizer':
        live = 3 if case['overflow'] != 'WRAP' else 1  # bit-widths that the training branch reads: k, i, f or f alone
        return {'bytes': 4 * case['n'] * (2 + live + 4), 'flops': 0}
    layers, (n_in, n_out), variables = _layers(case)
    rows = case['batch']
    forward = sum(2 * r * k * n * c for r, k, n, c in layers)
    if case['use'] == 'predict':
        return {'bytes': 4 * rows * (n_in + n_out) + 4 * variables, 'flops': forward}
    r, k, n, c = layers[0]  # no gradient of the inputs
    target = 4 * n_out if case['net'] == 'attention' else 8
    first = (3 if case['net'] == 'attention' else 1) * 2 * r * k * n * c
    return {'bytes': rows * (4 * n_in + target) + 8 * variables, 'flops': 3 * forward - first}


def tolerance(case):
    # Activations and weights are fixed-point numbers whose sums fit fp32's 24 bits, so a forward pass comes out the same in
    # any order of summation; what differs are fp32 sums of gradients and batch moments over up to 10^6 rows.  The
    # contractions on the other matrix instruction (fp32 instead of bf16 parts: other orders of summation) gave at most
    # 2.0e-6 (2-norm) and 3.7e-6 (largest entry) over the listed and twenty-four drawn cases, two passes each.
    if case['net'] == 'quantizer':  # one rounding per product of the surrogate gradients, nothing is summed
        return {'rel': 1e-6, 'max': 1e-5}
    return {'rel': 1e-5, 'max': 1e-4}
