"""Convolutions over few input values per pixel (one-pass backward, matrix-core forward) against 64-bit sums.

Bound: any order of n fp32 products differs from the exact sum by at most n u / (1 - n u) of the sum of magnitudes, u = 2^-24;
the bf16 parts of an operand add up to it exactly.  The tests allow 2 (n + 16) u of that sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from hgq2_amd import _lib, ops  # noqa: E402


def _conv64(x, w, b, pad):
    return torch.nn.functional.conv2d(x.permute(0, 3, 1, 2), w.permute(3, 2, 0, 1), b, padding=pad).permute(0, 2, 3, 1)


def _close(got, exact, magnitude, n, what):
    worst = ((got.double().cpu() - exact).abs() / (2.0 * (n + 16) * 2.0**-24 * magnitude + 1e-30)).max().item()
    assert worst <= 1.0, f'{what}: {worst} times the bound'


# one band and several, a last short band, one row per band, rows beyond the last, the widest map, F around 32 and 64, 1 .. 31 inputs
@pytest.mark.parametrize('B,H,W,C,k,F,padding', [(1, 3, 3, 1, 3, 1, 'valid'), (2, 12, 12, 3, 3, 40, 'valid'), (3, 28, 28, 1, 3, 32, 'valid'),
                                                 (2, 24, 24, 3, 3, 33, 'valid'), (1, 31, 30, 3, 3, 64, 'same'), (2, 17, 64, 2, 3, 48, 'same'),
                                                 (1, 5, 66, 3, 3, 37, 'valid'), (2, 20, 21, 1, 5, 47, 'same'), (1, 32, 32, 1, 5, 7, 'valid'),
                                                 (300, 9, 8, 3, 3, 5, 'same'), (1, 7, 68, 3, 3, 40, 'valid')])
@pytest.mark.parametrize('relu,bits', [(True, 4), (False, None)])
def test_forward_and_gradients(B, H, W, C, k, F, padding, relu, bits):
    g = torch.Generator().manual_seed(H * W + F)
    x, w, b = torch.randn((B, H, W, C), generator=g), 0.3 * torch.randn((k, k, C, F), generator=g), torch.randn(F, generator=g)
    if bits:
        x, w, b = (torch.round(t * 2**bits) / 2**bits for t in (x, w, b))
    pad = (k - 1) // 2 if padding == 'same' else 0
    xg, wg, bg = (t.cuda().requires_grad_() for t in (x, w, b))
    y = ops.conv2d(xg, wg, bg, (1, 1), padding, (1, 1), _lib.ACT_RELU if relu else _lib.ACT_NONE)
    dy = torch.randn(y.shape, generator=g)
    grads = torch.autograd.grad(y, (xg, wg, bg), dy.cuda())
    xd, wd, bd = x.double(), w.double(), b.double()
    z = _conv64(xd, wd, bd, pad)
    n = k * k * C
    _close(y, z.relu() if relu else z, _conv64(xd.abs(), wd.abs(), bd.abs(), pad), n, 'forward')
    dz = dy.double() * (y.detach().cpu() > 0) if relu else dy.double()

    def exact(xv, wv, dv):
        xv, wv, bv = xv.clone().requires_grad_(), wv.clone().requires_grad_(), bd.clone().requires_grad_()
        return torch.autograd.grad(_conv64(xv, wv, bv, pad), (xv, wv, bv), dv)

    for what, got, e, m, terms in zip(('dx', 'dw', 'db'), grads, exact(xd, wd, dz), exact(xd.abs(), wd.abs(), dz.abs()),
                                      (k * k * F, dy[..., 0].numel(), dy[..., 0].numel())):
        _close(got, e, m, terms, what)


def test_gradients_that_are_not_finite_stay_where_they_belong():
    g = torch.Generator().manual_seed(4)
    x, w = torch.randn((2, 20, 22, 3), generator=g).cuda().requires_grad_(), torch.randn((3, 3, 3, 40), generator=g).cuda().requires_grad_()
    y = ops.conv2d(x, w, None, (1, 1), 'valid', (1, 1), 0)
    dy = torch.randn(y.shape, generator=g).cuda()
    dy[1, 7, 5, 33], dy[0, 17, 19, 2] = float('inf'), float('nan')
    dx, dw = torch.autograd.grad(y, (x, w), dy)
    assert set(torch.nonzero(~torch.isfinite(dw).all(0).all(0).all(0)).flatten().tolist()) == {2, 33}
    assert torch.isinf(dw[..., 33]).all() and torch.isnan(dw[..., 2]).all()
    bad = torch.zeros_like(dx, dtype=torch.bool)
    bad[1, 7:10, 5:8], bad[0, 17:20, 19:22] = True, True
    assert torch.equal(~torch.isfinite(dx), bad) and torch.isinf(dx[1, 7:10, 5:8]).all()


# inputs of one bf16 part, kernels of two (zero parts among them): one block of filters and two, one batch of taps and two
@pytest.mark.parametrize('C,k,F', [(1, 3, 40), (3, 3, 64), (1, 5, 48), (2, 3, 33)])
def test_infinite_inputs_as_on_the_fp32_instruction(C, k, F):
    g = torch.Generator().manual_seed(F)
    x, w = torch.round(4 * torch.randn((2, 12, 15, C), generator=g)) / 4, torch.round(2**12 * torch.randn((k, k, C, F), generator=g)) / 2**12
    x[0, 5, 5, 0], x[1, 2, 3, C - 1], x[1, 9, 9, 0] = float('inf'), float('-inf'), float('nan')
    lib = _lib.load()
    got = ops.conv2d(x.cuda(), w.cuda(), None, (1, 1), 'valid', (1, 1), 0)
    before = lib.hgq_dense_use_bf16_parts(0)
    try:
        want = ops.conv2d(x.cuda(), w.cuda(), None, (1, 1), 'valid', (1, 1), 0)
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(kind(got), kind(want)) and kind(want).any()
