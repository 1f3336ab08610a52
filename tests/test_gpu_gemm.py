"""The bf16-part matrix products behind dense layers of more than 64 inputs or units, against 64-bit products.

Bound: a sum of n fp32 products in any order differs from the exact one by at most n u / (1 - n u) times the sum of the
products' magnitudes, u = 2^-24; the bf16 parts of an operand add up to it exactly, so splitting adds terms (at most nine per
product, of rapidly falling magnitude) but no other error.  The test allows 2 (n + 8) u of that sum."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from hgq2_amd import _lib, ops  # noqa: E402


def _operand(g, shape, bits):
    t = torch.randn(shape, generator=g)
    return t if bits is None else torch.round(t * 2.0**bits) / 2.0**bits


def _close(got, exact, magnitude, n, what):
    err = (got.double().cpu() - exact).abs()
    bound = 2.0 * (n + 8) * 2.0**-24 * magnitude + 1e-30
    worst = (err / bound).max().item()
    assert worst <= 1.0, f'{what}: {worst} times the bound'


# tile edges (64 / 128 outputs, 32 / 64 contraction steps), remainders that are not multiples of four, few and many columns;
# operands of one, two and three parts
@pytest.mark.parametrize('rows,K,N', [(1, 65, 1), (63, 100, 70), (64, 64, 128), (65, 66, 65), (129, 257, 33), (300, 8, 500),
                                      (257, 128, 10), (1031, 511, 130), (6500, 72, 129), (16500, 96, 385), (20, 2050, 40)])
@pytest.mark.parametrize('bits_x,bits_w,act', [(3, 3, 1), (3, 10, 0), (10, 3, 1), (9, 14, 0), (None, None, 1)])
def test_matmul_bias_act(rows, K, N, bits_x, bits_w, act):
    g = torch.Generator().manual_seed(rows * 7 + K + N)
    x, w, b = _operand(g, (rows, K), bits_x), _operand(g, (K, N), bits_w), _operand(g, (N,), 6)
    dy = torch.randn((rows, N), generator=g)
    xg, wg, bg = (t.cuda().requires_grad_() for t in (x, w, b))
    y = ops.matmul_bias_act(xg, wg, bg, act)
    gx, gw, gb = torch.autograd.grad(y, (xg, wg, bg), dy.cuda())
    xd, wd, bd = x.double(), w.double(), b.double()
    exact = xd @ wd + bd
    _close(y, exact.relu() if act else exact, xd.abs() @ wd.abs() + bd.abs(), K, 'forward')
    dz = dy.double() * (y.detach().cpu() > 0) if act else dy.double()
    _close(gx, dz @ wd.T, dz.abs() @ wd.abs().T, N, 'data gradient')
    _close(gw, xd.T @ dz, xd.abs().T @ dz.abs(), rows, 'weight gradient')
    _close(gb, dz.sum(0), dz.abs().sum(0), rows, 'bias gradient')


@pytest.mark.parametrize('bits', [3, None])
def test_operands_off_a_sixteen_byte_boundary(bits):
    g = torch.Generator().manual_seed(5)
    rows, K, N = 150, 90, 75
    x = _operand(g, (rows * K + 1,), bits).cuda()[1:].view(rows, K)
    w = _operand(g, (K * N + 3,), bits).cuda()[3:].view(K, N)
    y = ops.matmul_bias_act(x, w, None, 0)
    xd, wd = x.double().cpu(), w.double().cpu()
    _close(y, xd @ wd, xd.abs() @ wd.abs(), K, 'forward')


def test_infinities_and_nans_as_on_the_fp32_instruction():
    g = torch.Generator().manual_seed(6)
    x, w, dy = torch.randn((200, 96), generator=g), torch.randn((96, 80), generator=g), torch.randn((200, 80), generator=g)
    x[3, 5], x[100, 7], dy[17, 9], dy[150, 70] = float('inf'), float('nan'), float('-inf'), float('nan')

    def grads():
        xg, wg = x.cuda().requires_grad_(), w.cuda().requires_grad_()
        y = ops.matmul_bias_act(xg, wg, None, 0)
        return (y,) + torch.autograd.grad(y, (xg, wg), dy.cuda())

    lib = _lib.load()
    got = grads()
    before = lib.hgq_dense_use_bf16_parts(0)
    try:
        want = grads()
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    for a, b in zip(got, want):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isposinf(a), torch.isposinf(b))
        assert torch.equal(torch.isneginf(a), torch.isneginf(b)) and not torch.isfinite(b).all()


def test_contractions_beyond_the_tiled_products():
    # more inputs than the tiled products state: the general dense kernel
    g = torch.Generator().manual_seed(9)
    rows, K, N = 3, 2**20 + 3, 2
    x, w = _operand(g, (rows, K), 3).cuda(), _operand(g, (K, N), 3).cuda()
    y = torch.empty((rows, N), device='cuda')
    rc = _lib.load().hgq_qdense_fwd(x.data_ptr(), None, None, None, 0, w.data_ptr(), None, y.data_ptr(), None, rows, K, N, 0, 0,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    xd, wd = x.double().cpu(), w.double().cpu()
    _close(y, xd @ wd, xd.abs() @ wd.abs(), K, 'forward')


def test_data_gradient_in_large_tiles():
    # 384 tiles of 128 x 128 for the data gradient, both sides ragged
    g = torch.Generator().manual_seed(10)
    rows, K, N = 49100, 100, 70
    x, w = _operand(g, (rows, K), 3).cuda().requires_grad_(), _operand(g, (K, N), 10).cuda()
    dy = torch.randn((rows, N), generator=g).cuda()
    y = ops.matmul_bias_act(x, w, None, 1)
    (gx,) = torch.autograd.grad(y, (x,), dy)
    dz, wd = dy.double().cpu() * (y.detach().cpu() > 0), w.double().cpu()
    _close(gx, dz @ wd.T, dz.abs() @ wd.abs().T, N, 'data gradient')
