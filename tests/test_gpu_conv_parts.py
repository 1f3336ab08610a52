"""Convolutions on the tiled bf16-part products: any channel and filter count, stride, dilation and padding, against 64-bit
sums, with the bound of two orders of summation (2 (n + 16) 2^-24 of the sum of the products' magnitudes)."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

from hgq2_amd import _lib, ops  # noqa: E402


def _conv64(x, w, b, geom):
    _, H, W, _, kh, kw, sy, sx, py, px, dly, dlx, OH, OW = geom
    # padding may differ between the sides: pad by hand, to what the last window reads
    py1, px1 = (OH - 1) * sy + (kh - 1) * dly + 1 - H - py, (OW - 1) * sx + (kw - 1) * dlx + 1 - W - px
    xp = torch.nn.functional.pad(x.permute(0, 3, 1, 2), (px, max(px1, 0), py, max(py1, 0)))
    return torch.nn.functional.conv2d(xp, w.permute(3, 2, 0, 1), b, stride=(sy, sx), dilation=(dly, dlx))[..., :OH, :OW].permute(0, 2, 3, 1)


def _close(got, exact, magnitude, n, what):
    worst = ((got.double().cpu() - exact).abs() / (2.0 * (n + 16) * 2.0**-24 * magnitude + 1e-30)).max().item()
    assert worst <= 1.0, f'{what}: {worst} times the bound'


# depths around multiples of four and around 32 / 64 columns, remainders of the tiles, one pixel, strides and dilations, even kernels
CASES = [(2, 9, 9, 33, (3, 3), 5, (1, 1), 'valid', (1, 1)), (1, 3, 3, 40, (3, 3), 40, (1, 1), 'valid', (1, 1)), (3, 11, 10, 37, (3, 3), 65, (1, 1), 'same', (1, 1)),
         (5, 8, 13, 6, (2, 3), 130, (1, 1), 'valid', (1, 1)), (2, 12, 9, 34, (3, 2), 7, (2, 1), 'same', (1, 1)), (2, 15, 14, 35, (3, 3), 33, (1, 1), 'valid', (2, 3)),
         (1, 17, 18, 9, (5, 5), 31, (3, 2), 'same', (1, 1)), (40, 6, 7, 64, (3, 3), 64, (1, 1), 'same', (1, 1)), (2, 7, 5, 1, (7, 5), 3, (1, 1), 'same', (1, 1)),
         (3, 10, 10, 39, (1, 1), 41, (2, 2), 'valid', (1, 1))]


@pytest.mark.parametrize('case', CASES)
@pytest.mark.parametrize('relu,bits', [(True, 4), (False, None)])
def test_forward_and_gradients(case, relu, bits):
    B, H, W, C, k, F, strides, padding, dilation = case
    g = torch.Generator().manual_seed(C + F)
    x, w, b = torch.randn((B, H, W, C), generator=g), 0.3 * torch.randn(k + (C, F), generator=g), torch.randn(F, generator=g)
    if bits:
        x, w, b = (torch.round(t * 2**bits) / 2**bits for t in (x, w, b))
    geom = ops.conv_geometry((B, H, W, C), k + (C, F), strides, padding, dilation)
    xg, wg, bg = (t.cuda().requires_grad_() for t in (x, w, b))
    y = ops.conv2d(xg, wg, bg, strides, padding, dilation, _lib.ACT_RELU if relu else _lib.ACT_NONE)
    dy = torch.randn(y.shape, generator=g)
    grads = torch.autograd.grad(y, (xg, wg, bg), dy.cuda())
    xd, wd, bd = x.double(), w.double(), b.double()
    z = _conv64(xd, wd, bd, geom)
    _close(y, z.relu() if relu else z, _conv64(xd.abs(), wd.abs(), bd.abs(), geom), k[0] * k[1] * C, 'forward')
    dz = dy.double() * (y.detach().cpu() > 0) if relu else dy.double()

    def exact(xv, wv, dv):
        xv, wv, bv = xv.clone().requires_grad_(), wv.clone().requires_grad_(), bd.clone().requires_grad_()
        return torch.autograd.grad(_conv64(xv, wv, bv, geom), (xv, wv, bv), dv)

    for what, got, e, m, terms in zip(('dx', 'dw', 'db'), grads, exact(xd, wd, dz), exact(xd.abs(), wd.abs(), dz.abs()),
                                      (k[0] * k[1] * F, dy[..., 0].numel(), dy[..., 0].numel())):
        _close(got, e, m, terms, what)


def test_infinities_and_nans_as_on_the_fp32_instruction():
    g = torch.Generator().manual_seed(6)
    x, w, dy = torch.randn((2, 9, 9, 34), generator=g), torch.randn((3, 3, 34, 35), generator=g), torch.randn((2, 7, 7, 35), generator=g)
    x[1, 3, 5, 33], x[0, 8, 8, 0], dy[1, 2, 3, 34], dy[0, 6, 6, 1] = float('inf'), float('nan'), float('-inf'), float('nan')

    def results():
        xg, wg = x.cuda().requires_grad_(), w.cuda().requires_grad_()
        y = ops.conv2d(xg, wg, None, (1, 1), 'valid', (1, 1), 0)
        return (y,) + torch.autograd.grad(y, (xg, wg), dy.cuda())

    lib = _lib.load()
    got = results()
    before = lib.hgq_dense_use_bf16_parts(0)
    try:
        want = results()
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    for a, b in zip(got, want):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isposinf(a), torch.isposinf(b))
        assert torch.equal(torch.isneginf(a), torch.isneginf(b)) and not torch.isfinite(b).all()


# the choice of matrix instruction changes between the question for slices and the launch
@pytest.mark.parametrize('shape,k,F', [((7, 24, 24, 3), 3, 40), ((9, 28, 28, 1), 3, 32), ((5, 11, 11, 16), 3, 32), ((6, 11, 11, 37), 3, 37),
                                       ((40, 9, 9, 5), 3, 7), ((30, 6, 6, 100), 1, 70), ((3, 12, 12, 4), 3, 8), ((2, 9, 9, 40), 3, 36)])
@pytest.mark.parametrize('asked', [1, 0])
def test_slices_hold_when_the_matrix_instruction_changes(shape, k, F, asked):
    g = torch.Generator().manual_seed(F)
    geom = ops.conv_geometry(shape, (k, k, shape[-1], F), (1, 1), 'valid', (1, 1))
    x, w = torch.randn(shape, generator=g), torch.randn((k, k, shape[-1], F), generator=g)
    dy = torch.randn((shape[0], geom[12], geom[13], F), generator=g)
    xg, wg, dyg, dx = x.cuda(), w.cuda(), dy.cuda(), torch.empty(shape, device='cuda')
    lib, desc = _lib.load(), _lib.ConvGeom(*geom)
    at, stream = ctypes.addressof(desc), torch.cuda.current_stream().cuda_stream
    before = lib.hgq_dense_use_bf16_parts(asked)
    try:
        n, need = lib.hgq_conv2d_bwd_slice_count(at, F), lib.hgq_conv2d_bwd_workspace(at, F)
        lib.hgq_dense_use_bf16_parts(1 - asked)
        ws = torch.full((need,), float('nan'), device='cuda')
        rc = lib.hgq_conv2d_bwd_slices(dyg.data_ptr(), None, xg.data_ptr(), wg.data_ptr(), dx.data_ptr(), ws.data_ptr(), at, F, 0, stream)
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    assert rc == 0
    width = w.numel() + F
    total = ws[:n * width].view(n, width).double().sum(0).cpu()

    def exact(xv, wv, dv):
        xv, wv, bv = xv.clone().requires_grad_(), wv.clone().requires_grad_(), torch.zeros(F, dtype=torch.float64, requires_grad=True)
        return torch.autograd.grad(_conv64(xv, wv, bv, geom), (xv, wv, bv), dv)

    terms = dy[..., 0].numel()
    want, size = exact(x.double(), w.double(), dy.double()), exact(x.double().abs(), w.double().abs(), dy.double().abs())
    for what, got, e, m, count in (('dx', dx, want[0], size[0], k * k * F), ('dw', total[:w.numel()].view(w.shape), want[1], size[1], terms),
                                   ('db', total[w.numel():], want[2], size[2], terms)):
        _close(got, e, m, count, what)
