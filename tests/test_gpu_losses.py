"""Losses at the sizes where their kernels change, against 64-bit sums: sparse cross-entropy over the class counts at which its
rows change place (registers of 4, 8, 16 values, memory), the squared error around the length from which it leaves the cache
alone.

Bounds, u = 2^-24: a softmax value carries a few roundings of the exponential and of a sum of C terms; a row's loss the same
through a logarithm, times the size of the logits' spread; the rows of a workgroup (at most 256 here) are added in fp32."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from hgq2_amd import _lib, ops  # noqa: E402


@pytest.mark.parametrize('C', [1, 2, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize('rows', [1, 255, 3000])
def test_around_the_rows_kept_in_registers(rows, C):
    g = torch.Generator().manual_seed(rows + C)
    z, labels = 4 * torch.randn((rows, C), generator=g), torch.randint(0, C, (rows,), generator=g)
    zd = z.double().requires_grad_()
    want = torch.nn.functional.cross_entropy(zd, labels)
    want.backward()
    zg = z.cuda().requires_grad_()
    loss = ops.sparse_ce(zg, labels.cuda())
    (dz,) = torch.autograd.grad(loss, zg)
    spread = (z.max(1).values - z.min(1).values).max().item() + 1.0
    assert abs(loss.item() - want.item()) <= (C + 32 + 256) * 2.0**-24 * spread
    assert (dz.double().cpu() - zd.grad).abs().max() <= (C + 32) * 2.0**-24 * spread / rows


@pytest.mark.parametrize('C', [3, 7, 12, 20])
def test_labels_outside_the_classes(C):
    z = torch.randn((9, C), generator=torch.Generator().manual_seed(C)).cuda().requires_grad_()
    labels = torch.zeros(9, dtype=torch.int64)
    labels[4], labels[7] = C, -1
    loss = ops.sparse_ce(z, labels.cuda())
    (dz,) = torch.autograd.grad(loss, z)
    assert torch.isnan(loss) and not dz[4].any() and not dz[7].any() and dz[3].any()


# both sides of 2^26 values, with and without the last vector
@pytest.mark.parametrize('n', [2**26 - 4, 2**26 - 1, 2**26, 2**26 + 5])
@pytest.mark.parametrize('with_target', [True, False])
def test_squared_error_beyond_the_cache(n, with_target):
    a = torch.randn(n, generator=torch.Generator('cuda').manual_seed(n), device='cuda')
    t = torch.randn(n, generator=torch.Generator('cuda').manual_seed(n + 1), device='cuda') if with_target else None
    lib = _lib.load()
    loss, d, ws = torch.empty(1, device='cuda'), torch.empty(n, device='cuda'), torch.empty(lib.hgq_mse_workspace(), device='cuda')
    rc = lib.hgq_mse_fwd_bwd(a.data_ptr(), t.data_ptr() if with_target else None, loss.data_ptr(), d.data_ptr(), ws.data_ptr(), n,
                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    diff = a - t if with_target else a
    want = diff.double().square().mean().item()
    # squares and sums of one sign: at most a rounding per addition of the longest chain (elements per thread, wavefronts, parts)
    assert abs(loss.item() - want) <= (n // (2048 * 256) + 64) * 2.0**-24 * want
    # n as a float, the quotient 2 / n and the product are rounded, u each
    exact = diff.double() * (2.0 / n)
    assert ((d - exact).abs() <= 3 * 2.0**-24 * exact.abs()).all()
