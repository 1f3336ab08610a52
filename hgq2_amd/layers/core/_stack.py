"""Inference of consecutive QDense layers in one call of the library (``hgq_dense_stack_predict``): without gradients and
outside training and tracing, a run of plain layers leaves no state behind, so nothing between them has to exist."""

from __future__ import annotations

import functools

import torch

from ... import _lib, ops
from ...quantizer.internal import FixedPointQuantizerKBI, FixedPointQuantizerKIF
from ...quantizer.internal.base import bw_layout
from ...quantizer.quantizer import Quantizer

@functools.lru_cache(maxsize=1024)
def _mode(round_mode, overflow_mode, training, kbi, symmetric):
    return _lib.mode_bits(round_mode, overflow_mode, training=training, kbi=kbi, round_params=True, k_u8=True, symmetric=symmetric)


def _describe(q, shape, device, out) -> bool:
    """Fill ``out`` with the variables of the quantizer wrapper ``q`` as its call on a tensor of ``shape`` outside training
    uses them; False where that call is anything but one deterministic fixed-point quantizer."""
    if type(q) is not Quantizer or not q.built or not q.plain or 'call' in q.__dict__:
        return False
    fq = q.quantizer
    kind = type(fq)
    if kind is FixedPointQuantizerKIF:
        kbi = False
    elif kind is FixedPointQuantizerKBI:
        kbi = True
    else:
        return False
    if not fq.built or fq.stochastic or 'call' in fq.__dict__:
        return False
    p = fq._parameters
    i, fb, k = p.get('_i'), p.get('_b' if kbi else '_f'), fq._buffers.get('_var_k')
    if k is not fq._k or k is None or i is None or fb is None or k.dtype is not torch.uint8 or i.dtype is not torch.float32 or fb.dtype is not torch.float32:
        return False
    if i.device != device or fb.device != device or k.device != device or not (i.is_contiguous() and fb.is_contiguous() and k.is_contiguous()):
        return False
    n = i.numel()
    if fb.numel() != n or k.numel() != n:
        return False
    layout = bw_layout(i.shape, shape)
    if layout is None or layout[0] != n:
        return False
    # a trainable WRAP quantizer of a weight rounds and does not wrap (`FixedPointQuantizerKIF.call`, `...KBI.call`)
    rounds = fq._overflow_mode == 'WRAP' and fq.trainable and fq._is_weight and (not kbi or fq._round_mode == 'RND')
    out.k, out.i, out.fb = k.data_ptr(), i.data_ptr(), fb.data_ptr()
    out.size, out.inner = layout
    out.mode = _mode(fq._round_mode, fq._overflow_mode, rounds, kbi, fq._symmetric)
    return True


def _contraction(layer, K, N, device, out) -> bool:
    """Fill ``out`` with the kernel, bias and activation of a layer that contracts ``[rows, K]`` with its variables' ``[K, N]``
    view; False where its call does more than quantize, contract, add, activate."""
    if not layer.built or 'call' in layer.__dict__:
        return False
    # as the layers' own calls do: a ReLU by name runs inside the contraction, any other activation object behind it
    if layer._act_name != 'relu' and layer.activation is not None:
        return False
    w, b = layer._parameters.get('_kernel'), layer._parameters.get('bias')
    if w is None or layer._kq is None or w.numel() != K * N or w.dtype is not torch.float32 or w.device != device or not w.is_contiguous():
        return False
    if not _describe(layer._kq, w.shape, device, out.kq):
        return False
    out.w, out.K, out.N = w.data_ptr(), K, N
    out.act = _lib.ACT_RELU if layer._act_name == 'relu' else _lib.ACT_NONE
    if b is not None:
        if layer._bq is None or b.dtype is not torch.float32 or b.device != device or not b.is_contiguous() or b.numel() != N:
            return False
        if not _describe(layer._bq, b.shape, device, out.bq):
            return False
        out.bias = b.data_ptr()
    return True


def _rows_quantizer(q, shape, width, device, out, rows) -> bool:
    """Fill ``out`` for a quantizer of the contraction's input or output: one entry, or a table of ``rows`` (None: any number
    of) rows of ``width`` columns."""
    if not _describe(q, shape, device, out):
        return False
    if out.size == 1:
        out.inner = 1
        return True
    return out.inner == 1 and (out.size % width == 0 if rows is None else out.size == rows * width)


def _layer(layer, rows, k_in, device, out, first) -> bool:
    """Fill ``out`` for one QDense layer of a run."""
    from .dense import QDense

    if type(layer) is not QDense or not layer.built or layer._enable_oq or not _contraction(layer, k_in, layer.units, device, out):
        return False
    return not layer._enable_iq or _rows_quantizer(layer._iq, (rows, k_in), k_in, device, out.iq, None if first else 1)


def _ordinary_call() -> bool:
    """No tracer, transform, dual level or mode wants to see the operators of this call."""
    return not (torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack() or torch.jit.is_tracing()
                or torch.compiler.is_compiling() or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0)


def _plain_input(x) -> bool:
    return (type(x) is torch.Tensor and x.is_cuda and x.dtype is torch.float32 and 0 < x.numel() < 2**31
            and x.device.index == torch.cuda.current_device() and _ordinary_call())


def predict_contraction(layer, x, K, N, out_shape):
    """Output of a contraction layer's whole call - input, kernel, bias and output quantizer, contraction, activation - outside
    training, tracing and gradients as one library call, or ``None``.  ``x`` [..., K] and the output are read as rows."""
    if not _plain_input(x) or x.dim() < 1 or x.numel() % K:  # (what is no whole number of rows is for the layer to refuse)
        return None
    rows, device = x.numel() // K, x.device
    descs = (_lib.StackLayer * 1)()
    if not _contraction(layer, K, N, device, descs[0]):
        return None
    if layer._enable_iq and not _rows_quantizer(layer._iq, x.shape, K, device, descs[0].iq, None):
        return None
    if layer._enable_oq and not _rows_quantizer(layer._oq, out_shape, N, device, descs[0].oq, None):
        return None
    y = ops.dense_stack_predict(x, descs, 1, rows, N)
    if y is None:
        return None
    layer._deferred, layer._oq_applied_in_call = None, True
    return y.view(out_shape)


def predict_run(layers, first, x):
    """``(output, index behind the last layer taken)`` for the longest run of layers from ``first`` on that one library call
    covers, or ``None``."""
    if type(x) is not torch.Tensor or x.dim() != 2 or not _plain_input(x):  # (lists and tuples pass between layers too)
        return None
    rows, width = x.shape
    descs = (_lib.StackLayer * _lib.STACK_MAX_LAYERS)()
    n, device = 0, x.device
    while n < _lib.STACK_MAX_LAYERS and first + n < len(layers):
        if not _layer(layers[first + n], rows, width, device, descs[n], n == 0):
            break
        width = descs[n].N
        n += 1
    if n == 0:
        return None
    y = ops.dense_stack_predict(x, descs, n, rows, width)
    if y is None:
        return None
    for layer in layers[first:first + n]:
        layer._losses = []
        layer._deferred, layer._oq_applied_in_call = None, False
    return y, first + n
