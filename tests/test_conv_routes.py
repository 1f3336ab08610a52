"""Which kernels a convolution's backward pass takes, read off the slice counts that the library states without a GPU (where it
assumes 256 CUs)."""

import ctypes

import pytest

from hgq2_amd import _lib, ops


def _slices(shape, k, F, strides=(1, 1), padding='valid', dilation=(1, 1)):
    geom = _lib.ConvGeom(*ops.conv_geometry(shape, (k, k, shape[-1], F), strides, padding, dilation))
    lib = _lib.load()
    n = lib.hgq_conv2d_bwd_slice_count(ctypes.addressof(geom), F)
    need = lib.hgq_conv2d_bwd_workspace(ctypes.addressof(geom), F)
    assert n >= 1 and need >= n * (k * k * shape[-1] * F + F)
    return n


# two workgroups per CU on the matrix cores, three with multiply-adds per pixel; one value per side of the line and the ends
@pytest.mark.parametrize('shape,k,F,slices', [((1024, 28, 28, 1), 3, 32, 512), ((1024, 28, 28, 1), 3, 8, 768), ((1024, 28, 28, 1), 3, 1, 768),
                                              ((1024, 32, 32, 1), 3, 16, 768), ((1024, 32, 32, 2), 3, 8, 768), ((128, 64, 64, 1), 3, 32, 768),
                                              ((1024, 12, 12, 1), 3, 4, 512), ((300, 24, 24, 3), 3, 4, 512), ((300, 24, 24, 3), 3, 40, 512),
                                              ((1024, 32, 32, 1), 3, 33, 512), ((1024, 28, 28, 1), 5, 4, 512)])
def test_first_layers_take_the_faster_backward(shape, k, F, slices):
    assert _slices(shape, k, F) == slices


# one pass for all gradients, staged maps, tiled products of odd depths, 1 x 1, the general kernels
@pytest.mark.parametrize('shape,k,F,kw', [((300, 24, 24, 3), 3, 40, {}), ((64, 28, 28, 1), 3, 32, {}), ((256, 28, 28, 1), 5, 48, {}),
                                          ((300, 11, 11, 16), 3, 32, {}), ((300, 11, 11, 37), 3, 37, {}), ((16, 9, 9, 5), 3, 7, dict(padding='same')),
                                          ((40, 16, 16, 33), 3, 70, dict(strides=(2, 2))), ((30, 16, 16, 100), 1, 70, {}), ((300, 11, 11, 40), 3, 40, {}),
                                          ((3, 12, 12, 4), 3, 8, {})])
def test_slices_do_not_depend_on_the_matrix_instruction(shape, k, F, kw):
    lib = _lib.load()
    before, seen = lib.hgq_dense_use_bf16_parts(-1), []
    geom = _lib.ConvGeom(*ops.conv_geometry(shape, (k, k, shape[-1], F), kw.get('strides', (1, 1)), kw.get('padding', 'valid'), (1, 1)))
    try:
        for on in (1, 0):
            lib.hgq_dense_use_bf16_parts(on)
            seen.append((_slices(shape, k, F, **kw), lib.hgq_conv2d_bwd_workspace(ctypes.addressof(geom), F)))
    finally:
        lib.hgq_dense_use_bf16_parts(before)
    assert seen[0] == seen[1]
