"""The descriptors that Python hands to the library, field by field against the C compiler's layout of include/hgq_hip.h."""

import ctypes
import os
import shutil
import subprocess

import pytest

from hgq2_amd import _lib, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PAIRS = {'hgq_conv_geom': _lib.ConvGeom, 'hgq_qdesc': _lib.QDesc, 'hgq_bits_desc': _lib.BitsDesc, 'hgq_stack_quant': _lib.StackQuant,
         'hgq_stack_layer': _lib.StackLayer, 'hgq_mlp_layer': _lib.MlpLayer, 'hgq_track_item': ops._TrackItem, 'hgq_reduce_item': ops._ReduceItem,
         'hgq_dense_ebops_item': ops._DenseEbopsItem, 'hgq_sgd_item': ops._SgdItem, 'hgq_quant_item': ops._QuantItem,
         'hgq_quant_grad_item': ops._QuantGradItem}
LIMITS = {'HGQ_STACK_MAX_LAYERS': _lib.STACK_MAX_LAYERS, 'HGQ_REDUCE_BATCH': ops.REDUCE_BATCH, 'HGQ_REDUCE_QUANTS': ops.REDUCE_QUANTS,
          'HGQ_SGD_SIDES': ops.SGD_SIDES, 'HGQ_SUM_BATCH': ops.SUM_BATCH, 'HGQ_STATIC_SCRATCH_FLOATS': _lib.STATIC_SCRATCH_FLOATS}


@pytest.mark.skipif(shutil.which('g++') is None, reason='no host compiler')
def test_layouts_match_the_header(tmp_path):
    lines = ['#include <cstddef>', '#include <cstdio>', f'#include "{ROOT}/include/hgq_hip.h"', 'int main() {']
    want = []
    for name, struct in PAIRS.items():
        lines.append(f'printf("{name} %zu\\n", sizeof({name}));')
        want.append(f'{name} {ctypes.sizeof(struct)}')
        for field, *_ in struct._fields_:
            lines.append(f'printf("{name}.{field} %zu %zu\\n", offsetof({name}, {field}), sizeof((({name} *)0)->{field}));')
            d = getattr(struct, field)
            want.append(f'{name}.{field} {d.offset} {d.size}')
    for name, value in LIMITS.items():
        lines.append(f'printf("{name} %ld\\n", (long)({name}));')
        want.append(f'{name} {value}')
    (tmp_path / 'layout.cpp').write_text('\n'.join(lines + ['return 0;', '}']))
    subprocess.run(['g++', '-o', str(tmp_path / 'layout'), str(tmp_path / 'layout.cpp')], check=True)
    assert subprocess.run([str(tmp_path / 'layout')], check=True, capture_output=True, text=True).stdout.split('\n')[:-1] == want
