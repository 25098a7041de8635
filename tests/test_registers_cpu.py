"""Registers of the pair kernels, from the metadata of the library as it was built here.

A SIMD of an MI355X has 512 VGPRs per lane: kernels of two bodies per lane need at most 64 for
eight wavefronts per SIMD, those of four bodies at most 128 for four.  A workgroup of eight
wavefronts puts two on each SIMD, so a few registers more cost it a whole workgroup per
compute unit.
"""

import re
import struct

import pytest

from gravitation_amd import build

msgpack = pytest.importorskip('msgpack')


def _kernels():
    """{mangled name: VGPRs} from the AMDGPU metadata notes of libgravhip.so."""
    with open(build.LIB_PATH, 'rb') as f:
        data = f.read()
    out = {}
    for m in re.finditer(rb'\x07\0\0\0(.{4})\x20\0\0\0AMDGPU\0\0', data, re.S):
        size = struct.unpack('<I', m.group(1))[0]
        note = msgpack.unpackb(data[m.end():m.end() + size], strict_map_key=False)
        for k in note['amdhsa.kernels']:
            out[k['.name']] = k['.vgpr_count']
    return out


@pytest.mark.parametrize('name, bodies, limit', [('k_stage1_vjp_f32', 2, 64),
                                                 ('k_stage1_vjp_f32', 4, 128),
                                                 ('k_step_items_f64m', 2, 64),
                                                 ('k_step_items_f64m', 4, 128)])
def test_pair_kernels_keep_their_wavefronts(name, bodies, limit):
    of = {k: v for k, v in _kernels().items() if re.search(r'%sILi%dE' % (name, bodies), k)}
    assert of and max(of.values()) <= limit, of
