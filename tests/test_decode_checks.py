"""What a decode call hands to the library for a compressed cache, on the CPU: its
descriptors follow the plan and the views that the cache has at the call."""

import torch

from reskv_amd import ResKVKernelConfig
from reskv_amd import _extension, _lib
from reskv_amd.tensors import CompressedTensor


def _plan(layout):
    return ResKVKernelConfig(sparsity=0.5, bits=16, layout=layout).resolve(1)


def _tensor(t=48):
    return CompressedTensor(torch.zeros(1, 2, 8, 128, dtype=torch.float16), torch.zeros(1, 2, t, dtype=torch.int8),
                            torch.zeros(1, 2, t, 64, dtype=torch.float16), torch.zeros(1, 2, t, 2, dtype=torch.int64),
                            None, _plan("unstructured"))


def test_a_replaced_plan_is_followed():
    ct = _tensor()
    assert _extension._descriptor(ct).format == _lib.FMT_BITMAP
    ct.plan = _plan("tiled")  # the same 16 metadata bytes a token, read as tile masks
    assert _extension._descriptor(ct).format == _lib.FMT_TILED


def test_replaced_views_are_followed():
    ct, other = _tensor(), _tensor(t=32)
    strides = [_extension._descriptor(x).t_stride for x in (ct, other)]
    ct._native = other._native
    d = _extension._descriptor(ct)
    assert (strides, d.t_stride, d.payload) == ([48, 32], 32, other._native[2].data_ptr())
