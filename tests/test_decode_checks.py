"""What a decode call hands to the library for a compressed cache, on the CPU: its
descriptors follow the plan and the views that the cache has at the call."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from reskv_amd import ResKVKernelConfig
from reskv_amd import _extension, _lib
from reskv_amd.tensors import CompressedKV, CompressedTensor


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


@pytest.fixture
def decode(monkeypatch):
    """decode_step with every tensor passing for a CUDA one and the library answering for itself."""
    calls = []

    class Library:
        def reskv_decode_workspace_bytes(self, *args):
            return 16

        def reskv_decode_rope(self, *args):
            calls.append(args)
            return 0

    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: -1, raising=False)
    monkeypatch.setattr(_extension, "_stream", lambda d: 0)
    monkeypatch.setattr(_extension._lib, "lib", lambda: Library())
    monkeypatch.setattr(_extension, "_rope", lambda *a: (torch.zeros(64), torch.zeros(16)))

    def call(query, cache):
        return _extension.decode_step(query, cache, 4, position=60, start_position=0, scaling=0.1, inv_freq=None,
                                      rope_theta=1e4)

    return call, calls


@pytest.mark.parametrize("side", ["key", "value"])
@pytest.mark.parametrize("which", range(4))
def test_every_view_is_on_the_querys_device(decode, side, which):
    call, calls = decode
    cache = CompressedKV(_tensor(), _tensor())
    query = torch.zeros(4, 128, dtype=torch.float16)
    assert call(query, cache).shape == (4, 128) and len(calls) == 1
    ct = getattr(cache, side)
    with FakeTensorMode():
        elsewhere = torch.zeros(ct._native[which].shape, dtype=ct._native[which].dtype, device="cuda")
    ct._native = ct._native[:which] + (elsewhere,) + ct._native[which + 1:]
    with pytest.raises(RuntimeError, match="same GPU"):
        call(query, cache)
    assert len(calls) == 1


def test_the_result_is_a_plain_tensor_whatever_the_query_is(decode):
    class Subclass(torch.Tensor):
        pass

    query = torch.zeros(4, 128, dtype=torch.float16).as_subclass(Subclass)
    out = decode[0](query, CompressedKV(_tensor(), _tensor()))
    assert type(out) is torch.Tensor and out.dtype == torch.float16 and out.is_contiguous()
