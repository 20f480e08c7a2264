"""Which tokens and rings the one-launch ring append takes, on the CPU: the library and
the device queries are replaced, so that what reaches the kernel is seen and nothing runs.
Everything else has to be left to torch's copies, which handle (or refuse) it."""

import pytest
import torch

from reskv_amd import _extension

f16 = dict(dtype=torch.float16)


@pytest.fixture
def append(monkeypatch):
    """ring_append with every tensor passing for one on the current GPU; returns whether
    it took the call, which has to agree with whether the library was called."""
    calls = []

    class Library:
        def reskv_ring_append(self, *args):
            calls.append(args)
            return 0

    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None, raising=False)
    monkeypatch.setattr(_extension, "_stream", lambda d: 0)
    monkeypatch.setattr(_extension._lib, "lib", lambda: Library())

    def call(rings, tokens, slot=0):
        before = len(calls)
        taken = _extension.ring_append(rings, tokens, slot)
        assert len(calls) - before == int(taken)
        return taken

    return call


def _rings(b=2, h=3, cap=8):
    return [torch.zeros(b, h, cap, 128, **f16) for _ in range(3)]


def _tokens(b=2, h=3):
    return [torch.ones(b, h, 1, 128, **f16) for _ in range(3)]


def test_ordinary_tokens_are_taken(append):
    assert append(_rings(), _tokens(), 7)


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("form", ["shorter", "fewer_heads", "transposed", "gap", "float32", "bfloat16", "misaligned"])
def test_every_ring_is_one_dense_buffer_of_the_same_kind(append, which, form):
    rings = _rings()
    x = rings[which]
    rings[which] = {
        "shorter": lambda: x[:, :, :4].contiguous(),
        "fewer_heads": lambda: x[:, :2].contiguous(),
        "transposed": lambda: x.transpose(1, 2).contiguous().transpose(1, 2),
        "gap": lambda: torch.zeros(2, 3, 16, 128, **f16)[:, :, :8],
        "float32": lambda: x.float(),
        "bfloat16": lambda: x.bfloat16(),
        "misaligned": lambda: torch.zeros(x.numel() + 1, **f16)[1:].view(x.shape),
    }[form]()
    assert not append(rings, _tokens())
