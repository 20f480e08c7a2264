"""Every native launch is issued with its tensors' GPU as the current device: a
kernel goes to the current device, whatever device its pointers belong to.  On the
CPU, with the library, the device switch and the stream lookup replaced by records."""

import contextlib

import pytest
import torch

from reskv_amd import llama

f16 = dict(dtype=torch.float16)


class _Library:
    """Takes any entry point and records (name, device in force)."""

    def __init__(self, entered):
        self.calls, self.entered = [], entered

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, self.entered[-1] if self.entered else None))
            return 0

        return call


@pytest.fixture
def library(monkeypatch):
    entered = []

    @contextlib.contextmanager
    def device(d):
        entered.append(d)
        yield
        entered.pop()

    lib = _Library(entered)
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(llama._lib, "lib", lambda: lib)
    monkeypatch.setattr(llama, "_stream", lambda t: 0)
    monkeypatch.setattr(llama, "_on_gpu", lambda *t: None)
    return lib


def test_fused_steps_make_their_tensors_device_current(library):
    x = torch.zeros(4, 64, **f16)
    llama.fused_rmsnorm(x, torch.ones(64, **f16), 1e-5, torch.empty_like(x))
    llama.fused_silu_mul(torch.zeros(4, 32, **f16), torch.zeros(4, 16, **f16))
    head = lambda h: torch.zeros(2, h, 128, **f16)  # noqa: E731
    llama.fused_qkv_rope(torch.zeros(2, 6 * 128, **f16), torch.zeros(8, 64), torch.zeros(8, 64),
                         torch.zeros(1, dtype=torch.int64), head(4), head(4), head(1), head(1), head(1))
    q, k, kr, v = llama.fused_prefill_split(torch.zeros(6, 6 * 128, **f16), torch.zeros(3, 64), torch.zeros(3, 64),
                                            2, 4, 1)
    llama.fused_prefill_attention(q, kr, v, 0.1)
    cpu = torch.device("cpu")
    assert library.calls == [("reskv_llama_" + n, cpu) for n in
                             ("rmsnorm", "silu_mul", "qkv_rope", "prefill_split", "prefill_attention")]
