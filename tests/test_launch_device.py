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


def test_step_decoder_makes_its_device_current(library, monkeypatch):
    from reskv_amd import _extension

    monkeypatch.setattr(_extension._lib, "lib", lambda: library)
    monkeypatch.setattr(_extension, "_stream", lambda d: 0)
    # device 1 current until the decoder switches to its own (the CPU's index is None)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None if library.entered else 1, raising=False)
    cpu = torch.device("cpu")
    step = object.__new__(_extension.StepDecoder)
    step.dev, step.b, step.nh, step.kh, step.t, step.scaling, step.splits = cpu, 1, 4, 1, 16, 0.1, 0
    step.kdesc = step.vdesc = None
    step.freq = step.table = step.m = step.l = torch.zeros(4)
    step.ws = torch.zeros(4, dtype=torch.uint8)
    step.out, step.merged = torch.zeros(4, 128, **f16), torch.zeros(4, 128, **f16)
    q = torch.zeros(1, 4, 1, 128, **f16)
    ring = torch.zeros(1, 1, 8, 128, **f16)
    assert step.run(q, 20).shape == (1, 4, 1, 128)
    assert step.run(q, 20, q, ring, ring, 3, 8).shape == (1, 4, 1, 128)
    assert library.calls == [("reskv_decode_rope", cpu), ("reskv_decode_recent", cpu)]


def test_greedy_decoder_steps_and_captures_on_its_device(library):
    seen = []
    dec = object.__new__(llama.GreedyDecoder)
    dec.x, dec.pos, dec.max_pos = torch.zeros(1, 8), 0, 2
    dec._step = lambda events: seen.append(("step", library.entered[-1]))
    dec._capture = lambda: seen.append(("capture", library.entered[-1]))
    dec.step()
    dec.capture()
    assert seen == [("step", torch.device("cpu")), ("capture", torch.device("cpu"))]
