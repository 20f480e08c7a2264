"""Which tokens and rings the one-launch ring append takes, on the CPU: the library and
the device queries are replaced, so that what reaches the kernel is seen and nothing runs.
Everything else has to be left to torch's copies, which handle (or refuse) it."""

import pytest
import torch
import torch.autograd.forward_ad as forward_ad
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

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
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: -1, raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda d: 0, raising=False)
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


class _Subclass(torch.Tensor):
    pass


class _Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("form", ["fake", "subclass", "negated", "gradient"])
def test_tokens_that_are_not_plain_values_are_left_to_torch(append, form):
    for at in range(3):
        tokens, rings = _tokens(), _rings()
        if form == "fake":
            with FakeTensorMode():
                tokens[at] = torch.ones(2, 3, 1, 128, **f16)
        elif form == "subclass":
            tokens[at] = tokens[at].as_subclass(_Subclass)
        elif form == "negated":
            tokens[at] = torch._neg_view(tokens[at])
        else:
            tokens[at].requires_grad_()
        assert not append(rings, tokens)


def test_calls_that_something_has_to_see_are_left_to_torch(append):
    rings, tokens = _rings(), _tokens()
    for mode in (_Dispatch(), _Function(), FakeTensorMode(), forward_ad.dual_level()):
        with mode:
            assert not append(rings, tokens)
    with torch.device("cpu"):  # a default device for new tensors
        assert append(rings, tokens)

    taken = []

    def inside(x):
        taken.append(append(rings, tokens))
        return x * 2

    torch.jit.trace(inside, torch.zeros(2), check_trace=False)
    torch.func.vmap(inside)(torch.zeros(2, 2))
    torch.func.functionalize(inside)(torch.zeros(2))
    torch.func.jvp(inside, (torch.zeros(2),), (torch.ones(2),))
    assert len(taken) >= 4 and not any(taken)
    assert append(rings, tokens)


def test_rings_that_autograd_follows_are_left_to_torch(append):
    rings = _rings()
    rings[1].requires_grad_()
    assert not append(rings, _tokens())
    with torch.inference_mode():
        inner = _rings()
        assert append(inner, _tokens())
    assert not append(inner, _tokens())  # copies refuse an in-place update outside inference mode
    plain = _rings()
    before = [r._version for r in plain]
    assert append(plain, _tokens())
    assert all(r._version > v for r, v in zip(plain, before))


@pytest.mark.parametrize("b,h", [(0, 3), (2, 0)])
def test_an_empty_batch_is_left_to_torch(append, b, h):
    assert not append(_rings(b, h), _tokens(b, h))


def test_more_rows_than_the_kernel_indexes_are_left_to_torch(append):
    rows = 1 << 24
    ring = torch.empty(rows, 1, 1, 128, **f16)  # 4 GiB of addresses, no page of it touched
    token = torch.empty(1, 1, 1, 128, **f16).expand(rows, 1, 1, 128)
    assert not append([ring] * 3, [token] * 3)


@pytest.mark.parametrize("slot", [-1, 8])
def test_a_slot_past_the_ring_is_left_to_torch(append, slot):
    assert not append(_rings(), _tokens(), slot)


def test_tokens_that_lie_in_a_ring_are_left_to_torch(append):
    # the copies run one after the other, the launch writes all three at once
    rings, tokens = _rings(), _tokens()
    tokens[1] = rings[0][:, :, 3:4]
    assert not append(rings, tokens, 3)


def test_a_compiled_call_takes_the_other_path_in_one_graph():
    """torch.compile follows the question itself without a graph break."""
    def which(x):
        return x + (1.0 if _extension.eager() else 2.0)

    assert torch.compile(which, backend="eager", fullgraph=True)(torch.zeros(2)).tolist() == [2.0, 2.0]
    assert which(torch.zeros(2)).tolist() == [1.0, 1.0]
