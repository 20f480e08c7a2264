"""Unpacking of INT4 / INT2 codes in the decode kernel: with one token, a zero
centroid and a unit scale the output is the codes themselves, exactly; with two
tokens and a one-channel query the weights give every key code of that channel."""

import pytest
import torch

from reskv_amd import ResKVKernelConfig, attention
from reskv_amd.tensors import CompressedKV, CompressedTensor
from tests.gpu_helpers import seeded

pytestmark = pytest.mark.gpu


def _codes(words, bits):
    """Signed codes [..., 128] of packed words, lowest bits first."""
    fields = torch.stack([(words >> (bits * i)) & ((1 << bits) - 1) for i in range(32 // bits)], dim=-1)
    return torch.where(fields >= 1 << (bits - 1), fields - (1 << bits), fields).flatten(-2).float()


def _tensor(words, plan, device):
    b, h, t, _ = words.shape
    return CompressedTensor(torch.zeros(b, h, 1, 128, dtype=torch.float16, device=device),
                            torch.zeros(b, h, t, dtype=torch.int8, device=device), words.int().to(device), None,
                            torch.ones(b, h, t, dtype=torch.float16, device=device), plan)


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("gqa", [1, 4, 8])
def test_codes_of_every_channel(device, bits, gqa):
    g = seeded(bits + gqa)
    b, h = 8, 8
    plan = ResKVKernelConfig(sparsity=0.5, bits=bits, layout="unstructured").resolve(b)
    random = lambda t: torch.randint(-(1 << 31), 1 << 31, (b, h, t, 4 * bits), generator=g)  # noqa: E731
    kw, vw = random(1), random(1)
    q = torch.randn(b, h * gqa, 1, 128, generator=g).half().to(device)
    out = attention(q, CompressedKV(_tensor(kw, plan, device), _tensor(vw, plan, device)), position=1)
    want = _codes(vw, bits).repeat_interleave(gqa, dim=1)
    assert torch.equal(out.float().cpu().reshape(want.shape), want)


@pytest.mark.parametrize("bits", [4, 2])
def test_key_codes(device, bits):
    """Batch row d asks for channel d: two tokens at angles of no rotation (zero
    frequencies), V codes of +1 and 0, so the output is sigmoid(code_0 - code_1).
    The weight is rounded to fp16 (2^-11), once more in the output."""
    g = seeded(bits)
    plan = ResKVKernelConfig(sparsity=0.5, bits=bits, layout="unstructured").resolve(128)
    kw = torch.randint(-(1 << 31), 1 << 31, (128, 1, 2, 4 * bits), generator=g)
    vw = torch.zeros(128, 1, 2, 4 * bits, dtype=torch.int64)
    vw[:, :, 0] = sum(1 << (bits * i) for i in range(32 // bits))
    q = torch.zeros(128, 1, 1, 128, dtype=torch.float16)
    q[torch.arange(128), 0, 0, torch.arange(128)] = 1.0
    out = attention(q.to(device), CompressedKV(_tensor(kw, plan, device), _tensor(vw, plan, device)), position=2,
                    scaling=1.0, inv_freq=torch.zeros(64, device=device))
    k = _codes(kw, bits)[torch.arange(128), 0, :, torch.arange(128)]
    want = torch.sigmoid(k[:, 0] - k[:, 1])
    assert (out.float().cpu()[:, 0, 0, :] - want[:, None]).abs().max().item() < 2 ** -9
