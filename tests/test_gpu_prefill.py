"""The prompt kernels of the end-to-end decoder (include/reskv_llama.h): causal
attention against float64, the split and rotation bit for bit against the torch
formulas, and the fused prompt pass against the unfused one."""

import pytest
import torch

from reskv_amd.llama import LlamaShape, RandomLlama, _rotate, fused_prefill_attention, fused_prefill_split

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


# edges of the 32-query and 64-key tiles, each split of a workgroup over query heads
@pytest.mark.parametrize("t", [1, 2, 31, 32, 33, 63, 64, 65, 127, 129, 200, 1027])
@pytest.mark.parametrize("b,hk,g", [(2, 1, 1), (1, 3, 2), (1, 2, 4), (1, 1, 8)])
@pytest.mark.parametrize("scale", [0.5, 6.0])
def test_prefill_attention_matches_float64(device, t, b, hk, g, scale):
    gen = _gen(t + 10 * g)
    q = (torch.randn(b, hk * g, t, 128, device=device, generator=gen) * scale).half()
    k = torch.randn(b, hk, t, 128, device=device, generator=gen).half()
    v = torch.randn(b, hk, t, 128, device=device, generator=gen).half()
    got = fused_prefill_attention(q, k, v, 128 ** -0.5).double()
    assert got.shape == (b, t, hk * g, 128)
    kd, vd = (x.double().repeat_interleave(g, dim=1) for x in (k, v))
    score = torch.matmul(q.double(), kd.transpose(2, 3).contiguous()) * 128 ** -0.5
    score.masked_fill_(torch.ones(t, t, dtype=torch.bool, device=device).triu(1), float("-inf"))
    w = torch.softmax(score, dim=-1)
    ref = torch.matmul(w, vd).transpose(1, 2)
    # weights rounded to fp16 (relative 2^-11, or 2^-25 of the largest one), the result once more
    bound = 2.0 ** -11 * (torch.matmul(w, vd.abs()).transpose(1, 2) + ref.abs()) + 2.0 ** -24 * (t + 1) * 8 + 1e-5
    assert ((got - ref).abs() <= bound).all()


def test_prefill_attention_checks(device):
    q = torch.zeros(1, 3, 4, 128, device=device, dtype=torch.float16)
    with pytest.raises(ValueError, match="ratio"):
        fused_prefill_attention(q, q[:, :1].contiguous(), q[:, :1].contiguous(), 1.0)
    with pytest.raises(ValueError, match="contiguous fp16"):
        fused_prefill_attention(q.float(), q, q, 1.0)
    with pytest.raises(RuntimeError, match="scaling"):
        fused_prefill_attention(q, q, q, 0.0)


@pytest.mark.parametrize("b,t,hq,hk", [(1, 1, 4, 1), (2, 37, 8, 2), (1, 130, 3, 3)])
def test_prefill_split_matches_torch_bitwise(device, b, t, hq, hk):
    gen = _gen(t)
    qkv = (torch.randn(b * t, (hq + 2 * hk) * 128, device=device, generator=gen) * 3).half()
    ang = torch.arange(t, device=device).float()[:, None] * (torch.rand(64, device=device, generator=gen) + 0.01)
    cos, sin = torch.cos(ang), torch.sin(ang)
    qr, k, kr, v = fused_prefill_split(qkv, cos, sin, b, hq, hk)
    heads = qkv.view(b, t, hq + 2 * hk, 128).transpose(1, 2)
    eq, ek, ev = heads[:, :hq], heads[:, hq: hq + hk], heads[:, hq + hk:]
    assert torch.equal(k, ek) and torch.equal(v, ev)
    assert torch.equal(qr, _rotate(eq, cos, sin)) and torch.equal(kr, _rotate(ek, cos, sin))


@pytest.mark.parametrize("shape,b,t", [
    (LlamaShape(layers=2, hidden=512, heads=4, kv_heads=1, ffn=1024, vocab=1000), 2, 150),
    (LlamaShape(layers=1, hidden=1024, heads=8, kv_heads=4, ffn=2816, vocab=500), 1, 77),
])
def test_fused_prompt_pass_matches_the_unfused_one(device, monkeypatch, shape, b, t):
    model = RandomLlama(shape, device, seed=9)
    ids = torch.randint(shape.vocab, (b, t), device=device, generator=_gen(1))

    def run():
        kept = []
        logits = model.prefill(ids, lambda *a: kept.append(a[1:]), q_rows=64, logits=True)
        return logits.double(), kept

    got, kept = run()
    monkeypatch.setattr(RandomLlama, "_fused", lambda self, t: False)
    ref, ref_kept = run()
    # fp16 layers that round at different places: a few fp16 steps of the largest logit
    assert (got - ref).abs().max().item() <= 2e-2 * ref.abs().max().item()
    for a, c in zip(kept, ref_kept):
        for x, y in zip(a, c):
            assert x.shape == y.shape and x.is_contiguous()
            assert (x.double() - y.double()).abs().max().item() <= 2e-2 * y.double().abs().max().item()
