"""Causal attention of a prompt whose first keys score minus infinity (an fp16 overflow
in a key channel): later queries weigh the others, as a softmax does, and a query with
no other key gives NaN."""

import pytest
import torch

from reskv_amd.llama import fused_prefill_attention

pytestmark = pytest.mark.gpu


# within, at and past the 64-key tiles that a wave takes at a time
@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 150])
@pytest.mark.parametrize("hk,g", [(2, 1), (1, 2), (1, 4)])
def test_keys_of_minus_infinity_weigh_nothing(device, n, hk, g):
    gen = torch.Generator(device=device).manual_seed(n)
    t = 200
    q = torch.randn(1, hk * g, t, 128, device=device, generator=gen).half()
    q[..., 0] = 1.0
    k = torch.randn(1, hk, t, 128, device=device, generator=gen).half()
    k[:, :, :n, 0] = float("-inf")
    v = torch.randn(1, hk, t, 128, device=device, generator=gen).half()
    got = fused_prefill_attention(q, k, v, 128 ** -0.5).double()
    kd, vd = (x.double().repeat_interleave(g, dim=1) for x in (k, v))
    score = torch.matmul(q.double(), kd.transpose(2, 3).contiguous()) * 128 ** -0.5
    score.masked_fill_(torch.ones(t, t, dtype=torch.bool, device=device).triu(1), float("-inf"))
    w = torch.softmax(score, dim=-1)
    ref = torch.matmul(w, vd).transpose(1, 2)
    assert ref[:, :n].isnan().all() and ref[:, n:].isfinite().all()
    assert got[:, :n].isnan().all()
    # weights rounded to fp16 (relative 2^-11, or 2^-25 of the largest one), the result once more
    bound = 2.0 ** -11 * (torch.matmul(w, vd.abs()).transpose(1, 2) + ref.abs()) + 2.0 ** -24 * (t + 1) * 8 + 1e-5
    assert ((got - ref).abs() <= bound)[:, n:].all()
