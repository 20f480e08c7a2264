"""One-launch append of a decode token to the ring against the strided copies it
replaces, and which tensors still take those copies."""

import pytest
import torch

from reskv_amd import ResKVKernelConfig
from reskv_amd._extension import ring_append
from reskv_amd.cache import ResKVLayerCache
from tests.gpu_helpers import seeded

pytestmark = pytest.mark.gpu


def _token(form, b, h, g, device):
    x = torch.randn(b, h, 1, 128, generator=g).half().to(device)
    if form == "transposed":  # a projection's view: [B, 1, H, 128] memory
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "sliced":  # heads of a wider fused projection
        wide = torch.zeros(b, 3 * h, 1, 128, dtype=torch.float16, device=device)
        wide[:, h: 2 * h] = x
        return wide[:, h: 2 * h]
    if form == "odd":  # rows that start two bytes off
        return torch.empty(b * h * 128 + 1, dtype=torch.float16, device=device)[1:].view(b, h, 1, 128).copy_(x)
    if form == "expanded":
        return x[:, :1].expand(b, h, 1, 128)
    return x


@pytest.mark.parametrize("b,h,cap", [(1, 1, 1), (3, 5, 96), (16, 8, 96)])
@pytest.mark.parametrize("forms,taken", [
    (("plain", "plain", "plain"), True), (("transposed", "sliced", "plain"), True),
    (("expanded", "plain", "transposed"), True), (("plain", "odd", "plain"), False)])
def test_ring_append_equals_the_copies(device, b, h, cap, forms, taken):
    g = seeded(b + cap)
    rings = [torch.full((b, h, cap, 128), 7.0, dtype=torch.float16, device=device) for _ in range(3)]
    want = [r.clone() for r in rings]
    tokens = [_token(f, b, h, g, device) for f in forms]
    for slot in {0, cap // 2, cap - 1}:
        assert ring_append(rings, tokens, slot) is taken
        for w, x in zip(want, tokens):
            w[:, :, slot: slot + 1].copy_(x)
    if taken:
        assert all(torch.equal(r, w) for r, w in zip(rings, want))
    else:
        assert all((r == 7.0).all() for r in rings)


def test_ring_append_leaves_other_tensors_to_torch(device):
    ring = [torch.zeros(2, 3, 8, 128, dtype=torch.float16, device=device) for _ in range(3)]
    x = torch.ones(2, 3, 1, 128, dtype=torch.float16, device=device)
    assert not ring_append(ring, (x, x.float(), x), 0)
    assert not ring_append(ring, (x, x[:1], x), 0)
    assert not ring_append(ring, (x, x, x.clone().requires_grad_()), 0)
    assert not ring_append([r.cpu() for r in ring], (x.cpu(), x.cpu(), x.cpu()), 0)
    wide = [torch.zeros(2, 3, 8, 64, dtype=torch.float16, device=device) for _ in range(3)]
    assert not ring_append(wide, (x[..., :64], x[..., :64], x[..., :64]), 0)
    assert all((r == 0).all() for r in ring)


@pytest.mark.parametrize("form", ["plain", "transposed", "odd"])
def test_layer_cache_holds_the_same_tokens_either_way(device, form):
    cfg = ResKVKernelConfig(sparsity=0.75, num_clusters=8, kmeans_iterations=2)
    layer = ResKVLayerCache(cfg)
    prompt = torch.randn(2, 2, 150, 128, generator=seeded(1)).half().to(device)
    layer.update(prompt, prompt, {"raw_keys": prompt})
    live, seen = layer.live, []
    g = seeded(2)
    for _ in range(5):
        k, raw, v = (_token(form, 2, 2, g, device) for _ in range(3))
        seen.append((k, raw, v))
        layer.update(k, v, {"raw_keys": raw})
    for i, (k, raw, v) in enumerate(seen):
        assert torch.equal(layer.keys[:, :, live + i: live + i + 1], k)
        assert torch.equal(layer.raw_keys[:, :, live + i: live + i + 1], raw)
        assert torch.equal(layer.values[:, :, live + i: live + i + 1], v)
