"""Splits in whole 16-token tiles: automatic and given split counts at lengths
around tile, wave and split boundaries (waves and splits without tokens among
them) against the float64 oracle, for a format that works on single tiles, one
that works on pairs, and dense K and V."""

import numpy as np
import pytest
import torch

from reskv_amd import ResKVKernelConfig, attention, compress
from reskv_amd._extension import decode_splits, dense_decode
from tests.gpu_helpers import ATOL, expected_attention, np_, reference_test_inputs, seeded, theta_freq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparsity,bits", [(0.5, 16), (0.5, 4), (0.75, 4)])
@pytest.mark.parametrize("t", [1, 15, 16, 17, 63, 65, 127, 129, 200, 257, 960, 1041])
def test_lengths_around_the_tile_boundaries(device, sparsity, bits, t):
    k, v, q, clustering = reference_test_inputs(b=2, t=t, heads=2, gqa=4, seed=t, device=device)
    cache = compress(k, v, ResKVKernelConfig(sparsity=sparsity, bits=bits), clustering=clustering)
    freq = theta_freq(device=device)
    ref = expected_attention(q, cache, position=t + 5, start_position=3, inv_freq=freq)
    auto = decode_splits(cache, q.shape[1])
    assert 1 <= auto <= max(1, -(-t // 128))
    for splits in {0, 1, 2, 3, min(t, 7), min(t, 64), t}:
        out = attention(q, cache, position=t + 5, start_position=3, inv_freq=freq, splits=splits)
        assert float(np.abs(np_(out).astype(np.float64) - ref).max()) <= ATOL, splits


@pytest.mark.parametrize("t,splits", [(33, 0), (33, 33), (250, 0), (250, 9), (1000, 0)])
def test_dense_lengths(device, t, splits):
    g = seeded(t)
    q = torch.randn(1, 8, 1, 128, generator=g).half().to(device)
    k = (torch.randn(1, 2, t, 128, generator=g) * 0.5).half().to(device)
    v = torch.randn(1, 2, t, 128, generator=g).half().to(device)
    freq = theta_freq(device=device)
    out = dense_decode(q, k, v, freq, position=t, splits=splits).double()
    ang = lambda p: (p[:, None].float() * freq).double()  # noqa: E731

    def rot(x, p):
        a, b, c, s = x[..., :64], x[..., 64:], torch.cos(ang(p)), torch.sin(ang(p))
        return torch.cat((a * c - b * s, b * c + a * s), -1)

    qr = rot(q.double(), torch.full((1,), t, device=device))
    kr = rot(k.double(), torch.arange(t, device=device)).repeat_interleave(4, 1)
    w = torch.softmax(torch.matmul(qr, kr.transpose(2, 3).contiguous()) * 128 ** -0.5, -1)
    assert (out - torch.matmul(w, v.double().repeat_interleave(4, 1))).abs().max().item() <= ATOL
