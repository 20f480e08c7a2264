"""K-means gives the same bits however its work is split: a problem run alone
(one workgroup per chunk, 16 waves up to 32 centres), among a few (four or eight
waves per chunk) and among many (one workgroup per interleaved part of its
chunks), for K and for V, at the edges of sub-tiles, chunks and parts."""

import pytest
import torch

from tests.gpu_helpers import seeded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [64, 255, 257, 1024, 1025, 1296, 2063])
@pytest.mark.parametrize("count", [1, 16, 17, 32, 33, 64])
def test_results_do_not_depend_on_the_split(device, t, count):
    from reskv_amd._extension import kmeans, kmeans_kv

    g = seeded(1000 * count + t)
    scale = torch.exp(torch.randn(3, 1, 128, generator=g))
    base = (torch.randn(3, t, 128, generator=g) * scale).half().to(device)
    for value in (False, True):
        alone = [kmeans(base[i: i + 1].contiguous(), None, 4, value, count) for i in range(3)]
        for copies in (8, 48):  # 24 and 144 problems
            centres, ids = kmeans(base.repeat(copies, 1, 1), None, 4, value, count)
            for i in range(3):
                assert all(torch.equal(ids[i + 3 * j], alone[i][1][0]) for j in (0, copies - 1)), (value, copies, i)
                assert all(torch.equal(centres[i + 3 * j], alone[i][0][0]) for j in (0, copies - 1)), (value, copies, i)
    (kc, ki), (vc, vi) = kmeans_kv(base, base.flip(1).contiguous(), None, None, 4, count)
    k1, v1 = kmeans(base, None, 4, False, count), kmeans(base.flip(1).contiguous(), None, 4, True, count)
    assert torch.equal(kc, k1[0]) and torch.equal(ki, k1[1]) and torch.equal(vc, v1[0]) and torch.equal(vi, v1[1])
