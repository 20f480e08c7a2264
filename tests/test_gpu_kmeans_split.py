"""K-means gives the same bits however its work is split: a problem run alone
(one workgroup per chunk, 16 waves up to 32 centres), among a few (four or eight
waves per chunk) and among many (one workgroup per interleaved part of its
chunks), for K and for V, at the edges of sub-tiles, chunks and parts."""

import numpy as np
import pytest
import torch

from oracle import reskv_oracle as o
from tests.gpu_helpers import np_, seeded
from tests.test_gpu_kmeans_sweep import _within_one_fp16_step

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


@pytest.mark.parametrize("problems,t,count", [(40, 2339, 8), (40, 2339, 16), (24, 3000, 17), (144, 1100, 16)])
def test_many_problems_follow_lloyd(device, problems, t, count):
    """K against a 64-bit Lloyd loop on grids of more than one workgroup per CU, at
    the smallest centre tables (an earlier kernel read its tables past its LDS there,
    and gave wrong ids without any error).  Gaussian tokens on 128 channels: two fp32
    distances are closer than their rounding for fewer than one token in 1000."""
    from reskv_amd._extension import kmeans

    g = seeded(count + t)
    x = (torch.randn(problems, t, 128, generator=g) * torch.exp(torch.randn(problems, 1, 128, generator=g))).half()
    x = x.to(device)
    centres, ids = kmeans(x, None, 3, False, count)
    wide = x.double()
    c = wide[:, torch.linspace(0, t - 1, count).long()]
    for _ in range(3):
        near = ((c * c).sum(-1)[:, None] - 2 * torch.bmm(wide, c.transpose(1, 2).contiguous())).argmin(-1)
        member = torch.nn.functional.one_hot(near, count).double().transpose(1, 2).contiguous()
        n = member.sum(-1, keepdim=True)
        c = torch.where(n > 0, torch.bmm(member, wide) / n.clamp(min=1), c)
    assert (near != ids).float().mean().item() < 1e-3
    # every centre is the mean of its own ids' tokens: one rounding to fp16 (2^-11 of the value,
    # 2^-25 below the normal range) after fp32 sums (2^-24 for each of at most t additions)
    member = torch.nn.functional.one_hot(ids.long(), count).double().transpose(1, 2).contiguous()
    n = member.sum(-1, keepdim=True)
    mean = torch.bmm(member, wide) / n.clamp(min=1)
    size = torch.bmm(member, wide.abs()) / n.clamp(min=1)
    bound = 2.0 ** -11 * mean.abs() + 2.0 ** -25 + (t + 2) * 2.0 ** -24 * size
    assert (((centres.double() - mean).abs() <= bound) | (n == 0)).all()
    # and the 64-bit loop's, where the members are the same
    same = (torch.nn.functional.one_hot(near, count).double().transpose(1, 2) == member).all(-1, keepdim=True) & (n > 0)
    assert (((centres.double() - c).abs() <= bound) | ~same).all() and same.float().mean().item() > 0.3


@pytest.mark.parametrize("problems,t,count", [(40, 2339, 8), (24, 3000, 17), (144, 1100, 16), (48, 1500, 33)])
@pytest.mark.parametrize("n", [2, 3])
def test_many_value_problems_follow_the_fp16_rule(device, problems, t, count, n):
    """V on the same kind of grids: the n-th ids against the oracle's fp16 distances to the
    centres of n - 1 iterations (from the second iteration on the tokens' norms are the
    stored ones), away from roundings that fp32 sums may make either way, and the n-th
    centres within one fp16 step of those ids' means."""
    from reskv_amd._extension import kmeans

    g = seeded(count + t)
    x = (torch.randn(problems, t, 128, generator=g) * torch.exp(0.5 * torch.randn(problems, t, 1, generator=g))).half()
    before = np_(kmeans(x.to(device), None, n - 1, True, count)[0])
    centres, ids = (np_(r) for r in kmeans(x.to(device), None, n, True, count))
    unsure = o.value_ambiguous(np_(x), before)
    assert unsure.mean() < 0.02
    assert np.array_equal(ids[~unsure], o.assign_value(np_(x), before)[~unsure])
    means = o.update_centres(np_(x).astype(np.float64), ids.astype(np.int64), before, count, value=True)
    assert _within_one_fp16_step(centres, means)
