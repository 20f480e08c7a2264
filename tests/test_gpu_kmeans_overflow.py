"""Decode groups whose V tokens have an infinite fp16 norm (the square sum exceeds
65504): every distance of such a token is then infinite, and the nearest centre is the
lowest index, as an argmin over equal values gives it."""

import numpy as np
import pytest
import torch

from oracle import reskv_oracle as o
from reskv_amd import ResKVKernelConfig, compress
from reskv_amd._extension import kmeans_assign
from tests.gpu_helpers import np_, seeded

pytestmark = pytest.mark.gpu


def _with_large_tokens(x, g):
    """Every third token gets a channel of 300 (its square exceeds fp16), every fifth an rms of 30."""
    x[..., ::3, 5] = 300.0
    x[..., ::5, :] = torch.randn(x[..., ::5, :].shape, generator=g) * 30.0
    return x.half()


@pytest.mark.parametrize("count", [1, 2, 12, 16, 17, 33, 64])
@pytest.mark.parametrize("t", [15, 64, 257])
def test_tokens_of_infinite_norm_take_the_lowest_index(device, count, t):
    g = seeded(100 * count + t)
    x = _with_large_tokens(torch.randn(3, t, 128, generator=g), g)
    centres = torch.randn(3, count, 128, generator=g).half()
    ids = np_(kmeans_assign(x.to(device), centres.float().to(device), value=True))
    d = o.incremental_value_distances(np_(x), np_(centres))
    want = np.argmin(d, axis=-1)
    infinite = np.isinf(d).all(-1)
    assert infinite[:, ::3].all() and not infinite[:, 1::15].any()
    assert ids.min() >= 0 and ids.max() < count
    assert (ids[infinite] == want[infinite]).all() and (want[infinite] == 0).all()
    # elsewhere the products differ from the oracle's exact ones by fp32 rounding alone
    got = np.take_along_axis(d, ids[..., None].astype(np.int64), -1)[..., 0][~infinite]
    scale = np.abs(np_(x).astype(np.float64)).sum(-1)[~infinite] * float(np.abs(np_(centres)).max())
    assert (got - d.min(-1)[~infinite] <= 2.0 ** -20 * scale).all()


def test_appended_groups_are_decoded_with_the_centroid_that_they_were_encoded_with(device):
    g = seeded(3)
    cfg = ResKVKernelConfig(sparsity=0.5, num_clusters=8, kmeans_iterations=2)
    k, v = (torch.randn(2, 2, 128, 128, generator=g).half().to(device) for _ in range(2))
    gk, gv = (_with_large_tokens(torch.randn(2, 2, 64, 128, generator=g), g).to(device) for _ in range(2))
    cache = compress(gk, gv, cfg, previous=compress(k, v, cfg))
    for x, ct in ((gk, cache.key), (gv, cache.value)):
        ids = np_(ct.cluster_ids)[:, :, -64:].astype(np.int64)
        assert ids.min() >= 0 and ids.max() < ct.centroids.shape[2]
        # the stored residuals are x - centroid of that id, on the kept channels
        cent = np_(ct.centroids).astype(np.float64)
        base = np.take_along_axis(cent, ids[..., None].repeat(128, -1), 2)
        whole = o.reconstruct("bitmap", np_(ct.centroids), np_(ct.cluster_ids).astype(np.int64), np_(ct.payload),
                              np_(ct.metadata))[:, :, -64:]
        kept = whole != base
        err = np.abs(whole - np_(x).astype(np.float64))[kept]
        # one rounding of the residual to fp16: half a unit in the last place of at most 512
        assert kept.mean() > 0.45 and err.max() <= 0.25


@pytest.mark.parametrize("count", [16, 33])
def test_centres_without_a_distance_are_passed_over(device, count):
    """A NaN centre is nobody's nearest one, wherever it stands in a lane's scan; a token
    without any finite distance takes the lowest index."""
    g = seeded(count)
    x = torch.randn(2, 70, 128, generator=g).half()
    centres = torch.randn(2, count, 128, generator=g).half()
    nan = [0, 4, 5, 15, count - 1]
    clean = np_(centres).copy()
    centres[:, nan, 3] = float("nan")
    x[:, 9] = float("nan")
    ids = np_(kmeans_assign(x.to(device), centres.float().to(device), value=True))
    d = o.incremental_value_distances(np_(x), clean)
    d[:, :, nan] = np.inf
    finite = np.isfinite(d).any(-1) & ~np.isnan(d).any(-1)
    assert not finite[:, 9].any() and finite.sum() == 2 * 69
    assert (ids[:, 9] == 0).all() and not np.isin(ids[finite], nan).any()
    got = np.take_along_axis(d, ids[..., None].astype(np.int64), -1)[..., 0][finite]
    # an fp16 norm that rounds the other way moves a distance by two fp16 steps of at most 512
    assert (got - d.min(-1)[finite] <= 4 * 0.25).all()
