"""Ids of decode groups (the assignment without member sums): token counts at the edges of
the waves' sub-tiles and of the turns that a short group leaves out, for a workgroup of
sixteen waves (few problems), of four and of eight."""

import numpy as np
import pytest
import torch

from oracle import reskv_oracle as o
from reskv_amd._extension import kmeans_assign
from tests.gpu_helpers import np_, seeded

pytestmark = pytest.mark.gpu


def _ambiguous_norms(a):
    """Rows whose fp16 norm an fp32 sum may round either way: within its error (33 additions
    at most in a row, 2^-24 each) of the midpoint between two fp16 values."""
    exact = o._half_norm_exact(a)
    slack = 34 * 2.0 ** -24 * exact
    return (exact - slack).astype(np.float16) != (exact + slack).astype(np.float16)


@pytest.mark.parametrize("problems", [1, 300])
@pytest.mark.parametrize("t", [1, 16, 17, 63, 64, 65, 128, 129, 255, 256, 257, 400])
@pytest.mark.parametrize("count", [16, 33, 64])
def test_group_ids_are_nearest_for_both_rules(device, problems, t, count):
    g = seeded(1000 * count + t)
    x = torch.randn(problems, t, 128, generator=g).half()
    centres = torch.randn(problems, count, 128, generator=g).half()
    xd, cd = np_(x).astype(np.float64), np_(centres).astype(np.float64)
    for value in (False, True):
        ids = kmeans_assign(x.to(device), centres.float().to(device), value)
        assert ids.shape == (problems, t) and int(ids.min()) >= 0 and int(ids.max()) < count
        if value:
            d = o.incremental_value_distances(np_(x), np_(centres))
        else:
            d = (cd * cd).sum(-1)[:, None, :] - 2.0 * (xd @ np.swapaxes(cd, 1, 2))
        index = np_(ids).astype(np.int64)
        got = np.take_along_axis(d, index[..., None], -1)[..., 0]
        # fp32 sums of 128 products of at most |x| |c|: 2^-20 of that is beyond their rounding
        allowed = 2.0 ** -20 * np.abs(xd).sum(-1) * np.abs(cd).max()
        if value:
            # a norm that rounds the other way moves fp16(|x|^2 + |c|^2) by at most two fp16
            # steps (its own and the sum's; 2^-10 of the value each), on either distance
            unsure_c = _ambiguous_norms(np_(centres))
            unsure = (_ambiguous_norms(np_(x)) | np.take_along_axis(unsure_c, index, 1)
                      | np.take_along_axis(unsure_c, d.argmin(-1), 1))
            assert unsure.sum() <= 3 + 0.05 * unsure.size
            largest = (o.half_norms(np_(x)).astype(np.float64)[..., None] + o.half_norms(np_(centres))[:, None, :]).max(-1)
            allowed = allowed + unsure * 4 * 2.0 ** -10 * largest
        assert (got - d.min(-1) <= allowed).all()
