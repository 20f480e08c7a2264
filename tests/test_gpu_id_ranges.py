"""Range check of an external clustering: one launch for K and V, the same refusals
in the same order as tensor by tensor, whatever the ids' type and layout."""

import pytest
import torch

from reskv_amd import ResKVKernelConfig, compress
from reskv_amd._extension import ids_in_range
from tests.gpu_helpers import reference_test_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 4095, 4096, 4097, 300001])
@pytest.mark.parametrize("offset", [0, 1])
def test_one_bad_id_is_found_anywhere(device, n, offset):
    good = torch.randint(7, (n + offset,), device=device, dtype=torch.int32)[offset:]
    assert ids_in_range([(good, 7), (good, 7)]) == [True, True]
    for at in {0, n // 2, n - 1}:
        for value in (-1, 7, 1 << 30, -(1 << 31)):
            bad = good.clone() if offset == 0 else torch.cat((good[:1], good))[1:]
            bad[at] = value
            assert ids_in_range([(bad, 7), (good, 7)]) == [False, True]
            assert ids_in_range([(good, 7), (bad, 7)]) == [True, False]


@pytest.mark.parametrize("dtype", [torch.int8, torch.int16, torch.int32, torch.int64])
@pytest.mark.parametrize("layout", ["contiguous", "strided"])
def test_refusals_and_their_order(device, dtype, layout):
    k, v, _, ((kc, ki), (vc, vi)) = reference_test_inputs(t=70, heads=2, device=device)
    cfg = ResKVKernelConfig()

    def ids(x, bad=False):
        x = x.to(dtype)
        if bad:
            x = x.clone()
            x[..., -1] = 32
        return x if layout == "contiguous" else x.transpose(1, 2).contiguous().transpose(1, 2)

    ok = compress(k, v, cfg, clustering=((kc, ids(ki)), (vc, ids(vi))))
    want = compress(k, v, cfg, clustering=((kc, ki), (vc, vi)))
    assert torch.equal(ok.key.payload, want.key.payload) and torch.equal(ok.value.metadata, want.value.metadata)
    for pair in (((kc, ids(ki, True)), (vc, ids(vi))), ((kc, ids(ki)), (vc, ids(vi, True))),
                 ((kc, ids(ki, True)), (vc, ids(vi)[..., :-1]))):
        with pytest.raises(ValueError, match="out of range"):
            compress(k, v, cfg, clustering=pair)
    with pytest.raises(ValueError, match="incompatible sizes"):
        compress(k, v, cfg, clustering=((kc, ids(ki)), (vc, ids(vi)[..., :-1])))
