"""Which sizes the allocation-free decode takes: a rule of the sizes alone, restated here
from include/reskv_hip.h.  On the CPU a call that passes it fails later, for want of a
device; one that does not is refused by the rule's own message."""

import itertools

import pytest

from reskv_amd import _lib

RECORDS = (8 << 20) // 776  # split records that the array holds


def _refused(b, hq, h, t, splits):
    lib = _lib.lib()
    ct = _lib.CTensor()
    status = lib.reskv_decode_recent_noalloc(16, ct, ct, 16, 16, b, hq, h, t, 0, t, 0.1, splits, None, None, None, 0, 0,
                                             16, None)
    assert status != 0
    return b"allocation-free" in lib.reskv_last_error()


@pytest.fixture(scope="module", autouse=True)
def no_device():
    import torch

    if torch.cuda.device_count():
        pytest.skip("the calls that pass would be issued")


@pytest.mark.parametrize("g", [1, 2, 4, 8])
def test_automatic_counts(g):
    for rows, t in itertools.product((1, 8, 100, 255, 256, 257, 338, 341, 342, 700, 1023, 1025, 1351, 1352, 2703, 10811),
                                     (1, 127, 128, 200, 256, 383, 400, 512, 8192, 1 << 20)):
        counted = max(1, min(-(-1024 // rows), t // 128))
        assert _refused(rows, g, 1, t, 0) is (rows * g * counted > RECORDS), (rows, g, t)
        assert not (_refused(rows, g, 1, t, 0) and rows * g + 1024 * g <= 10810)


@pytest.mark.parametrize("splits", [1, 2, 16, 1024, 5000])
def test_given_counts(splits):
    for rows, t in itertools.product((1, 10, 11, 675, 676, 10810, 10811), (1, 16, 1000, 1 << 20)):
        assert _refused(rows, 1, 1, t, splits) is (rows * min(splits, t, 1024) > RECORDS), (rows, t)
