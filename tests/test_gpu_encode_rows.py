"""Which encoder a call takes follows its row count and the tokens per (batch, head) row:
four lanes per token where there are many rows, one wave per token for few rows and for
rows of a few tokens.  On both sides of each line the bytes are those of the
one-wave-per-token kernels, which inputs off the 16-byte alignment always take."""

import pytest
import torch

from tests.test_gpu_encode_paths import KINDS, _case, _same, _unaligned

pytestmark = pytest.mark.gpu


def _calls(ext, c, ids):
    return {
        "int4": lambda k: ext.compress_quantized(k, c, ids, 64, 4),
        "int4/32": lambda k: ext.compress_quantized(k, c, ids, 32, 4),
        "int2": lambda k: ext.compress_quantized(k, c, ids, 64, 2),
        "int2/32": lambda k: ext.compress_quantized(k, c, ids, 32, 2),
        "sint4": lambda k: ext.compress_structured_int4(k, c, ids),
        "tile8": lambda k: ext.compress_fp16(k, c, ids, 8, False),
        "tile64": lambda k: ext.compress_fp16(k, c, ids, 64, False),
        "tile120": lambda k: ext.compress_fp16(k, c, ids, 120, False),
        "bitmap1": lambda k: ext.compress_bitmap(k, c, ids, 1),
        "bitmap32": lambda k: ext.compress_bitmap(k, c, ids, 32),
        "bitmap64": lambda k: ext.compress_bitmap(k, c, ids, 64),
        "bitmap127": lambda k: ext.compress_bitmap(k, c, ids, 127),
    }


def _check(ext, x, c, ids, calls):
    slow = _unaligned(x)
    for name, call in calls.items():
        for got, want in zip(call(x), call(slow)):
            assert _same(got, want), name


# past both row counts, with whole and partial waves and workgroups
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("b,h,t", [(91, 3, 16), (64, 1, 65), (9, 4, 147)])
def test_many_rows_equal_the_general_kernels(device, kind, b, h, t):
    from reskv_amd._extension import load_extension

    ext = load_extension("compression")
    x, c, ids = _case(kind, b, h, t, 5, device)
    _check(ext, x, c, ids, _calls(ext, c, ids))


# the row counts' edges (2048, 4096) and the token counts' (3, 4, 8), single and paired
@pytest.mark.parametrize("b,h,t", [(32, 1, 64), (683, 1, 3), (1025, 1, 2), (1366, 1, 3), (513, 1, 4), (64, 1, 64),
                                   (241, 1, 17), (1025, 1, 4), (900, 1, 5), (586, 1, 7), (513, 1, 8)])
def test_both_sides_of_each_line(device, b, h, t):
    from reskv_amd._extension import load_extension

    ext = load_extension("compression")
    x, c, ids = _case("near_tied", b, h, t, 3, device)
    x = x + torch.randn(x.shape, device=device, generator=torch.Generator(device=device).manual_seed(t)).half()
    _check(ext, x, c, ids, _calls(ext, c, ids))
    y = x.flip(2).contiguous()
    for pair, one in ((lambda: ext.compress_bitmap_kv(x, c, ids, y, c, ids, 64), lambda k: ext.compress_bitmap(k, c, ids, 64)),
                      (lambda: ext.compress_fp16_kv(x, c, ids, y, c, ids, 64, False),
                       lambda k: ext.compress_fp16(k, c, ids, 64, False))):
        for got, k in zip(pair(), (x, y)):
            assert all(_same(a, w) for a, w in zip(got, one(_unaligned(k))))
