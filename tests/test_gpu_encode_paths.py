"""The encoders that work on bit planes (four lanes per token) against the
one-wave-per-token kernels that inputs off the 16-byte alignment still take:
the same bytes for every format, also for residuals that are not finite, for
subnormal and overflowing scales, and for quotients on rounding boundaries.
At these row counts an aligned call takes the one-wave kernels too; the same inputs
at the counts that take the bit planes are in test_gpu_encode_rows.py."""

import pytest
import torch

from tests.gpu_helpers import seeded

pytestmark = pytest.mark.gpu

KINDS = ["nan", "inf", "tiny", "huge", "boundary", "all_tied", "near_tied"]


def _case(kind, b, h, t, c, device):
    g = seeded(sum(map(ord, kind)) + t)
    x = torch.randn(b, h, t, 128, generator=g).half()
    cen = (torch.randn(b, h, c, 128, generator=g) * 0.1).half()
    ids = torch.randint(c, (b, h, t), generator=g, dtype=torch.int32)
    hit = torch.rand(x.shape, generator=g) < 0.02
    sign = torch.where(torch.rand(x.shape, generator=g) < 0.5, -1.0, 1.0)
    if kind == "nan":
        x[hit] = float("nan")
    elif kind == "inf":
        x = torch.where(hit, sign * float("inf"), x.float()).half()
    elif kind == "tiny":  # multiples of the smallest subnormal, scales that round to zero or to few bits
        x = (torch.randint(-9, 10, x.shape, generator=g).float() * 2.0 ** -24).half()
        cen = torch.zeros_like(cen)
    elif kind == "huge":  # |x - c| up to 131008: the fp16 residual and the INT2 scale overflow
        x = torch.where(hit, sign * 65504.0, x.float()).half()
        cen = torch.where(torch.rand(cen.shape, generator=g) < 0.1, -65504.0, cen.float()).half()
    elif kind == "boundary":  # residuals at and next to (k + 1/2) times the scale
        cen = torch.zeros_like(cen)
        step = (torch.rand(b, h, t, 1, generator=g) + 0.5).half().float()
        k = torch.randint(0, 8, x.shape, generator=g).float() - 0.5
        x = (sign * k * step).half()
        x[..., 0] = (7.0 * step[..., 0]).half()
    elif kind == "all_tied":  # every magnitude equal: the largest is the threshold itself
        x = (sign * 0.75).half()
        cen = torch.zeros_like(cen)
    elif kind == "near_tied":  # one fp16 magnitude from several fp32 residuals (x is coarser than x - c)
        x = (sign * 512.0).half()
        cen = torch.where(torch.rand(cen.shape, generator=g) < 0.5, 0.01, -0.01).half()
    return x.to(device), cen.to(device), ids.to(device)


def _unaligned(x):
    """x's values in a contiguous tensor that starts two bytes off a 16-byte boundary."""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    out = flat[1:].view(x.shape)
    out.copy_(x)
    assert out.is_contiguous() and out.data_ptr() % 16 == 2
    return out


def _same(a, b):
    return a.shape == b.shape and torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("t", [1, 15, 64, 65, 147])
def test_plane_encoders_equal_the_general_kernels(device, kind, t):
    from reskv_amd._extension import load_extension

    ext = load_extension("compression")
    x, c, ids = _case(kind, 2, 3, t, 5, device)
    calls = {f"quant{bits}/{nnz}": (lambda k, nnz=nnz, bits=bits: ext.compress_quantized(k, c, ids, nnz, bits))
             for bits in (4, 2) for nnz in (32, 64)}
    calls.update({f"tile{nnz}": (lambda k, nnz=nnz: ext.compress_fp16(k, c, ids, nnz, False)) for nnz in (8, 64, 120)})
    calls.update({f"bitmap{nnz}": (lambda k, nnz=nnz: ext.compress_bitmap(k, c, ids, nnz)) for nnz in (1, 32, 64, 127)})
    calls["sint4"] = lambda k: ext.compress_structured_int4(k, c, ids)
    slow = _unaligned(x)
    for name, call in calls.items():
        for got, want in zip(call(x), call(slow)):
            assert _same(got, want), (name, got.dtype)
