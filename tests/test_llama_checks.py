"""Input checks of the end-to-end harness's fused steps (reskv_amd/llama.py),
on the CPU: every mismatch is refused in Python before a pointer reaches the
library (shape, dtype and layout first, then the device)."""

import pytest
import torch
import torch.autograd.forward_ad as forward_ad
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from reskv_amd.llama import LlamaShape, RandomLlama, fused_qkv_rope, fused_rmsnorm, fused_silu_mul

f16 = dict(dtype=torch.float16)


def test_rmsnorm_checks():
    x = torch.zeros(4, 64, **f16)
    w = torch.ones(64, **f16)
    with pytest.raises(ValueError, match="out has 3 rows"):
        fused_rmsnorm(x, w, 1e-5, torch.zeros(3, 64, **f16))
    with pytest.raises(ValueError, match="out has 32 columns"):
        fused_rmsnorm(x, w, 1e-5, torch.zeros(4, 32, **f16))
    with pytest.raises(ValueError, match="x must be a contiguous fp16 matrix"):
        fused_rmsnorm(x.float(), w, 1e-5, torch.zeros(4, 64, **f16))
    with pytest.raises(ValueError, match="x must be a contiguous fp16 matrix"):
        fused_rmsnorm(torch.zeros(64, 4, **f16).t(), w, 1e-5, torch.zeros(4, 64, **f16))
    with pytest.raises(ValueError, match="w must be"):
        fused_rmsnorm(x, torch.ones(32, **f16), 1e-5, torch.zeros(4, 64, **f16))
    with pytest.raises(ValueError, match="CUDA"):
        fused_rmsnorm(x, w, 1e-5, torch.zeros(4, 64, **f16))


def test_silu_mul_checks():
    out = torch.zeros(4, 16, **f16)
    with pytest.raises(ValueError, match="gu has 24 columns, expected 32"):
        fused_silu_mul(torch.zeros(4, 24, **f16), out)
    with pytest.raises(ValueError, match="gu has 5 rows"):
        fused_silu_mul(torch.zeros(5, 32, **f16), out)
    with pytest.raises(ValueError, match="gu must be a contiguous fp16 matrix"):
        fused_silu_mul(torch.zeros(4, 32), out)
    with pytest.raises(ValueError, match="CUDA"):
        fused_silu_mul(torch.zeros(4, 32, **f16), out)


def _qkv_args(b=2, hq=4, hk=1, p=8):
    return dict(qkv=torch.zeros(b, (hq + 2 * hk) * 128, **f16), cos=torch.zeros(p, 64), sin=torch.zeros(p, 64),
                pos=torch.zeros(1, dtype=torch.int64), q=torch.zeros(b, hq, 128, **f16),
                qr=torch.zeros(b, hq, 128, **f16), k=torch.zeros(b, hk, 128, **f16),
                kr=torch.zeros(b, hk, 128, **f16), v=torch.zeros(b, hk, 128, **f16))


@pytest.mark.parametrize("field,value,match", [
    ("qkv", torch.zeros(2, 5 * 128, **f16), "qkv has 640 columns, expected 768"),
    ("qkv", torch.zeros(3, 6 * 128, **f16), "qkv has 3 rows"),
    ("qr", torch.zeros(2, 4, 64, **f16), r"qr must be a contiguous fp16 tensor \[2, 4, 128\]"),
    ("kr", torch.zeros(2, 1, 128), r"kr must be a contiguous fp16 tensor"),
    ("v", torch.zeros(2, 2, 128, **f16), r"v must be a contiguous fp16 tensor \[2, 1, 128\]"),
    ("cos", torch.zeros(8, 64, dtype=torch.float16), "cos and sin must be contiguous fp32 tables"),
    ("sin", torch.zeros(4, 64), "cos and sin must be contiguous fp32 tables"),
    ("sin", torch.zeros(64, 8).t(), "cos and sin must be contiguous fp32 tables"),
    ("pos", torch.zeros(1, dtype=torch.int32), "pos must be an int64 tensor"),
])
def test_qkv_rope_checks(field, value, match):
    args = _qkv_args()
    args[field] = value
    with pytest.raises(ValueError, match=match):
        fused_qkv_rope(**args)


def test_qkv_rope_append_target_checks():
    args = _qkv_args()
    slot = torch.zeros(1, dtype=torch.int64)
    cache = torch.zeros(2, 1, 16, 128, **f16)
    with pytest.raises(ValueError, match="slot must be an int64 tensor"):
        fused_qkv_rope(**args, targets=(cache, cache, cache, None))
    with pytest.raises(ValueError, match="one \\[B, Hk, cap, 128\\] layout"):
        fused_qkv_rope(**args, targets=(cache, cache.float(), cache, slot))
    with pytest.raises(ValueError, match="one \\[B, Hk, cap, 128\\] layout"):
        fused_qkv_rope(**args, targets=(torch.zeros(2, 2, 16, 128, **f16), None, None, slot))
    with pytest.raises(ValueError, match="CUDA"):
        fused_qkv_rope(**args, targets=(cache, cache, cache, slot))


def _cuda_model():
    model = object.__new__(RandomLlama)
    model.shape, model.device, model.scaling = LlamaShape(), torch.device("cuda", 0), 128 ** -0.5
    model.layers = []
    return model


def test_prompts_that_torch_has_to_see_take_the_torch_formulas():
    """Raw-pointer launches are not seen by tracing, modes, transforms or forward-mode levels."""
    model = _cuda_model()
    assert model._fused(64)
    for mode in (FakeTensorMode(), forward_ad.dual_level()):
        with mode:
            assert not model._fused(64)
    seen = []

    def inside(x):
        seen.append(model._fused(64))
        return x * 2

    torch.jit.trace(inside, torch.zeros(2), check_trace=False)
    make_fx(inside)(torch.zeros(2))
    torch.func.vmap(inside)(torch.zeros(2, 2))
    assert len(seen) >= 3 and not any(seen)


@pytest.mark.parametrize("scaling", [0.0, -0.5, float("nan")])
def test_scalings_that_the_prompt_kernel_refuses_take_the_torch_formulas(scaling):
    model = _cuda_model()
    model.scaling = scaling
    assert not model._fused(64)


@pytest.mark.parametrize("name", ["n1", "n2"])
@pytest.mark.parametrize("gains", [torch.ones(4096), torch.ones(8192, **f16)[::2], torch.ones(4104, **f16)[1:4097]])
def test_norm_gains_that_the_kernel_refuses_take_the_torch_formulas(name, gains):
    model = _cuda_model()
    model.layers = [{n: torch.ones(4096, **f16) for n in ("n1", "n2")} for _ in range(2)]
    assert model._fused(64)
    model.layers[1][name] = gains
    assert not model._fused(64)


def test_an_empty_batch_of_prompts_takes_the_torch_formulas(monkeypatch):
    shape = LlamaShape(layers=1, hidden=256, heads=2, kv_heads=1, ffn=64, vocab=50)
    model = RandomLlama(shape, "cpu")
    ids = torch.zeros(0, 5, dtype=torch.int64)
    want = model.prefill(ids, lambda *a: None, logits=True)
    assert want.shape == (0, 50)
    monkeypatch.setattr(RandomLlama, "_fused", lambda self, t: True)
    assert model.prefill(ids, lambda *a: None, logits=True).shape == (0, 50)
