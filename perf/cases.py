"""What this framework's users have it do, as cases that can be timed and compared.

Six kinds, each through an entry point that a program calls:

* ``decode``   -- ``attention``: one decode step of one layer over a compressed history, for every residual
  format, with or without a dense recent window (the step that a served token pays for in each layer);
* ``encode``   -- ``compress`` with a given clustering: the residual encoders alone;
* ``compress`` -- ``compress`` of a prompt's K and V of one layer: K-means and encoding (prefill);
* ``layer``    -- a ``ResKVLayerCache`` from its prompt through decode steps, long enough that the ring of
  recent tokens fills and a group is compressed into the history;
* ``prefill``  -- ``RandomLlama.prefill``: the prompt pass of the end-to-end decoder;
* ``model``    -- ``ResKVForCausalLM``: prompt and teacher-forced continuation steps of a transformers model.

Shapes are the Llama-3.1-8B layer's (32 query heads, 8 KV heads, 128 channels, theta 500000) unless a case
says otherwise; keys have per-channel scales with a few outlier channels, values are N(0, 1).
"""

import math

import torch

from reskv_amd import ResKVKernelConfig, attention, compress
from reskv_amd.cache import ResKVLayerCache
from reskv_amd.llama import LlamaShape, RandomLlama

D = 128
THETA = 500000.0
DEVICE = "cuda"

# residual formats: (sparsity, bits, layout)
FORMATS = {
    "bitmap50": (0.5, 16, "unstructured"),  # default at 50%
    "bitmap75": (0.75, 16, "unstructured"),
    "struct75": (0.75, 16, "structured"),  # default at 75%
    "tiled50": (0.5, 16, "tiled"),
    "int4": (0.5, 4, "unstructured"),
    "int2": (0.5, 2, "unstructured"),
    "sint4": (0.75, 4, "structured"),  # structured INT4
}


def listed():
    return [
        # a single short conversation: one sequence, 1K tokens with its recent window; latency and launches
        {"name": "decode_b1_t960_bitmap50", "kind": "decode", "fmt": "bitmap50", "b": 1, "kv": 8, "gqa": 4,
         "t": 960, "start": 0, "recent": 64},
        # a few sequences at the 8K context, default format at 75%, ring in use
        {"name": "decode_b4_t8192_struct75", "kind": "decode", "fmt": "struct75", "b": 4, "kv": 8, "gqa": 4,
         "t": 8192, "start": 0, "recent": 48},
        # full serving batch at the 8K context, default format at 50%
        {"name": "decode_b32_t8192_bitmap50", "kind": "decode", "fmt": "bitmap50", "b": 32, "kv": 8, "gqa": 4,
         "t": 8192, "start": 0, "recent": 0},
        # long context with quantised residuals
        {"name": "decode_b8_t16384_int4", "kind": "decode", "fmt": "int4", "b": 8, "kv": 8, "gqa": 4,
         "t": 16384, "start": 0, "recent": 0},
        # odd batch and length, structured INT4, 8 query heads per KV head, sink tokens in front
        {"name": "decode_b5_t5003_sint4_gqa8", "kind": "decode", "fmt": "sint4", "b": 5, "kv": 4, "gqa": 8,
         "t": 5003, "start": 4, "recent": 31},
        # residual encoders at the long context, INT4
        {"name": "encode_b8_t16384_int4", "kind": "encode", "fmt": "int4", "b": 8, "kv": 8, "t": 16384, "c": 32},
        # prefill compression of one prompt, 75%
        {"name": "compress_b1_t8192_struct75", "kind": "compress", "fmt": "struct75", "b": 1, "kv": 8, "t": 8192,
         "c": 32, "iterations": 10},
        # prefill compression of a batch of prompts (8192 less the recent window, whole groups), 75%
        {"name": "compress_b16_t8128_struct75", "kind": "compress", "fmt": "struct75", "b": 16, "kv": 8, "t": 8128,
         "c": 32, "iterations": 10},
        # a short ragged prompt with more centroids and iterations, 50%
        {"name": "compress_b3_t1999_bitmap50", "kind": "compress", "fmt": "bitmap50", "b": 3, "kv": 8, "t": 1999,
         "c": 48, "iterations": 15},
        # one layer of a decode loop: prompt, then 72 tokens (one group compression on the way)
        {"name": "layer_b16_t1056_struct75", "kind": "layer", "fmt": "struct75", "b": 16, "kv": 8, "gqa": 4,
         "t": 1056, "steps": 72, "c": 32, "iterations": 10},
        # prompt pass of the end-to-end decoder, one full-size layer
        {"name": "prefill_b1_t4096", "kind": "prefill", "b": 1, "t": 4096, "hidden": 4096, "kv": 8, "gqa": 4,
         "ffn": 14336, "vocab": 1000, "layers": 1},
        # a transformers model over the cache: prompt and 64 continuation tokens
        {"name": "model_b2_t300", "kind": "model", "fmt": "struct75", "b": 2, "t": 300, "steps": 64, "hidden": 512,
         "kv": 1, "gqa": 4, "ffn": 1024, "vocab": 1000, "layers": 2, "c": 8, "iterations": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["encode"] * 2 + ["compress"] * 3 + ["layer", "prefill"])
    fmt = rng.choice(sorted(FORMATS))
    if kind == "decode":
        kv = rng.choice([1, 2, 4, 8, 8, 8])
        t = _log(rng, 64, 32768)
        most = max(1, min(32, 32 * 8 * 8192 // (kv * t)))
        return {"kind": kind, "fmt": fmt, "b": _log(rng, 1, most), "kv": kv, "gqa": rng.choice([1, 4, 4, 4, 8]),
                "t": t, "start": rng.choice([0, 0, 4]), "recent": rng.choice([0, rng.randint(1, 200)])}
    if kind == "encode":
        kv, t = rng.choice([1, 4, 8]), _log(rng, 64, 16384)
        most = max(1, min(16, 16 * 8 * 8192 // (kv * t)))
        return {"kind": kind, "fmt": fmt, "b": _log(rng, 1, most), "kv": kv, "t": t, "c": rng.randint(4, 64)}
    if kind == "compress":
        kv, t = rng.choice([1, 4, 8, 8]), _log(rng, 64, 16384)
        most = max(1, min(16, 16 * 8 * 8128 // (2 * kv * t)))
        return {"kind": kind, "fmt": fmt, "b": _log(rng, 1, most), "kv": kv, "t": t,
                "c": rng.choice([16, 32, 32, 48, 64]), "iterations": rng.choice([5, 10, 15])}
    if kind == "layer":
        return {"kind": kind, "fmt": fmt, "b": _log(rng, 1, 16), "kv": 8, "gqa": 4, "t": _log(rng, 128, 2048),
                "steps": rng.randint(8, 80), "c": 32, "iterations": 10}
    return {"kind": kind, "b": rng.choice([1, 1, 2]), "t": _log(rng, 200, 2048), "hidden": rng.choice([1024, 4096]),
            "kv": 2, "gqa": 4, "ffn": rng.choice([2816, 14336]), "vocab": 1000, "layers": rng.choice([1, 2])}


def _config(case):
    sparsity, bits, layout = FORMATS[case["fmt"]]
    extra = {}
    if "c" in case:
        extra.update(num_clusters=case["c"])
    if "iterations" in case:
        extra.update(kmeans_iterations=case["iterations"])
    return ResKVKernelConfig(sparsity=sparsity, bits=bits, layout=layout, **extra)


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _kv(g, b, kv, t):
    """Keys N(0, 1) with log-normal channel scales and four outlier channels per head; values N(0, 1)."""
    scale = torch.exp(torch.randn(1, kv, 1, D, device=DEVICE, generator=g))
    outlier = torch.rand(1, kv, 1, D, device=DEVICE, generator=g).argsort(-1) < 4
    scale = torch.where(outlier, scale * 10.0, scale)
    k = torch.empty(b, kv, t, D, device=DEVICE, dtype=torch.float16)
    v = torch.empty_like(k)
    for i in range(b):
        k[i] = (torch.randn(kv, t, D, device=DEVICE, generator=g) * scale[0]).half()
        v[i] = torch.randn(kv, t, D, device=DEVICE, generator=g).half()
    return k, v


def _clusters(g, x, c):
    """Centroids near some of the tokens' mean directions and a random assignment, as a controlled benchmark has them."""
    b, kv, t, _ = x.shape
    pick = torch.randint(t, (c,), device=DEVICE, generator=g)
    centers = (x[:, :, pick].float() * 0.25).half()
    return centers, torch.randint(c, (b, kv, t), device=DEVICE, dtype=torch.int32, generator=g)


def _frequencies():
    return (THETA ** (-torch.arange(64, device=DEVICE).float() / 64)).float()


def _rotate(x, pos, freq):
    """Rotate-half RoPE of x [..., 128] at positions broadcastable to x.shape[:-1]."""
    ang = pos[..., None].to(x.dtype) * freq.to(x.dtype)
    c, s = torch.cos(ang), torch.sin(ang)
    a, b = x[..., :64], x[..., 64:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _decode_inputs(case, seed):
    """(K, V, clusterings, pre-RoPE query, recent window or None, query position)."""
    g = _gen(seed)
    b, kv, t, hq = case["b"], case["kv"], case["t"], case["kv"] * case["gqa"]
    k, v = _kv(g, b, kv, t)
    clusters = _clusters(g, k, 32), _clusters(g, v, 32)
    # queries as large as scaled attention logits of a few units need them with these keys
    q = (torch.randn(b, hq, 1, D, device=DEVICE, generator=g) * 0.5).half()
    pos = case["start"] + t + case["recent"]
    recent = None
    if case["recent"]:
        rk, rv = _kv(g, b, kv, case["recent"])
        at = case["start"] + t + torch.arange(case["recent"], device=DEVICE)
        q_rot = _rotate(q.float(), torch.full((1,), pos, device=DEVICE), _frequencies()).half()
        recent = (q_rot, _rotate(rk.float(), at, _frequencies()).half(), rv)
    return k, v, clusters, q, recent, pos


def _encode_inputs(case, seed):
    g = _gen(seed)
    k, v = _kv(g, case["b"], case["kv"], case["t"])
    kc = _clusters(g, k, case["c"])
    return (k, kc), (v, _clusters(g, v, case["c"]))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        k, v, clusters, q, recent, pos = _decode_inputs(case, seed)
        cache = compress(k, v, _config(case), clustering=clusters)
        return {"kind": kind, "cache": cache, "q": q, "recent": recent, "position": pos, "start": case["start"],
                "freq": _frequencies()}
    g = _gen(seed)
    if kind == "encode":
        (k, kc), (v, vc) = _encode_inputs(case, seed)
        return {"kind": kind, "k": k, "v": v, "config": _config(case), "clusters": (kc, vc)}
    if kind == "compress":
        k, v = _kv(g, case["b"], case["kv"], case["t"])
        return {"kind": kind, "k": k, "v": v, "config": _config(case)}
    if kind == "layer":
        b, kv, t, steps = case["b"], case["kv"], case["t"], case["steps"]
        k, v = _kv(g, b, kv, t + steps)
        rot = _rotate(k.float(), torch.arange(t + steps, device=DEVICE), _frequencies()).half()
        q = (torch.randn(b, kv * case["gqa"], steps, D, device=DEVICE, generator=g) * 0.5).half()
        q_rot = _rotate(q.float(), t + torch.arange(steps, device=DEVICE), _frequencies()).half()
        one = lambda x, i: x[:, :, i: i + 1].contiguous()  # noqa: E731
        return {"kind": kind, "config": _config(case), "freq": _frequencies(),
                "prompt": tuple(x[:, :, :t].contiguous() for x in (rot, v, k)),
                "tokens": [tuple(one(x, t + i) for x in (rot, v, k)) + (one(q, i), one(q_rot, i))
                           for i in range(steps)]}
    if kind == "prefill":
        shape = LlamaShape(layers=case["layers"], hidden=case["hidden"], heads=case["hidden"] // D,
                           kv_heads=case["kv"], ffn=case["ffn"], vocab=case["vocab"])
        ids = torch.randint(case["vocab"], (case["b"], case["t"]), device=DEVICE, generator=g)
        return {"kind": kind, "model": RandomLlama(shape, DEVICE, seed=seed), "ids": ids}
    return {"kind": kind, **_transformers_model(case, seed)}


def _transformers_model(case, seed):
    from transformers import LlamaConfig

    from reskv_amd import ResKVForCausalLM

    torch.manual_seed(seed)
    config = LlamaConfig(vocab_size=case["vocab"], hidden_size=case["hidden"], intermediate_size=case["ffn"],
                         num_hidden_layers=case["layers"], num_attention_heads=case["hidden"] // D,
                         num_key_value_heads=case["kv"], max_position_embeddings=8192)
    model = ResKVForCausalLM(config, _config(case)).half().to(DEVICE).eval()
    ids = torch.randint(case["vocab"], (case["b"], case["t"] + case["steps"]), device=DEVICE, generator=_gen(seed))
    return {"model": model, "ids": ids, "prompt": case["t"]}


def _stored(cache):
    return [{"centroids": x.centroids, "ids": x.cluster_ids, "payload": x.payload, "metadata": x.metadata,
             "scale": x.scale} for x in (cache.key, cache.value)]


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind == "decode":
        return attention(state["q"], state["cache"], position=state["position"], start_position=state["start"],
                         inv_freq=state["freq"], recent=state["recent"])
    if kind == "encode":
        return _stored(compress(state["k"], state["v"], state["config"], clustering=state["clusters"]))
    if kind == "compress":
        return _stored(compress(state["k"], state["v"], state["config"]))
    if kind == "layer":
        layer = ResKVLayerCache(state["config"])
        rot, v, raw = state["prompt"]
        layer.update(rot, v, {"raw_keys": raw})
        out = []
        for rot, v, raw, q, q_rot in state["tokens"]:
            layer.update(rot, v, {"raw_keys": raw})
            if layer.compressed is not None:  # else the ring alone: dense attention, not this path
                out.append(layer.attend(q, q_rot, scaling=D ** -0.5, inv_freq=state["freq"],
                                        out=torch.empty_like(q)))
        return {"out": torch.stack(out) if out else None, "ring": layer.keys[:, :, : layer.live]}
    if kind == "prefill":
        kept = []
        logits = state["model"].prefill(state["ids"], lambda li, raw, rot, v: kept.append((raw, rot, v)), logits=True)
        return {"logits": logits, "kv": kept}
    ids, n = state["ids"], state["prompt"]
    got = state["model"](ids[:, :n], use_cache=True)
    logits = [got.logits[:, -1]]
    for i in range(n, ids.shape[1]):
        got = state["model"](ids[:, i: i + 1], past_key_values=got.past_key_values, use_cache=True)
        logits.append(got.logits[:, -1])
    return torch.stack(logits, dim=1)


# ---------------------------------------------------------------------------
# work, tolerance, exact results
# ---------------------------------------------------------------------------

def _token_bytes(fmt):
    """Stored bytes per token of one tensor: int8 id, payload, metadata, scale."""
    sparsity, bits, layout = FORMATS[fmt]
    if bits == 16:
        return 1 + 2 * int(D * (1 - sparsity)) + 16
    return 1 + 16 + 8 + 2 if layout == "structured" else 1 + 16 * bits + 2


def _decode_work(fmt, b, kv, gqa, t, recent, c=32):
    rows, hq = b * kv, b * kv * gqa
    return (rows * (2 * t * _token_bytes(fmt) + 2 * c * D * 2 + 2 * recent * D * 2) + (3 if recent else 2) * hq * D * 2,
            4 * hq * (t + recent) * D)


def _compress_work(fmt, b, kv, t, c, iterations):
    rows = 2 * b * kv
    return rows * (t * (2 * D + _token_bytes(fmt)) + c * D * 2), rows * t * (2 * D * c * iterations + 4 * D)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        by, fl = _decode_work(case["fmt"], case["b"], case["kv"], case["gqa"], case["t"], case["recent"])
    elif kind == "encode":
        rows = 2 * case["b"] * case["kv"]
        by = rows * (case["t"] * (2 * D + 4 + _token_bytes(case["fmt"])) + case["c"] * D * 2)
        fl = rows * case["t"] * D * 4
    elif kind == "compress":
        by, fl = _compress_work(case["fmt"], case["b"], case["kv"], case["t"], case["c"], case["iterations"])
    elif kind == "layer":
        kept = max(0, case["t"] - 32) // 64 * 64
        by, fl = _compress_work(case["fmt"], case["b"], case["kv"], kept, case["c"], case["iterations"])
        for i in range(case["steps"]):
            recent = case["t"] + i + 1 - kept
            if recent >= 96:
                kept, recent = kept + 64, recent - 64
            a, f = _decode_work(case["fmt"], case["b"], case["kv"], case["gqa"], kept, recent)
            by, fl = by + a, fl + f
    else:
        b, t, h, f, kvd = case["b"], case["t"], case["hidden"], case["ffn"], case["kv"] * D
        per = h * (2 * h + 2 * kvd) + 3 * h * f
        head = case["vocab"] * h
        steps = case.get("steps", 0)
        by = (1 + steps) * 2 * (case["layers"] * per + head) + 2 * b * t * h
        fl = 2 * b * ((t + steps) * case["layers"] * per + (1 + steps) * head) + case["layers"] * 2 * b * t * t * h
        if kind == "prefill":
            by += case["layers"] * 3 * b * t * kvd * 2
    return {"bytes": by, "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 2e-3, "max": 2e-2}  # fp16 results of weights rounded to fp16: 11 bits
    if kind == "encode":
        return "exact"  # masks, codes and stored residuals are determined bit for bit
    if kind == "compress":
        # Another order of the centroid sums moves a token that lies between two centroids now and then
        # (none to 0.09% of a tensor's ids), and with it the whole stored row.
        return {"rel": 0.03, "max": 0.99, "differ": 0.004}
    if kind == "layer":
        return {"rel": 4e-3, "max": 0.1}
    return {"rel": 8e-3, "max": 0.1}  # fp16 layers: the prompt pass is within 2e-3 of 64 bits


def _kept(x, centers, ids, fmt):
    """(fp32 residuals, kept mask) of x [H, T, 128] against its centroids: the largest |fp16(residual)| per
    token (unstructured), per 16 channels (tiled, 4:16) or per 4 (structured INT4), lower channels on ties."""
    sparsity, bits, layout = FORMATS[fmt]
    r = x.float() - torch.gather(centers, 1, ids.long()[..., None].expand_as(x)).float()
    mag = r.half().abs()
    h, t, _ = r.shape
    if layout == "unstructured":
        width, keep = D, int(D * (1 - sparsity))
    elif bits == 4:
        width, keep = 4, 1
    else:
        width, keep = 16, int(16 * (1 - sparsity))
    groups = mag.view(h, t, D // width, width)
    order = groups.sort(dim=-1, descending=True, stable=True).indices
    mask = torch.zeros_like(groups, dtype=torch.bool).scatter_(-1, order[..., :keep], True)
    return r, mask.view(h, t, D)


def _scale(r, mask, bits, layout):
    """fp32 magnitude that one code step stands for, before its rounding to fp16 (all-zero rows: 1)."""
    amax = torch.where(mask, r, torch.zeros_like(r)).abs().amax(-1, keepdim=True)
    step = amax * (1.0 / 7.0) if layout == "structured" else amax / float((1 << (bits - 1)) - 1)
    return torch.where(amax > 0, step, torch.ones_like(step))


def _reconstructed(x, centers, ids, fmt):
    """float64 [H, T, 128]: centroid + stored residual."""
    sparsity, bits, layout = FORMATS[fmt]
    r, mask = _kept(x, centers, ids, fmt)
    base = torch.gather(centers, 1, ids.long()[..., None].expand_as(x)).double()
    if bits == 16:
        stored = r.half().double()
    else:
        step = _scale(r, mask, bits, layout)
        top = (1 << (bits - 1)) - 1
        divide = step if layout == "structured" else step.half().float()
        stored = torch.round(r / divide).clamp(-top, top).double() * step.half().double()
    return base + torch.where(mask, stored, torch.zeros_like(stored))


def _exact_decode(case, seed):
    k, v, clusters, q, recent, pos = _decode_inputs(case, seed)
    (kc, ki), (vc, vi) = clusters
    gqa, kv, t = case["gqa"], case["kv"], case["t"]
    freq = _frequencies().double()
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    at = case["start"] + torch.arange(t, device=DEVICE)
    for i in range(case["b"]):
        qd = _rotate(q[i].double(), torch.full((1,), pos, device=DEVICE), freq).view(kv, gqa, D)
        keys = _rotate(_reconstructed(k[i], kc[i], ki[i], case["fmt"]), at, freq)
        vals = _reconstructed(v[i], vc[i], vi[i], case["fmt"])
        score = torch.matmul(qd, keys.transpose(1, 2).contiguous())
        if recent is not None:
            qr = recent[0][i].double().view(kv, gqa, D)
            score = torch.cat((score, torch.matmul(qr, recent[1][i].double().transpose(1, 2).contiguous())), dim=-1)
            vals = torch.cat((vals, recent[2][i].double()), dim=1)
        out[i] = torch.matmul(torch.softmax(score * D ** -0.5, dim=-1), vals).view(kv * gqa, 1, D)
    return out


def _exact_encode(case, seed):
    sparsity, bits, layout = FORMATS[case["fmt"]]
    out = []
    for x, (centers, ids) in _encode_inputs(case, seed):
        payload, scale = [], []
        for i in range(x.shape[0]):
            r, mask = _kept(x[i], centers[i], ids[i], case["fmt"])
            if bits == 16:
                exact = x[i].double() - torch.gather(centers[i], 1, ids[i].long()[..., None].expand_as(x[i])).double()
                payload.append(exact[mask].view(*mask.shape[:2], -1))
            else:
                scale.append(_scale(r.double(), mask, bits, layout)[..., 0])
        out.append({"centroids": centers.double(), "ids": None, "payload": torch.stack(payload) if payload else None,
                    "metadata": None, "scale": torch.stack(scale) if scale else None})
    return out


def _exact_prefill(case, seed):
    """The prompt pass in float64, from the weights that the same seed gives."""
    shape = LlamaShape(layers=case["layers"], hidden=case["hidden"], heads=case["hidden"] // D, kv_heads=case["kv"],
                       ffn=case["ffn"], vocab=case["vocab"])
    model = RandomLlama(shape, DEVICE, seed=seed)  # its weights only
    b, t, hq, kv = case["b"], case["t"], case["hidden"] // D, case["kv"]
    ids = torch.randint(case["vocab"], (b, t), device=DEVICE, generator=_gen(seed))
    freq, at = model.inv_freq.double(), torch.arange(t, device=DEVICE)
    norm = lambda y, w: y * torch.rsqrt(y.square().mean(-1, keepdim=True) + shape.rms_eps) * w.double()  # noqa: E731
    x = model.embed[ids].double()
    kept = []
    for p in model.layers:
        y = torch.matmul(norm(x, p["n1"]), p["wqkv"].double().t())
        q, k, v = y.split((hq * D, kv * D, kv * D), dim=-1)
        q, k, v = (z.view(b, t, -1, D).transpose(1, 2) for z in (q, k, v))
        q, rot = _rotate(q, at, freq), _rotate(k, at, freq)
        kept.append((k, rot, v))
        a = torch.empty(b, t, hq, D, dtype=torch.float64, device=DEVICE)
        mask = torch.ones(t, t, dtype=torch.bool, device=DEVICE).triu(1)
        for i in range(b):
            for h in range(hq):
                j = h // (hq // kv)
                s = torch.mm(q[i, h], rot[i, j].t().contiguous()).mul_(D ** -0.5).masked_fill_(mask, float("-inf"))
                a[i, :, h] = torch.mm(torch.softmax(s, dim=-1), v[i, j])
        x = x + torch.matmul(a.view(b, t, -1), p["wo"].double().t())
        gate, up = torch.matmul(norm(x, p["n2"]), p["wgu"].double().t()).split(case["ffn"], dim=-1)
        x = x + torch.matmul(gate * torch.sigmoid(gate) * up, p["wd"].double().t())
    return {"logits": torch.matmul(norm(x[:, -1], model.norm), model.lm_head.double().t()), "kv": kept}


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "decode":
        return _exact_decode(case, seed)
    if case["kind"] == "encode":
        return _exact_encode(case, seed)
    if case["kind"] == "prefill":
        return _exact_prefill(case, seed)
    return None  # clustering is a sequence of choices: 64 bits make others of them
