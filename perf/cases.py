"""The work that programs using this framework have it do, as measured cases.

Sizes are those of a Llama-3-8B decoder (hidden 4096, intermediate 14336, 32
query and 8 key/value heads of 128, vocabulary 128256), which the benchmark
and the tests use, and smaller ones of the same kind in ``draw``.  A case is a
dict of plain values; its ``kind`` names the entry point it goes through:

  linear   quantized_linear                          (one projection)
  mlp      quantized_mlp_block                       (norm, gate/up, SwiGLU, down)
  attn     paged_gqa_decode_attention                (decode over fp16/bf16 pages)
  qattn    paged_quantized_kv_gqa_decode_attention   (decode over q8/q4 pages)
  verify   paged_verify_attention                    (W draft rows a sequence)
  stack    llama_stack_decode_step                   (layers, and the head if vocab > 0)
  codec    quantize_kv_pages, dequantize_kv_pages    (cache pages to codes and back)

A serving loop checks its positions and lengths once, on the host, where it
makes them; it runs with MK_SKIP_DEVICE_RANGE_CHECKS=1, so that a decode call
does not read them back from the device.
"""

import dataclasses
import math
import os
import sys

os.environ.setdefault("MK_SKIP_DEVICE_RANGE_CHECKS", "1")
sys.path.insert(0, os.path.join(os.getcwd(), "mlx-metal-kernels_amd"))

import torch

from mk import gqa_ops, llama_layer_ops, llama_stack_ops, mlp_block_ops, paged_quantized_kv_ops, quantize_weights
from mk import speculative_verify_ops

DEV = "cuda"
EPS = 1e-5
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32}


def listed():
    mlp = {"kind": "mlp", "hidden": 4096, "inter": 14336, "group": 64, "dtype": "float16", "scale": "float16"}
    heads = {"hq": 32, "hkv": 8, "d": 128, "page": 16}
    return [
        # the smallest call: one projection (o-proj) of a single decoding sequence
        {"name": "linear_q4_m1", "kind": "linear", "rows": 1, "n": 4096, "k": 4096, "bits": 4, "group": 64,
         "dtype": "float16", "scale": "float16"},
        # the MLP block of one decoding sequence: the benchmark's own step
        {"name": "mlp_q4_m1", **mlp, "rows": 1, "bits": 4},
        # four sequences in bf16, the type most checkpoints of this size come in
        {"name": "mlp_q4_bf16_m4", **mlp, "rows": 4, "bits": 4, "dtype": "bfloat16"},
        # a small batch over 8-bit weights in the entry point's default groups of 32
        {"name": "mlp_q8_g32_m8", **mlp, "rows": 8, "bits": 8, "group": 32},
        # a full decode batch
        {"name": "mlp_q4_m32", **mlp, "rows": 32, "bits": 4},
        # a prompt's rows through the block: an odd number of them
        {"name": "mlp_q4_rows509", **mlp, "rows": 509, "bits": 4},
        # attention of one sequence at a short context: latency
        {"name": "attn_b1_2k", "kind": "attn", **heads, "batch": 1, "ctx": 2048, "least": 2048, "dtype": "float16"},
        # sixteen sequences of very different lengths
        {"name": "attn_b16_8k", "kind": "attn", **heads, "batch": 16, "ctx": 8192, "least": 512, "dtype": "float16"},
        # long contexts over a 4-bit cache
        {"name": "qattn_q4_b8_32k", "kind": "qattn", **heads, "batch": 8, "ctx": 32768, "least": 32000, "bits": 4,
         "group": 64, "dtype": "float16"},
        # speculative decoding: five draft rows a sequence, in bf16
        {"name": "verify_w5_bf16_b16", "kind": "verify", **heads, "batch": 16, "ctx": 8192, "least": 512, "width": 5,
         "dtype": "bfloat16"},
        # a decode step of a batch: two layers and the head (the layers repeat)
        {"name": "stack_q4_b32", "kind": "stack", **heads, "batch": 32, "ctx": 2048, "least": 1024, "layers": 2,
         "inter": 14336, "vocab": 128256, "bits": 4, "group": 64, "dtype": "float16"},
        # a prompt's cache pages quantized to 8 bits, and back
        {"name": "codec_q8_b4_8k", "kind": "codec", **heads, "batch": 4, "ctx": 8192, "bits": 8, "group": 64,
         "dtype": "float16"},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "mlp", "attn", "qattn", "verify", "stack", "codec"])
    dtype = rng.choice(["float16", "bfloat16"])
    c = {"kind": kind, "dtype": dtype}
    if kind in ("linear", "mlp"):
        c.update(rows=_log(rng, 1, 509), bits=rng.choice([4, 4, 8]), group=rng.choice([32, 64, 64, 128]),
                 scale=rng.choice(["float16"] * 5 + ["float32"]))
        if kind == "linear":  # rows of any number (a vocabulary's head), columns in whole 32s
            return {**c, "n": _log(rng, 512, 33000), "k": 32 * _log(rng, 32, 448)}
        return {**c, "hidden": 128 * rng.randint(8, 32), "inter": 32 * _log(rng, 64, 448)}
    d, hkv = rng.choice([64, 128, 128]), rng.choice([1, 2, 4, 8, 8])
    c.update(d=d, hkv=hkv, hq=hkv * rng.choice([1, 4, 4, 7, 8]), page=rng.choice([8, 16, 16, 32, 64]))
    if kind == "stack":
        hidden_heads = {64: [16, 32, 48], 128: [8, 16, 32]}[d]
        hq = rng.choice(hidden_heads)
        ctx = _log(rng, 64, 2048)
        return {**c, "hq": hq, "hkv": rng.choice([h for h in (2, 4, 8) if hq % h == 0]), "page": rng.choice([16, 32]),
                "batch": _log(rng, 1, 32), "ctx": ctx, "least": max(1, ctx // 2), "layers": rng.randint(1, 2),
                "inter": 64 * rng.randint(hq * d // 64 + 1, 224),
                "vocab": rng.choice([0, 1000, 32000]), "bits": rng.choice([4, 4, 8]), "group": rng.choice([32, 64, 128])}
    batch = _log(rng, 1, 32)
    ctx = _log(rng, 100, min(32768, 131072 // batch))
    c.update(batch=batch, ctx=ctx)
    if kind == "codec":
        return {**c, "bits": rng.choice([4, 8]), "group": rng.choice([32, 64])}
    c["least"] = max(1, ctx // rng.choice([1, 2, 16]))
    if kind == "verify":
        return {**c, "width": rng.choice([2, 3, 4, 5, 8]), "least": max(16, c["least"])}
    if kind == "qattn":
        return {**c, "bits": rng.choice([4, 8]), "group": rng.choice([32, 64]), "dtype": "float16"}
    return c


# ----------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * int(seed) + 17)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32).to(dtype)


def _weight(gen, n, k, c):
    """A projection as a checkpoint's would be: N(0, 0.02), quantized by the framework."""
    w = torch.randn((n, k), generator=gen, device=DEV, dtype=torch.float32).mul_(0.02)
    q = quantize_weights.quantize_weight_groupwise(
        w, quantize_weights.QuantizationConfig(bits=c["bits"], group_size=c["group"], dtype=c["scale"]))
    return q.packed_weight, q.scales, q.kernel_zeros()


def _lengths(gen, c):
    return torch.randint(c["least"], c["ctx"] + 1, (c["batch"],), generator=gen, device=DEV, dtype=torch.int32)


def _table(gen, batch, positions, page):
    """A block table whose pages lie in any order, as in a cache in use."""
    mb = -(-positions // page)
    return torch.randperm(batch * mb, generator=gen, device=DEV).to(torch.int32).reshape(batch, mb)


def _pages(gen, c, table):
    shape = (table.numel(), c["page"], c["hkv"], c["d"])
    return _randn(gen, shape, DTYPES[c["dtype"]]), _randn(gen, shape, DTYPES[c["dtype"]])


def prepare(case, seed):
    c, gen = case, _gen(seed)
    dtype = DTYPES[c["dtype"]]
    kind = c["kind"]
    if kind == "linear":
        w = _weight(gen, c["n"], c["k"], c)
        return {"case": c, "w": w, "x": _randn(gen, (c["rows"], c["k"]), dtype)}
    if kind == "mlp":
        h, i = c["hidden"], c["inter"]
        gate, up, down = _weight(gen, i, h, c), _weight(gen, i, h, c), _weight(gen, h, i, c)
        # decode batches are rows of one position each, a prompt is one sequence
        shape = (c["rows"], 1, h) if c["rows"] <= 64 else (1, c["rows"], h)
        norm = (1.0 + 0.1 * torch.randn(h, generator=gen, device=DEV)).to(dtype)
        return {"case": c, "gate": gate, "up": up, "down": down, "norm": norm, "x": _randn(gen, shape, dtype),
                "residual": _randn(gen, shape, dtype)}
    if kind == "stack":
        cfg = _config(c)
        weights = llama_stack_ops.create_random_quantized_llama_stack_weights(
            cfg, vocab_size=c["vocab"] or None, bits=c["bits"], group_size=c["group"], dtype=dtype, seed=int(seed),
            device=DEV, include_embedding=False, include_lm_head=c["vocab"] > 0)
        for layer in weights.layers:
            layer.input_layernorm_weight.add_(0.1 * _randn(gen, (cfg.hidden_size,), dtype))
            layer.post_attention_layernorm_weight.add_(0.1 * _randn(gen, (cfg.hidden_size,), dtype))
        table = _table(gen, c["batch"], c["ctx"] + 1, c["page"])
        cache = llama_stack_ops.init_llama_stack_cache(cfg, c["batch"], c["ctx"] + 1, cache_layout="paged", dtype=dtype,
                                                       page_size=c["page"], device=DEV, block_table=table)
        for k, v, _ in cache.layer_caches:
            k.normal_(generator=gen)
            v.normal_(generator=gen)
        cos, sin = llama_layer_ops.build_rope_tables(cfg, device=DEV)
        return {"case": c, "cfg": cfg, "weights": weights, "cache": cache, "cos": cos, "sin": sin,
                "pos": _lengths(gen, c), "x": _randn(gen, (c["batch"], 1, cfg.hidden_size), dtype)}
    table = _table(gen, c["batch"], c["ctx"], c["page"])
    k, v = _pages(gen, c, table)
    if kind == "codec":
        return {"case": c, "k": k, "v": v, "table": table,
                "lengths": torch.full((c["batch"],), c["ctx"], dtype=torch.int32, device=DEV),
                "config": paged_quantized_kv_ops.PagedQuantizedKVConfig(bits=c["bits"], page_size=c["page"],
                                                                        group_size=c["group"])}
    lengths = _lengths(gen, c)
    q = _randn(gen, (c["batch"], c.get("width", 1), c["hq"], c["d"]), dtype)
    state = {"case": c, "q": q, "table": table, "lengths": lengths}
    if kind == "qattn":
        state["cache"] = paged_quantized_kv_ops.quantize_kv_pages(
            k, v, table, lengths, paged_quantized_kv_ops.PagedQuantizedKVConfig(
                bits=c["bits"], page_size=c["page"], group_size=c["group"]))
    else:
        state.update(k=k, v=v)
    return state


def _config(c):
    cfg = llama_layer_ops.llama3_8b_like()
    return dataclasses.replace(cfg, hidden_size=c["hq"] * c["d"], intermediate_size=c["inter"],
                               num_attention_heads=c["hq"], num_key_value_heads=c["hkv"], head_dim=c["d"],
                               num_hidden_layers=c["layers"], vocab_size=c["vocab"] or None)


# ----------------------------------------------------------------- one pass


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "linear":
        w, scales, zeros = s["w"]
        return mlp_block_ops.quantized_linear(s["x"], w, scales, zeros, bits=c["bits"], group_size=c["group"])
    if kind == "mlp":
        (gw, gs, gz), (uw, us, uz), (dw, ds, dz) = s["gate"], s["up"], s["down"]
        return mlp_block_ops.quantized_mlp_block(
            s["x"], s["residual"], s["norm"], gw, gs, uw, us, dw, ds, gate_zeros=gz, up_zeros=uz, down_zeros=dz,
            bits=c["bits"], group_size=c["group"], eps=EPS, backend_preset="fused_experimental")
    if kind == "attn":
        return gqa_ops.paged_gqa_decode_attention(s["q"], s["k"], s["v"], s["table"], s["lengths"])
    if kind == "qattn":
        return paged_quantized_kv_ops.paged_quantized_kv_gqa_decode_attention(s["q"], s["cache"],
                                                                              backend=f"metal_q{c['bits']}")
    if kind == "verify":
        return speculative_verify_ops.paged_verify_attention(s["q"], s["k"], s["v"], s["table"], s["lengths"])
    if kind == "stack":
        got = llama_stack_ops.llama_stack_decode_step(s["x"], s["weights"], s["cache"], s["cos"], s["sin"], s["pos"],
                                                      s["cfg"])
        pages = [(k, v) for k, v, _ in got[-1].layer_caches]
        return {"outputs": list(got[:-1]), "pages": pages}
    cache = paged_quantized_kv_ops.quantize_kv_pages(s["k"], s["v"], s["table"], s["lengths"], s["config"])
    k, v = paged_quantized_kv_ops.dequantize_kv_pages(cache)
    return {"codes": [cache.k_pages_q, cache.v_pages_q], "scales": [cache.k_scales, cache.v_scales], "pages": [k, v]}


# ----------------------------------------------------------------- what a pass cannot do without


def _weight_bytes(n, k, c):
    scale = 4 if c.get("scale") == "float32" else 2
    return n * math.ceil(k * c["bits"] / 8) + 2 * scale * n * math.ceil(k / c["group"])


def _kv_bytes(c):
    """Bytes of one position of K and V of every kv head."""
    if c["kind"] == "qattn":
        return 2 * c["hkv"] * (c["d"] * c["bits"] // 8 + 2 * math.ceil(c["d"] / c["group"]))
    return 2 * c["hkv"] * c["d"] * 2


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        m, n, k = c["rows"], c["n"], c["k"]
        return {"bytes": _weight_bytes(n, k, c) + 2 * m * (n + k), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, i = c["rows"], c["hidden"], c["inter"]
        return {"bytes": 2 * _weight_bytes(i, h, c) + _weight_bytes(h, i, c) + 2 * (3 * m * h + h),
                "flops": 6 * m * h * i}
    if kind == "codec":
        values = 2 * c["batch"] * math.ceil(c["ctx"] / c["page"]) * c["page"] * c["hkv"] * c["d"]
        # pages in, codes and scales out; the codes and scales in again, pages out
        return {"bytes": 4 * values + 2 * (values * c["bits"] // 8 + 2 * values // c["group"]), "flops": 0}
    seen = c["batch"] * (c["least"] + c["ctx"]) / 2  # positions, on the average over the lengths drawn
    rows = c["batch"] * c.get("width", 1)
    heads = rows * c["hq"] * c["d"]
    flops = 4 * seen * c.get("width", 1) * c["hq"] * c["d"]
    if kind != "stack":
        return {"bytes": seen * _kv_bytes(c) + 4 * heads, "flops": flops}
    h, i, kv = c["hq"] * c["d"], c["inter"], c["hkv"] * c["d"]
    shapes = [(h + 2 * kv, h), (h, h), (i, h), (i, h), (h, i)]
    weights = sum(_weight_bytes(n, k, c) for n, k in shapes)
    products = sum(n * k for n, k in shapes)
    total = c["layers"] * (weights + seen * _kv_bytes(c) + c["batch"] * _kv_bytes(c))
    ops = c["layers"] * (2 * c["batch"] * products + flops)
    if c["vocab"]:
        total += _weight_bytes(c["vocab"], h, c) + 4 * c["batch"] * c["vocab"]
        ops += 2 * c["batch"] * c["vocab"] * h
    return {"bytes": total + 2 * 2 * c["batch"] * h, "flops": ops}


def tolerance(case):
    """About four times the error against ``exact`` that was measured for each kind."""
    c = case
    if c["kind"] == "codec":  # codes and the values they stand for
        return "exact"
    half = c["dtype"] == "float16"
    if c["kind"] == "linear":  # weights and results rounded once each: 2.1e-4, 2.0e-3
        return {"rel": 1e-3 if half else 8e-3}
    if c["kind"] == "mlp":  # and the intermediates: 6.5e-4, 5.4e-3
        return {"rel": 2.6e-3 if half else 2e-2}
    if c["kind"] == "stack":  # the roundings of every stage of one or two layers: 1.0e-3
        return {"rel": 4e-3 if half else 3e-2}
    return {"rel": 1.6e-3 if half else 1e-2}  # attention: the probabilities and the results, 4.1e-4, 2.3e-3


# ----------------------------------------------------------------- the same in 64 bits


def _dequant(w, c, k):
    codes, scales, zeros = w
    if c["bits"] == 4:
        codes = torch.stack((codes & 15, codes >> 4), dim=-1).reshape(codes.shape[0], -1)[:, :k]
    full = scales.double().repeat_interleave(c["group"], dim=1)[:, :k]
    zero = zeros.double().repeat_interleave(c["group"], dim=1)[:, :k]
    return codes.double().sub_(zero).mul_(full)


def _product(x, w, c):
    return x @ _dequant(w, c, x.shape[-1]).t()


def _norm(x, weight):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + EPS) * weight.double()


def _mlp(z, norm, gate, up, down, c):
    n = _norm(z, norm)
    return z + _product(torch.nn.functional.silu(_product(n, gate, c)) * _product(n, up, c), down, c)


def _attend(q, k, v, table, lengths, width=1):
    """q [B,W,Hq,D] over pages; row w sees the positions below its length - (W - 1 - w)."""
    out = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
    hkv, d = k.shape[2], k.shape[3]
    for b, n in enumerate(lengths.tolist()):
        pages = table[b, : -(-n // k.shape[1])].long()
        ks = k[pages].reshape(-1, hkv, d)[:n].double().permute(1, 0, 2)
        vs = v[pages].reshape(-1, hkv, d)[:n].double().permute(1, 0, 2)
        rows = q[b].double().reshape(width, hkv, -1, d).permute(1, 0, 2, 3)  # [Hkv, W, G, D]
        scores = rows.reshape(hkv, -1, d).contiguous() @ ks.transpose(1, 2).contiguous() / math.sqrt(d)
        scores = scores.reshape(hkv, width, -1, n)
        end = n - (width - 1 - torch.arange(width, device=DEV))
        scores.masked_fill_((torch.arange(n, device=DEV)[None, :] >= end[:, None])[None, :, None, :], -math.inf)
        got = torch.softmax(scores, dim=-1).reshape(hkv, -1, n) @ vs.contiguous()
        out[b] = got.reshape(hkv, width, -1, d).permute(1, 0, 2, 3).reshape(width, -1, d)
    return out


def _rope(x, cos, sin):
    """x [B,H,D], the even and odd neighbours turned by cos, sin [B,D/2]."""
    e, o, cos, sin = x[..., 0::2], x[..., 1::2], cos[:, None], sin[:, None]
    return torch.stack((e * cos - o * sin, e * sin + o * cos), dim=-1).reshape(x.shape)


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    kind = c["kind"]
    if kind == "linear":
        return _product(s["x"].double(), s["w"], c)
    if kind == "mlp":
        z = s["x"].double() + s["residual"].double()
        return _mlp(z, s["norm"], s["gate"], s["up"], s["down"], c)
    if kind in ("attn", "verify"):
        return _attend(s["q"], s["k"], s["v"], s["table"], s["lengths"], c.get("width", 1))
    if kind == "qattn":
        cache = s["cache"]
        off = 128 if c["bits"] == 8 else 8

        def pages(codes, scales):
            if c["bits"] == 4:
                codes = torch.stack((codes & 15, codes >> 4), dim=-1).reshape(*codes.shape[:-1], -1)
            return (codes.float() - off) * scales.float().repeat_interleave(c["group"], dim=-1)[..., : c["d"]]

        return _attend(s["q"], pages(cache.k_pages_q, cache.k_scales), pages(cache.v_pages_q, cache.v_scales),
                       s["table"], s["lengths"])
    if kind == "codec":
        top = 127 if c["bits"] == 8 else 7

        def scales(x):
            return x.double().unflatten(-1, (-1, c["group"])).abs().amax(dim=-1).clamp(min=1e-8) / top

        return {"codes": [None, None], "scales": [scales(s["k"]), scales(s["v"])], "pages": [None, None]}
    x, b, hq, hkv, d = s["x"][:, 0].double(), c["batch"], c["hq"], c["hkv"], c["d"]
    pos = s["pos"].long()
    cos, sin = s["cos"][pos].double(), s["sin"][pos].double()
    slot = torch.arange(b, device=DEV), pos // c["page"], pos % c["page"]
    done = []
    for lw, (kp, vp, table) in zip(s["weights"].layers, s["cache"].layer_caches):
        qkv = _product(_norm(x, lw.input_layernorm_weight), (lw.qkv_w, lw.qkv_scales, lw.qkv_zeros), c)
        q, k, v = qkv.split([hq * d, hkv * d, hkv * d], dim=1)
        kp, vp, page = kp.double(), vp.double(), table[slot[0], slot[1]].long()
        kp[page, slot[2]] = _rope(k.reshape(b, hkv, d), cos, sin)
        vp[page, slot[2]] = v.reshape(b, hkv, d)
        att = _attend(_rope(q.reshape(b, hq, d), cos, sin)[:, None], kp, vp, table, s["pos"] + 1)
        h = x + _product(att.reshape(b, -1), (lw.o_w, lw.o_scales, lw.o_zeros), c)
        x = _mlp(h, lw.post_attention_layernorm_weight, (lw.gate_w, lw.gate_scales, lw.gate_zeros),
                 (lw.up_w, lw.up_scales, lw.up_zeros), (lw.down_w, lw.down_scales, lw.down_zeros), c)
        done.append((kp, vp))
    final = _norm(x, s["weights"].final_norm_weight)
    outputs = [final[:, None]]
    head = s["weights"].lm_head
    if head is not None:
        outputs = [_product(final, (head.w, head.scales, head.zeros), c)[:, None]] + outputs
    return {"outputs": outputs, "pages": done}
