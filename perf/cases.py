"""What is timed: the work an engine has this framework do, through its public
entry points, from a single short decode call to a whole model step.

Families (``kind``):

* ``decode``       one paged decode attention call over one layer's cache
* ``decode_step``  the attention part of a decode step, captured: metadata
                   advance, then per layer q/k norm + RoPE + append + decode
* ``append``       one slot-mapped KV append (copy or quantising)
* ``prefill``      one chunked-prefill call over the paged cache
* ``mixed``        one Attention.forward of a mixed decode + prefill batch
* ``flash``        one full-prefill call over fresh contiguous q / k / v
* ``model``        one captured decode step of a decoder with Qwen3-0.6B layers

Cache formats (``fmt``): ``fp32``, ``bf16``, ``fp16`` (plain), ``fp8``
(per-tensor scales), ``fp8_token`` and ``int8_token`` (one scale per token and
KV head).  A case's sequence lengths follow from its sizes alone; the seed
decides their order, the block tables and every value.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent.parent / "mini-kvllm_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

import mkv  # noqa: E402
from mkv.decode_state import DecodeGraphs, DecodeMetadata  # noqa: E402
from mkv.engine import ModelConfig, Qwen3Model  # noqa: E402
from mkv.producer import qkv_norm_rope_append_decode  # noqa: E402

DEV = "cuda"
CACHE_DTYPE = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16,
               "fp8": torch.float8_e4m3fn, "fp8_token": torch.float8_e4m3fn,
               "int8_token": torch.int8}
ROW_DTYPE = {"fp32": torch.float32, "fp16": torch.float16}  # q / k / v rows; bf16 otherwise
MODE = {"fp8": "fp8_per_tensor", "fp8_token": "fp8_per_token_head",
        "int8_token": "int8_per_token_head"}  # kv_cache_dtype; "auto" otherwise
FP8_SCALE = 5.5 / 448  # a calibrated per-tensor scale of N(0, 1) values
EPS = 1e-5
ROPE_BASE = 1e6
MAX_POSITION = 32768
HIDDEN, INTER, VOCAB = 1024, 3072, 151936  # the Qwen3-0.6B shape


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a lone request's decode call: launch and host latency are all there is
        dict(name="decode_b1_fp8", kind="decode", fmt="fp8", batch=1, lo=700, hi=700,
             heads=16, kv_heads=8, head_dim=128, block=256),
        # the precision the reference engine runs by default, a mid-sized batch
        dict(name="decode_b32_fp32", kind="decode", fmt="fp32", batch=32, lo=64, hi=2048,
             heads=16, kv_heads=8, head_dim=128, block=256),
        # a mid-sized batch of mixed contexts, scales per token and head
        dict(name="decode_b32_fp8_token", kind="decode", fmt="fp8_token", batch=32, lo=256,
             hi=4096, heads=32, kv_heads=8, head_dim=128, block=256),
        # ragged contexts at the Llama-3.2-1B head shape, 16-bit cache
        dict(name="decode_b48_bf16_d64", kind="decode", fmt="bf16", batch=48, lo=10, hi=3000,
             heads=32, kv_heads=8, head_dim=64, block=256),
        # the large-batch serving step: the bandwidth-bound end
        dict(name="decode_b256_fp8", kind="decode", fmt="fp8", batch=256, lo=512, hi=8192,
             heads=32, kv_heads=8, head_dim=128, block=256),
        # the attention part of the end-to-end engine's decode step, captured
        dict(name="decode_step_b60_fp8", kind="decode_step", fmt="fp8", batch=60, lo=288, hi=768,
             heads=16, kv_heads=8, head_dim=128, block=256, layers=8),
        # one prefill step's KV append
        dict(name="append_fp8_t4096", kind="append", fmt="fp8", tokens=4096, kv_heads=8,
             head_dim=128, block=256),
        # chunked prefill: eight 512-row chunks behind cached contexts
        dict(name="prefill_chunks_bf16", kind="prefill", fmt="bf16", seqs=8, chunk_lo=512,
             chunk_hi=512, lo=0, hi=4096, heads=32, kv_heads=8, head_dim=128, block=256),
        # chunked prefill in the reference engine's default precision, ragged chunks
        dict(name="prefill_chunks_fp32", kind="prefill", fmt="fp32", seqs=6, chunk_lo=37,
             chunk_hi=512, lo=0, hi=2048, heads=16, kv_heads=8, head_dim=128, block=256),
        # a continuous-batching step: prefill chunks beside many decode rows
        dict(name="mixed_fp8", kind="mixed", fmt="fp8", seqs=8, chunk_lo=512, chunk_hi=512, lo=0,
             hi=4096, rows=120, row_lo=256, row_hi=4096, heads=32, kv_heads=8, head_dim=128,
             block=256),
        # full prefill of the end-to-end workload's prompts
        dict(name="flash_prompts_bf16", kind="flash", fmt="bf16", seqs=60, lo=32, hi=512,
             heads=16, kv_heads=8, head_dim=128),
        # the end-to-end engine's decode step through the LM head, on 8 of its 28
        # layers (through all 28 the 16-bit roundings of two correct programs
        # part by 3% of the logits)
        dict(name="model_decode_b60_fp8", kind="model", fmt="fp8", batch=60, lo=288, hi=768,
             block=256, layers=8),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _heads(rng):
    h = rng.choice([(16, 8, 128), (32, 8, 128), (32, 8, 128), (32, 8, 64)])
    return dict(heads=h[0], kv_heads=h[1], head_dim=h[2])


def _draw_one(rng):
    kind = rng.choice(["decode"] * 4 + ["decode_step", "append"] + ["prefill"] * 2
                      + ["mixed", "flash", "model"])
    block = rng.choice([256, 256, 256, 128, 64, 16])
    any_fmt = rng.choice(["fp32", "bf16", "fp16", "fp8", "fp8", "fp8_token", "int8_token"])
    if kind == "decode":
        lo = _log_int(rng, 1, 2000)
        return dict(kind=kind, fmt=any_fmt, batch=_log_int(rng, 1, 256), lo=lo,
                    hi=_log_int(rng, max(lo, 40), 8192), **_heads(rng), block=block)
    if kind == "decode_step":
        lo = _log_int(rng, 20, 500)
        return dict(kind=kind, fmt=rng.choice(["fp8", "fp8", "bf16", "fp8_token", "int8_token"]),
                    batch=_log_int(rng, 1, 128), lo=lo, hi=_log_int(rng, lo + 20, 2000),
                    heads=rng.choice([16, 32]), kv_heads=8, head_dim=128, block=block, layers=8)
    if kind == "append":
        return dict(kind=kind, fmt=any_fmt, tokens=_log_int(rng, 1, 16384), kv_heads=8,
                    head_dim=rng.choice([64, 128, 128]), block=block)
    if kind == "prefill":
        lo = _log_int(rng, 1, 600)
        return dict(kind=kind, fmt=any_fmt, seqs=_log_int(rng, 1, 16), chunk_lo=lo,
                    chunk_hi=_log_int(rng, lo, 1024), lo=rng.choice([0, rng.randint(0, 2000)]),
                    hi=rng.randint(2000, 4096), **_heads(rng), block=block)
    if kind == "mixed":
        lo = _log_int(rng, 16, 512)
        return dict(kind=kind, fmt=rng.choice(["fp8", "bf16", "fp8_token"]),
                    seqs=rng.randint(1, 8), chunk_lo=lo, chunk_hi=_log_int(rng, lo, 1024), lo=0,
                    hi=rng.randint(200, 4096), rows=_log_int(rng, 4, 120), row_lo=rng.randint(1, 300),
                    row_hi=rng.randint(1000, 4096), **_heads(rng), block=block)
    if kind == "flash":
        lo = _log_int(rng, 1, 400)
        return dict(kind=kind, fmt=rng.choice(["bf16", "bf16", "fp16", "fp32"]),
                    seqs=_log_int(rng, 1, 60), lo=lo, hi=_log_int(rng, max(lo, 32), 4096), **_heads(rng))
    lo = _log_int(rng, 20, 500)
    return dict(kind=kind, fmt=rng.choice(["fp8", "fp8", "bf16", "fp8_token"]),
                batch=_log_int(rng, 1, 64), lo=lo, hi=_log_int(rng, lo + 20, 1024), block=block,
                layers=8)


def draw(rng):
    """A case of the listed families; one that would move or compute more than
    the largest listed one of its kind (fp32: of the fp32 one) is drawn again."""
    while True:
        case = _draw_one(rng)
        w = work(case)
        if w["bytes"] <= (3e9 if case["kind"] == "model" else 1.4e9) and w["flops"] <= (3e10 if case["fmt"] == "fp32" else 2e11):
            return case


# ---------------------------------------------------------------------------
# Sizes that follow from a case alone
# ---------------------------------------------------------------------------
def _spread(n, lo, hi):
    """n lengths over [lo, hi]: evenly over the values, or over their
    logarithm where the range spans more than a factor of ten."""
    at = [(i + 0.5) / n for i in range(n)]
    if lo > 0 and hi > 10 * lo:
        return [min(hi, max(lo, int(lo * (hi / lo) ** t))) for t in at]
    return [lo + int((hi - lo + 1) * t) if hi > lo else lo for t in at]


def _items(case):
    """(query rows, context length) of every sequence of a batch."""
    if case["kind"] in ("decode", "decode_step", "model"):
        return [(1, c) for c in _spread(case["batch"], case["lo"], case["hi"])]
    if case["kind"] == "flash":
        return [(c, c) for c in _spread(case["seqs"], case["lo"], case["hi"])]
    n = case["seqs"]
    chunks = _spread(n, case["chunk_lo"], case["chunk_hi"])
    priors = _spread(n, case["lo"], case["hi"])
    items = [(c, priors[(5 * i + 2) % n] + c) for i, c in enumerate(chunks)]
    if case["kind"] == "mixed":
        items += [(1, c) for c in _spread(case["rows"], case["row_lo"], case["row_hi"])]
    return items


def _elem(fmt):
    return torch.empty(0, dtype=CACHE_DTYPE[fmt]).element_size()


def _model_shape(case):
    return dict(heads=16, kv_heads=8, head_dim=128) if case["kind"] == "model" else \
        dict(heads=case.get("heads", 0), kv_heads=case["kv_heads"], head_dim=case["head_dim"])


def work(case):
    s = _model_shape(case)
    Hq, Hkv, D, fmt = s["heads"], s["kv_heads"], s["head_dim"], case["fmt"]
    row = Hkv * D  # elements of one token's K (or V) row
    ein = torch.empty(0, dtype=ROW_DTYPE.get(fmt, torch.bfloat16)).element_size()
    kv_row = 2 * (row * _elem(fmt) + (4 * Hkv if fmt.endswith("_token") else 0))
    if case["kind"] == "append":
        return dict(bytes=case["tokens"] * (2 * row * ein + kv_row + 8), flops=0)
    items = _items(case)
    rows = sum(n for n, _ in items)
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for n, c in items)  # (query row, visible key)
    flops = 4 * pairs * Hq * D
    ctx = sum(c for _, c in items)
    if case["kind"] == "flash":
        return dict(bytes=rows * (2 * Hq * D + 2 * row) * ein, flops=flops)
    tables = sum(-(-c // case["block"]) for _, c in items) * 4 + 8 * len(items)
    qo = 2 * rows * Hq * D * ein
    if case["kind"] in ("decode", "prefill"):
        return dict(bytes=ctx * kv_row + qo + tables, flops=flops)
    if case["kind"] == "mixed":  # the new rows come in and go to the cache
        return dict(bytes=ctx * kv_row + qo + tables + rows * (2 * row * ein + kv_row), flops=flops)
    step = (ctx + rows) * kv_row + tables + rows * (2 * Hq * D + 2 * row) * ein
    if case["kind"] == "decode_step":
        return dict(bytes=case["layers"] * step, flops=case["layers"] * flops)
    weights = (Hq + 2 * Hkv) * D * HIDDEN + HIDDEN * Hq * D + 3 * INTER * HIDDEN
    # weights once, K/V once, the new rows, the logits
    return dict(bytes=case["layers"] * (2 * weights + ctx * kv_row + rows * kv_row)
                + 2 * VOCAB * (HIDDEN + rows),
                flops=case["layers"] * (flops + 2 * rows * weights) + 2 * rows * VOCAB * HIDDEN)


# About four times the measured difference between the framework's result and
# the 64-bit one on these inputs.  16-bit outputs (0.0017): their own rounding;
# 32-bit outputs (7e-7): the order of 32-bit sums; a step from qkv rows
# (0.0029): q's rounding too.  A model's logits carry the roundings of every
# layer: 0.020 from the 64-bit ones, and 0.0125 from those of the same program
# with its matrix products summed in another order, which also moves 2e-4 of
# all K and V codes (new rows whose rounding is nearly a tie).
def tolerance(case):
    if case["kind"] == "append":
        return "exact"
    if case["kind"] == "model":
        return {"rel": 0.03, "max": 0.3, "differ": 0.005}
    if case["fmt"] == "fp32":
        return {"rel": 3e-6, "max": 3e-5, "differ": 0.0}
    if case["kind"] == "decode_step":
        return {"rel": 1.2e-2, "max": 0.1, "differ": 0.0}
    return {"rel": 7e-3, "max": 0.05, "differ": 0.0}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _quantise(x, fmt):
    """Codes and scales of rows (..., D) in a cache format: the framework's
    append rules in torch."""
    f = x.float()
    if fmt == "fp8":
        s = torch.tensor(FP8_SCALE, dtype=torch.float32, device=x.device)
        return (f / s).clamp(-448, 448).to(torch.float8_e4m3fn), None
    amax = f.abs().amax(dim=-1, keepdim=True)
    if fmt == "fp8_token":
        s = torch.where(amax > 0, amax / 448, torch.ones_like(amax))
        return (f / s).clamp(-448, 448).to(torch.float8_e4m3fn), s[..., 0].contiguous()
    s = (amax / 127).clamp(min=1e-6)
    y = f * (1 / s)
    y = torch.where(y >= 0, y + 0.5, y - 0.5).clamp(-128, 127).trunc()
    return y.to(torch.int8), s[..., 0].contiguous()


def _pool(blocks, block, kv_heads, head_dim, fmt, g):
    """A (blocks, block, kv_heads, head_dim) pool of N(0, 1) values in a cache
    format, and its scales; where every token has scales of its own, its
    magnitude spreads over a factor of sixteen."""
    dt = CACHE_DTYPE[fmt]
    pool = torch.empty(blocks, block, kv_heads, head_dim, dtype=dt, device=DEV)
    scale = None
    if fmt.endswith("_token"):
        scale = torch.empty(blocks, block, kv_heads, device=DEV)
    step = max(1, (1 << 26) // (block * kv_heads * head_dim))
    for i in range(0, blocks, step):
        n = min(step, blocks - i)
        x = torch.randn(n, block, kv_heads, head_dim, generator=g, device=DEV)
        if scale is not None:
            x *= torch.exp2(torch.rand(n, block, kv_heads, 1, generator=g, device=DEV) * 4 - 2)
        if fmt in MODE:
            pool[i:i + n], s = _quantise(x.to(torch.bfloat16), fmt)
            if scale is not None:
                scale[i:i + n] = s
        else:
            pool[i:i + n] = x.to(dt)
    if fmt == "fp8":
        scale = torch.full((1,), FP8_SCALE, device=DEV)
    return pool, scale


def _batch(case, seed):
    """Lengths in a seeded order, and block tables that are slices of one
    permutation of the pool, padded with -1 to the longest sequence."""
    g = torch.Generator().manual_seed(seed)
    items = _items(case)
    order = torch.randperm(len(items), generator=g).tolist()
    items = [items[i] for i in order]
    block = case["block"]
    need = [-(-c // block) for _, c in items]
    blocks = sum(need) + max(4, sum(need) // 16)
    perm = torch.randperm(blocks, generator=g).to(torch.int32)
    bt = torch.full((len(items), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = perm[at:at + n]
        at += n
    return items, bt, blocks


def _rows_of(items, bt, block):
    """Absolute positions and cache slots of every query row."""
    pos = torch.cat([torch.arange(c - n, c) for n, c in items])
    seq = torch.repeat_interleave(torch.arange(len(items)), torch.tensor([n for n, _ in items]))
    slots = bt[seq, pos // block].to(torch.int64) * block + pos % block
    return pos, slots


def _cos_sin(head_dim):
    inv = 1.0 / (ROPE_BASE ** (torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim))
    f = torch.outer(torch.arange(MAX_POSITION, dtype=torch.float32), inv)
    return torch.cat([f.cos(), f.sin()], dim=-1).to(DEV)


def _weights(case, g):
    """Random decoder weights N(0, 0.02), norms around one, as one dict a layer."""
    s = _model_shape(case)
    Hq, Hkv, D = s["heads"], s["kv_heads"], s["head_dim"]

    def w(*shape):
        return (torch.randn(*shape, generator=g, device=DEV) * 0.02).to(torch.bfloat16)

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16)

    layers = [dict(in_norm=norm(HIDDEN), qkv=w((Hq + 2 * Hkv) * D, HIDDEN), q_norm=norm(D),
                   k_norm=norm(D), o=w(HIDDEN, Hq * D), post_norm=norm(HIDDEN),
                   gate_up=w(2 * INTER, HIDDEN), down=w(HIDDEN, INTER))
              for _ in range(case["layers"])]
    return dict(embed=w(VOCAB, HIDDEN), layers=layers, final_norm=norm(HIDDEN))


def _inputs(case, seed):
    """Everything a pass reads, on the GPU, in plain torch."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind, fmt = case["kind"], case["fmt"]
    s = _model_shape(case)
    Hq, Hkv, D = s["heads"], s["kv_heads"], s["head_dim"]
    dt = ROW_DTYPE.get(fmt, torch.bfloat16)
    x = dict(fmt=fmt, heads=Hq, kv_heads=Hkv, head_dim=D, scale=1 / math.sqrt(D))

    def rows(n, heads):
        return torch.randn(n, heads, D, generator=g, device=DEV).to(dt)

    if kind == "append":
        T, block = case["tokens"], case["block"]
        blocks = -(-5 * T // (4 * block)) + 2
        for name in ("k", "v"):
            r = torch.randn(T, Hkv, D, generator=g, device=DEV)
            out = torch.rand(r.shape, generator=g, device=DEV) < 0.01
            x[name] = torch.where(out, 20 * r, r).to(dt)
            x[name + "_pool"] = torch.zeros(blocks, block, Hkv, D, dtype=CACHE_DTYPE[fmt], device=DEV)
            if fmt == "fp8":
                x[name + "_scale"] = torch.full((1,), 20 * FP8_SCALE, device=DEV)
            elif fmt in MODE:
                x[name + "_scale"] = torch.zeros(blocks, block, Hkv, device=DEV)
        slots = torch.randperm(blocks * block, generator=g, device=DEV)[:T]
        pad = torch.rand(T, generator=g, device=DEV) < 0.05  # padding rows
        x["slots"] = torch.where(pad, torch.full_like(slots, -1), slots)
        x["block"] = block
        return x
    if kind == "flash":
        order = torch.randperm(case["seqs"], generator=torch.Generator().manual_seed(seed))
        lens = torch.tensor([n for n, _ in _items(case)])[order]
        x["cu"] = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(torch.int32).to(DEV)
        x["lens"] = lens.tolist()
        total = int(lens.sum())
        x["q"], x["k"], x["v"] = rows(total, Hq), rows(total, Hkv), rows(total, Hkv)
        return x

    items, bt, blocks = _batch(case, seed)
    block = case["block"]
    pos, slots = _rows_of(items, bt, block)
    n_rows = int(pos.numel())
    x.update(items=items, block=block, blocks=blocks, bt=bt.to(DEV), pos=pos.to(DEV),
             slots=slots.to(DEV), ctx=torch.tensor([c for _, c in items], device=DEV))
    if kind in ("decode_step", "model"):
        L = case["layers"]
        pools = [[_pool(blocks, block, Hkv, D, fmt, g) for _ in range(L)] for _ in "kv"]
        for name, per_layer in zip(("k", "v"), pools):
            # one allocation for all layers, as a runner makes it
            x[name + "_pool"] = torch.stack([p.view(torch.uint8) if fmt in MODE else p
                                             for p, _ in per_layer]).view(CACHE_DTYPE[fmt])
            x[name + "_scale"] = [sc for _, sc in per_layer]
        del pools, per_layer
        x["cos_sin"] = _cos_sin(D)
        if kind == "model":
            x["weights"] = _weights(case, g)
            x["ids"] = torch.randint(0, VOCAB, (n_rows,), generator=g, device=DEV)
        else:
            x["qkv"] = torch.randn(L, n_rows, (Hq + 2 * Hkv) * D, generator=g, device=DEV).to(dt)
            x["q_norm"] = (1 + 0.1 * torch.randn(L, D, generator=g, device=DEV)).to(dt)
            x["k_norm"] = (1 + 0.1 * torch.randn(L, D, generator=g, device=DEV)).to(dt)
        return x
    x["k_pool"], x["k_scale"] = _pool(blocks, block, Hkv, D, fmt, g)
    x["v_pool"], x["v_scale"] = _pool(blocks, block, Hkv, D, fmt, g)
    x["q"] = rows(n_rows, Hq)
    if kind != "decode":
        lens = torch.tensor([0] + [n for n, _ in items])
        x["cu"] = lens.cumsum(0).to(torch.int32).to(DEV)
    if kind == "mixed":
        x["k"], x["v"] = rows(n_rows, Hkv), rows(n_rows, Hkv)
    return x


def prepare(case, seed):
    x = _inputs(case, seed)
    x["kind"] = case["kind"]
    if "k_pool" in x:  # what a pass leaves in the caches, as bytes where they are codes
        x["state"] = [x[n].view(torch.uint8) if case["fmt"] in MODE else x[n] for n in ("k_pool", "v_pool")]
        if case["fmt"].endswith("_token"):
            for n in ("k_scale", "v_scale"):
                x["state"].append(torch.stack(x[n]) if isinstance(x[n], list) else x[n])
                if isinstance(x[n], list):
                    x[n] = list(x["state"][-1].unbind(0))
    if case["kind"] == "mixed":
        att = mkv.Attention(x["heads"], x["head_dim"], num_kv_heads=x["kv_heads"], block_size=x["block"])
        att.k_cache, att.v_cache = x["k_pool"], x["v_pool"]
        att.kv_cache_dtype = MODE.get(case["fmt"], "auto")
        att.k_scale, att.v_scale = x["k_scale"], x["v_scale"]
        x["layer"] = att
    elif case["kind"] in ("decode_step", "model"):
        _plan_step(case, x)
    return x


def _plan_step(case, x):
    """The captured decode step a serving program keeps: its metadata, its
    buffers and one graph, over this batch's sequences."""
    B, L, bs = len(x["items"]), case["layers"], x["block"]
    Hq, Hkv, D = x["heads"], x["kv_heads"], x["head_dim"]
    mode = MODE.get(case["fmt"], "auto")
    meta = DecodeMetadata(B, x["bt"].shape[1], bs, x["blocks"], x["bt"].device)
    meta.block_tables.copy_(x["bt"].clamp(min=0))
    x["seq_lens"] = x["ctx"] - 1  # before the step's token
    scales = []
    if mode == "fp8_per_tensor":
        scales = [s for n in ("k_scale", "v_scale") for s in x[n]]
    if case["kind"] == "model":
        w = x["weights"]
        cfg = ModelConfig(vocab_size=VOCAB, hidden_size=HIDDEN, num_layers=L, num_heads=Hq,
                          num_kv_heads=Hkv, head_dim=D, intermediate_size=INTER,
                          rope_base=ROPE_BASE, max_position=MAX_POSITION, eps=EPS)
        model = Qwen3Model(cfg, DEV, block_size=bs)
        model.embed.copy_(w["embed"])
        model.final_norm.copy_(w["final_norm"])
        model.kv_cache_dtype = mode
        for i, lay in enumerate(model.layers):
            for n, t in w["layers"][i].items():
                lay[n].copy_(t)
            att = lay["attn"]
            att.kv_cache_dtype = mode
            att.k_cache, att.v_cache = x["k_pool"][i], x["v_pool"][i]
            att.k_scale, att.v_scale = x["k_scale"][i], x["v_scale"][i]
        del x["weights"], w
        x["out"] = torch.empty(B, VOCAB, dtype=torch.bfloat16, device=DEV)

        def step(rows, slots, ctx, bt):
            mkv.set_context(False, slot_mapping=slots, context_lens=ctx, block_tables=bt)
            try:
                hidden = model(x["ids"], (ctx - 1).clamp_(min=0), slots)
                x["out"].copy_(model.logits(hidden))
            finally:
                mkv.reset_context()
    else:
        x["out"] = torch.empty(L, B, Hq, D, dtype=x["qkv"].dtype, device=DEV)

        def step(rows, slots, ctx, bt):
            pos = (ctx - 1).clamp_(min=0)
            for i in range(L):
                qkv_norm_rope_append_decode(
                    x["qkv"][i], pos, Hq, Hkv, D, x["cos_sin"], x["k_pool"][i], x["v_pool"][i], slots,
                    bs, bt, ctx, x["scale"], q_norm_weight=x["q_norm"][i],
                    k_norm_weight=x["k_norm"][i], eps=EPS, kv_cache_dtype=mode,
                    k_scale=x["k_scale"][i], v_scale=x["v_scale"][i], out=x["out"][i])
    graphs = DecodeGraphs(meta, step, buckets=[B])
    graphs.capture(scales=scales)
    x["meta"], x["graphs"] = meta, graphs


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(x):
    kind, fmt = x["kind"], x["fmt"]
    dims = (x["heads"], x["kv_heads"], x["head_dim"])
    if kind == "decode":
        if fmt in MODE:
            return mkv.paged_attention_decode_quantized(
                x["q"], x["k_pool"], x["v_pool"], x["k_scale"], x["v_scale"], x["bt"], x["ctx"],
                x["scale"], *dims, x["block"], MODE[fmt])
        return mkv.paged_attention_decode(x["q"], x["k_pool"], x["v_pool"], x["bt"], x["ctx"],
                                          x["scale"], *dims, x["block"])
    if kind == "append":
        if fmt == "int8_token":
            mkv.store_kvcache_int8(x["k"], x["v"], x["k_pool"], x["v_pool"], x["k_scale"],
                                   x["v_scale"], x["slots"], x["block"])
        elif fmt in MODE:
            mkv.store_kvcache_fp8(x["k"], x["v"], x["k_pool"], x["v_pool"], x["k_scale"],
                                  x["v_scale"], x["slots"], x["block"], MODE[fmt])
        else:
            mkv.store_kvcache(x["k"], x["v"], x["k_pool"], x["v_pool"], x["slots"], x["block"])
        return x["state"]
    if kind == "prefill":
        quant = dict(k_scale=x["k_scale"], v_scale=x["v_scale"], kv_cache_dtype=MODE[fmt]) if fmt in MODE else {}
        return mkv.paged_attention_prefill_triton(x["q"], x["k_pool"], x["v_pool"], x["bt"], x["ctx"],
                                                  x["cu"], x["pos"], x["scale"], *dims, x["block"], **quant)
    if kind == "flash":
        return mkv.flash_attention_prefill(x["q"], x["k"], x["v"], x["cu"], x["scale"], *dims)
    if kind == "mixed":
        mkv.set_context(True, cu_seqlens_q=x["cu"], slot_mapping=x["slots"], context_lens=x["ctx"],
                        block_tables=x["bt"], positions=x["pos"])
        try:
            o = x["layer"](x["q"], x["k"], x["v"])
        finally:
            mkv.reset_context()
        return [o] + x["state"]
    # a captured step over the same sequences: their lengths as before it
    x["meta"].seq_lens.copy_(x["seq_lens"])
    x["graphs"].run(len(x["items"]))
    return [x["out"]] + x["state"]


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _dense(pool, scale, fmt, entries, n):
    """The first n tokens of a sequence, (kv_heads, n, head_dim) in 64 bits."""
    t = pool[entries].flatten(0, 1)[:n].to(torch.float32).double()
    if fmt == "fp8":
        t = t * scale.double()
    elif fmt in MODE:
        t = t * scale[entries].flatten(0, 1)[:n].double()[..., None]
    return t.transpose(0, 1)


def _attend(q, k, v, first, scale):
    """q (rows, heads, D) at positions first, first + 1, ...; k, v (kv_heads, n, D)."""
    rows, heads, D = q.shape
    kv_heads, n = k.shape[:2]
    q = q.double().view(rows, kv_heads, heads // kv_heads, D).permute(1, 2, 0, 3)
    hidden = torch.arange(n, device=q.device)[None] > first + torch.arange(rows, device=q.device)[:, None]
    out = []
    for h in range(kv_heads):
        p = (q[h] @ k[h].transpose(0, 1).contiguous()) * scale
        out.append(p.masked_fill_(hidden, -math.inf).softmax(dim=-1) @ v[h])
    return torch.stack(out).permute(2, 0, 1, 3).reshape(rows, heads, D)


def _attend_paged(x, q, k_pool, v_pool, k_scale, v_scale):
    out, at = [], 0
    for i, (n, c) in enumerate(x["items"]):
        entries = x["bt"][i, :-(-c // x["block"])].long()
        k = _dense(k_pool, k_scale, x["fmt"], entries, c)
        v = _dense(v_pool, v_scale, x["fmt"], entries, c)
        out.append(_attend(q[at:at + n], k, v, c - n, x["scale"]))
        at += n
    return torch.cat(out)


def _store(x, k, v, k_pool, v_pool, k_scale, v_scale):
    """The rows' K and V in their slots, in the cache's format."""
    keep = x["slots"] >= 0
    slots = x["slots"][keep]
    for r, pool, scale in ((k, k_pool, k_scale), (v, v_pool, v_scale)):
        flat = pool.view(-1, *pool.shape[2:])
        r = r[keep].float()
        if x["fmt"] not in MODE:
            flat[slots] = r.to(pool.dtype)
            continue
        codes, s = _quantise(r, x["fmt"])
        flat.view(torch.uint8)[slots] = codes.view(torch.uint8)
        if s is not None:
            scale.view(-1, scale.shape[-1])[slots] = s


def _norm(t, w):
    return t / (t.square().mean(dim=-1, keepdim=True) + EPS).sqrt() * w.double()


def _rotate(t, cos_sin, pos):
    half = t.shape[-1] // 2
    cs = cos_sin[pos].double()[:, None]
    c, s = cs[..., :half], cs[..., half:]
    a, b = t[..., :half], t[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], dim=-1)


def _attention_step(x, i, qkv, q_norm, k_norm):
    """One layer's q/k norm, rotation, append and decode from its qkv rows."""
    Hq, Hkv, D = x["heads"], x["kv_heads"], x["head_dim"]
    q, k, v = qkv.double().view(-1, Hq + 2 * Hkv, D).split([Hq, Hkv, Hkv], dim=1)
    q = _rotate(_norm(q, q_norm), x["cos_sin"], x["pos"])
    k = _rotate(_norm(k, k_norm), x["cos_sin"], x["pos"])
    pools = [x[n][i] for n in ("k_pool", "v_pool", "k_scale", "v_scale")]
    _store(x, k, v, *pools)
    return _attend_paged(x, q, *pools)


def _model_step(x):
    w = x["weights"]
    h = w["embed"][x["ids"]].double()
    for i, lay in enumerate(w["layers"]):
        o = _attention_step(x, i, _norm(h, lay["in_norm"]) @ lay["qkv"].double().t(), lay["q_norm"], lay["k_norm"])
        h = h + o.flatten(1) @ lay["o"].double().t()
        gate, up = (_norm(h, lay["post_norm"]) @ lay["gate_up"].double().t()).chunk(2, dim=-1)
        h = h + (torch.nn.functional.silu(gate) * up) @ lay["down"].double().t()
    return _norm(h, w["final_norm"]) @ w["embed"].double().t()


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "append":
        return None  # codes and copies are compared byte by byte
    if kind == "flash":
        out, at = [], 0
        for n in x["lens"]:
            k, v = (x[m][at:at + n].double().transpose(0, 1) for m in ("k", "v"))
            out.append(_attend(x["q"][at:at + n], k, v, 0, x["scale"]))
            at += n
        return torch.cat(out)
    if kind in ("decode_step", "model"):
        state = [None] * (4 if case["fmt"].endswith("_token") else 2)
        if kind == "model":
            return [_model_step(x)] + state
        return [torch.stack([_attention_step(x, i, x["qkv"][i], x["q_norm"][i], x["k_norm"][i])
                             for i in range(case["layers"])])] + state
    pools = [x[n] for n in ("k_pool", "v_pool", "k_scale", "v_scale")]
    if kind == "mixed":
        _store(x, x["k"], x["v"], *pools)
        state = [None] * (4 if case["fmt"].endswith("_token") else 2)
        return [_attend_paged(x, x["q"], *pools).flatten(1)] + state
    return _attend_paged(x, x["q"], *pools)
