"""The work that programs built on this package have the GPU do, as timed cases.

Each case is a dict of plain values. Sizes are those of the package's own
configurations, tests and benchmark: the attention geometries of the
benchmark (32 query / 8 KV heads, head_dim 128 or 64, blocks of 16 slots),
its decode and packed steps, the Llama-3-8B-architecture engine, and, in the
drawn cases, the head counts of the random-shape tests. Values are N(0, 1),
block tables are shuffled, weights are the random-initialised model's.

Kinds:
  model   one decode step of the engine's model through its captured graph
          (`DecodeGraphs.run`): token ids and addresses in, logits and the
          written caches out.
  layer   one layer's attention part of a decode step, called eagerly: RoPE
          and the slot-write (`update_rotated`), then `paged_attention`.
  decode  `paged_decode` of one layer, writing the step's newest K / V rows.
  packed  `paged_attention` over a packed pass: prompt chunks over what the
          cache holds, with or without one-query (decode) rows beside them.
  rope    RoPE with the slot-write of a packed pass (`rotate_and_scatter`).
"""

from __future__ import annotations

import math
import random

import torch

from liteinfer_amd.attention import PagedKV, paged_attention
from liteinfer_amd.cache.block_pool import BlockPool, newest_slots, packed_addresses, slot_table
from liteinfer_amd.cache.kv_cache import KVCache
from liteinfer_amd.engine.model import LlamaShape, RandomLlama
from liteinfer_amd.engine.runner import DecodeGraphs
from liteinfer_amd.paged_kernels import paged_decode

BLOCK = 16
DEVICE = torch.device("cuda")
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
K_SCALE, V_SCALE = 0.02, 0.015  # of the fp8 pools: N(0, 1) rows reach 250 .. 340 of e4m3's 448
ROPE_THETA = 500000.0

# The engine's model, cut so that its parts keep their proportions: an eighth
# of the Llama-3-8B architecture (4 of 32 layers, an eighth of the
# vocabulary), a quarter of the Llama-3.2-1B one.
SHAPES = {
    "8b": LlamaShape(num_layers=4, vocab_size=128256 // 8),
    "1b": LlamaShape(hidden_size=2048, num_layers=4, num_heads=32, num_kv_heads=8, head_dim=64,
                     intermediate_size=8192, vocab_size=128256 // 4),
}
MAX_MODEL_LEN = 4352  # the engine's default: the width of its captured slot table
MAX_NUM_SEQS = 256


def listed():
    return [
        # One user at a chat prompt: the engine's decode step at batch 1,
        # bound by reading the weights.
        {"name": "model_decode_1", "kind": "model", "shape": "8b", "batch": 1, "median": 1100, "pool": "same", "lens": 1},
        # A small model serving a moderate, odd batch (padded to the next captured width).
        {"name": "model_decode_24", "kind": "model", "shape": "1b", "batch": 24, "median": 512, "pool": "same", "lens": 2},
        # The end-to-end configuration's decode step: 256 sequences, contexts
        # lognormal around the prompt median plus half the output.
        {"name": "model_decode_256", "kind": "model", "shape": "8b", "batch": 256, "median": 640, "pool": "same", "lens": 3},
        # The smallest call: four short contexts, eager, where launches and
        # the host count (a program without captured graphs).
        {"name": "layer_decode_4", "kind": "layer", "batch": 4, "lo": 37, "hi": 1023, "kv_heads": 8, "groups": 4,
         "dim": 64, "dtype": "bf16", "pool": "same", "lens": 4},
        # The benchmark's headline: a layer's decode step over 64 sequences of 512 .. 8192 keys.
        {"name": "decode_64", "kind": "decode", "batch": 64, "lo": 512, "hi": 8192, "kv_heads": 8, "groups": 4,
         "dim": 128, "dtype": "bf16", "pool": "same", "lens": 5},
        # Long contexts at a small batch over the quantised cache, what it is used for.
        {"name": "decode_long_fp8", "kind": "decode", "batch": 8, "lo": 32768, "hi": 131072, "kv_heads": 8, "groups": 4,
         "dim": 128, "dtype": "bf16", "pool": "fp8", "lens": 6},
        # A continuous-batching step: prompt chunks beside decode rows, as the
        # benchmark's mixed step draws them.
        {"name": "packed_mixed", "kind": "packed", "chunks": 8, "qlo": 64, "qhi": 2048, "plo": 0, "phi": 4096, "rows": 56,
         "rlo": 256, "rhi": 4096, "kv_heads": 8, "groups": 4, "dim": 128, "dtype": "bf16", "pool": "same", "lens": 7},
        # Long prompts in chunks of the token budget: 2048 queries over 8192 cached keys.
        {"name": "packed_long", "kind": "packed", "chunks": 4, "qlo": 2048, "qhi": 2048, "plo": 8192, "phi": 8192,
         "rows": 0, "rlo": 1, "rhi": 1, "kv_heads": 8, "groups": 4, "dim": 128, "dtype": "f16", "pool": "same", "lens": 8},
        # Ragged prompt chunks over the quantised cache.
        {"name": "packed_fp8", "kind": "packed", "chunks": 6, "qlo": 64, "qhi": 2048, "plo": 0, "phi": 4096, "rows": 0,
         "rlo": 1, "rhi": 1, "kv_heads": 8, "groups": 4, "dim": 128, "dtype": "bf16", "pool": "fp8", "lens": 9},
        # A follow-up question: one short chunk over a cached conversation, small heads.
        {"name": "packed_small", "kind": "packed", "chunks": 1, "qlo": 100, "qhi": 100, "plo": 4096, "phi": 4096,
         "rows": 0, "rlo": 1, "rhi": 1, "kv_heads": 8, "groups": 4, "dim": 64, "dtype": "bf16", "pool": "same", "lens": 10},
        # A float32 model's mixed step (the exact mode, what 16-bit runs are checked against).
        {"name": "packed_f32", "kind": "packed", "chunks": 3, "qlo": 50, "qhi": 400, "plo": 0, "phi": 1200, "rows": 5,
         "rlo": 256, "rhi": 1500, "kv_heads": 8, "groups": 4, "dim": 64, "dtype": "f32", "pool": "same", "lens": 11},
        # RoPE and the slot-write of a packed pass near the token budget.
        {"name": "rope_packed", "kind": "rope", "tokens": 5942, "kv_heads": 8, "groups": 4, "dim": 128, "dtype": "bf16",
         "pool": "same", "lens": 12},
    ]


def draw(rng):
    """One more case: sizes spread over the ranges the listed cases stand for."""
    def spread(lo, hi):  # log-uniform whole number
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def geometry(dims, fp8_share):
        kv_heads, groups = (8, 4) if rng.random() < 0.5 else (rng.choice([1, 2, 3, 4, 8]), rng.choice([1, 2, 4, 5, 8, 16]))
        fp8 = rng.random() < fp8_share
        return {"kv_heads": kv_heads, "groups": groups, "dim": 128 if fp8 else rng.choice(dims),
                "pool": "fp8" if fp8 else "same", "dtype": "bf16" if rng.random() < 0.7 else "f16"}

    kind = rng.choice(["model", "model", "layer", "decode", "decode", "decode", "packed", "packed", "packed", "rope"])
    lens = rng.randrange(1 << 30)
    if kind == "model":
        batch = spread(1, 256)
        return {"kind": kind, "shape": rng.choice(["8b", "1b"]), "batch": batch, "median": spread(64, min(900, 160000 // batch)),
                "pool": "fp8" if rng.random() < 0.25 else "same", "lens": lens}
    if kind == "layer":
        return {"kind": kind, "batch": spread(1, 64), "lo": 1, "hi": spread(64, 2000), "lens": lens} | geometry([64, 128], 0.2)
    if kind == "decode":
        case = {"kind": kind, "lens": lens} | geometry([64, 128], 0.3)
        if rng.random() < 0.15:
            case |= {"dtype": "f32", "pool": "same", "batch": spread(1, 32), "lo": 1, "hi": spread(64, 2048)}
            return case
        case["hi"] = spread(100, 131072)
        # Values of the pools held to those of the largest listed call.
        most = 280000 * 8 * 128 // (case["kv_heads"] * case["dim"]) // ((case["hi"] + 1) // 2 + 1)
        return case | {"batch": spread(1, max(1, min(256, most))), "lo": max(1, case["hi"] // 16)}
    if kind == "packed":
        case = {"kind": kind, "lens": lens} | geometry([64, 128], 0.3)
        exact_mode = rng.random() < 0.15
        if exact_mode:
            case |= {"dtype": "f32", "pool": "same", "kv_heads": 8, "groups": 4}
        qhi, phi = (spread(16, 400), spread(1, 1200)) if exact_mode else (spread(16, 2048), spread(1, 8192))
        chunks = rng.randint(1, 3) if exact_mode else rng.randint(1, 8)
        # Pairs of the chunks held under those of the largest listed pass.
        while chunks > 1 and chunks * qhi * (phi + qhi) * case["kv_heads"] * case["groups"] * case["dim"] > 2.4e11:
            chunks -= 1
        rows = rng.choice([0, 0, spread(1, 8 if exact_mode else 64)])
        return case | {"chunks": chunks, "qlo": max(2, qhi // 8), "qhi": qhi, "plo": 0, "phi": phi, "rows": rows,
                       "rlo": 1, "rhi": spread(64, 1500 if exact_mode else 4096)}
    return {"kind": kind, "tokens": spread(1, 8192), "lens": lens} | geometry([64, 128], 0.3)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _lengths(case):
    """Context lengths (and, for packed passes, query counts): functions of the case alone."""
    rng = random.Random(case["lens"])
    kind = case["kind"]
    if kind == "model":
        got = [int(round(case["median"] * math.exp(rng.gauss(0.0, 0.7)))) for _ in range(case["batch"])]
        return [min(MAX_MODEL_LEN - 1, max(16, n)) for n in got], None
    if kind in ("layer", "decode"):
        return [rng.randint(case["lo"], case["hi"]) for _ in range(case["batch"])], None
    if kind == "packed":
        counts = [rng.randint(case["qlo"], case["qhi"]) for _ in range(case["chunks"])]
        totals = [q + rng.randint(case["plo"], case["phi"]) for q in counts]
        totals += [rng.randint(case["rlo"], case["rhi"]) for _ in range(case["rows"])]
        return totals, counts + [1] * case["rows"]
    # rope: whole prompts that add up to the pass's tokens
    totals, left = [], case["tokens"]
    while left:
        totals.append(min(left, rng.randint(16, 2048)))
        left -= totals[-1]
    return totals, list(totals)


def _tables(totals, seed, spare=0):
    """Shuffled block tables that hold `totals`, and the pool's blocks (the last `spare` of them unused)."""
    need = [-(-n // BLOCK) for n in totals]
    order = list(range(sum(need)))
    random.Random(seed).shuffle(order)
    tables, at = [], 0
    for n in need:
        tables.append(order[at:at + n])
        at += n
    return tables, sum(need) + spare


def _normal(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype)


def _fill(pool_tensor, gen, scale):
    """N(0, 1) rows into a pool (divided by the scale for an fp8 one), a part at a time."""
    flat = pool_tensor.view(-1)
    for part in flat.split(1 << 28):
        if pool_tensor.dtype == torch.float8_e4m3fn:
            x = torch.randn(part.shape, generator=gen, device=DEVICE)
            part.copy_((x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn))
        else:
            part.normal_(generator=gen)


def _pools(case, blocks, gen):
    dtype = torch.float8_e4m3fn if case["pool"] == "fp8" else DTYPES[case["dtype"]]
    shape = (blocks * BLOCK, case["kv_heads"], case["dim"])
    pools = [torch.empty(shape, device=DEVICE, dtype=dtype) for _ in range(2)]
    for t, s in zip(pools, (K_SCALE, V_SCALE)):
        _fill(t, gen, s)
    return pools


def _scales(case):
    return {"k_scale": K_SCALE, "v_scale": V_SCALE} if case["pool"] == "fp8" else {}


def _rotary(positions, dim, dtype):
    inv = 1.0 / (ROPE_THETA ** (torch.arange(0, dim, 2, dtype=torch.float32, device=DEVICE) / dim))
    freqs = positions[..., None].float() * inv
    emb = torch.cat((freqs, freqs), dim=-1)
    return emb.cos().to(dtype), emb.sin().to(dtype)


def _block_pool(case, blocks, layers, kv_heads, dim, dtype, gen):
    pool = BlockPool(blocks, BLOCK, layers, kv_heads, dim, dtype, DEVICE,
                     cache_quant="fp8" if case["pool"] == "fp8" else None, **_scales(case))
    for layer in range(layers):
        for t, s in zip(pool.slots(layer), (K_SCALE, V_SCALE)):
            _fill(t, gen, s)
    return pool


def _projections(case, gen, batch, tokens):
    """q, k, v as a layer's fused projection gives them: views of one tensor."""
    nkv, nq, dim = case["kv_heads"], case["kv_heads"] * case["groups"], case["dim"]
    qkv = _normal(gen, (batch, tokens, nq + 2 * nkv, dim), DTYPES[case["dtype"]])
    q, k, v = qkv.split([nq, nkv, nkv], dim=2)
    return [t.transpose(1, 2) for t in (q, k, v)]


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    kind = case["kind"]
    totals, counts = _lengths(case)
    tables, blocks = _tables(totals, seed, spare=1 if kind == "model" else 0)
    state = {"case": case, "totals": totals, "counts": counts}
    if kind == "model":
        shape = SHAPES[case["shape"]]
        model = RandomLlama(shape, seed=seed)
        cache = KVCache(_block_pool(case, blocks, shape.num_layers, shape.num_kv_heads, shape.head_dim, model.dtype, gen))
        graphs = DecodeGraphs(model, cache, MAX_NUM_SEQS, MAX_MODEL_LEN, pad_slot=(blocks - 1) * BLOCK)
        ids = torch.randint(0, shape.vocab_size, (len(totals), 1), generator=gen, device=DEVICE)
        positions = torch.tensor(totals, device=DEVICE).unsqueeze(1) - 1
        state |= {"model": model, "cache": cache, "graphs": graphs,
                  "step": (ids, positions, newest_slots(tables, [n - 1 for n in totals], BLOCK, DEVICE),
                           slot_table(tables, totals, BLOCK, DEVICE),
                           torch.tensor(totals, dtype=torch.int32, device=DEVICE))}
        run(state)  # captures the batch width's graph, as the engine does before it serves
        return state
    dtype = DTYPES[case["dtype"]]
    dim, nkv, groups = case["dim"], case["kv_heads"], case["groups"]
    state["scaling"] = dim ** -0.5
    if kind in ("layer", "rope"):
        cache = KVCache(_block_pool(case, blocks, 1, nkv, dim, dtype, gen))
        state["cache"] = cache
        if kind == "rope":
            addr = packed_addresses(tables, [0] * len(totals), counts, BLOCK, DEVICE)
            positions, state["slots"] = addr.positions, addr.slots
            state["qkv"] = _projections(case, gen, 1, sum(counts))
        else:
            positions = torch.tensor(totals, device=DEVICE).unsqueeze(1) - 1
            state["table"] = slot_table(tables, totals, BLOCK, DEVICE)
            state["payload"] = cache.make_decode_payload(
                newest_slots(tables, [n - 1 for n in totals], BLOCK, DEVICE), state["table"],
                torch.tensor(totals, dtype=torch.int32, device=DEVICE))
            state["qkv"] = _projections(case, gen, len(totals), 1)
        state["rotary"] = _rotary(positions, dim, dtype)
        return state
    keys, values = _pools(case, blocks, gen)
    if kind == "decode":
        new = [_normal(gen, (len(totals), nkv, dim), dtype) for _ in range(2)]
        return state | {"q": _normal(gen, (len(totals), nkv * groups, dim), dtype), "keys": keys, "values": values,
                        "table": slot_table(tables, totals, BLOCK, DEVICE), "new": new,
                        "lens": torch.tensor(totals, dtype=torch.int32, device=DEVICE)}
    addr = packed_addresses(tables, [n - q for n, q in zip(totals, counts)], counts, BLOCK, DEVICE)
    kv = PagedKV(keys, values, addr.slot_table, addr.context_lens, query_start_loc=addr.query_start_loc,
                 max_query_len=max(counts), host_context_lens=tuple(totals), host_query_lens=tuple(counts),
                 **_scales(case))
    q = _normal(gen, (1, sum(counts), nkv * groups, dim), dtype).transpose(1, 2)  # as RoPE returns it
    return state | {"q": q, "kv": kv}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "model":
        logits = state["graphs"].run(*state["step"])
        layers = [state["cache"].layer_storage(i) for i in range(state["model"].shape.num_layers)]
        return {"logits": logits, "keys": [k for k, _ in layers], "values": [v for _, v in layers]}
    if kind == "layer":
        q, kv = state["payload"].update_rotated(*state["qkv"], *state["rotary"], 0)
        out = paged_attention(q, kv, state["scaling"], case["groups"])
        return {"out": out, "keys": kv.key_pool, "values": kv.value_pool}
    if kind == "rope":
        q = state["cache"].rotate_and_scatter(0, state["slots"], *state["qkv"], *state["rotary"])
        keys, values = state["cache"].layer_storage(0)
        return {"q": q, "keys": keys, "values": values}
    if kind == "decode":
        out = paged_decode(state["q"], state["keys"], state["values"], state["table"], state["lens"], state["scaling"],
                           case["groups"], new_key=state["new"][0], new_value=state["new"][1], **_scales(case))
        return {"out": out, "keys": state["keys"], "values": state["values"]}
    return {"out": paged_attention(state["q"], state["kv"], state["scaling"], case["groups"])}


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far correct results may differ
# ---------------------------------------------------------------------------


def work(case):
    totals, counts = _lengths(case)
    kind = case["kind"]
    if kind == "model":
        s = SHAPES[case["shape"]]
        b = len(totals)
        row = s.num_kv_heads * s.head_dim
        per_layer = (s.num_heads + 2 * s.num_kv_heads) * s.head_dim * s.hidden_size + \
            s.num_heads * s.head_dim * s.hidden_size + 3 * s.intermediate_size * s.hidden_size
        weights = s.num_layers * per_layer + s.vocab_size * s.hidden_size
        size = 1 if case["pool"] == "fp8" else 2
        return {"bytes": 2 * weights + s.num_layers * sum(totals) * (2 * row * size + 8)
                + 2 * b * (s.hidden_size + s.vocab_size),
                "flops": 2 * b * weights + 4 * s.num_layers * s.num_heads * s.head_dim * sum(totals)}
    dim, nkv, nq = case["dim"], case["kv_heads"], case["kv_heads"] * case["groups"]
    size = 4 if case["dtype"] == "f32" else 2
    psize = 1 if case["pool"] == "fp8" else size
    if kind == "rope":
        t = case["tokens"]
        return {"bytes": t * (2 * nq * dim * size + 2 * nkv * dim * (size + psize) + 2 * dim * size + 8),
                "flops": 3 * t * (nq + nkv) * dim}
    counts = counts or [1] * len(totals)
    pairs = sum(q * (n - q) + q * (q + 1) // 2 for n, q in zip(totals, counts))
    got = sum(totals) * (2 * nkv * dim * psize + 8) + 2 * sum(counts) * nq * dim * size
    if kind in ("layer", "decode"):
        got += sum(counts) * 2 * nkv * dim * (size + psize)
    if kind == "layer":
        got += 2 * sum(counts) * nq * dim * size
    return {"bytes": got, "flops": 4 * nq * dim * pairs}


def tolerance(case):
    if case["kind"] == "model":
        return {"rel": 0.03}
    if case["kind"] == "rope":
        return {"rel": 0.01}
    return {"rel": {"bf16": 0.01, "f16": 0.002, "f32": 1e-5}[case["dtype"]]}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ---------------------------------------------------------------------------


def _rows64(pool, slots, scale):
    rows = pool[slots]
    return rows.float().double() * scale if pool.dtype == torch.float8_e4m3fn else rows.double()


def _attend64(q, keys, values, scaling):
    """q [Q, Hq, D], the last positions of a context whose rows are keys / values [N, Hkv, D]; in float64."""
    nq, ctx, nkv = q.shape[0], keys.shape[0], keys.shape[1]
    groups = q.shape[1] // nkv
    out = torch.empty_like(q)
    hidden = None
    if nq > 1:
        hidden = torch.arange(ctx, device=DEVICE)[None, :] > torch.arange(ctx - nq, ctx, device=DEVICE)[:, None]
    for h in range(q.shape[1]):
        scores = torch.mm(q[:, h], keys[:, h // groups].t()) * scaling
        if hidden is not None:
            scores.masked_fill_(hidden, float("-inf"))
        out[:, h] = torch.mm(torch.softmax(scores, dim=-1), values[:, h // groups])
    return out


def _rotate64(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat((-x[..., half:], x[..., :half]), dim=-1) * sin


def _contexts64(keys, values, table, totals, new_k, new_v, scales):
    """Each sequence's dequantised rows, the last one replaced by its newest K / V."""
    for i, n in enumerate(totals):
        k, v = (_rows64(p, table[i, :n], s) for p, s in zip((keys, values), scales))
        if new_k is not None:
            k[-1], v[-1] = new_k[i], new_v[i]
        yield k, v


def exact(case, seed):
    state = prepare(case, seed) if case["kind"] != "model" else _model_state(case, seed)
    kind = case["kind"]
    totals, counts = state["totals"], state["counts"]
    scales = (K_SCALE, V_SCALE) if case["pool"] == "fp8" else (1.0, 1.0)
    if kind == "model":
        return {"logits": _model64(state, scales), "keys": None, "values": None}
    scaling = state["scaling"]
    if kind == "rope":
        q, k, v = (t.double() for t in state["qkv"])
        cos, sin = (t.double().unsqueeze(1) for t in state["rotary"])
        if case["pool"] == "fp8":
            return {"q": _rotate64(q, cos, sin), "keys": None, "values": None}
        keys, values = (t.double() for t in state["cache"].layer_storage(0))
        slots = state["slots"].reshape(-1)
        keys[slots] = _rotate64(k, cos, sin)[0].transpose(0, 1)
        values[slots] = v[0].transpose(0, 1)
        return {"q": _rotate64(q, cos, sin), "keys": keys, "values": values}
    if kind == "layer":
        q, k, v = (t.double()[:, :, 0] for t in state["qkv"])  # [B, H, D]
        cos, sin = (t.double() for t in state["rotary"])
        q, k = _rotate64(q, cos, sin), _rotate64(k, cos, sin)
        keys, values = state["cache"].layer_storage(0)
        out = [_attend64(q[i:i + 1], kk, vv, scaling) for i, (kk, vv) in
               enumerate(_contexts64(keys, values, state["table"], totals, k, v, scales))]
        return {"out": torch.cat(out).unsqueeze(2), "keys": None, "values": None}
    if kind == "decode":
        q = state["q"].double()
        out = [_attend64(q[i:i + 1], kk, vv, scaling) for i, (kk, vv) in
               enumerate(_contexts64(state["keys"], state["values"], state["table"], totals,
                                     state["new"][0].double(), state["new"][1].double(), scales))]
        return {"out": torch.cat(out), "keys": None, "values": None}
    kv = state["kv"]
    q = state["q"][0].transpose(0, 1).double()  # [T, H, D]
    out, at = [], 0
    for (kk, vv), n in zip(_contexts64(kv.key_pool, kv.value_pool, kv.slot_table, totals, None, None, scales), counts):
        out.append(_attend64(q[at:at + n], kk, vv, scaling))
        at += n
    return {"out": torch.cat(out).transpose(0, 1).unsqueeze(0)}


def _model_state(case, seed):
    state = prepare(case, seed)
    del state["graphs"]
    return state


def _model64(state, scales):
    model, cache = state["model"], state["cache"]
    s = model.shape
    ids, positions, _, table, _ = state["step"]
    b, nq, nkv = len(state["totals"]), s.num_heads, s.num_kv_heads

    def linear(x, w):
        return torch.mm(x, w.double().t())

    def norm(x, w):
        return w.double() * x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + s.rms_norm_eps)

    inv = 1.0 / (s.rope_theta ** (torch.arange(0, s.head_dim, 2, dtype=torch.float64, device=DEVICE) / s.head_dim))
    freqs = positions.double() * inv
    emb = torch.cat((freqs, freqs), dim=-1)
    cos, sin = emb.cos().unsqueeze(1), emb.sin().unsqueeze(1)
    h = model.embed[ids[:, 0]].double()
    for i, layer in enumerate(model.layers):
        qkv = linear(norm(h, layer.attn_norm), layer.w_qkv).view(b, nq + 2 * nkv, s.head_dim)
        q, k = _rotate64(qkv[:, :nq], cos, sin), _rotate64(qkv[:, nq:nq + nkv], cos, sin)
        keys, values = cache.layer_storage(i)
        out = [_attend64(q[j:j + 1], kk, vv, model.scaling) for j, (kk, vv) in
               enumerate(_contexts64(keys, values, table, state["totals"], k, qkv[:, nq + nkv:], scales))]
        h = h + linear(torch.cat(out).reshape(b, nq * s.head_dim), layer.w_o)
        gate, up = linear(norm(h, layer.mlp_norm), layer.w_gate_up).chunk(2, dim=-1)
        h = h + linear(torch.nn.functional.silu(gate) * up, layer.w_down)
    return linear(norm(h, model.final_norm), model.lm_head)
