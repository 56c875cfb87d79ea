"""The work that programs have this package do, as cases that can be timed and checked.

A case is a dict of plain values. prepare() makes what a program holds before the call (pools,
block tables, handles), run() makes one pass through the public entry points, exact() gives the
same outputs in float64 from plain torch. Kinds of cases:

  decode   one layer of a decode step: paged attention over packed rows (PagedKVCache.decode_batch)
  step     a whole decode step of every layer at small batch, as a captured graph
           (DecodeAttentionGraphs.run: token writes and attention)
  prefill  one layer of a prefill chunk over its paged history
  swap     blocks of every layer out to pinned host memory and back into other blocks
           (NativeBackend), BF16 or FP8 records
  records  the FP8 record kernels alone: blocks to records, records to other blocks

Unless a case says otherwise the shape is Qwen3-4B's: 36 layers, 32 query heads over 8 KV heads,
head_dim 128, 16-token blocks. Q, K and V are N(0, 1); blocks are a random permutation of the pool's.
"""

from __future__ import annotations

import math
import random

import torch

from layover_amd.config import ModelConfig
from layover_amd.kernels import fp8
from layover_amd.kernels.hip_decode import Fp8KVPool, paged_decode_attention_hip_trusted
from layover_amd.kernels.hip_prefill import prefill_attention
from layover_amd.kv.decode_graphs import DecodeAttentionGraphs
from layover_amd.kv.paged_cache import BlockTable, PagedKVCache
from layover_amd.kv.transfer import NativeBackend

DEVICE = "cuda"
TORCH_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32, "fp8": torch.bfloat16}
DTYPE_BYTES = {"bf16": 2, "fp32": 4, "fp8": 1}
QWEN = {"layers": 36, "kv_heads": 8, "groups": 4, "head_dim": 128, "slots": 16}


def listed():
    return [
        # One chat's decode: the smallest call, bound by latency and launches.
        {"name": "decode_one_short", "kind": "decode", "kv": "bf16", "batch": 1, "low": 1000, "high": 1000, **QWEN},
        # A serving batch of mixed contexts in BF16: bound by HBM.
        {"name": "decode_batch_mixed", "kind": "decode", "kv": "bf16", "batch": 32, "low": 512, "high": 8192, **QWEN},
        # One long context over FP8 records.
        {"name": "decode_one_long_fp8", "kind": "decode", "kv": "fp8", "batch": 1, "low": 32768, "high": 32768, **QWEN},
        # Full precision, as when a served model is checked against its FP32 self.
        {"name": "decode_fp32", "kind": "decode", "kv": "fp32", "batch": 4, "low": 700, "high": 2500, **QWEN},
        # Another model's shape: 64-dim heads.
        {"name": "decode_dim64", "kind": "decode", "kv": "bf16", "batch": 16, "low": 300, "high": 6000, "layers": 24, "kv_heads": 8,
         "groups": 4, "head_dim": 64, "slots": 16},
        # Three chats' decode step through every layer, launched as one graph.
        {"name": "step_three_chats", "kind": "step", "kv": "bf16", "batch": 3, "low": 600, "high": 2000, **QWEN},
        # The first chunk of a prompt, a chunk far into a long one, and the ragged end of a
        # middling one whose history is held as FP8 records.
        {"name": "prefill_first", "kind": "prefill", "kv": "bf16", "tokens": 2048, "start": 0, **QWEN},
        {"name": "prefill_long", "kind": "prefill", "kv": "bf16", "tokens": 2048, "start": 30720, **QWEN},
        {"name": "prefill_tail_fp8", "kind": "prefill", "kv": "fp8", "tokens": 509, "start": 8203, **QWEN},
        # A short session parked in BF16, and a 4,096-token one parked as FP8 records.
        {"name": "swap_short", "kind": "swap", "kv": "bf16", "blocks": 3, **QWEN},
        {"name": "swap_fp8", "kind": "swap", "kv": "fp8", "blocks": 256, **QWEN},
        # Records of 64-dim heads' groups (1,024 values each).
        {"name": "records_dim64", "kind": "records", "kv": "fp8", "blocks": 300, "layers": 24, "kv_heads": 8, "groups": 4, "head_dim": 64,
         "slots": 16},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 3 + ["records"] * 2 + ["step", "swap"])
    if kind == "decode":
        shape = dict(QWEN)
        if rng.random() < 0.4:
            shape.update(layers=rng.randint(4, 28), kv_heads=rng.choice([2, 4, 8]), groups=rng.choice([1, 2, 4, 7, 8]),
                         head_dim=rng.choice([24, 32, 64, 128, 256]), slots=rng.choice([8, 16, 16, 32]))
        kv = rng.choice(["bf16", "bf16", "fp8", "fp8", "fp32"])
        batch = _log(rng, 1, 48)
        # As many tokens in all as the largest listed batch reads at most.
        most = min(32768, int(130000 * 128 / (batch * shape["head_dim"] * (2 if kv == "fp32" else 1))))
        high = _log(rng, 64, max(most, 65))
        return {"kind": kind, "kv": kv, "batch": batch, "low": rng.randint(max(1, high // 8), high), "high": high, **shape}
    if kind == "step":
        high = _log(rng, 64, 4000)
        return {"kind": kind, "kv": rng.choice(["bf16", "fp8"]), "batch": rng.randint(1, 8), "low": rng.randint(1, high), "high": high, **QWEN}
    if kind == "prefill":
        return {"kind": kind, "kv": rng.choice(["bf16", "bf16", "fp8"]), "tokens": _log(rng, 16, 2048),
                "start": rng.choice([0, _log(rng, 1, 30000)]), **QWEN}
    if kind == "swap":
        return {"kind": kind, "kv": rng.choice(["bf16", "fp8"]), "blocks": _log(rng, 1, 128), **QWEN}
    shape = dict(QWEN)
    if rng.random() < 0.6:
        shape.update(layers=rng.randint(4, 28), kv_heads=rng.choice([2, 4, 8]), head_dim=rng.choice([24, 32, 64, 128, 256]),
                     slots=rng.choice([8, 16, 32]))
    block = 2 * shape["layers"] * shape["kv_heads"] * shape["slots"] * shape["head_dim"]
    return {"kind": kind, "kv": "fp8", "blocks": _log(rng, 1, max(2, 250_000_000 // block)), **shape}


# ---- inputs -------------------------------------------------------------------------------


def _lengths(case):
    """The rows' contexts, a property of the case: `high` once, the others spread over [low, high]."""
    rng = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    return [case["high"]] + [rng.randint(case["low"], case["high"]) for _ in range(case["batch"] - 1)]


def _config(case):
    return ModelConfig(num_hidden_layers=case["layers"], num_attention_heads=case["kv_heads"] * case["groups"],
                       num_key_value_heads=case["kv_heads"], head_dim=case["head_dim"])


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _fill(pool, generator, piece=1 << 28):
    flat = pool.view(-1)
    for at in range(0, flat.numel(), piece):
        flat[at : at + piece].normal_(generator=generator)


def _group_shifts(groups):
    """The record format's shift per group of BF16 values [..., n]: the largest finite nonzero
    exponent field minus 134, 0 without one."""
    raw = (groups.view(torch.int16).to(torch.int32) >> 7) & 0xFF
    raw = torch.where(raw == 0xFF, torch.zeros_like(raw), raw).amax(dim=-1)
    return torch.where(raw > 0, raw - 134, torch.zeros_like(raw))


def _encode(groups):
    """BF16 groups [..., n] of ordinary values as E4M3 bytes and int16 shifts."""
    shifts = _group_shifts(groups)
    scaled = groups.to(torch.float32) * torch.pow(2.0, -shifts.to(torch.float32))[..., None]
    return scaled.to(torch.float8_e4m3fn).view(torch.uint8), shifts.to(torch.int16)


def _decode(codes, shifts):
    values = codes.view(torch.float8_e4m3fn).to(torch.float32) * torch.pow(2.0, shifts.to(torch.float32))[..., None]
    return values.to(torch.bfloat16)


def _fill_records(records, groups, elems, generator, piece=1 << 26):
    """FP8 records of N(0, 1) blocks."""
    data = groups * elems
    per = max(1, piece // data)
    for at in range(0, records.shape[0], per):
        n = min(per, records.shape[0] - at)
        values = torch.empty(n, groups, elems, dtype=torch.bfloat16, device=DEVICE).normal_(generator=generator)
        codes, shifts = _encode(values)
        records[at : at + n, :data] = codes.view(n, data)
        records[at : at + n, data:] = shifts.view(n, groups).contiguous().view(torch.uint8).view(n, 2 * groups)


def _pool(case, blocks, generator):
    """A cache of `blocks` blocks, and the pool that is read: its own, or FP8 records beside it."""
    kv = case["kv"]
    cache = PagedKVCache(_config(case), blocks, device=DEVICE, dtype=TORCH_DTYPES[kv], block_tokens=case["slots"], fill=False)
    if kv != "fp8":
        _fill(cache.pool, generator)
        return cache, cache.pool
    pool = Fp8KVPool.empty(blocks, case["layers"], case["kv_heads"], case["slots"], case["head_dim"], DEVICE)
    _fill_records(pool.records, pool.layout.groups_per_block, pool.layout.group_elems, generator)
    return cache, pool


def _tables(cache, ids, lengths):
    tables, at = [], 0
    for length in lengths:
        blocks = cache.blocks_for(length)
        tables.append(BlockTable(ids[at : at + blocks], length))
        at += blocks
    return tables


def _blocks_of(case, lengths):
    return sum(-(-length // case["slots"]) for length in lengths)


def prepare(case, seed):
    generator, rng = _generator(seed), random.Random(seed)
    heads = case["kv_heads"] * case["groups"]
    kind, dim, layers = case["kind"], case["head_dim"], case["layers"]

    def normal(*shape, dtype=torch.bfloat16):
        return torch.empty(*shape, dtype=dtype, device=DEVICE).normal_(generator=generator)

    if kind == "decode":
        lengths = _lengths(case)
        cache, pool = _pool(case, _blocks_of(case, lengths), generator)
        ids = list(range(cache.allocator.num_blocks))
        rng.shuffle(ids)
        batch = cache.decode_batch(_tables(cache, ids, lengths))
        q = normal(case["batch"], heads, dim, dtype=TORCH_DTYPES[case["kv"]])
        return {"kind": kind, "q": q, "pool": pool, "layer": layers // 2, "batch": batch, "groups": case["groups"]}
    if kind == "step":
        lengths = _lengths(case)
        size = next(s for s in (1, 2, 4, 8) if s >= case["batch"])
        cache, pool = _pool(case, _blocks_of(case, lengths) + size, generator)
        graphs = DecodeAttentionGraphs(cache, heads, pool=None if case["kv"] != "fp8" else pool, sizes=(size,),
                                       max_tokens=-(-max(lengths) // 1024) * 1024)
        ids = [i for i in range(cache.allocator.num_blocks) if i not in graphs.scratch_blocks]
        rng.shuffle(ids)
        q = normal(layers, case["batch"], heads, dim)
        k, v = (normal(layers, case["batch"], case["kv_heads"], dim) for _ in range(2))
        # The allocator hands out its lowest ids first: the padding rows' blocks are 0 .. size - 1.
        storage = (pool.records if case["kv"] == "fp8" else pool)[size:]
        return {"kind": kind, "graphs": graphs, "tables": _tables(cache, ids, lengths), "q": q, "k": k, "v": v, "storage": storage,
                "size": size}
    if kind == "prefill":
        end = case["start"] + case["tokens"]
        cache, pool = _pool(case, -(-end // case["slots"]), generator)
        ids = list(range(cache.allocator.num_blocks))
        rng.shuffle(ids)
        chunk = cache.chunk(BlockTable(ids, end), case["start"], case["tokens"])
        q = normal(heads, case["tokens"], dim)
        # Already written to the pool, as a model does before it attends.
        k, v = (normal(case["kv_heads"], case["tokens"], dim) for _ in range(2))
        if case["kv"] != "fp8":
            cache.write_at(chunk.write_blocks, chunk.write_slots, layers // 2, k, v)
        return {"kind": kind, "q": q, "k": k, "v": v, "cache": cache, "pool": pool, "layer": layers // 2, "chunk": chunk,
                "groups": case["groups"]}
    # swap and records: blocks of the pool's first half go out, and come back into its second half.
    n = case["blocks"]
    cache = PagedKVCache(_config(case), 2 * n, device=DEVICE, block_tokens=case["slots"], fill=False)
    _fill(cache.pool[:n], generator)
    cache.pool[n:].zero_()
    source, target = list(range(n)), list(range(n, 2 * n))
    rng.shuffle(source)
    rng.shuffle(target)
    if kind == "swap":
        backend = NativeBackend(DEVICE)
        backend.prepare(cache, fp8=case["kv"] == "fp8")
        return {"kind": kind, "cache": cache, "backend": backend, "source": source, "target": target, "fp8": case["kv"] == "fp8",
                "payload": None, "restored": cache.pool[n:]}
    layout = fp8.Fp8Layout.from_cache(cache)
    stage = torch.empty(n * layout.record_bytes, dtype=torch.uint8, device=DEVICE)
    source, target = (torch.tensor(ids, dtype=torch.int32, device=DEVICE) for ids in (source, target))
    return {"kind": kind, "pool": cache.pool, "layout": layout, "stage": stage, "source": source, "target": target,
            "restored": cache.pool[n:]}


def run(state):
    kind = state["kind"]
    if kind == "decode":
        batch = state["batch"]
        return paged_decode_attention_hip_trusted(state["q"], state["pool"], state["layer"], batch.table, batch.lengths, state["groups"])
    if kind == "step":
        return [state["graphs"].run(state["tables"], state["q"], state["k"], state["v"]), state["storage"]]
    if kind == "prefill":
        return prefill_attention(state["q"], state["k"], state["v"], state["cache"], state["layer"], state["chunk"], state["groups"],
                                 pool=state["pool"])
    if kind == "swap":
        backend, cache = state["backend"], state["cache"]
        if state["payload"] is not None:
            backend.free(state["payload"])
        out = backend.start_out(cache, state["source"], fp8=state["fp8"])
        out.wait()
        state["payload"] = out.payload
        backend.start_in(cache, state["target"], out.payload).wait()
        parked = out.payload.memory.view(-1)
        parked.owner = backend  # the payload's pinned memory lives as long as its backend
        return [parked, state["restored"]]
    fp8.quantize_blocks(state["pool"], state["source"], state["stage"], state["layout"])
    fp8.dequantize_blocks(state["stage"], state["target"], state["pool"], state["layout"])
    return [state["stage"], state["restored"]]


# ---- what a pass cannot do without, and what it should give --------------------------------


def work(case):
    heads, dim = case["kv_heads"] * case["groups"], case["head_dim"]
    element = DTYPE_BYTES[case["kv"]]
    wide = 4 if case["kv"] == "fp32" else 2
    token = 2 * case["kv_heads"] * dim * element + (2 * 2 * case["kv_heads"] / case["slots"] if case["kv"] == "fp8" else 0)
    kind = case["kind"]
    if kind in ("decode", "step"):
        lengths = _lengths(case)
        layers = case["layers"] if kind == "step" else 1
        rows = case["batch"] * dim * wide * (2 * heads + (4 * case["kv_heads"] if kind == "step" else 0))
        return {"bytes": layers * (sum(lengths) * token + rows) + 4 * _blocks_of(case, lengths),
                "flops": layers * 4.0 * heads * dim * sum(lengths)}
    if kind == "prefill":
        tokens, start = case["tokens"], case["start"]
        pairs = tokens * start + tokens * (tokens + 1) / 2
        return {"bytes": (start + tokens) * token + 2 * heads * tokens * dim * 2, "flops": 4.0 * heads * dim * pairs}
    elements = case["blocks"] * 2 * case["layers"] * case["kv_heads"] * case["slots"] * dim
    shifts = 2 * case["blocks"] * 2 * case["layers"] * case["kv_heads"] if case["kv"] == "fp8" else 0
    # Out: blocks read, records (or blocks) written; in: the reverse.
    return {"bytes": 2 * (2 * elements + elements * element + shifts), "flops": 0}


def tolerance(case):
    if case["kind"] in ("swap", "records"):
        return "exact"
    if case["kv"] == "fp32":
        return {"rel": 5e-6, "max": 1e-4}
    # BF16 results (2^-9 of rounding each); prefill's weights are BF16 too.
    return {"rel": 1e-2, "max": 0.1}


def _attend(q, k, v):
    """q [heads, tokens, dim], k and v [kv_heads, keys, dim], float64; each query token t of T sees
    the first keys - T + 1 + t keys."""
    heads, tokens, dim = q.shape
    kv_heads, keys, _ = k.shape
    out = torch.empty_like(q)
    visible = torch.arange(keys, device=q.device)[None, :] <= torch.arange(keys - tokens, keys, device=q.device)[:, None]
    for head in range(heads):
        kk, vv = k[head * kv_heads // heads], v[head * kv_heads // heads]
        scores = (q[head] @ kk.t().contiguous()) / math.sqrt(dim)
        out[head] = torch.softmax(scores.masked_fill(~visible, -math.inf), dim=-1) @ vv
    return out


def _read(case, pool, ids, layer, tokens):
    """K and V of a sequence's first tokens, float64 [kv_heads, tokens, dim]."""
    ids = ids.long()
    slots, dim, heads, layers = case["slots"], case["head_dim"], case["kv_heads"], case["layers"]
    if case["kv"] == "fp8":
        groups, elems = 2 * layers * heads, slots * dim
        shape = (-1, 2, layers, heads)
        codes = pool.records[:, : groups * elems].unflatten(1, (2, layers, heads, elems))[:, :, layer].index_select(0, ids)
        shifts = pool.records[:, groups * elems :].contiguous().view(torch.int16).view(shape)[:, :, layer].index_select(0, ids)
        picked = _decode(codes.contiguous(), shifts).view(-1, 2, heads, slots, dim)
    else:
        picked = pool[:, :, layer].index_select(0, ids)
    flat = picked.to(torch.float64).permute(1, 2, 0, 3, 4).reshape(2, heads, -1, dim)[:, :, :tokens]
    return flat[0], flat[1]


def _append(case, storage, block, slot, k, v):
    """The new token of every layer, k and v [layers, kv_heads, dim], into one block of a pool."""
    if case["kv"] != "fp8":
        storage[block, 0, :, :, slot], storage[block, 1, :, :, slot] = k, v
        return
    layers, heads, slots, dim = case["layers"], case["kv_heads"], case["slots"], case["head_dim"]
    data = 2 * layers * heads * slots * dim
    codes = storage[block, :data].view(2, layers, heads, slots * dim)
    shifts = storage[block, data:].clone().view(torch.int16).view(2, layers, heads)
    values = _decode(codes, shifts).view(2, layers, heads, slots, dim)
    values[:, :, :, slot] = torch.stack([k, v])
    values[:, :, :, slot + 1 :] = 0
    codes, shifts = _encode(values.view(2, layers, heads, slots * dim))
    storage[block, :data] = codes.reshape(-1)
    storage[block, data:] = shifts.contiguous().view(-1).view(torch.uint8)


def exact(case, seed):
    state = prepare(case, seed)
    kind = state["kind"]
    if kind == "decode":
        batch, out = state["batch"], []
        for row, length in enumerate(_lengths(case)):
            ids = batch.table[row, : -(-length // case["slots"])]
            k, v = _read(case, state["pool"], ids, state["layer"], length)
            out.append(_attend(state["q"][row].to(torch.float64)[:, None], k, v)[:, 0])
        return torch.stack(out)
    if kind == "step":
        graphs, out = state["graphs"], torch.empty(state["q"].shape, dtype=torch.float64, device=DEVICE)
        storage = graphs.pool.records if case["kv"] == "fp8" else graphs.pool
        for row, table in enumerate(state["tables"]):
            where, slot = divmod(table.num_tokens - 1, case["slots"])
            _append(case, storage, table.blocks[where], slot, state["k"][:, row], state["v"][:, row])
        for row, table in enumerate(state["tables"]):
            ids = torch.tensor(table.blocks, device=DEVICE)
            for layer in range(case["layers"]):
                k, v = _read(case, graphs.pool, ids, layer, table.num_tokens)
                out[layer, row] = _attend(state["q"][layer, row].to(torch.float64)[:, None], k, v)[:, 0]
        return [out, state["storage"].to(torch.float64) if case["kv"] != "fp8" else None]
    if kind == "prefill":
        chunk = state["chunk"]
        k, v = _read(case, state["pool"], chunk.block_ids, state["layer"], chunk.end)
        return _attend(state["q"].to(torch.float64), k, v)
    # Blocks come back as they were, or as their records hold them.
    n, pool = case["blocks"], state["cache"].pool if kind == "swap" else state["pool"]
    restored = state["restored"].to(torch.float64)
    for source, target in zip(*(state[side] if kind == "swap" else state[side].tolist() for side in ("source", "target"))):
        values = pool[source]
        if case["kv"] == "fp8":
            groups = values.reshape(-1, case["slots"] * case["head_dim"])
            values = _decode(*_encode(groups)).view(values.shape)
        restored[target - n] = values.to(torch.float64)
    return [None, restored]
