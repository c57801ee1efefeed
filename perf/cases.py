"""What is measured of this package: its calls at the sizes programs make them with.

Eight kinds of call, each through a public entry point:

prefill     ``ccpe_prefill_paged``: a batch of prompts (or of prompt chunks: the
            last ``rows`` positions of each context) over the paged cache.
attention   ``cope_attention`` of one request on dense K/V, no policies: the
            recompute call of a layer, in every element type a model runs in.
reuse       ``cope_attention`` of one request whose reused chunks keep their
            calibrated positions: with WCA's selected rows (every layer after
            the calibration layer) or with all rows (the calibration layer).
decode      ``ccpe_decode_paged``: one new token per request.
shared      ``ccpe_decode_shared``: the same over chunks that the batch shares.
step        ``PagedDecoder.step``: one token per request through a whole
            decoder, to its logits.
selective   the layers of one request's selective prefill around attention:
            ``WCAState.initialize``, then per layer ``next_layer_rows`` and
            ``WCAState.update``, and ``scatter_rows`` at the end.
relocate    a SLIDE step: pages and single records move, the token map is
            rewritten and read back, slots return to the free list.

The shapes are this repository's own: 32 query heads over 8 KV heads (and
halves of that), head size 128 (64 for smaller models), 64 or 128 contextual
positions, blocks of 16 or 32 tokens, chunks of up to 2048 tokens.
"""

import math
import random

import numpy as np
import torch

from cacheslide_amd import (CCPEProfile, CanonicalPositionPolicy, ChunkIdentity, CoPE, RequestPlan,
                            SelectedAssociationPolicy, WCAConfig, WCAState, cope_attention)
from cacheslide_amd import _hip, relocate
from cacheslide_amd.ccpe import (SharedRuns, ccpe_decode_paged, ccpe_decode_shared, ccpe_prefill_paged,
                                 decode_shared_workspace, decode_workspace)
from cacheslide_amd.decode_model import DecoderShape, PagedDecoder
from cacheslide_amd.runtime_rows import next_layer_rows, scatter_rows

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
FRACTION = 0.15          # of the reused tokens are corrected per layer
DEVICE = "cuda"


def listed():
    return [
        # eight prompts of four 1024-token chunks in one batch: the headline prefill
        dict(name="prefill_batch", op="prefill", batch=8, context=4096, rows=4096, ragged=False, heads=32,
             kv_heads=8, positions=64, block=16),
        # chunked prefill: a few requests of unlike lengths, each with its next piece of the prompt
        dict(name="prefill_ragged", op="prefill", batch=5, context=2900, rows=333, ragged=True, heads=32,
             kv_heads=8, positions=64, block=16),
        # a short prompt recomputed alone: launches and checks count, not the arithmetic
        dict(name="attention_short", op="attention", tokens=211, dtype="bfloat16", heads=32, kv_heads=8, dim=128,
             positions=64),
        # an ordinary prompt of a float16 model
        dict(name="attention_half", op="attention", tokens=1000, dtype="float16", heads=32, kv_heads=8, dim=128,
             positions=64),
        # the reuse call of every layer after the calibration layer, long context
        dict(name="reuse_long", op="reuse", fixed=16128, dynamic=256, selected=True, per_head=False, heads=32,
             kv_heads=8, positions=64),
        # one request generating alone: latency
        dict(name="decode_single", op="decode", batch=1, context=1500, ragged=False, heads=32, kv_heads=8,
             positions=64, block=16),
        # a small serving batch of unlike lengths
        dict(name="decode_ragged", op="decode", batch=12, context=9000, ragged=True, heads=32, kv_heads=8,
             positions=64, block=16),
        # 64 requests of 32k tokens, one layer of distinct K/V: bandwidth
        dict(name="decode_batch", op="decode", batch=64, context=32769, ragged=False, heads=32, kv_heads=8,
             positions=64, block=16),
        # 32 requests over the same eight 1024-token chunks, each in its own order
        dict(name="decode_shared", op="shared", batch=32, chunks=8, chunk=1024, own=45, heads=32, kv_heads=8,
             positions=64, block=16),
        # one token of each of eight requests through a four-layer decoder
        dict(name="decoder_step", op="step", batch=8, context=1900, layers=4, heads=16, kv_heads=4, ffn=5632,
             vocab=32000, positions=64, block=16),
        # four layers of an 8k prompt's selective prefill
        dict(name="selective_layers", op="selective", tokens=8192, dynamic=250, layers=4, hidden=4096, kv_heads=8,
             dim=128, dtype="bfloat16"),
        # 64 chunks of 64 to 2048 tokens moved in four layers' caches
        dict(name="relocate_chunks", op="relocate", layers=4, blocks=10000, chunks=64, kv_heads=8, block=16),
    ]


def _log(rng, low, high):
    """An integer of [low, high], even over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    op = rng.choice(["prefill", "attention", "attention", "reuse", "decode", "decode", "shared", "step", "selective",
                     "relocate"])
    heads, kv_heads = rng.choice([(32, 8), (32, 8), (16, 4), (32, 4), (16, 16)])
    positions = rng.choice([64, 64, 128])
    block = rng.choice([16, 16, 32])
    if op == "prefill":
        context = _log(rng, 100, 4096)
        rows = context if rng.random() < 0.5 else _log(rng, 17, context)
        return dict(op=op, batch=rng.randint(1, 8), context=context, rows=rows, ragged=rows < context, heads=heads,
                    kv_heads=kv_heads, positions=positions, block=block)
    if op == "attention":
        return dict(op=op, tokens=_log(rng, 17, 2048), dtype=rng.choice(["bfloat16", "float16", "float32"]),
                    heads=heads, kv_heads=kv_heads, dim=rng.choice([128, 128, 64]), positions=positions)
    if op == "reuse":
        fixed = _log(rng, 300, 8000)
        return dict(op=op, fixed=fixed, dynamic=_log(rng, 16, 500), selected=fixed > 4096 or rng.random() < 0.7,
                    per_head=fixed <= 2048, heads=heads, kv_heads=kv_heads, positions=positions)
    if op == "decode":
        batch = _log(rng, 1, 64)
        most = 64 * 32000 * 8 // (batch * kv_heads)        # the largest batch's bytes
        return dict(op=op, batch=batch, context=min(_log(rng, 40, 32000), most), ragged=rng.random() < 0.6, heads=heads,
                    kv_heads=kv_heads, positions=positions, block=block)
    if op == "shared":
        return dict(op=op, batch=_log(rng, 4, 64), chunks=rng.randint(4, 12), chunk=rng.choice([256, 512, 1024, 2048]),
                    own=_log(rng, 1, 300), heads=heads, kv_heads=kv_heads, positions=positions, block=block)
    if op == "step":
        heads, kv_heads = rng.choice([(8, 2), (16, 4), (16, 8)])
        return dict(op=op, batch=_log(rng, 1, 32), context=_log(rng, 50, 4000), layers=rng.randint(2, 5), heads=heads,
                    kv_heads=kv_heads, ffn=heads * 352, vocab=32000, positions=64, block=block)
    if op == "selective":
        return dict(op=op, tokens=_log(rng, 256, 16384), dynamic=_log(rng, 16, 250), layers=rng.randint(2, 6),
                    hidden=rng.choice([2048, 4096]), kv_heads=rng.choice([4, 8]), dim=rng.choice([64, 128]),
                    dtype=rng.choice(["bfloat16", "bfloat16", "float16"]))
    return dict(op=op, layers=rng.randint(1, 6), blocks=10000, chunks=_log(rng, 4, 70), kv_heads=rng.choice([4, 8]),
                block=block)


# ---------------------------------------------------------------- inputs
def _gen(seed, stream=0):
    return torch.Generator(device=DEVICE).manual_seed(1_000_003 * seed + stream)


def _normal(gen, *shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=gen)


def _cope(gen, dim, positions):
    cope = CoPE(dim, positions, device=torch.device(DEVICE, torch.cuda.current_device()))
    with torch.no_grad():
        cope.position_embeddings.normal_(0.0, 0.1, generator=gen)
    return cope


def _lengths(case):
    """Keys of each request: ``context``, or unlike lengths up to it."""
    batch, context = case["batch"], case["context"]
    if not case["ragged"]:
        return [context] * batch
    spread = random.Random(f"{batch} {context}")
    low = max(case.get("rows", 1), context // 10, 1)
    return [context] + [spread.randint(low, context) for _ in range(batch - 1)]


def _paged(case, gen, seed, lengths):
    """A cache of K/V ~ N(0, 1) with block tables of a random permutation of its blocks."""
    block = case["block"]
    per = [(n + block - 1) // block for n in lengths]
    total = sum(per)
    cache = _normal(gen, total, case["kv_heads"], block, 2 * 128)
    ids = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    table = torch.zeros((len(lengths), max(per)), dtype=torch.int32)
    at = 0
    for b, count in enumerate(per):
        table[b, :count] = ids[at:at + count]
        at += count
    return cache, table.to(DEVICE)


def _plan(case):
    fixed, dynamic = case["fixed"], case["dynamic"]
    half = fixed // 2
    spans = [("first", "reuse", 0, half), ("second", "reuse", half, fixed),
             ("question", "recompute", fixed, fixed + dynamic)]
    doc = {"version": 1, "namespace": "cases", "task_id": "reuse", "operation": "reuse",
           "chunks": [dict(id=i, role=r, start=a, end=b) for i, r, a, b in spans]}
    return RequestPlan.parse(doc, [(7 * i) % 32000 for i in range(fixed + dynamic)])


def _chunk_moves(case, seed):
    """Blocks and slots of a relocation: chunks of 64 .. 2048 tokens (sizes from
    the case, places from the seed)."""
    sizes = np.random.default_rng(case["chunks"]).integers(64, 2049, case["chunks"])
    block = case["block"]
    pages = [(int(n) + block - 1) // block for n in sizes]
    need = sum(pages)
    perm = np.random.default_rng(seed).permutation(case["blocks"])
    source, target = perm[:need], perm[need:2 * need]
    page_src, page_dst, slot_src, slot_dst, slots = [], [], [], [], []
    at = 0
    for n, count in zip(sizes.tolist(), pages):
        src, dst = source[at:at + count], target[at:at + count]
        at += count
        full = n // block
        page_src.append(src[:full])
        page_dst.append(dst[:full])
        tail = np.arange(full * block, n)
        slot_src.append(src[tail // block] * block + tail % block)
        slot_dst.append(dst[tail // block] * block + tail % block)
        tokens = np.arange(n)
        slots.append(dst[tokens // block] * block + tokens % block)
    freed = (source[:, None] * block + np.arange(block)).reshape(-1)
    lists = [np.concatenate(x) for x in (page_src, page_dst, slot_src, slot_dst, slots)] + [freed]
    return sizes, [torch.from_numpy(x.astype(np.int64)).to(DEVICE) for x in lists]


def prepare(case, seed):
    op = case["op"]
    gen = _gen(seed)
    device = torch.device(DEVICE, torch.cuda.current_device())
    state = dict(case=case)
    if op in ("prefill", "decode"):
        lengths = _lengths(case)
        batch = len(lengths)
        state["cache"], state["table"] = _paged(case, gen, seed, lengths)
        state["cope"] = _cope(gen, 128, case["positions"])
        state["lens"] = torch.tensor(lengths, dtype=torch.int32, device=device)
        if op == "prefill":
            rows = case["rows"]
            state["query"] = _normal(gen, batch, rows, case["heads"], 128)
            starts = torch.tensor(lengths, device=device) - rows
            state["qpos"] = (starts[:, None] + torch.arange(rows, device=device)).contiguous()
        else:
            state["query"] = _normal(gen, batch, case["heads"], 128)
            state["workspace"] = decode_workspace(batch, case["heads"], case["context"], 1024, device)
            state["flags"] = _hip.new_flags(device)
    elif op == "attention":
        dtype, n = DTYPES[case["dtype"]], case["tokens"]
        state["query"] = _normal(gen, n, case["heads"], case["dim"], dtype=dtype)
        state["key"] = _normal(gen, n, case["kv_heads"], case["dim"], dtype=dtype)
        state["value"] = _normal(gen, n, case["kv_heads"], case["dim"], dtype=dtype)
        state["cope"] = _cope(gen, case["dim"], case["positions"])
        state["rows"] = torch.arange(n, device=device)
    elif op == "reuse":
        fixed, n = case["fixed"], case["fixed"] + case["dynamic"]
        state["rows"], state["selected"] = _reuse_rows(case, seed)
        state["query"] = _normal(gen, len(state["rows"]), case["heads"], 128)
        state["key"] = _normal(gen, n, case["kv_heads"], 128)
        state["value"] = _normal(gen, n, case["kv_heads"], 128)
        state["cope"] = _cope(gen, 128, case["positions"])
        state["plan"] = _plan(case)
        state["profile"] = CCPEProfile(
            trained_profile_version="v1", checkpoint_id="ckpt",
            chunks=tuple(ChunkIdentity(*c) for c in state["plan"].fixed_layout),
            query_positions=torch.arange(fixed), key_positions=torch.arange(fixed),
            canonical_positions=_canonical(case), max_positions=case["positions"], histogram_bin_width=0.25,
            sample_count=1)
    elif op == "shared":
        block, chunks, batch = case["block"], case["chunks"], case["batch"]
        chunk_blocks = case["chunk"] // block
        own = (case["own"] + block - 1) // block
        state["cache"] = _normal(gen, chunks * chunk_blocks + batch * own, case["kv_heads"], block, 2 * 128)
        rotation = (torch.arange(chunks)[None, :] + torch.arange(batch)[:, None] + seed) % chunks
        runs = torch.arange(chunks * chunk_blocks, dtype=torch.int32).view(chunks, chunk_blocks)
        private = chunks * chunk_blocks + torch.arange(batch * own).view(batch, own)
        table = torch.cat([runs[rotation].reshape(batch, -1), private], dim=1).to(torch.int32).to(device)
        state["table"] = table
        state["shared"] = SharedRuns(table, runs, rotation, block, margin=128 if case["chunk"] < 512 else 256)
        state["context"] = chunks * case["chunk"] + case["own"]
        state["lens"] = torch.full((batch,), state["context"], dtype=torch.int32, device=device)
        state["tail"] = state["shared"].tail_lens(state["lens"])
        state["query"] = _normal(gen, batch, case["heads"], 128)
        state["cope"] = _cope(gen, 128, case["positions"])
        state["workspace"] = decode_shared_workspace(batch, case["heads"], state["shared"], state["context"], 1024,
                                                     device)
        state["flags"] = _hip.new_flags(device)
    elif op == "step":
        batch, block = case["batch"], case["block"]
        shape = DecoderShape(layers=case["layers"], hidden=128 * case["heads"], heads=case["heads"],
                             kv_heads=case["kv_heads"], ffn=case["ffn"], vocab=case["vocab"], npos=case["positions"])
        state["model"] = PagedDecoder(shape, device, seed=seed)
        lengths = _lengths(dict(case, ragged=True))
        per = case["context"] // block + 1
        state["caches"] = state["model"].new_caches(batch * per, block)
        for cache in state["caches"]:
            cache.normal_(generator=gen)
        ids = torch.randperm(batch * per, generator=torch.Generator().manual_seed(seed))
        state["table"] = ids.to(torch.int32).view(batch, per).to(device)
        state["positions"] = torch.tensor(lengths, dtype=torch.long, device=device)
        state["ids"] = torch.randint(0, case["vocab"], (batch,), generator=torch.Generator().manual_seed(seed + 1)
                                     ).to(device)
        state["workspace"] = decode_workspace(batch, case["heads"], case["context"] + 1, 1024, device)
        state["flags"] = _hip.new_flags(device)
    elif op == "selective":
        dtype, n = DTYPES[case["dtype"]], case["tokens"]
        shape = (n, case["kv_heads"], case["dim"])
        state["fresh_k"] = _normal(gen, *shape, dtype=dtype)
        state["fresh_v"] = _normal(gen, *shape, dtype=dtype)
        # the cached rows drifted, each token by its own amount
        drift = 0.02 + 0.3 * torch.rand((n, 1, 1), generator=gen, device=device)
        state["cached_k"] = (state["fresh_k"].float() + drift * _normal(gen, *shape, dtype=torch.float32)).to(dtype)
        state["cached_v"] = (state["fresh_v"].float() + drift * _normal(gen, *shape, dtype=torch.float32)).to(dtype)
        reused = torch.arange(n, device=device) < n - case["dynamic"]
        state["reused"], state["mandatory"] = reused, ~reused
        state["cached_k"] = torch.where(reused[:, None, None], state["cached_k"], state["fresh_k"])
        state["fixed"] = torch.arange(n - case["dynamic"], device=device)
        state["hidden"] = _normal(gen, n, case["hidden"], dtype=dtype)
        state["residual"] = _normal(gen, n, case["hidden"], dtype=dtype)
        count = n - case["dynamic"]
        state["snapshot"] = {"hidden": _normal(gen, count, case["hidden"], dtype=dtype),
                             "residual": _normal(gen, count, case["hidden"], dtype=dtype)}
        state["config"] = WCAConfig(correction_fraction=FRACTION)
    elif op == "relocate":
        sizes, lists = _chunk_moves(case, seed)
        state["lists"] = lists
        state["cache"] = _normal(gen, case["layers"], case["blocks"], case["kv_heads"], case["block"], 2 * 128)
        tokens = int(sizes.sum())
        state["tokens"] = torch.randperm(tokens, generator=torch.Generator().manual_seed(seed)).to(device)
        state["mapping"] = torch.full((tokens,), -1, dtype=torch.long, device=device)
        state["free"] = relocate.SlotFreeList(case["blocks"] * case["block"], device)
    return state


def _reuse_rows(case, seed):
    """Query rows of a reuse call, and the selected ones among them."""
    fixed, n = case["fixed"], case["fixed"] + case["dynamic"]
    if not case["selected"]:
        return torch.arange(n, device=DEVICE), None
    gen = torch.Generator().manual_seed(seed)
    chosen = torch.randperm(fixed, generator=gen)[:math.ceil(FRACTION * fixed)].sort().values
    return torch.cat([chosen, torch.arange(fixed, n)]).to(DEVICE), chosen.to(DEVICE)


def _canonical(case):
    """Calibrated positions [heads, fixed, fixed]: a steady path per token, one
    for all heads (a broadcast view) or one per head."""
    fixed, heads, top = case["fixed"], case["heads"], case["positions"] - 1
    ords = torch.arange(fixed, device=DEVICE, dtype=torch.float32)
    base = (ords[:, None] - ords[None, :] + 1).clamp_(min=0)
    if not case["per_head"]:
        return base.mul_(0.5).clamp_(max=top).expand(heads, fixed, fixed)
    out = torch.empty((heads, fixed, fixed), dtype=torch.float32, device=DEVICE)
    for h in range(heads):
        torch.mul(base, 0.4 + 0.01 * h, out=out[h]).clamp_(max=top)
    return out


# ---------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    op = case["op"]
    if op == "prefill":
        return ccpe_prefill_paged(state["query"], state["cache"], state["table"], state["lens"], state["cope"],
                                  state["qpos"])
    if op == "attention":
        return cope_attention(state["query"], state["key"], state["value"], state["cope"], state["rows"])
    if op == "reuse":
        policy = CanonicalPositionPolicy(state["plan"], state["profile"], "ckpt")
        visible = (SelectedAssociationPolicy(state["plan"].fixed_indices, state["selected"])
                   if state["selected"] is not None else None)
        return cope_attention(state["query"], state["key"], state["value"], state["cope"], state["rows"],
                              positions_transform=policy, visibility_transform=visible, query_chunk_size=64)
    if op == "decode":
        return ccpe_decode_paged(state["query"], state["cache"], state["table"], state["lens"], state["cope"],
                                 max_context=case["context"], workspace=state["workspace"], flags=state["flags"],
                                 check=False)
    if op == "shared":
        return ccpe_decode_shared(state["query"], state["cache"], state["table"], state["lens"], state["cope"],
                                  state["shared"], max_context=state["context"], tail=state["tail"],
                                  workspace=state["workspace"], flags=state["flags"], check=False)
    if op == "step":
        logits = state["model"].step(state["ids"], state["positions"], state["caches"], state["table"],
                                     max_context=case["context"] + 1, workspace=state["workspace"],
                                     flags=state["flags"])
        return logits, state["caches"]
    if op == "selective":
        return _run_selective(state)
    page_src, page_dst, slot_src, slot_dst, slots, freed = state["lists"]
    cache, free = state["cache"], state["free"]
    relocate.copy_pages(cache, page_src, page_dst, check=False)   # disjoint: two parts of one permutation
    relocate.copy_slots(cache, slot_src, slot_dst, check=False)
    relocate.scatter_mapping(state["mapping"], state["tokens"], slots)
    found = relocate.gather_mapping(state["mapping"], state["tokens"])
    free.release(freed)
    taken = free.acquire(slots.numel() // 2)     # the next request's slots, given back when it retires
    free.release(taken)
    return cache, state["mapping"], found, taken


def _run_selective(state):
    case = state["case"]
    wca = WCAState.initialize(state["cached_k"], state["fresh_k"], state["reused"], state["mandatory"],
                              state["config"])
    hidden, residual = state["hidden"], state["residual"]
    previous = torch.arange(case["tokens"], device=hidden.device)
    out = []
    for layer in range(2, 2 + case["layers"]):
        active = wca.active_indices
        rows = next_layer_rows(hidden, residual, previous, active, state["fixed"], state["snapshot"])
        hidden, residual = rows.hidden, rows.residual
        update = wca.update(layer, state["cached_k"], state["cached_v"],
                            state["fresh_k"].index_select(0, active), state["fresh_v"].index_select(0, active),
                            computed_indices=active)
        out.append((hidden, residual, update.fused_k, update.fused_v, update.alpha, update.next_indices))
        previous = active
    return out, scatter_rows(hidden, previous, case["tokens"])


# ---------------------------------------------------------------- what a pass cannot do without
def _pairs(case):
    """(query row, visible key) pairs of one head."""
    op = case["op"]
    if op == "prefill":
        rows = case["rows"]
        return sum(rows * (n - rows) + rows * (rows + 1) // 2 for n in _lengths(case))
    if op == "attention":
        return case["tokens"] * (case["tokens"] + 1) // 2
    fixed, dynamic = case["fixed"], case["dynamic"]
    question = dynamic * fixed + dynamic * (dynamic + 1) // 2
    if case["selected"]:
        # a corrected row sees itself; nothing it attends depends on the other reused keys
        return question + math.ceil(FRACTION * fixed)
    return question + fixed * (fixed + 1) // 2


def work(case):
    op = case["op"]
    if op in ("prefill", "attention", "reuse"):
        dim, size = case.get("dim", 128), 4 if case.get("dtype") == "float32" else 2
        heads, kv_heads = case["heads"], case["kv_heads"]
        if op == "prefill":
            rows, keys = case["batch"] * case["rows"], sum(_lengths(case))
        elif op == "attention":
            rows = keys = case["tokens"]
        else:
            keys = case["fixed"] + case["dynamic"]
            rows = (math.ceil(FRACTION * case["fixed"]) + case["dynamic"]) if case["selected"] else keys
        moved = size * dim * (2 * rows * heads + 2 * keys * kv_heads)
        if op == "reuse":
            # the strict policy checks every causal canonical cell of the fixed rows
            fixed = case["fixed"]
            cells = (math.ceil(FRACTION * fixed) * (fixed + 1) / 2) if case["selected"] else fixed * (fixed + 1) / 2
            moved += 4 * cells * (heads if case["per_head"] else 1)
        return dict(bytes=moved, flops=4.0 * heads * dim * _pairs(case) + 2.0 * rows * heads * dim * case["positions"])
    if op in ("decode", "shared"):
        heads, kv_heads, batch = case["heads"], case["kv_heads"], case["batch"]
        if op == "decode":
            keys = stored = sum(_lengths(case))
        else:
            stored = case["chunks"] * case["chunk"] + batch * case["own"]
            keys = batch * (case["chunks"] * case["chunk"] + case["own"])
        return dict(bytes=4 * 128 * kv_heads * stored + 4 * 128 * batch * heads, flops=4.0 * heads * 128 * keys)
    if op == "step":
        hidden, heads, kv_heads = 128 * case["heads"], case["heads"], case["kv_heads"]
        weights = case["layers"] * ((heads + 2 * kv_heads) * 128 * hidden + hidden * hidden
                                    + 3 * case["ffn"] * hidden) + case["vocab"] * hidden
        keys = sum(_lengths(dict(case, ragged=True)))
        return dict(bytes=2 * weights + case["layers"] * 4 * 128 * kv_heads * keys + 2 * case["batch"] * case["vocab"],
                    flops=2.0 * case["batch"] * weights + case["layers"] * 4.0 * heads * 128 * keys)
    if op == "selective":
        n, row = case["tokens"], case["kv_heads"] * case["dim"] * 2
        active = math.ceil(FRACTION * (n - case["dynamic"])) + case["dynamic"]
        layer = 2 * n * row + 4 * active * row + 4 * active * case["hidden"] * 2
        return dict(bytes=2 * n * row + case["layers"] * layer + (n + active) * case["hidden"] * 2,
                    flops=4.0 * n * row)
    sizes = np.random.default_rng(case["chunks"]).integers(64, 2049, case["chunks"])
    tokens = int(sizes.sum())
    return dict(bytes=2 * tokens * case["layers"] * case["kv_heads"] * 512 + 5 * 8 * tokens, flops=0)


def tolerance(case):
    """Relative 2-norm error of a correct implementation at the same precision,
    about four times what the present one shows against ``exact``."""
    op = case["op"]
    if op == "relocate":
        return "exact"
    if op == "attention" and case["dtype"] != "bfloat16":
        return {"rel": 1e-5 if case["dtype"] == "float32" else 1e-3}
    if op == "selective":
        # rounding of the blended rows; the index lists are whole numbers
        return {"rel": 6e-3, "differ": 0.0}
    if op == "step":
        # bf16 rounding of every layer travels to the logits
        return {"rel": 5e-2}
    if op == "reuse" and case["selected"]:
        # a corrected row returns its own value exactly; the question's rows,
        # means over about a fifth of their keys, carry the error
        question = 5.0 * case["dynamic"] / (case["fixed"] + case["dynamic"])
        return {"rel": 9e-3 * math.sqrt(question / (math.ceil(FRACTION * case["fixed"]) + question))}
    return {"rel": 9e-3}


# ---------------------------------------------------------------- in 64 bits
def _attend(q, k, v, table, qpos, canonical=None, fixed=0, selected=None):
    """Contextual-position attention of query rows [r, heads, D] over keys
    [n, kv_heads, D] at positions 0 .. n - 1, in float64, a few rows and one head at
    a time.  canonical [heads, fixed, fixed]: positions of the reused rows'
    reused keys; selected: rows that see of the reused keys only their own."""
    heads, n = q.shape[1], k.shape[0]
    group = heads // k.shape[1]
    out = torch.empty(q.shape[0], heads, v.shape[2], dtype=torch.float64, device=q.device)
    keys = torch.arange(n, device=q.device)
    top = table.shape[1] - 1
    table = table.double()
    step = max(1, min(q.shape[0], (1 << 25) // n))
    for h in range(heads):
        kh = k[:, h // group].double().t().contiguous()
        vh = v[:, h // group].double().contiguous()
        for a in range(0, q.shape[0], step):
            qh, pos = q[a:a + step, h].double(), qpos[a:a + step]
            logits = (qh @ kh) / math.sqrt(q.shape[2])
            causal = keys[None, :] <= pos[:, None]
            gates = torch.sigmoid(logits).masked_fill_(~causal, 0.0)
            place = gates.flip(-1).cumsum(-1).flip(-1).clamp_(0, top)
            if canonical is not None:
                own = pos < fixed
                place[own, :fixed] = canonical[h, pos[own]].double()
            low = place.floor().long()
            qe = qh @ table
            left, right = qe.gather(1, low), qe.gather(1, (low + 1).clamp_(max=top))
            logits += left + (place - low) * (right - left)
            if selected is not None:
                hide = selected[a:a + step, None] & (keys < fixed)[None, :] & (keys[None, :] != pos[:, None])
                causal &= ~hide
            out[a:a + step, h] = torch.softmax(logits.masked_fill_(~causal, -math.inf), dim=-1) @ vh
    return out


def _records(cache, row, n):
    """K and V [n, kv_heads, 128] of a request's first n tokens."""
    block = cache.shape[2]
    rec = cache[row[:(n + block - 1) // block].long()].permute(0, 2, 1, 3).reshape(-1, cache.shape[1], 256)[:n]
    return rec[..., :128], rec[..., 128:]


def exact(case, seed):
    op = case["op"]
    if op == "relocate":
        return _exact_relocate(case, seed)
    state = prepare(case, seed)
    if op == "selective":
        return _exact_selective(state)
    if op == "step":
        return _exact_step(state)
    table = state["cope"].position_embeddings.detach()
    if op == "attention":
        return _attend(state["query"], state["key"], state["value"], table, state["rows"])
    if op == "reuse":
        selected = None
        if state["selected"] is not None:
            selected = state["rows"] < case["fixed"]
        return _attend(state["query"], state["key"], state["value"], table, state["rows"],
                       state["profile"].canonical_positions, case["fixed"], selected)
    lengths = state["lens"].tolist()
    out = []
    for b, n in enumerate(lengths):
        k, v = _records(state["cache"], state["table"][b], n)
        if op == "prefill":
            out.append(_attend(state["query"][b], k, v, table, state["qpos"][b]))
        else:
            at = torch.tensor([n - 1], device=k.device)
            out.append(_attend(state["query"][b:b + 1], k, v, table, at)[0])
    return torch.stack(out)


def _exact_step(state):
    """The decoder in float64 on its own weights: norm, projections, attention
    over the cached keys and the new one, gated MLP, head."""
    model, case = state["model"], state["case"]
    shape, block = model.shape, case["block"]
    positions, batch = state["positions"], case["batch"]
    slots = [(int(state["table"][b, p // block]), p % block) for b, p in enumerate(positions.tolist())]

    def norm(x, weight):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + shape.eps) * weight.double()

    residual = model.embed[state["ids"]].double()
    q_end = shape.heads * 128
    k_end = q_end + shape.kv_heads * 128
    caches = []
    for layer, cache in zip(model.layers, state["caches"]):
        qkv = norm(residual, layer.in_norm) @ layer.qkv.double().t()
        q, k, v = (qkv[:, a:b].reshape(batch, -1, 128) for a, b in ((0, q_end), (q_end, k_end), (k_end, None)))
        wide = cache.double()
        rows = []
        for b, (blk, at) in enumerate(slots):
            wide[blk, :, at, :128], wide[blk, :, at, 128:] = k[b], v[b]
            keys, values = _records(wide, state["table"][b], int(positions[b]) + 1)
            rows.append(_attend(q[b:b + 1], keys, values, layer.cope.position_embeddings.detach(),
                                positions[b:b + 1])[0])
        caches.append(wide)
        residual = torch.stack(rows).reshape(batch, -1) @ layer.o.double().t() + residual
        gate, up = (norm(residual, layer.post_norm) @ layer.gate_up.double().t()).split(shape.ffn, dim=-1)
        residual = (torch.nn.functional.silu(gate) * up) @ layer.down.double().t() + residual
    return norm(residual, model.norm) @ model.lm_head.double().t(), caches


def _exact_selective(state):
    case, config = state["case"], state["config"]
    old_k, old_v = state["cached_k"].double(), state["cached_v"].double()
    new_k, new_v = state["fresh_k"].double(), state["fresh_v"].double()
    n, fixed = case["tokens"], state["fixed"]
    deviation = (new_k - old_k).square().sum((1, 2))
    weight = deviation / (old_k.square().sum((1, 2)) + config.epsilon)
    mandatory, candidate = state["mandatory"], state["reused"] & (deviation > 0)
    budget = min(math.ceil(config.correction_fraction * int(state["reused"].sum())), int(candidate.sum()))
    selected, removed = torch.zeros_like(candidate), torch.zeros_like(candidate)

    def promote():
        open_rows = (candidate & ~selected & ~removed).nonzero().flatten()
        order = torch.argsort(-deviation[open_rows], stable=True)
        selected[open_rows[order[:max(0, budget - int(selected.sum()))]]] = True

    promote()
    next_weight = weight.clone()
    hidden, residual = state["hidden"], state["residual"]
    previous = torch.arange(n, device=hidden.device)
    out = []
    for layer in range(2, 2 + case["layers"]):
        active = (selected | mandatory).nonzero().flatten()
        place = torch.full((n,), -1, dtype=torch.long, device=hidden.device)
        place[previous] = torch.arange(len(previous), device=hidden.device)
        kept = place[active]
        rows = []
        for old, name in ((hidden, "hidden"), (residual, "residual")):
            spare = state["snapshot"][name].new_zeros((n, case["hidden"]))
            spare[fixed] = state["snapshot"][name]
            rows.append(torch.where((kept >= 0)[:, None], old[kept.clamp(min=0)], spare[active]))
        hidden, residual = rows
        used = torch.where(mandatory[active], torch.ones_like(next_weight[active]), next_weight[active])
        w = used[:, None, None]
        fused = [w * new[active] + (1 - w) * old[active] for new, old in ((new_k, old_k), (new_v, old_v))]
        gone = active[:0]
        if layer % config.gate_interval == 0:
            a = torch.nn.functional.normalize(new_k[active], dim=-1)
            b = torch.nn.functional.normalize(old_k[active], dim=-1)
            cosine = (a * b).sum(-1).clamp(-1, 1).mean(-1)
            gone = active[selected[active] & (cosine < config.convergence_threshold)]
        next_weight[active] = weight[active]
        selected[gone], candidate[gone], removed[gone] = False, False, True
        promote()
        out.append((hidden, residual, *fused, used, (selected | mandatory).nonzero().flatten()))
        previous = active
    final = hidden.new_zeros((n, case["hidden"]))
    final[previous] = hidden
    return out, final


def _exact_relocate(case, seed):
    state = prepare(case, seed)
    page_src, page_dst, slot_src, slot_dst, slots, freed = state["lists"]
    cache, block = state["cache"], case["block"]
    cache[:, page_dst] = cache[:, page_src]
    cache[:, slot_dst // block, :, slot_dst % block] = cache[:, slot_src // block, :, slot_src % block]
    mapping = state["mapping"]
    mapping[state["tokens"]] = slots
    return cache, mapping, mapping[state["tokens"]], freed.sort().values[:slots.numel() // 2]
