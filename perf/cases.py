"""Performance cases of the LIFetch path: the calls a serving engine makes per step, through
the package's public entry points.

Kinds of case:
  decode     kvip_amd.LIFetch over a ContiguousFetch: score, TopK-2048, gather of the selected
             656-byte KV rows (forward() with no arguments, inputs already in the binding).
  resident   kvip_amd.LIFetch over a ResidentIndexUpdate with attached LRU chains: score,
             TopK-2048, the hot-cache round with misses read from pinned host memory, the LRU
             commit. Every pass takes the next query set of a random walk.
  prefill    kvip_amd.PrefillIndexer (plan kept) or kvip_amd.quant_lightning_indexer (one
             functional call): causal scoring and TopK-2048 of packed prompt chunks.
  attention  kvip_amd.SparseAttention over the selected rows.
  lidu       kvip_amd.lidu and the LRU commit that feeds its next victims. Every pass takes
             the next TopK rows of a cycle that no cache of that budget can hold.

Context and prompt lengths are drawn per request between a case's bounds, so batches are
ragged as served batches are.
"""
import math

import numpy as np
import torch

import kvip_amd
from kvip_amd import synthetic

DEVICE = "cuda"
TOPK = 2048
BLOCK = 128
ROW_BYTES = 656
DIM = 128
KEY_DIM, VALUE_DIM = 576, 512
LRU_CAPACITY = (1 << 17) + 20 * 128  # lidu's victim bitmap covers this many slots
WALK = 16                            # query sets of a resident walk
LIDU_HOT = 4096                      # tokens of a request that its TopK rows keep coming back to

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # One interactive request just past the selection size: the smallest decode call.
        _decode("decode_single", batch=1, ctx_low=2500, ctx_high=4000, weights="bf16", query_scale=True),
        # The bf16 index-cache option at batch 4, context 4096 (the repository's configuration 1).
        _decode("decode_bf16_b4", batch=4, ctx_low=4096, ctx_high=4096, qk="bf16"),
        # The benchmark's decode step: batch 64, contexts 8K to 32K (configuration 2).
        _decode("decode_b64_32k", batch=64, ctx_low=8192, ctx_high=32768),
        # Speculative decoding: four query rows per request, very unequal contexts.
        _decode("decode_mtp4", batch=24, ctx_low=1000, ctx_high=65536, rows=4, weights="bf16", query_scale=True),
        # Few requests with very long contexts (history of configuration 4).
        _decode("decode_128k", batch=8, ctx_low=98304, ctx_high=131072, weights="bf16", query_scale=True),
        # A decode step on the resident cache with misses from host memory.
        _resident("resident_64k", batch=8, history=65536, resident=8192),
        # The long-prompt chunk: 4096 rows against 65536 tokens (configuration 3).
        _prefill("prefill_64k", sequences=1, q_low=4096, q_high=4096, k_low=65536, k_high=65536),
        # Several short ragged prompts in one functional call, as the selector's native call has it.
        _prefill("prefill_packed", sequences=6, q_low=33, q_high=900, k_low=900, k_high=9000, weights="bf16",
                 functional=True),
        # A mid-size chunk with unquantised Q/K.
        _prefill("prefill_bf16_16k", sequences=1, q_low=2048, q_high=2048, k_low=16384, k_high=16384, qk="bf16"),
        # Attention over the selected rows: 16 heads (8-way tensor parallel) and all 128 heads.
        _attention("attention_h16", rows=64, heads=16, slots=16384),
        _attention("attention_h128", rows=64, heads=128, slots=2048),
        # The batch transaction of the slot tables (configuration 4): 16 requests of four rows.
        _lidu("lidu_b16q4", batch=16, queries=4, budget=16384, tokens=131072),
    ]


def _decode(name, *, batch, ctx_low, ctx_high, rows=1, heads=64, qk="fp8", weights="fp32", query_scale=False):
    return _named(name, kind="decode", batch=batch, ctx_low=ctx_low, ctx_high=ctx_high, rows=rows, heads=heads, qk=qk,
                  weights=weights, query_scale=query_scale)


def _resident(name, *, batch, history, resident, rows=1, heads=64):
    return _named(name, kind="resident", batch=batch, history=history, resident=resident, rows=rows, heads=heads)


def _prefill(name, *, sequences, q_low, q_high, k_low, k_high, heads=64, qk="fp8", weights="fp32", functional=False):
    return _named(name, kind="prefill", sequences=sequences, q_low=q_low, q_high=q_high, k_low=k_low, k_high=k_high,
                  heads=heads, qk=qk, weights=weights, functional=functional)


def _attention(name, *, rows, heads, slots, per_request=1, short=False):
    return _named(name, kind="attention", rows=rows, heads=heads, slots=slots, per_request=per_request, short=short)


def _lidu(name, *, batch, queries, budget, tokens):
    return _named(name, kind="lidu", batch=batch, queries=queries, budget=budget, tokens=tokens)


def _named(name, **case):
    return case if name is None else {"name": name, **case}


def _log(rng, low, high):
    """A whole number between low and high, spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "attention", "attention", "resident", "lidu"])
    if kind == "decode":
        batch, rows, qk = _log(rng, 1, 256), rng.choice([1, 1, 2, 4]), rng.choice(["fp8", "fp8", "bf16"])
        while batch * rows > 384:
            batch //= 2
        top = min(131072, 2_000_000 // (batch * (2 if qk == "bf16" else 1)))
        high = _log(rng, 600, top)
        return _decode(None, batch=batch, ctx_low=_log(rng, min(64, high), high), ctx_high=high, rows=rows,
                       heads=rng.choice([32, 64, 64]), qk=qk, weights=rng.choice(["fp32", "bf16"]),
                       query_scale=qk == "fp8" and rng.random() < 0.5)
    if kind == "prefill":
        qk, sequences = rng.choice(["fp8", "fp8", "bf16"]), _log(rng, 1, 12)
        q_high = _log(rng, 40, 4096 // sequences)
        k_high = _log(rng, max(q_high, 600), max(q_high, min(65536, 120_000_000 // (sequences * q_high))))
        return _prefill(None, sequences=sequences, q_low=_log(rng, max(1, q_high // 8), q_high), q_high=q_high,
                        k_low=_log(rng, q_high, k_high), k_high=k_high, heads=rng.choice([32, 64, 64]), qk=qk,
                        weights=rng.choice(["fp32", "bf16"]), functional=rng.random() < 0.5)
    if kind == "attention":
        per_request = rng.choice([1, 1, 2, 4])
        return _attention(None, rows=_log(rng, 1, 48) * per_request, heads=rng.choice([8, 16, 20, 32, 64, 128]),
                          slots=rng.choice([2048, 4096, 16384]), per_request=per_request, short=rng.random() < 0.3)
    if kind == "resident":
        resident = rng.choice([4096, 6144, 8192])
        return _resident(None, batch=_log(rng, 1, 8), history=BLOCK * _log(rng, 3 * resident // BLOCK, 65536 // BLOCK),
                         resident=resident, rows=rng.choice([1, 1, 2, 4]), heads=rng.choice([32, 64]))
    budget = BLOCK * rng.randint(64, 128)
    return _lidu(None, batch=_log(rng, 1, 24), queries=rng.randint(1, 4), budget=budget,
                 tokens=BLOCK * _log(rng, 512, 1024))


# --- inputs -------------------------------------------------------------------------------


def prepare(case, seed):
    return {"decode": _prepare_decode, "resident": _prepare_resident, "prefill": _prepare_prefill,
            "attention": _prepare_attention, "lidu": _prepare_lidu}[case["kind"]](case, seed)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(shape, generator=gen, device=DEVICE)


def _cast(x, qk):
    return synthetic.saturating_fp8(torch, x) if qk == "fp8" else x.to(torch.bfloat16)


def _prepare_decode(case, seed):
    rows = case["rows"]
    wl = synthetic.decode_workload(
        torch, batch=case["batch"], device=DEVICE, ctx_low=case["ctx_low"], ctx_high=case["ctx_high"],
        heads=case["heads"], qk=case["qk"], weight_dtype=_DTYPES[case["weights"]], key_scale=case["qk"] == "fp8",
        query_scale=case["query_scale"], rows_per_request=rows, seed=seed, max_context=case["ctx_high"])
    ends = None
    if rows > 1:  # row q of a request sees the tokens up to its own position
        ends = np.maximum(np.repeat(wl.ctx, rows) - rows + 1 + np.tile(np.arange(rows), len(wl.ctx)), 0)
    _, update, forward = synthetic.bind(torch, kvip_amd, wl, query_ends=ends)
    return {"kind": "decode", "forward": forward, "update": update}


def _prepare_resident(case, seed):
    rotating, update, forward = synthetic.resident_workload(
        torch, kvip_amd, torch.device(DEVICE), seed=seed, batch=case["batch"], history=case["history"],
        resident=case["resident"], q_rows=case["rows"], heads=case["heads"], fill_pool=True)
    gen = _generator(seed + 1)
    for owner in range(update.owners):
        update.keys[owner].copy_(_cast(_normal(gen, case["history"], DIM), "fp8"))
    update.attach_lru(kvip_amd.SlotLRUChains(torch, case["batch"], case["resident"], DEVICE, slots=update.lru_slots))
    values = _normal(gen, *rotating.query.shape)
    queries = torch.empty((WALK, *rotating.query.shape), dtype=rotating.query.dtype, device=DEVICE)
    for k in range(WALK):
        queries[k].copy_(_cast(values, "fp8"))
        values = 0.95 * values + math.sqrt(1 - 0.95 ** 2) * _normal(gen, *rotating.query.shape)
    return {"kind": "resident", "rotating": rotating, "update": update, "forward": forward, "queries": queries,
            "step": 0}


def _prepare_prefill(case, seed):
    rng, gen = np.random.default_rng(seed), _generator(seed)
    n, heads, qk = case["sequences"], case["heads"], case["qk"]
    # The rows to score are the case's, so that every seed gives the same shapes.
    q_lens = np.random.default_rng([n, case["q_low"], case["q_high"]]).integers(case["q_low"], case["q_high"] + 1, size=n)
    k_lens = np.maximum(rng.integers(case["k_low"], case["k_high"] + 1, size=n), q_lens)
    blocks = -(-k_lens // BLOCK)
    pages = rng.permutation(int(blocks.sum())).astype(np.int32)
    table = np.zeros((n, -(-case["k_high"] // BLOCK)), np.int32)
    at = 0
    for s, count in enumerate(blocks):
        table[s, :count] = pages[at:at + count]
        at += count
    rows = int(q_lens.sum())
    state = {
        "kind": "prefill", "functional": case["functional"],
        "query": _cast(_normal(gen, rows, heads, DIM), qk), "keys": _cast(_normal(gen, at, BLOCK, DIM), qk),
        "weights": (_normal(gen, rows, heads) / 8).to(_DTYPES[case["weights"]]), "query_scale": None, "key_scale": None,
        "starts": torch.from_numpy(np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)).to(DEVICE),
        "k_lens": torch.from_numpy(k_lens.astype(np.int32)).to(DEVICE), "table": torch.from_numpy(table).to(DEVICE)}
    if qk == "fp8":
        state["query_scale"] = torch.rand((rows, heads), generator=gen, device=DEVICE) + 0.5
        state["key_scale"] = torch.rand((at, BLOCK), generator=gen, device=DEVICE) * 1.5 + 0.5
    if not case["functional"]:
        state["indexer"] = kvip_amd.PrefillIndexer(
            torch, max_rows=n * case["q_high"], max_context=case["k_high"], max_sequences=n, device=DEVICE, heads=heads,
            weight_dtype=_DTYPES[case["weights"]])
    return state


def _kv_rows(gen, count):
    """uint8 [count, 656]: 512 fp8 features of N(0, 1) values with one scale per 128, 64 bf16
    rope features, the four scales."""
    rows = torch.empty((count, ROW_BYTES), dtype=torch.uint8, device=DEVICE)
    for at in range(0, count, 1 << 17):
        part = rows[at:at + (1 << 17)]
        values = _normal(gen, len(part), 4, DIM)
        scales = values.abs().amax(2) / 448
        part[:, :512] = synthetic.saturating_fp8(torch, values / scales[:, :, None]).view(torch.uint8).view(-1, 512)
        part[:, 512:640] = _normal(gen, len(part), 64).to(torch.bfloat16).view(torch.uint8)
        part[:, 640:] = scales.view(torch.uint8)
    return rows


def _prepare_attention(case, seed):
    gen = _generator(seed)
    rows, heads, slots = case["rows"], case["heads"], case["slots"]
    requests = rows // case["per_request"]
    kv = _kv_rows(gen, requests * slots).view(-1, BLOCK, ROW_BYTES)
    per = slots // BLOCK
    table = torch.randperm(requests * per, generator=gen, device=DEVICE).to(torch.int32).view(requests, per)
    indices = torch.rand((rows, slots), generator=gen, device=DEVICE).argsort(1)[:, :TOPK].to(torch.int32).contiguous()
    if case["short"]:  # rows that see fewer tokens than the selection holds
        seen = torch.randint(1, TOPK + 1, (rows, 1), generator=gen, device=DEVICE)
        indices[torch.arange(TOPK, device=DEVICE)[None, :] >= seen] = -1
    query = _normal(gen, rows, heads, KEY_DIM).to(torch.bfloat16)
    op = kvip_amd.SparseAttention(torch, rows=rows, heads=heads, device=DEVICE, rows_per_request=case["per_request"])
    return {"kind": "attention", "op": op, "query": query, "kv": kv, "table": table, "indices": indices}


def _lidu_steps(case):
    """TopK sets whose tokens together are half as many again as the budget."""
    fresh = 410 + 102 * (case["queries"] - 1)
    return -(-3 * case["budget"] // (2 * fresh)), fresh


def _prepare_lidu(case, seed):
    gen = _generator(seed)
    batch, queries, budget, tokens = case["batch"], case["queries"], case["budget"], case["tokens"]
    steps, fresh = _lidu_steps(case)
    order = torch.rand((batch, tokens), generator=gen, device=DEVICE).argsort(1).to(torch.int32)
    resident = order[:, :budget]
    slots = torch.rand((batch, budget), generator=gen, device=DEVICE).argsort(1)
    token_to_slot = torch.full((batch + 1, tokens), -1, dtype=torch.int32, device=DEVICE)
    slot_to_token = torch.full((batch + 1, budget), -1, dtype=torch.int32, device=DEVICE)
    token_to_slot[:batch].scatter_(1, resident.long(), slots.to(torch.int32))
    slot_to_token[:batch].scatter_(1, slots, resident)
    topk = torch.empty((steps, batch, queries, TOPK), dtype=torch.int32, device=DEVICE)
    for k in range(steps):
        # Each row: tokens of the hot set, and cold ones of which the request's rows share most.
        hot = torch.rand((batch, queries, LIDU_HOT), generator=gen, device=DEVICE).argsort(2)[:, :, :TOPK - 410]
        hot = torch.gather(order[:, None, :LIDU_HOT].expand(batch, queries, LIDU_HOT), 2, hot)
        at = LIDU_HOT + (k * fresh) % (tokens - LIDU_HOT - fresh)
        for q in range(queries):
            topk[k, :, q, :TOPK - 410] = hot[:, q]
            topk[k, :, q, TOPK - 410:] = order[:, at + 102 * q:at + 102 * q + 410]
        shuffle = torch.rand((batch, queries, TOPK), generator=gen, device=DEVICE).argsort(2)
        topk[k] = torch.gather(topk[k], 2, shuffle)

    def zeros(*shape, dtype=torch.int32):
        return torch.zeros(shape, dtype=dtype, device=DEVICE)

    def full(value, *shape):
        return torch.full(shape, value, dtype=torch.int32, device=DEVICE)

    lru = kvip_amd.SlotLRUChains(torch, batch, LRU_CAPACITY, DEVICE, active=budget)
    blocks = torch.randperm(batch * (budget // BLOCK), generator=gen, device=DEVICE).to(torch.int32).view(batch, -1)
    capacity = batch * 4 * TOPK
    return {
        "kind": "lidu", "topk": topk.view(steps, batch * queries, 1, TOPK), "step": 0, "lru": lru, "batch": batch,
        "inputs": (torch.arange(1, batch + 1, dtype=torch.int32, device=DEVICE) * queries,
                   torch.arange(batch, dtype=torch.int32, device=DEVICE), token_to_slot, slot_to_token, zeros(batch + 1),
                   full(budget, batch), full(tokens, batch), lru.slots, lru.bitmap, blocks, full(tokens + 1, batch),
                   zeros(1)),
        "outputs": (zeros(batch * queries, 1, TOPK), zeros(batch + 1), zeros(capacity), zeros(capacity), zeros(capacity),
                    zeros(batch), zeros(batch, 8, 32, dtype=torch.int64)),
        "sizes": (7, 61, batch + 1, -(-tokens // BLOCK))}


# --- one pass -----------------------------------------------------------------------------


def run(state):
    return {"decode": _run_decode, "resident": _run_resident, "prefill": _run_prefill, "attention": _run_attention,
            "lidu": _run_lidu}[state["kind"]](state)


def _run_decode(state):
    state["forward"]()
    update = state["update"]
    return [update.logical_output, update.output]


def _run_resident(state):
    update, queries = state["update"], state["queries"]
    state["rotating"].query.copy_(queries[state["step"] % len(queries)])
    state["step"] += 1
    state["forward"]()
    return [update.outputs, update.hot_cache, update.hot_valid, update.keys, update.scales, update.addresses,
            update.logical_ids, update.lru_slots]


def _run_prefill(state):
    s = state
    if s["functional"]:
        return kvip_amd.quant_lightning_indexer(s["query"], s["keys"], s["weights"], s["query_scale"], s["key_scale"],
                                                s["starts"][1:], s["k_lens"], s["table"])
    return s["indexer"](s["query"], s["weights"], s["query_scale"], s["keys"], s["key_scale"], s["starts"], s["k_lens"],
                        s["table"])


def _run_attention(state):
    return state["op"].bind(state["query"], state["kv"], state["table"], state["indices"])()


def _run_lidu(state):
    topk = state["topk"][state["step"] % len(state["topk"])]
    state["step"] += 1
    outputs = kvip_amd.lidu(topk, *state["inputs"], *state["outputs"], *state["sizes"])
    state["lru"].commit(outputs[0].view(state["batch"], -1))
    return [*outputs, state["inputs"][2], state["inputs"][3], state["lru"].slots]


# --- what a pass cannot do without ----------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "decode":
        size = 1 if case["qk"] == "fp8" else 2
        rows, heads = case["batch"] * case["rows"], case["heads"]
        seen = case["batch"] * (case["ctx_low"] + case["ctx_high"]) / 2
        chosen = min(TOPK, (case["ctx_low"] + case["ctx_high"]) / 2)
        bytes_ = seen * (DIM * size + (4 if size == 1 else 0) + 4 / BLOCK)
        bytes_ += rows * heads * (DIM * size + (4 if case["weights"] == "fp32" else 2) + 4 * case["query_scale"])
        bytes_ += rows * TOPK * (4 + ROW_BYTES) + rows * chosen * ROW_BYTES
        return {"bytes": bytes_, "flops": 2 * heads * DIM * seen * case["rows"]}
    if kind == "resident":
        seen, rows = case["batch"] * case["history"], case["batch"] * case["rows"]
        return {"bytes": seen * (DIM + 4) + rows * case["heads"] * (DIM + 8) + rows * TOPK * 8,
                "flops": 2 * case["heads"] * DIM * seen * case["rows"]}
    if kind == "prefill":
        size = 1 if case["qk"] == "fp8" else 2
        q, k = (case["q_low"] + case["q_high"]) / 2, (case["k_low"] + case["k_high"]) / 2
        rows, tokens, heads = case["sequences"] * q, case["sequences"] * k, case["heads"]
        bytes_ = tokens * (DIM * size + (4 if size == 1 else 0)) + rows * TOPK * 4
        bytes_ += rows * heads * (DIM * size + (4 if case["weights"] == "fp32" else 2) + (4 if size == 1 else 0))
        return {"bytes": bytes_, "flops": 2 * heads * DIM * rows * max(k - q / 2, q / 2)}
    if kind == "attention":
        rows, heads = case["rows"], case["heads"]
        chosen = TOPK / 2 if case["short"] else TOPK
        read = min(rows * chosen, rows // case["per_request"] * case["slots"])
        return {"bytes": read * ROW_BYTES + rows * TOPK * 4 + rows * heads * (KEY_DIM * 2 + VALUE_DIM * 4),
                "flops": 2 * rows * heads * chosen * (KEY_DIM + VALUE_DIM)}
    rows = case["batch"] * case["queries"]
    _, fresh = _lidu_steps(case)
    # The rows and their slots, a table entry per token, the descriptors of the misses, the LRU
    # order read and written.
    return {"bytes": rows * TOPK * 12 + case["batch"] * (fresh * 32 + case["budget"] * 8 + TOPK * 8), "flops": 0}


def tolerance(case):
    # Selections, slots and copied bytes are whole numbers: the score keys they follow from are
    # defined bit by bit. Attention rounds keys, values and probabilities to bf16: 0.002 off in 64 bits.
    return {"rel": 8e-3, "max": 0.05} if case["kind"] == "attention" else "exact"


def exact(case, seed):
    if case["kind"] != "attention":
        return None
    s = _prepare_attention(case, seed)
    rows = s["kv"].view(-1, ROW_BYTES)
    out = torch.zeros((case["rows"], case["heads"], VALUE_DIM), dtype=torch.float64, device=DEVICE)
    for r in range(case["rows"]):
        at = s["indices"][r][s["indices"][r] >= 0].long()
        picked = rows[s["table"][r // case["per_request"]].long()[at // BLOCK] * BLOCK + at % BLOCK]
        scales = picked[:, 640:].contiguous().view(torch.float32).double()
        values = picked[:, :512].contiguous().view(torch.float8_e4m3fn).double() * scales.repeat_interleave(DIM, 1)
        rope = picked[:, 512:640].contiguous().view(torch.bfloat16).double()
        logits = s["query"][r].double() @ torch.cat([values, rope], 1).T.contiguous() * KEY_DIM ** -0.5
        out[r] = torch.softmax(logits, 1) @ values
    return out
