"""The work this framework is measured on, through its public entry points.

Kinds of case, and what each one is in a user's program:

  attend_api     KVAllocator + paged_attention / paged_attention_batch: the drop-in call, one layer,
                 with its checks and its read of the fault word.
  attend         Paged decode attention of a ragged batch in every layer (planned_decode_attention),
                 replayed as one graph, as a decode step issues it.
  append_attend  The same with each sequence's newest token appended in the attention launch.
  append         One prompt's K and V of 22 layers scattered into the pool (kv_append).
  prompt_attend  Causal attention of one prompt in every layer (prefill_attention), replayed as one
                 graph, as a captured prefill issues it.
  mlp            The MLP half of a decode step in every layer: SwiGLU projection, down projection as
                 split-K partials, residual add and RMSNorm, at the step's row count.
  project        The attention half's projections in every layer: q|k|v partials, RoPE + KV append,
                 o_proj partials, residual add and RMSNorm.
  prefill        prefill_paged of one prompt through the whole model (admit, prefill, release).
  serve          Requests admitted through PrefillGraphs and decoded together through a DecodeGraph
                 for some steps, then released: a whole serving episode, with given token ids so
                 that the logits of every step can be compared.

Sizes are the TinyLlama architecture of the decoder (22 layers, hidden 2048, 32 query and 4 kv
heads of 64, MLP 5632, vocabulary 32000) and the batches, contexts and prompts of the benchmark and
the tests: contexts of 1 to 2048 tokens, batches of 1 to 256, decode GEMMs of 1 to 128 rows. All
data is fp16 (the one type the pool takes); weights N(0, 0.02), K/V and queries N(0, 1).
"""

from __future__ import annotations

import math

import numpy as np
import torch

from pagedcore_amd import _hip
from pagedcore_amd.attention import paged_attention, paged_attention_batch
from pagedcore_amd.decoder import (
    DecodeGraph,
    LayerWeights,
    PrefillGraph,
    TinyLlamaWeights,
    capture_graph,
    prefill_paged,
    rope_table,
)
from pagedcore_amd.engine_types import KVReservation, RequestId
from pagedcore_amd.kv_cache import KVAllocator

DEVICE = "cuda:0"
LAYERS, BLOCK, Q_HEADS, KV_HEADS, DIM = 22, 16, 32, 4, 64
HIDDEN, QKV, MLP, VOCAB = 2048, 2560, 5632, 32000
EPS = 1e-5
LAYER_WEIGHTS = QKV * HIDDEN + HIDDEN * HIDDEN + 3 * MLP * HIDDEN + 2 * HIDDEN  # elements of one layer
PREFILL_SIZES = (64, 128, 256, 512, 1024, 2048)  # PrefillGraph sizes of a serving episode


def listed():
    return [
        # One row of the reference's own decode loop: a 128-token sequence, one layer.
        {"name": "attend_api_b1_c128", "kind": "attend_api", "batch": 1, "lo": 128, "hi": 128},
        # The benchmark's headline: 64 sequences of 1 to 2048 tokens, 22 layers.
        {"name": "attend_b64", "kind": "attend", "batch": 64, "lo": 1, "hi": 2048, "layers": 22},
        # High occupancy: 256 sequences at the full context, each step also writing its token.
        {"name": "append_attend_b256", "kind": "append_attend", "batch": 256, "lo": 2048, "hi": 2048, "layers": 4},
        # A full-length prompt's K/V written into a fragmented pool.
        {"name": "append_2048", "kind": "append", "tokens": 2048},
        # Prompt attention of a full-length prompt and of an ordinary, ragged one.
        {"name": "prompt_attend_2048", "kind": "prompt_attend", "tokens": 2048},
        {"name": "prompt_attend_333", "kind": "prompt_attend", "tokens": 333},
        # Decode projections: the full batch of the decode workload, a small batch, an odd one.
        {"name": "mlp_b128", "kind": "mlp", "rows": 128},
        {"name": "mlp_b7", "kind": "mlp", "rows": 7},
        {"name": "project_b37", "kind": "project", "rows": 37},
        # The longest prompt through the whole model.
        {"name": "prefill_2048", "kind": "prefill", "tokens": 2048},
        # One user's short exchange: everything at one row.
        {"name": "serve_one", "kind": "serve", "requests": 1, "rows": 1, "lo": 61, "hi": 61, "steps": 24},
        # A serving batch: 45 requests of 100 to 500 prompt tokens in a 48-row graph.
        {"name": "serve_b45", "kind": "serve", "requests": 45, "rows": 48, "lo": 100, "hi": 500, "steps": 32},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("attend_api", "attend", "append_attend", "append", "prompt_attend", "mlp", "project", "prefill", "serve"))
    if kind == "append" or kind == "prompt_attend" or kind == "prefill":
        return {"kind": kind, "tokens": _log(rng, 1 if kind == "append" else 16, 2047)}
    if kind == "mlp" or kind == "project":
        return {"kind": kind, "rows": _log(rng, 1, 128)}
    if kind == "serve":
        requests = _log(rng, 1, 40)
        hi = _log(rng, 16, 500)
        return {"kind": kind, "requests": requests, "rows": requests + rng.randint(0, 3), "lo": rng.randint(1, hi), "hi": hi,
                "steps": rng.randint(4, 24)}
    case = {"kind": kind, "batch": _log(rng, 1, 64 if kind == "attend_api" else 255), "hi": _log(rng, 16, 2047)}
    case["lo"] = rng.randint(1, case["hi"])
    if kind != "attend_api":
        case["layers"] = 4 if kind == "append_attend" or case["batch"] > 64 else 22
    return case


# ---------------------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(gen, shape, std=1.0):
    return torch.empty(shape, dtype=torch.float16, device=DEVICE).normal_(0.0, std, generator=gen)


def _sequences(case, seed):
    """Context lengths, fragmented block tables and the pool's block count of a batch."""
    rng = np.random.Generator(np.random.PCG64(seed))
    lengths = rng.integers(case["lo"], case["hi"] + 1, size=case["batch"], dtype=np.int32)
    need = (lengths + BLOCK - 1) // BLOCK
    blocks = max(64, case["batch"] * _credits(case["hi"]))  # the pool does not depend on the seed
    if case["lo"] == case["hi"]:
        blocks += blocks // 4
    order = rng.permutation(blocks).astype(np.int32)
    tables = np.zeros((case["batch"], int(need.max())), dtype=np.int32)
    at = 0
    for row, n in enumerate(need):
        tables[row, :n] = order[at : at + n]
        at += int(n)
    return lengths, tables, blocks


def _pool(blocks):
    return torch.empty((LAYERS, 2, blocks, BLOCK, KV_HEADS, DIM), dtype=torch.float16, device=DEVICE)


def _attend_inputs(case, seed):
    lengths, tables, blocks = _sequences(case, seed)
    gen = _gen(seed)
    pool = _pool(blocks)
    pool[: case["layers"]].normal_(0.0, 1.0, generator=gen)
    query = _normal(gen, (case["layers"], case["batch"], Q_HEADS, DIM))
    new = _normal(gen, (2, case["layers"], case["batch"], KV_HEADS, DIM)) if case["kind"] == "append_attend" else None
    return lengths, tables, pool, query, new


def _append_inputs(case, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    tokens = case["tokens"]
    blocks = 1024 if tokens <= 1024 else 4096
    table = rng.permutation(blocks)[: (tokens + BLOCK - 1) // BLOCK].astype(np.int64)
    position = np.arange(tokens)
    slots = torch.from_numpy(table[position // BLOCK] * BLOCK + position % BLOCK).to(DEVICE)
    gen = _gen(seed)
    key, value = (_normal(gen, (LAYERS, tokens, KV_HEADS, DIM)) for _ in range(2))
    return blocks, slots, key, value


def _prompt_inputs(case, seed):
    gen = _gen(seed)
    tokens = case["tokens"]
    return (_normal(gen, (LAYERS, tokens, Q_HEADS, DIM)), _normal(gen, (LAYERS, tokens, KV_HEADS, DIM)),
            _normal(gen, (LAYERS, tokens, KV_HEADS, DIM)))


def _norm_weight(gen):
    return 1 + _normal(gen, (HIDDEN,), 0.1)


def _mlp_inputs(case, seed):
    gen = _gen(seed)
    rows = case["rows"]
    x, hidden = _normal(gen, (rows, HIDDEN)), _normal(gen, (rows, HIDDEN))
    layers = [(_normal(gen, (2 * MLP, HIDDEN), 0.02), _normal(gen, (HIDDEN, MLP), 0.02), _norm_weight(gen)) for _ in range(LAYERS)]
    return x, hidden, layers


def _project_inputs(case, seed):
    gen = _gen(seed)
    rows = case["rows"]
    rng = np.random.Generator(np.random.PCG64(seed))
    x, hidden, attended = (_normal(gen, (rows, HIDDEN)) for _ in range(3))
    layers = [(_normal(gen, (QKV, HIDDEN), 0.02), _normal(gen, (HIDDEN, HIDDEN), 0.02), _norm_weight(gen)) for _ in range(LAYERS)]
    positions = torch.from_numpy(rng.integers(0, 2048, size=rows)).to(DEVICE)
    slots = torch.from_numpy(rng.permutation(rows * BLOCK)[:rows].astype(np.int64)).to(DEVICE)
    return x, hidden, attended, layers, positions, slots


def _model(seed):
    """The architecture's weights with q|k|v and gate|up stacked, as random_weights lays them out."""
    gen = _gen(seed)
    layers = []
    for _ in range(LAYERS):
        qkv, gate_up = _normal(gen, (QKV, HIDDEN), 0.02), _normal(gen, (2 * MLP, HIDDEN), 0.02)
        layers.append(LayerWeights(
            input_norm=_norm_weight(gen), q_proj=qkv[:HIDDEN], k_proj=qkv[HIDDEN : HIDDEN + 256], v_proj=qkv[HIDDEN + 256 :],
            o_proj=_normal(gen, (HIDDEN, HIDDEN), 0.02), post_attention_norm=_norm_weight(gen), gate_proj=gate_up[:MLP],
            up_proj=gate_up[MLP:], down_proj=_normal(gen, (HIDDEN, MLP), 0.02)))
    return TinyLlamaWeights(_normal(gen, (VOCAB, HIDDEN), 0.02), tuple(layers), _norm_weight(gen), _normal(gen, (VOCAB, HIDDEN), 0.02))


def _serve_ids(case, seed):
    """Each request's prompt ids and the ids it is fed at every decode step."""
    rng = np.random.Generator(np.random.PCG64(seed))
    lengths = rng.integers(case["lo"], case["hi"] + 1, size=case["requests"])
    return [rng.integers(0, VOCAB, size=int(n)) for n in lengths], rng.integers(0, VOCAB, size=(case["steps"], case["requests"]))


def _credits(tokens):
    return (tokens + BLOCK - 1) // BLOCK


def _allocator(tables, lengths, blocks, seed):
    """An allocator whose requests hold N(0, 1) K/V of the given lengths (layer 0 is read)."""
    gen = _gen(seed)
    allocator = KVAllocator(_pool(blocks))
    requests = tuple(RequestId("r%d" % i) for i in range(len(lengths)))
    for request, n in zip(requests, lengths):
        allocator.create(KVReservation(request, _credits(int(n))))
        kv = _normal(gen, (2, 1, int(n), KV_HEADS, DIM)).expand(2, LAYERS, int(n), KV_HEADS, DIM)
        allocator.append(request, kv[0], kv[1])
    return allocator, requests, _normal(gen, (len(lengths), Q_HEADS, 1, DIM))


# ---------------------------------------------------------------------------------------
# What a program holds, and one pass
# ---------------------------------------------------------------------------------------


def prepare(case, seed):
    kind, device = case["kind"], torch.device(DEVICE)
    if kind == "attend_api":
        lengths, tables, blocks = _sequences(case, seed)
        allocator, requests, query = _allocator(tables, lengths, blocks, seed)
        return {"kind": kind, "allocator": allocator, "requests": requests, "query": query}
    if kind == "attend" or kind == "append_attend":
        lengths, tables, pool, query, new = _attend_inputs(case, seed)
        batch, width = tables.shape
        plan = torch.from_numpy(_hip.decode_plan(lengths, tables)).to(device)
        lens = torch.from_numpy(lengths).to(device)
        workspace = torch.zeros(_hip.workspace_bytes(batch, width), dtype=torch.uint8, device=device)
        out = torch.zeros_like(query)

        def step():
            for layer in range(case["layers"]):
                more = {} if new is None else {"new_key": new[0, layer], "new_value": new[1, layer]}
                _hip.planned_decode_attention(out[layer], query[layer], pool, layer, lens, plan, width, workspace, **more)

        graph, _ = capture_graph(step, device)
        result = out if new is None else [out, pool[: case["layers"]]]
        return {"kind": kind, "graph": graph, "out": result, "keep": (pool, query, new, plan, lens, workspace)}
    if kind == "append":
        blocks, slots, key, value = _append_inputs(case, seed)
        pool = _pool(blocks).zero_()
        return {"kind": kind, "pool": pool, "slots": slots, "key": key, "value": value}
    if kind == "prompt_attend":
        query, key, value = _prompt_inputs(case, seed)
        out = torch.zeros_like(query)

        def step():
            for layer in range(LAYERS):
                _hip.prefill_attention(out[layer], query[layer], key[layer], value[layer])

        graph, _ = capture_graph(step, device)
        return {"kind": kind, "graph": graph, "out": out, "keep": (query, key, value)}
    if kind == "mlp":
        x, hidden, layers = _mlp_inputs(case, seed)
        rows = case["rows"]
        activated = torch.empty((rows, MLP), dtype=torch.float16, device=device)
        parts = torch.empty((8, rows, HIDDEN), dtype=torch.float32, device=device)
        sums = torch.empty((LAYERS, rows, HIDDEN), dtype=torch.float16, device=device)
        out = torch.empty_like(sums)

        def step():
            sums.copy_(hidden.expand_as(sums))
            for layer, (gate_up, down, norm) in enumerate(layers):
                _hip.gemm_m128(activated, x, gate_up, epilogue=_hip.GEMM_SWIGLU)
                _hip.gemm_m128(parts, activated, down, splits=8)
                _hip.add_rms_norm_parts(out[layer], sums[layer], parts, norm, EPS)

        step()
        graph, _ = capture_graph(step, device)
        return {"kind": kind, "graph": graph, "out": [out, sums], "keep": (x, hidden, layers, activated, parts)}
    if kind == "project":
        x, hidden, attended, layers, positions, slots = _project_inputs(case, seed)
        rows = case["rows"]
        table = rope_table(device)
        pool = _pool(rows).zero_()
        qkv = torch.empty((2, rows, QKV), dtype=torch.float32, device=device)
        parts = torch.empty((4, rows, HIDDEN), dtype=torch.float32, device=device)
        query = torch.empty((LAYERS, rows, Q_HEADS, DIM), dtype=torch.float16, device=device)
        sums = torch.empty((LAYERS, rows, HIDDEN), dtype=torch.float16, device=device)
        out = torch.empty_like(sums)

        def step():
            sums.copy_(hidden.expand_as(sums))
            for layer, (w_qkv, w_o, norm) in enumerate(layers):
                _hip.gemm_m128(qkv, x, w_qkv, splits=2)
                _hip.rope_kv_append_parts(query[layer], qkv, positions, table, pool=pool, layer=layer, slot_mapping=slots)
                _hip.gemm_m128(parts, attended, w_o, splits=4)
                _hip.add_rms_norm_parts(out[layer], sums[layer], parts, norm, EPS)

        step()
        graph, _ = capture_graph(step, device)
        return {"kind": kind, "graph": graph, "out": [query, pool, out, sums],
                "keep": (x, hidden, attended, layers, positions, slots, qkv, parts, table)}
    if kind == "prefill":
        weights = _model(seed)
        rng = np.random.Generator(np.random.PCG64(seed))
        ids = torch.from_numpy(rng.integers(0, VOCAB, size=(1, case["tokens"]))).to(device)
        allocator = KVAllocator(_pool(_credits(case["tokens"]) + 32).zero_())
        return {"kind": kind, "weights": weights, "ids": ids, "allocator": allocator,
                "reservation": KVReservation(RequestId("prompt"), _credits(case["tokens"]))}
    prompts, fed = _serve_ids(case, seed)
    weights = _model(seed)
    credits = [_credits(len(p) + case["steps"]) for p in prompts]
    allocator = KVAllocator(_pool(sum(credits) + 16).zero_())
    graphs = {}
    for prompt in prompts:
        size = next(s for s in PREFILL_SIZES if s >= len(prompt))
        if size not in graphs:
            graphs[size] = PrefillGraph(weights, allocator, size)
    requests = tuple(RequestId("r%d" % i) for i in range(len(prompts)))
    admissions = [(KVReservation(r, c), graphs[next(s for s in PREFILL_SIZES if s >= len(p))],
                   torch.from_numpy(p[None]).to(device)) for r, c, p in zip(requests, credits, prompts)]
    return {"kind": kind, "allocator": allocator, "requests": requests, "admissions": admissions,
            "decode": DecodeGraph(weights, allocator, case["rows"]), "fed": torch.from_numpy(fed[:, :, None]).to(device)}


def run(state):
    kind = state["kind"]
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if kind == "attend_api":
        if len(state["requests"]) == 1:
            return paged_attention(state["query"], state["allocator"], state["requests"][0], layer_index=0)
        return paged_attention_batch(state["query"], state["allocator"], state["requests"], layer_index=0)
    if kind == "append":
        _hip.kv_append(state["pool"], 0, state["key"], state["value"], state["slots"])
        return state["pool"]
    allocator = state["allocator"]
    if kind == "prefill":
        allocator.create(state["reservation"])
        logits = prefill_paged(state["ids"], state["weights"], allocator, state["reservation"].request_id)
        allocator.release_all(state["reservation"].request_id)
        return [logits, allocator.pool]
    first, decode, requests = [], state["decode"], state["requests"]
    for reservation, graph, ids in state["admissions"]:
        allocator.create(reservation)
        first.append(graph.step(ids, reservation.request_id))
    later = [decode.step(ids, requests) for ids in state["fed"]]
    decode.check_faults()
    for request in requests:
        allocator.release_all(request)
    return [torch.cat(first), torch.cat(later)]


# ---------------------------------------------------------------------------------------
# What a pass cannot do without, and how exact it is
# ---------------------------------------------------------------------------------------


def _attend_work(lengths):
    tokens = int(lengths.sum())
    blocks = int(((lengths + BLOCK - 1) // BLOCK).sum())
    return tokens * 1024 + len(lengths) * (2 * Q_HEADS * DIM * 2 + 4) + blocks * 4, tokens * Q_HEADS * DIM * 4


def _causal_flops(tokens):
    return tokens * (tokens + 1) // 2 * Q_HEADS * DIM * 4


def work(case):
    kind = case["kind"]
    if kind in ("attend_api", "attend", "append_attend"):
        # The mean context: work() has no seed, and a batch's lengths are drawn from it.
        mean = np.full(case["batch"], (case["lo"] + case["hi"]) // 2, dtype=np.int64)
        bytes_, flops = _attend_work(mean)
        if kind == "append_attend":
            bytes_ += case["batch"] * 2 * 1024
        layers = case.get("layers", 1)
        return {"bytes": layers * bytes_, "flops": layers * flops}
    if kind == "append":
        return {"bytes": case["tokens"] * (LAYERS * 2 * 1024 + 8), "flops": 0}
    if kind == "prompt_attend":
        tokens = case["tokens"]
        return {"bytes": LAYERS * tokens * (2 * Q_HEADS + 2 * KV_HEADS) * DIM * 2, "flops": LAYERS * _causal_flops(tokens)}
    if kind == "mlp":
        rows = case["rows"]
        return {"bytes": LAYERS * (3 * MLP * HIDDEN * 2 + 3 * rows * HIDDEN * 2), "flops": LAYERS * rows * 3 * MLP * HIDDEN * 2}
    if kind == "project":
        rows = case["rows"]
        elements = (QKV + HIDDEN) * HIDDEN
        return {"bytes": LAYERS * (elements * 2 + rows * (QKV + 4 * HIDDEN) * 2), "flops": LAYERS * rows * elements * 2}
    model = LAYERS * LAYER_WEIGHTS
    if kind == "prefill":
        tokens = case["tokens"]
        return {"bytes": 2 * (model + VOCAB * HIDDEN) + tokens * (VOCAB * 2 + HIDDEN * 2 + LAYERS * 1024),
                "flops": 2 * tokens * (model + VOCAB * HIDDEN) + LAYERS * _causal_flops(tokens)}
    # serve: every prompt and every step reads the weights; each step reads the cached K/V.
    requests, steps, mean = case["requests"], case["steps"], (case["lo"] + case["hi"]) // 2
    passes = requests + steps
    cached = steps * requests * (mean + steps // 2)
    return {"bytes": passes * 2 * (model + VOCAB * HIDDEN) + (cached + requests * mean) * LAYERS * 1024 + (requests + steps * requests) * VOCAB * 2,
            "flops": 2 * model * requests * (mean + steps) + 2 * VOCAB * HIDDEN * requests * (1 + steps)
            + LAYERS * (requests * _causal_flops(mean) + cached * Q_HEADS * DIM * 4)}


def tolerance(case):
    kind = case["kind"]
    if kind == "append":
        return "exact"  # bytes are moved, nothing is computed
    # About four times the error against 64 bits measured for each kind.
    if kind in ("attend_api", "attend", "append_attend"):
        return {"rel": 8.5e-4}  # one fp16 rounding of the outputs: 2.1e-4
    if kind == "prompt_attend":
        return {"rel": 1e-3}  # probabilities enter the product as fp16: 2.5e-4
    if kind == "mlp" or kind == "project":
        return {"rel": 1.9e-3}  # fp16 roundings of the projection, the sum and the norm: 3e-4 to 4.7e-4
    return {"rel": 1.5e-2}  # fp16 roundings carried through 22 layers: 3.1e-3 to 3.6e-3


# ---------------------------------------------------------------------------------------
# The same in 64 bits, with torch alone
# ---------------------------------------------------------------------------------------


def _attention64(query, key, value, mask=None):
    """softmax(q k^T / 8) v for q [T, 32, 64] and k, v [L, 4, 64], all float64."""
    q = query.reshape(query.shape[0], KV_HEADS, Q_HEADS // KV_HEADS, DIM).permute(1, 2, 0, 3).contiguous()  # [4, 8, T, 64]
    k, v = (t.permute(1, 2, 0).contiguous() for t in (key, value))  # [4, 64, L]
    out = torch.empty_like(q)
    for h in range(KV_HEADS):
        scores = (q[h].reshape(-1, DIM) @ k[h] / 8).view(Q_HEADS // KV_HEADS, -1, key.shape[0])
        if mask is not None:
            scores = scores.masked_fill(mask, float("-inf"))
        out[h] = (torch.softmax(scores, -1).reshape(-1, key.shape[0]) @ v[h].T.contiguous()).view_as(out[h])
    return out.permute(2, 0, 1, 3).reshape(query.shape)


def _causal_mask(tokens):
    return torch.ones(tokens, tokens, dtype=torch.bool, device=DEVICE).triu(1)


def _history(pool, layer, table, length):
    rows = pool[layer, :, torch.from_numpy(table.astype(np.int64)).to(DEVICE)]  # [2, n, 16, 4, 64]
    return rows.reshape(2, -1, KV_HEADS, DIM)[:, :length].double()


def _norm64(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _rope64(x, positions):
    """Rotate [T, heads, 64] by the model's fp16 cos/sin table at the given positions."""
    inverse = 1.0 / (10000.0 ** (torch.arange(0, DIM, 2).float() / DIM))
    angles = torch.arange(2048).float()[:, None] * inverse
    c, s = (t.half().double().to(DEVICE)[positions][:, None, :] for t in (angles.cos(), angles.sin()))
    lo, hi = x[..., : DIM // 2], x[..., DIM // 2 :]
    return torch.cat((lo * c - hi * s, hi * c + lo * s), -1)


def _forward64(weights, ids, positions_out):
    """Float64 logits at `positions_out` of a causal forward over `ids`, and each layer's K and V."""
    ids = torch.as_tensor(ids, device=DEVICE)
    tokens = ids.shape[0]
    positions = torch.arange(tokens, device=DEVICE)
    mask = _causal_mask(tokens)
    hidden = weights.embedding[ids].double()
    cache = []
    for w in weights.layers:
        x = _norm64(hidden, w.input_norm)
        q = _rope64((x @ w.q_proj.double().T).view(tokens, Q_HEADS, DIM), positions)
        k = _rope64((x @ w.k_proj.double().T).view(tokens, KV_HEADS, DIM), positions)
        v = (x @ w.v_proj.double().T).view(tokens, KV_HEADS, DIM)
        cache.append((k, v))
        hidden = hidden + _attention64(q, k, v, mask).reshape(tokens, HIDDEN) @ w.o_proj.double().T
        x = _norm64(hidden, w.post_attention_norm)
        hidden = hidden + (torch.nn.functional.silu(x @ w.gate_proj.double().T) * (x @ w.up_proj.double().T)) @ w.down_proj.double().T
    return _norm64(hidden[positions_out], weights.final_norm) @ weights.lm_head.double().T, cache


def exact(case, seed):
    kind = case["kind"]
    if kind == "attend_api":
        lengths, tables, blocks = _sequences(case, seed)
        gen = _gen(seed)
        kv = [_normal(gen, (2, 1, int(n), KV_HEADS, DIM))[:, 0].double() for n in lengths]
        query = _normal(gen, (len(lengths), Q_HEADS, 1, DIM)).double()
        return torch.stack([_attention64(q.view(1, Q_HEADS, DIM), k, v).reshape(Q_HEADS, 1, DIM) for q, (k, v) in zip(query, kv)])
    if kind == "attend" or kind == "append_attend":
        lengths, tables, pool, query, new = _attend_inputs(case, seed)
        if new is not None:
            last = lengths - 1
            blocks = torch.from_numpy(tables[np.arange(len(lengths)), last // BLOCK].astype(np.int64)).to(DEVICE)
            slots = torch.from_numpy((last % BLOCK).astype(np.int64)).to(DEVICE)
            for layer in range(case["layers"]):
                for which in range(2):
                    pool[layer, which, blocks, slots] = new[which, layer]
        out = torch.empty(query.shape, dtype=torch.float64, device=DEVICE)
        for layer in range(case["layers"]):
            for row, n in enumerate(lengths):
                history = _history(pool, layer, tables[row, : _credits(int(n))], int(n))
                out[layer, row] = _attention64(query[layer, row : row + 1].double(), history[0], history[1])[0]
        return out if new is None else [out, None]
    if kind == "append":
        return None
    if kind == "prompt_attend":
        query, key, value = _prompt_inputs(case, seed)
        mask = _causal_mask(case["tokens"])
        return torch.stack([_attention64(query[i].double(), key[i].double(), value[i].double(), mask) for i in range(LAYERS)])
    if kind == "mlp":
        x, hidden, layers = _mlp_inputs(case, seed)
        x = x.double()
        sums = torch.stack([hidden.double() + (torch.nn.functional.silu(x @ gate_up[:MLP].double().T)
                                               * (x @ gate_up[MLP:].double().T)) @ down.double().T for gate_up, down, _ in layers])
        return [torch.stack([_norm64(s, norm) for s, (_, _, norm) in zip(sums, layers)]), sums]
    if kind == "project":
        x, hidden, attended, layers, positions, slots = _project_inputs(case, seed)
        rows = case["rows"]
        pool = torch.zeros((LAYERS, 2, rows * BLOCK, KV_HEADS, DIM), dtype=torch.float64, device=DEVICE)
        query = torch.empty((LAYERS, rows, Q_HEADS, DIM), dtype=torch.float64, device=DEVICE)
        for layer, (w_qkv, _, _) in enumerate(layers):
            qkv = (x.double() @ w_qkv.double().T).view(rows, -1, DIM)
            query[layer] = _rope64(qkv[:, :Q_HEADS], positions)
            pool[layer, 0, slots] = _rope64(qkv[:, Q_HEADS : Q_HEADS + KV_HEADS], positions)
            pool[layer, 1, slots] = qkv[:, Q_HEADS + KV_HEADS :]
        sums = torch.stack([hidden.double() + attended.double() @ w_o.double().T for _, w_o, _ in layers])
        out = torch.stack([_norm64(s, norm) for s, (_, _, norm) in zip(sums, layers)])
        return [query, pool.view(LAYERS, 2, rows, BLOCK, KV_HEADS, DIM), out, sums]
    if kind == "prefill":
        weights = _model(seed)
        rng = np.random.Generator(np.random.PCG64(seed))
        ids = rng.integers(0, VOCAB, size=(1, case["tokens"]))[0]
        logits, _ = _forward64(weights, ids, torch.arange(case["tokens"], device=DEVICE))
        return [logits[None], None]
    prompts, fed = _serve_ids(case, seed)
    weights = _model(seed)
    first, later = [], []
    for row, prompt in enumerate(prompts):
        ids = np.concatenate([prompt, fed[:, row]])
        logits, _ = _forward64(weights, ids, torch.arange(len(prompt) - 1, len(ids), device=DEVICE))
        first.append(logits[:1])
        later.append(logits[1:])
    return [torch.stack(first), torch.stack(later, 1).reshape(-1, 1, VOCAB)]
