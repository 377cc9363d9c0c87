"""The work a serving program gives this library, as timed cases.

Shapes are those of the package's own workloads (``mini_infra_qwen3_amd.workloads``) and the dense
Qwen3 head counts the kernels are built for: 8 KV heads of 128, 16 / 32 / 40 / 64 query heads,
16-token blocks, bf16.  Each case goes through an entry point a program calls:

* ``decode``  -- ``data_plane.paged_decode_attention_fused`` (q/k norm + RoPE, K/V append and
  attention of one decode layer) or, with ``append`` off, ``paged_decode_attention``; with the
  bandwidth kernels or with reference numerics (``exact``);
* ``prefill`` -- ``data_plane.chunked_prefill_attention``: left-padded prompt chunks with their
  history in the pool, either numerics;
* ``mixed``   -- ``data_plane.mixed_paged_attention``: ragged prompt chunks and decode rows of one step;
* ``store``   -- ``data_plane.reshape_and_cache``: prompts' K/V of every layer into their pool slots;
* ``model``   -- a whole decode step of the 28-layer model, captured in a HIP graph once and replayed,
  as ``PagedRunner`` serves it.

Context and chunk lengths belong to the case (``lengths_seed``), values and block tables to the seed.
"""

import math
import random

import torch

from mini_infra_qwen3_amd import data_plane
from mini_infra_qwen3_amd.model.config import qwen3_0_6b
from mini_infra_qwen3_amd.model.qwen3 import PagedAttentionMetadata, Qwen3ForCausalLM

HEAD_DIM = 128
BLOCK = 16
SCALE = HEAD_DIM ** -0.5
EPS = 1e-6
THETA = 1_000_000.0
LAYERS = 28


def listed():
    return [
        # One sequence decoding alone: the smallest call, launch and latency bound.
        {"name": "decode_one", "kind": "decode", "batch": 1, "dist": "uniform", "lo": 417, "hi": 417, "lengths_seed": 0,
         "heads": 16, "kv_heads": 8, "exact": False, "append": True},
        # A serving batch of the continuous-batching run (about 9 live requests, prompts U[32, 1024]
        # plus up to 128 new tokens) with the default, reference numerics.
        {"name": "decode_serving_exact", "kind": "decode", "batch": 9, "dist": "uniform", "lo": 32, "hi": 1150,
         "lengths_seed": 1, "heads": 16, "kv_heads": 8, "exact": True, "append": True},
        # A full serving batch with the bandwidth kernels.
        {"name": "decode_batch", "kind": "decode", "batch": 64, "dist": "uniform", "lo": 32, "hi": 1150,
         "lengths_seed": 2, "heads": 16, "kv_heads": 8, "exact": False, "append": True},
        # A larger GQA group (64 query heads on 8 KV heads) at longer contexts.
        {"name": "decode_group8", "kind": "decode", "batch": 21, "dist": "lognormal", "lo": 256, "hi": 8192,
         "lengths_seed": 3, "heads": 64, "kv_heads": 8, "exact": False, "append": True},
        # Decode at scale: one layer of the 256-sequence step, about 3 GB of K/V.
        {"name": "decode_scale", "kind": "decode", "batch": 256, "dist": "lognormal", "lo": 256, "hi": 8192,
         "lengths_seed": 4, "heads": 16, "kv_heads": 8, "exact": False, "append": False},
        # Two prompts of the serving run prefilled together, no history.
        {"name": "prefill_prompts", "kind": "prefill", "rows": 2, "lo": 250, "hi": 700, "start": 0, "lengths_seed": 5,
         "heads": 16, "kv_heads": 8, "exact": False},
        # The same kind of step with the default, reference numerics; ragged lengths, some history.
        {"name": "prefill_prompts_exact", "kind": "prefill", "rows": 2, "lo": 400, "hi": 1024, "start": 300,
         "lengths_seed": 6, "heads": 16, "kv_heads": 8, "exact": True},
        # Long prompts in 2048-token chunks, deep in their history: the largest prefill call.
        {"name": "prefill_long", "kind": "prefill", "rows": 4, "lo": 2048, "hi": 2048, "start": 10240,
         "lengths_seed": 7, "heads": 16, "kv_heads": 8, "exact": False},
        # A mixed step: one arriving prompt beside eight decoding requests.
        {"name": "mixed_step", "kind": "mixed", "rows": 1, "lo": 650, "hi": 800, "start": 0, "decode_rows": 8,
         "lengths_seed": 8, "heads": 16, "kv_heads": 8, "exact": False},
        {"name": "mixed_step_exact", "kind": "mixed", "rows": 1, "lo": 400, "hi": 650, "start": 0, "decode_rows": 7,
         "lengths_seed": 9, "heads": 16, "kv_heads": 8, "exact": True},
        # The prefill store: four prompts' K/V of all 28 layers into the pool.
        {"name": "store_prefill", "kind": "store", "rows": 4, "lo": 128, "hi": 2048, "layers": LAYERS,
         "lengths_seed": 10, "kv_heads": 8},
        # A whole decode step of the model (bandwidth numerics), replayed from its HIP graph.
        {"name": "model_decode", "kind": "model", "batch": 8, "lo": 32, "hi": 1150, "lengths_seed": 11},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode_exact", "prefill", "prefill", "prefill_exact", "mixed", "mixed_exact",
                       "store", "model"))
    seed = rng.randrange(1 << 30)
    heads = rng.choice((16, 16, 16, 32, 40, 64))
    if kind in ("decode", "decode_exact"):
        exact = kind == "decode_exact"
        lognormal = not exact and rng.random() < 0.5
        batch = _log_int(rng, 1, 40 if exact else 128)
        hi = 8192 if lognormal else rng.randrange(64, 1200)
        return {"kind": "decode", "batch": batch, "dist": "lognormal" if lognormal else "uniform",
                "lo": 256 if lognormal else rng.randrange(1, 64), "hi": hi, "lengths_seed": seed, "heads": heads,
                "kv_heads": 8, "exact": exact, "append": True}
    if kind in ("prefill", "prefill_exact"):
        exact = kind == "prefill_exact"
        hi = _log_int(rng, 24, 1024 if exact else 2048)
        return {"kind": "prefill", "rows": rng.randrange(1, 3 if exact else 4), "lo": max(hi // 2, 1), "hi": hi,
                "start": rng.choice((0, rng.randrange(1, 600 if exact else 6000))), "lengths_seed": seed, "heads": 16,
                "kv_heads": 8, "exact": exact}
    if kind in ("mixed", "mixed_exact"):
        exact = kind == "mixed_exact"
        hi = _log_int(rng, 24, 650 if exact else 1024)
        return {"kind": "mixed", "rows": rng.randrange(1, 3), "lo": max(hi // 2, 1), "hi": hi,
                "start": rng.choice((0, rng.randrange(1, 500))), "decode_rows": _log_int(rng, 1, 16 if exact else 32),
                "lengths_seed": seed, "heads": 16, "kv_heads": 8, "exact": exact}
    if kind == "store":
        return {"kind": "store", "rows": rng.randrange(1, 5), "lo": 1, "hi": _log_int(rng, 24, 2048), "layers": LAYERS,
                "lengths_seed": seed, "kv_heads": 8}
    return {"kind": "model", "batch": _log_int(rng, 1, 24), "lo": 32, "hi": 1150, "lengths_seed": seed}


# ------------------------------------------------------------------ lengths and block tables
def _lengths(case):
    """Decode: contexts (the new token included).  Prefill / mixed / store: chunk lengths."""
    rng = random.Random(case["lengths_seed"])
    n = case["batch"] if "batch" in case else case["rows"]
    if case.get("dist") == "lognormal":
        draws = [math.exp(math.log(2048.0) + 1.3 * rng.gauss(0.0, 1.0)) for _ in range(n)]
        return [int(min(max(round(x), case["lo"]), case["hi"])) for x in draws]
    return [rng.randint(case["lo"], case["hi"]) for _ in range(n)]


def _starts(case):
    """History lengths of the chunk rows: up to 20% below the case's start, not block aligned."""
    rng = random.Random(case["lengths_seed"] + 1)
    return [rng.randint(case["start"] * 4 // 5, case["start"]) if case["start"] else 0 for _ in range(case["rows"])]


def _mixed_contexts(case):
    rng = random.Random(case["lengths_seed"] + 2)
    return [rng.randint(33, 1150) for _ in range(case["decode_rows"])]


def _blocks(tokens):
    return -(-tokens // BLOCK)


def _tables(token_counts, gen):
    """Null-padded block tables of a scattered pool, one row per sequence, and the pool's block count."""
    need = [_blocks(n) for n in token_counts]
    num_blocks = 1 + sum(need) + 64
    perm = torch.randperm(num_blocks - 1, generator=gen) + 1
    width = max(max(need), 1)
    table = torch.zeros((len(need), width), dtype=torch.long)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return table, num_blocks


def _slot(table, row, position):
    return int(table[row, position // BLOCK]) * BLOCK + position % BLOCK


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda").to(torch.bfloat16)


def _generators(seed):
    return torch.Generator().manual_seed(seed), torch.Generator(device="cuda").manual_seed(seed + 1)


def _rope_tables(positions):
    inv = 1.0 / THETA ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float32) / HEAD_DIM)
    angles = torch.tensor(positions, dtype=torch.float32).unsqueeze(-1) * inv
    angles = torch.cat((angles, angles), dim=-1)
    return angles.cos().to(torch.bfloat16).cuda(), angles.sin().to(torch.bfloat16).cuda()


# --------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "mixed": _prepare_mixed, "store": _prepare_store,
            "model": _prepare_model}[case["kind"]](case, seed)


def _prepare_decode(case, seed):
    cpu, gpu = _generators(seed)
    ctx = _lengths(case)
    batch, heads, kv = case["batch"], case["heads"], case["kv_heads"]
    table, num_blocks = _tables(ctx, cpu)
    state = {"case": case, "ctx": torch.tensor(ctx).cuda(), "tables": table.cuda()}
    state["key_pool"] = _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM)
    state["value_pool"] = _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM)
    if case["append"]:
        qkv = _randn(gpu, batch, (heads + 2 * kv) * HEAD_DIM)  # one projection's rows, split into views
        state["q"], state["k"], state["v"] = qkv.split((heads * HEAD_DIM, kv * HEAD_DIM, kv * HEAD_DIM), dim=1)
        state["q_weight"] = (1 + 0.1 * torch.randn(HEAD_DIM, generator=gpu, device="cuda")).to(torch.bfloat16)
        state["k_weight"] = (1 + 0.1 * torch.randn(HEAD_DIM, generator=gpu, device="cuda")).to(torch.bfloat16)
        state["cos"], state["sin"] = _rope_tables([n - 1 for n in ctx])
        state["slots"] = torch.tensor([_slot(table, i, n - 1) for i, n in enumerate(ctx)]).cuda()
    else:
        state["query"] = _randn(gpu, batch, heads, HEAD_DIM)
    # One workspace per model forward, shared by its layers.
    need = max(data_plane.paged_decode_workspace_bytes(batch, table.shape[1], heads, HEAD_DIM, BLOCK, kv),
               data_plane.paged_decode_exact_workspace_bytes(batch, table.shape[1], heads, kv, BLOCK), 1)
    state["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    return state


def _prepare_prefill(case, seed):
    cpu, gpu = _generators(seed)
    lens, starts = _lengths(case), _starts(case)
    rows, heads, kv, width = case["rows"], case["heads"], case["kv_heads"], max(lens)
    table, num_blocks = _tables(starts, cpu)
    hist = table if any(starts) else table[:, :0]
    # Token-major rows seen as [B, heads, L, D], as the model hands them over.
    q = _randn(gpu, rows, width, heads, HEAD_DIM).transpose(1, 2)
    k = _randn(gpu, rows, width, kv, HEAD_DIM).transpose(1, 2)
    v = _randn(gpu, rows, width, kv, HEAD_DIM).transpose(1, 2)
    return {"case": case, "q": q, "k": k, "v": v, "key_pool": _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM),
            "value_pool": _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM), "hist": hist.contiguous().cuda(),
            "starts": torch.tensor(starts).cuda(), "lens": torch.tensor(lens).cuda()}


def _prepare_mixed(case, seed):
    cpu, gpu = _generators(seed)
    lens, starts, ctx = _lengths(case), _starts(case), _mixed_contexts(case)
    rows, heads, kv = case["rows"], case["heads"], case["kv_heads"]
    table, num_blocks = _tables(starts + ctx, cpu)
    hist = table[:rows, :max(_blocks(max(starts)), 0)].contiguous()
    dec = table[rows:, :_blocks(max(ctx))].contiguous()
    chunk_tokens = sum(lens)
    tokens = chunk_tokens + len(ctx)
    first = [sum(lens[:i]) for i in range(rows)]
    return {"case": case, "q": _randn(gpu, tokens, heads, HEAD_DIM), "k": _randn(gpu, tokens, kv, HEAD_DIM),
            "v": _randn(gpu, tokens, kv, HEAD_DIM), "key_pool": _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM),
            "value_pool": _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM), "rows": rows, "width": max(lens),
            "hist": hist.cuda(), "starts": torch.tensor(starts).cuda(), "lens": torch.tensor(lens).cuda(),
            "tables": dec.cuda(), "ctx": torch.tensor(ctx).cuda(), "first": torch.tensor(first).cuda(),
            "chunk_tokens": chunk_tokens,
            "slots": torch.tensor([_slot(dec, i, n - 1) for i, n in enumerate(ctx)]).cuda()}


def _prepare_store(case, seed):
    cpu, gpu = _generators(seed)
    lens = _lengths(case)
    rows, kv, width, layers = case["rows"], case["kv_heads"], max(lens), case["layers"]
    table, num_blocks = _tables(lens, cpu)
    triples = [(r, width - n + t, _slot(table, r, t)) for r, n in enumerate(lens) for t in range(n)]
    index = torch.tensor(triples).t().contiguous().cuda()
    keys = [_randn(gpu, rows, width, kv, HEAD_DIM).transpose(1, 2) for _ in range(layers)]
    values = [_randn(gpu, rows, width, kv, HEAD_DIM).transpose(1, 2) for _ in range(layers)]
    pools = [torch.zeros((2, num_blocks, BLOCK, kv, HEAD_DIM), dtype=torch.bfloat16, device="cuda")
             for _ in range(layers)]
    return {"case": case, "keys": keys, "values": values, "token_rows": index[0], "positions": index[1],
            "slots": index[2], "key_pools": [p[0] for p in pools], "value_pools": [p[1] for p in pools]}


def _prepare_model(case, seed):
    cpu, gpu = _generators(seed)
    config = qwen3_0_6b()
    with torch.device("cuda"):
        model = Qwen3ForCausalLM(config, exact=False)
    model = model.to("cuda", torch.bfloat16).eval()
    with torch.no_grad():
        for name, p in model.named_parameters():
            if p.ndim == 1:
                p.copy_(1 + 0.1 * torch.randn(p.shape, generator=gpu, device="cuda"))
            else:
                p.copy_(0.02 * torch.randn(p.shape, generator=gpu, device="cuda"))
    ctx = _lengths(case)
    table, num_blocks = _tables(ctx, cpu)
    kv = config.num_key_value_heads
    pools = tuple((_randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM), _randn(gpu, num_blocks, BLOCK, kv, HEAD_DIM))
                  for _ in range(config.num_hidden_layers))
    ids = torch.randint(1000, 100000, (case["batch"], 1), generator=cpu).cuda()
    positions = torch.tensor(ctx).unsqueeze(1).cuda() - 1
    slots = torch.tensor([_slot(table, i, n - 1) for i, n in enumerate(ctx)]).cuda()
    meta = PagedAttentionMetadata(slot_mapping=slots, block_tables=table.cuda(), context_lens=torch.tensor(ctx).cuda(),
                                  kv_pools=pools)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.inference_mode():
        for _ in range(2):  # warm-up outside the capture
            model(ids, position_ids=positions, attn_metadata=meta, last_logits_only=True)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph), torch.inference_mode():
        logits, _ = model(ids, position_ids=positions, attn_metadata=meta, last_logits_only=True)
    return {"case": case, "model": model, "ids": ids, "positions": positions, "meta": meta, "graph": graph,
            "logits": logits}


# ------------------------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        if not case["append"]:
            return data_plane.paged_decode_attention(state["query"], state["key_pool"], state["value_pool"],
                                                     state["tables"], state["ctx"], SCALE, workspace=state["workspace"],
                                                     exact=case["exact"])
        out = data_plane.paged_decode_attention_fused(
            state["q"], state["k"], state["v"], state["q_weight"], state["k_weight"], state["cos"], state["sin"], EPS,
            state["slots"], state["key_pool"], state["value_pool"], state["tables"], state["ctx"], SCALE,
            workspace=state["workspace"], exact=case["exact"])
        return out, state["key_pool"], state["value_pool"]
    if kind == "prefill":
        return data_plane.chunked_prefill_attention(state["q"], state["k"], state["v"], state["key_pool"],
                                                    state["value_pool"], state["hist"], state["starts"], state["lens"],
                                                    SCALE, exact=case["exact"])
    if kind == "mixed":
        out = data_plane.mixed_paged_attention(
            state["q"], state["k"], state["v"], state["key_pool"], state["value_pool"], state["rows"], state["width"],
            state["hist"], state["starts"], state["lens"], state["tables"], state["ctx"], state["slots"], SCALE,
            exact=case["exact"], chunk_first=state["first"], chunk_tokens=state["chunk_tokens"])
        return out, state["key_pool"], state["value_pool"]
    if kind == "store":
        data_plane.reshape_and_cache(state["keys"], state["values"], state["slots"], state["key_pools"],
                                     state["value_pools"], token_rows=state["token_rows"],
                                     token_positions=state["positions"])
        return state["key_pools"], state["value_pools"]
    state["graph"].replay()
    return state["logits"], [k for k, _ in state["meta"].kv_pools], [v for _, v in state["meta"].kv_pools]


# ------------------------------------------------------------------------ work and tolerance
def _attention_flops(heads, pairs):
    return 4.0 * HEAD_DIM * heads * pairs  # Q K^T and P V over the visible (query, key) pairs


def _chunk_pairs(lens, starts):
    return sum(n * s + n * (n + 1) // 2 for n, s in zip(lens, starts))


def work(case):
    kv_row = 2 * case.get("kv_heads", 8) * HEAD_DIM * 2  # one token's K and V, bf16
    kind = case["kind"]
    if kind == "decode":
        ctx = _lengths(case)
        rows = 2 * case["batch"] * case["heads"] * HEAD_DIM * 2  # queries in, outputs out
        rows += 2 * case["batch"] * kv_row if case["append"] else 0
        return {"bytes": sum(ctx) * kv_row + rows, "flops": _attention_flops(case["heads"], sum(ctx))}
    if kind == "prefill":
        lens, starts = _lengths(case), _starts(case)
        return {"bytes": (sum(lens) + sum(starts)) * kv_row + 2 * sum(lens) * case["heads"] * HEAD_DIM * 2,
                "flops": _attention_flops(case["heads"], _chunk_pairs(lens, starts))}
    if kind == "mixed":
        lens, starts, ctx = _lengths(case), _starts(case), _mixed_contexts(case)
        tokens = sum(lens) + len(ctx)
        return {"bytes": (sum(lens) + sum(starts) + sum(ctx) + len(ctx)) * kv_row + 2 * tokens * case["heads"] * HEAD_DIM * 2,
                "flops": _attention_flops(case["heads"], _chunk_pairs(lens, starts) + sum(ctx))}
    if kind == "store":
        return {"bytes": 2 * sum(_lengths(case)) * kv_row * case["layers"], "flops": 0}
    config = qwen3_0_6b()
    ctx = _lengths(case)
    q, kv = config.num_attention_heads * HEAD_DIM, config.num_key_value_heads * HEAD_DIM
    layer = config.hidden_size * (2 * q + 2 * kv + 3 * config.intermediate_size)
    weights = config.num_hidden_layers * layer + config.vocab_size * config.hidden_size
    return {"bytes": 2 * weights + config.num_hidden_layers * sum(ctx) * kv_row + 2 * case["batch"] * config.vocab_size,
            "flops": 2.0 * case["batch"] * weights
                     + config.num_hidden_layers * _attention_flops(config.num_attention_heads, sum(ctx))}


def tolerance(case):
    if case["kind"] == "store" or case.get("exact"):
        return "exact"  # a copy; reference numerics define every bit
    if case["kind"] == "model":
        # bf16 rounding of 28 layers' activations: one implementation's logits measured 0.054 away from
        # the 64-bit model's, so two of them can be 0.076 apart.
        return {"rel": 0.15, "max": 0.8}
    return {"rel": 1e-2, "max": 0.1}  # measured 2e-3 to 8e-3 against 64 bits (bf16 queries, p and output)


# ------------------------------------------------------------------------- 64-bit reference
def exact(case, seed):
    return {"decode": _exact_decode, "prefill": _exact_prefill, "mixed": _exact_mixed, "store": _exact_store,
            "model": _exact_model}[case["kind"]](case, seed)


def _bf16(x):
    return x.to(torch.bfloat16).double()


def _attend(q, k, v, visible=None):
    """q [H, n, D], k / v [H_kv, t, D] in float64: softmax attention with the scores at the two bf16
    rounding points that the entry points state, everything else in 64 bits.  Returns [n, H, D]."""
    group = q.shape[0] // k.shape[0]
    outs = []
    for h in range(q.shape[0]):
        s = _bf16(_bf16(q[h] @ k[h // group].t()) * SCALE)
        if visible is not None:
            s = s.masked_fill(~visible, float("-inf"))
        outs.append(torch.softmax(s, dim=-1) @ v[h // group])
    return torch.stack(outs, dim=1)


def _norm_rope(x, weight, cos, sin):
    """[B, heads, D] in float64: RMSNorm over the head, then the rotation."""
    y = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * weight
    half = HEAD_DIM // 2
    return y * cos.unsqueeze(1) + torch.cat((-y[..., half:], y[..., :half]), dim=-1) * sin.unsqueeze(1)


def _history(pool, table_row, n):
    """[H_kv, n, D] float64: the first n tokens behind a block table row."""
    return pool[table_row[:_blocks(n)]].flatten(0, 1)[:n].double().transpose(0, 1)


def _exact_decode(case, seed):
    s = _prepare_decode(case, seed)
    batch, heads, kv = case["batch"], case["heads"], case["kv_heads"]
    kp, vp = s["key_pool"], s["value_pool"]
    if case["append"]:
        cos, sin = s["cos"].double(), s["sin"].double()
        q = _norm_rope(s["q"].double().view(batch, heads, HEAD_DIM), s["q_weight"].double(), cos, sin)
        new_k = _norm_rope(s["k"].double().view(batch, kv, HEAD_DIM), s["k_weight"].double(), cos, sin)
        new_v = s["v"].double().view(batch, kv, HEAD_DIM)
    else:
        q = s["query"].double()
    out = torch.empty((batch, heads * HEAD_DIM), dtype=torch.float64, device="cuda")
    for b, n in enumerate(s["ctx"].tolist()):
        k, v = _history(kp, s["tables"][b], n), _history(vp, s["tables"][b], n)
        if case["append"]:
            k[:, -1], v[:, -1] = new_k[b], new_v[b]
        out[b] = _attend(q[b].unsqueeze(1), k, v).reshape(-1)
    if not case["append"]:
        return out
    kp, vp = kp.double(), vp.double()
    kp.view(-1, kv, HEAD_DIM)[s["slots"]] = new_k
    vp.view(-1, kv, HEAD_DIM)[s["slots"]] = new_v
    return out, kp, vp


def _chunk_row(q, k, v, hist_k, hist_v):
    """One chunk row: q [H, n, D], k / v [H_kv, n, D] behind their history."""
    n, start = q.shape[1], hist_k.shape[1]
    visible = torch.ones((n, start + n), dtype=torch.bool, device="cuda").tril(start)
    return _attend(q, torch.cat((hist_k, k), dim=1), torch.cat((hist_v, v), dim=1), visible)


def _exact_prefill(case, seed):
    s = _prepare_prefill(case, seed)
    rows, heads, width = case["rows"], case["heads"], s["q"].shape[2]
    out = torch.zeros((rows, width, heads * HEAD_DIM), dtype=torch.float64, device="cuda")
    for b, (n, start) in enumerate(zip(s["lens"].tolist(), s["starts"].tolist())):
        hk, hv = _history(s["key_pool"], s["hist"][b], start), _history(s["value_pool"], s["hist"][b], start)
        real = slice(width - n, width)
        out[b, real] = _chunk_row(s["q"][b, :, real].double(), s["k"][b, :, real].double(),
                                  s["v"][b, :, real].double(), hk, hv).reshape(n, -1)
    return out


def _exact_mixed(case, seed):
    s = _prepare_mixed(case, seed)
    kv, c = case["kv_heads"], s["chunk_tokens"]
    q, k, v = (s[x].double().transpose(0, 1) for x in ("q", "k", "v"))
    out = torch.empty((q.shape[1], case["heads"] * HEAD_DIM), dtype=torch.float64, device="cuda")
    for b, (n, start, at) in enumerate(zip(s["lens"].tolist(), s["starts"].tolist(), s["first"].tolist())):
        hk, hv = _history(s["key_pool"], s["hist"][b], start), _history(s["value_pool"], s["hist"][b], start)
        part = slice(at, at + n)
        out[part] = _chunk_row(q[:, part], k[:, part], v[:, part], hk, hv).reshape(n, -1)
    for b, n in enumerate(s["ctx"].tolist()):
        t = c + b
        hk, hv = _history(s["key_pool"], s["tables"][b], n - 1), _history(s["value_pool"], s["tables"][b], n - 1)
        out[t] = _attend(q[:, t:t + 1], torch.cat((hk, k[:, t:t + 1]), dim=1),
                         torch.cat((hv, v[:, t:t + 1]), dim=1)).reshape(-1)
    kp, vp = s["key_pool"].double(), s["value_pool"].double()
    kp.view(-1, kv, HEAD_DIM)[s["slots"]] = s["k"][c:].double()
    vp.view(-1, kv, HEAD_DIM)[s["slots"]] = s["v"][c:].double()
    return out, kp, vp


def _exact_store(case, seed):
    return None  # a copy: nothing is computed


def _exact_model(case, seed):
    s = _prepare_model(case, seed)
    config, model, meta = s["model"].config, s["model"].model, s["meta"]
    batch, heads, kv = case["batch"], config.num_attention_heads, config.num_key_value_heads

    def weight(linear):
        return linear.weight.detach().double().t()

    def norm(x, module):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * module.weight.detach().double()

    inv = 1.0 / THETA ** (torch.arange(0, HEAD_DIM, 2, dtype=torch.float64, device="cuda") / HEAD_DIM)
    angles = s["positions"].double() * inv
    angles = torch.cat((angles, angles), dim=-1)
    cos, sin = angles.cos(), angles.sin()
    hidden = model.embed_tokens.weight.detach()[s["ids"][:, 0]].double()
    keys, values = [], []
    for layer, (kp, vp) in zip(model.layers, meta.kv_pools):
        att, mlp = layer.self_attn, layer.mlp
        x = norm(hidden, layer.input_layernorm)
        q = _norm_rope((x @ weight(att.q_proj)).view(batch, heads, HEAD_DIM), att.q_norm.weight.detach().double(), cos, sin)
        k = _norm_rope((x @ weight(att.k_proj)).view(batch, kv, HEAD_DIM), att.k_norm.weight.detach().double(), cos, sin)
        v = (x @ weight(att.v_proj)).view(batch, kv, HEAD_DIM)
        out = torch.empty((batch, heads * HEAD_DIM), dtype=torch.float64, device="cuda")
        for b, n in enumerate(meta.context_lens.tolist()):
            hk, hv = _history(kp, meta.block_tables[b], n), _history(vp, meta.block_tables[b], n)
            hk[:, -1], hv[:, -1] = k[b], v[b]
            scores = torch.einsum("hd,htd->ht", q[b], hk.repeat_interleave(heads // kv, 0)) * SCALE
            out[b] = torch.einsum("ht,htd->hd", scores.softmax(-1), hv.repeat_interleave(heads // kv, 0)).reshape(-1)
        hidden = hidden + out @ weight(att.o_proj)
        x = norm(hidden, layer.post_attention_layernorm)
        gate, up = x @ weight(mlp.gate_proj), x @ weight(mlp.up_proj)
        hidden = hidden + (gate * torch.sigmoid(gate) * up) @ weight(mlp.down_proj)
        kp, vp = kp.double(), vp.double()
        kp.view(-1, kv, HEAD_DIM)[meta.slot_mapping] = k
        vp.view(-1, kv, HEAD_DIM)[meta.slot_mapping] = v
        keys.append(kp)
        values.append(vp)
    logits = norm(hidden, model.norm) @ weight(s["model"].lm_head)
    return logits.unsqueeze(1), keys, values
