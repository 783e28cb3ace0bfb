"""The work that a program asks of this framework, as cases to be timed and compared.

Every case is one call (or one captured decode step) of the token-by-token
decode path: paged attention over the cache in its layouts and head shapes, the
fused append of the current token, shared prefixes, RoPE + append, and a whole
multi-layer engine step.  K/V, queries and block tables are drawn from the
seed; blocks are handed out in random order, as a cache that has been serving
for a while holds them.
"""

import math
import random

import torch

import flashdec_amd as fd
from flashdec_amd.cascade import build_cascade_groups, paged_decode_attention_cascade_into
from flashdec_amd.rope import rope_cos_sin_table

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_MAX_KV_BYTES = 800 << 20  # of a drawn case: under the largest listed one's


# ------------------------------------------------------------------ cases --
def _attention(name=None, **over):
    case = {"kind": "attention", "batch": 8, "ctx": 2048, "lengths": "full", "q_heads": 16, "kv_heads": 2,
            "head_dim": 128, "block": 32, "dtype": "bf16", "layout": "token_major", "ragged": False, "index": "int32",
            "table_slack": 1}
    case.update(over)
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # One short chat turn: the smallest call, all latency and launches.
        _attention("one-request", batch=1, ctx=128, block=16),
        # The headline: eight requests of equal length.
        _attention("batch8-ctx2048"),
        # A large serving batch of short requests, with block tables as wide as
        # the server's longest allowed request and 64-bit indices.
        _attention("many-short", batch=193, ctx=511, lengths="half", q_heads=32, kv_heads=8, block=16, index="int64",
                   table_slack=4),
        # A large serving batch of long requests, somewhere in their second half: the largest.
        _attention("long-half-to-full", batch=64, ctx=4096, lengths="half", q_heads=32, kv_heads=8),
        # Requests of widely different lengths, said to be so by the caller.
        _attention("widely-mixed", batch=32, ctx=32768, lengths="log", ragged=True),
        # Small heads, seven query heads for each KV head (a 0.5B model's 14/2), fp16.
        _attention("head64-group7", batch=16, ctx=8192, q_heads=14, kv_heads=2, head_dim=64, dtype="fp16"),
        # One KV head for all 71 query heads.
        _attention("multi-query-71", batch=16, ctx=8192, q_heads=71, kv_heads=1, head_dim=64),
        # The dim-major cache layout.
        _attention("dim-major", batch=16, ctx=8192, block=16, layout="dim_major"),
        # A serving engine's hook: the current token's K/V are written by the
        # attention call, into a cache kept as [block, K/V, token, head, dim].
        {"name": "append-token", "kind": "append", "batch": 48, "ctx": 2048, "lengths": "half", "q_heads": 16,
         "kv_heads": 2, "block": 16, "dtype": "bf16"},
        # Many requests on one long system prompt.
        {"name": "shared-prefix", "kind": "prefix", "batch": 64, "prefix": 16384, "tail": 512, "q_heads": 16,
         "kv_heads": 2, "block": 32, "dtype": "bf16"},
        # A prompt's tokens rotated and written to the cache in one call.
        {"name": "rope-append-prompt", "kind": "rope", "rows": 4096, "q_heads": 32, "kv_heads": 8, "head_dim": 128,
         "rotary_dim": 128, "block": 32, "dtype": "bf16", "table": True},
        # A decode step of a 36-layer model: RoPE, append and attention of every
        # layer, replayed from the engine's captured step.
        {"name": "engine-step", "kind": "engine", "layers": 36, "batch": 8, "ctx": 2047, "q_heads": 16, "kv_heads": 2,
         "block": 32, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("attention", "append", "prefix", "rope", "engine"), (12, 2, 2, 2, 1))[0]
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    if kind == "rope":
        head_dim = rng.choice((64, 128, 128))
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "q_heads": rng.choice((14, 16, 32)),
                "kv_heads": rng.choice((2, 8)), "head_dim": head_dim,
                "rotary_dim": rng.choice((head_dim, head_dim, head_dim // 2)), "block": rng.choice((16, 32)),
                "dtype": dtype, "table": rng.choice((True, False))}
    q_heads, kv_heads = rng.choice(((16, 2), (16, 2), (32, 8), (32, 8), (32, 4), (16, 1)))
    if kind == "engine":
        layers = rng.choice((2, 8, 36))
        batch = _log_int(rng, 1, 32)
        most = min(8192, (_MAX_KV_BYTES // 2) // (layers * batch * kv_heads * 512))
        ctx = _log_int(rng, min(100, most), most)
        ctx -= ctx % 32 == 0  # the new token goes into a block that its request has (see run)
        return {"kind": kind, "layers": layers, "batch": batch, "ctx": ctx, "q_heads": q_heads, "kv_heads": kv_heads,
                "block": 32, "dtype": dtype}
    if kind == "prefix":
        return {"kind": kind, "batch": _log_int(rng, 8, 64), "prefix": 32 * _log_int(rng, 64, 512),
                "tail": _log_int(rng, 32, 1024), "q_heads": q_heads, "kv_heads": min(kv_heads, 4),
                "block": rng.choice((16, 32)), "dtype": dtype}
    batch = _log_int(rng, 1, 256)
    if kind == "append":
        most = min(16384, _MAX_KV_BYTES // (batch * kv_heads * 512))
        return {"kind": kind, "batch": batch, "ctx": _log_int(rng, min(100, most), most),
                "lengths": rng.choice(("full", "half", "log")), "q_heads": q_heads, "kv_heads": kv_heads, "block": 16,
                "dtype": dtype}
    head_dim = rng.choice((128, 128, 128, 64))
    if head_dim == 64:
        q_heads, kv_heads = rng.choice(((14, 2), (16, 2), (71, 1), (32, 8)))
    else:
        q_heads, kv_heads = rng.choice(((16, 2), (16, 2), (32, 8), (32, 8), (32, 4), (16, 16), (64, 2), (12, 4)))
    layout = rng.choice(("token_major",) * 5 + ("dim_major",))
    if q_heads // kv_heads > 16:
        layout = "token_major"
    lengths = rng.choice(("full", "half", "half", "log"))
    most = min(32768, _MAX_KV_BYTES // (batch * kv_heads * head_dim * 4))
    if q_heads // kv_heads > 16:
        most = min(most, (_MAX_KV_BYTES // 4) // (batch * kv_heads * head_dim * 4))
    ctx = _log_int(rng, min(64, most), most)
    return _attention(batch=batch, ctx=ctx, lengths=lengths, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
                      block=rng.choice((8, 16, 32, 32)), dtype=dtype, layout=layout,
                      ragged=lengths == "log" and rng.random() < 0.5, index=rng.choice(("int32", "int64")),
                      table_slack=rng.choice((1, 1, 2)))


# ----------------------------------------------------------------- inputs --
def _lengths(case, seed):
    """Tokens attended by each request.  Half: between half of ctx and ctx; log: spread evenly over
    the logarithm from ctx / 256 to ctx.  The lengths' sum is close to the same for every seed."""
    n, ctx = case["batch"], case["ctx"]
    if case.get("lengths", "full") == "full":
        return [ctx] * n
    rng = random.Random(seed)
    at = [(i + rng.random()) / n for i in range(n)]  # one from each n-th of the range
    rng.shuffle(at)
    low = max(1, ctx // 2 if case["lengths"] == "half" else ctx // 256)
    if case["lengths"] == "half":
        return [min(ctx, int(low + u * (ctx + 1 - low))) for u in at]
    return [max(1, min(ctx, int(round(low * (ctx / low) ** u)))) for u in at]


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(shape, dtype, gen, std=1.0):
    return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=gen)


def _tables(lens, block, slack, gen, shared=0):
    """(block table with -1 past each row's blocks, number of blocks); the first `shared` blocks of
    every row are the same ones."""
    need = [-(-n // block) for n in lens]
    width = max(need) * slack
    total = shared + sum(n - shared for n in need)
    order = torch.randperm(total, device="cuda", generator=gen).cpu()
    table = torch.full((len(lens), width), -1, dtype=torch.int64)
    at = shared
    for b, n in enumerate(need):
        table[b, :shared] = order[:shared]
        table[b, shared:n] = order[at : at + n - shared]
        at += n - shared
    return table, total


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    if kind == "rope":
        return _prepare_rope(case, gen)
    if kind == "engine":
        return _prepare_engine(case, seed, gen)
    dtype, hq, hkv, block = _DTYPES[case["dtype"]], case["q_heads"], case["kv_heads"], case["block"]
    head_dim = case.get("head_dim", 128)
    shared = 0
    if kind == "prefix":
        rng = random.Random(seed)
        n = case["batch"]
        at = [(i + rng.random()) / n for i in range(n)]
        rng.shuffle(at)
        lens = [case["prefix"] + max(1, int(math.ceil(u * case["tail"]))) for u in at]
        shared = case["prefix"] // block
    else:
        lens = _lengths(case, seed)
    index = torch.int64 if case.get("index") == "int64" else torch.int32
    table, blocks = _tables(lens, block, case.get("table_slack", 1), gen, shared)
    state = {"case": case, "tables": table.to("cuda", index), "lens": torch.tensor(lens, device="cuda", dtype=index),
             # queries of twice unit size: scores spread as a trained head's do, a few tokens weighing most
             "q": _normal((len(lens), hq, head_dim), dtype, gen, 2.0)}
    if kind == "append":
        blocks = len(lens) * table.shape[1]  # a pool that also holds every request at full length
        kv = _normal((blocks, 2, block, hkv, head_dim), dtype, gen)
        state["k"], state["v"] = kv[:, 0].permute(0, 2, 1, 3), kv[:, 1].permute(0, 2, 1, 3)
        state["new_k"] = _normal((len(lens), hkv, head_dim), dtype, gen)
        state["new_v"] = _normal((len(lens), hkv, head_dim), dtype, gen)
        last = torch.tensor(lens) - 1
        state["slots"] = (table.gather(1, (last // block)[:, None])[:, 0] * block + last % block).cuda()
        state["out"] = torch.empty_like(state["q"])
    else:
        shape = (blocks, hkv, block, head_dim)
        if case.get("layout") == "dim_major":
            shape = (blocks, hkv, head_dim, block)
        state["k"], state["v"] = _normal(shape, dtype, gen), _normal(shape, dtype, gen)
    if kind == "prefix":
        state["groups"] = build_cascade_groups(state["tables"], state["lens"], block, hq, hkv)
        state["out"] = torch.empty_like(state["q"])
    return state


def _prepare_rope(case, gen):
    dtype, block, d = _DTYPES[case["dtype"]], case["block"], case["head_dim"]
    rows, hq, hkv = case["rows"], case["q_heads"], case["kv_heads"]
    blocks = -(-rows // block)
    pos = torch.arange(rows, device="cuda")
    order = torch.randperm(blocks, device="cuda", generator=gen)
    state = {"case": case, "q": _normal((rows, hq, d), dtype, gen), "k": _normal((rows, hkv, d), dtype, gen),
             "v": _normal((rows, hkv, d), dtype, gen), "positions": pos, "block_ids": order[pos // block],
             "block_offsets": pos % block,
             "k_cache": torch.zeros((blocks, hkv, block, d), device="cuda", dtype=dtype),
             "v_cache": torch.zeros((blocks, hkv, block, d), device="cuda", dtype=dtype)}
    state["table"] = rope_cos_sin_table(max(rows, 4096), case["rotary_dim"]) if case["table"] else None
    return state


def _prepare_engine(case, seed, gen):
    layers, batch, hq, hkv, block = (case[k] for k in ("layers", "batch", "q_heads", "kv_heads", "block"))
    width = -(-(case["ctx"] + 1) // block)
    cache = fd.PagedKVCache(layers, hkv, 128, block, max_blocks=batch * width, dtype=_DTYPES[case["dtype"]],
                            device="cuda")
    cache.k_cache.normal_(generator=gen)
    cache.v_cache.normal_(generator=gen)
    cache.enable_graph_metadata(batch, width)
    engine = fd.DecodeEngine(cache)
    ids = list(range(batch))
    for rid in ids:
        engine.add_request(rid)
    engine.admit()
    cache.seed_context(ids, case["ctx"])
    graph = engine.capture_step_graph(batch, hq)
    graph.q.normal_(0.0, 2.0, generator=gen)
    graph.k.normal_(generator=gen)
    graph.v.normal_(generator=gen)
    return {"case": case, "engine": engine, "cache": cache, "graph": graph, "ids": ids}


# -------------------------------------------------------------------- run --
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attention":
        return fd.decode(state["q"], state["k"], state["v"], state["tables"], state["lens"],
                         kv_layout=case["layout"], ragged=case["ragged"])
    if kind == "append":
        fd.paged_decode_attention_into(state["q"], state["k"], state["v"], state["tables"], state["lens"],
                                       state["out"], append_k=state["new_k"], append_v=state["new_v"],
                                       slot_mapping=state["slots"])
        return {"out": state["out"], "k": state["k"], "v": state["v"]}
    if kind == "prefix":
        return paged_decode_attention_cascade_into(state["q"], state["k"], state["v"], state["tables"],
                                                   state["lens"], state["out"], state["groups"])
    if kind == "rope":
        q = fd.fused_rope_kv_append(state["q"], state["k"], state["v"], state["k_cache"], state["v_cache"],
                                    state["block_ids"], state["block_offsets"], state["positions"],
                                    rotary_dim=case["rotary_dim"], cos_sin_table=state["table"])
        return {"q": q, "k": state["k_cache"], "v": state["v_cache"]}
    # the token is rolled back after the step, so that the next pass decodes the same position again
    engine = state["engine"]
    step = engine.begin_step(state["ids"])
    out = engine.step_graph(step, state["graph"])
    engine.abort_step(step)
    return {"out": out, "k": state["cache"].k_cache, "v": state["cache"].v_cache}


# ------------------------------------------------------------------- work --
def work(case):
    kind = case["kind"]
    hq, hkv, d = case["q_heads"], case["kv_heads"], case.get("head_dim", 128)
    if kind == "rope":
        return {"bytes": case["rows"] * 2 * d * 2 * (hq + 2 * hkv), "flops": case["rows"] * (hq + hkv) * 3 * d}
    if kind == "prefix":
        n, tail = case["batch"], case["tail"] / 2
        return {"bytes": (case["prefix"] + n * tail) * hkv * d * 4 + n * hq * d * 4,
                "flops": n * (case["prefix"] + tail) * hq * d * 4}
    if kind == "engine":
        tokens = case["batch"] * (case["ctx"] + 1) * case["layers"]
        rows = case["batch"] * case["layers"]
    else:
        tokens, rows = sum(_lengths(case, 0)), case["batch"]
    appended = 4 * rows * hkv * d * 2 if kind in ("append", "engine") else 0
    return {"bytes": tokens * hkv * d * 4 + rows * hq * d * 4 + appended, "flops": tokens * hq * d * 4}


def tolerance(case):
    # Results leave in the 16-bit type, and the probabilities enter the second
    # product in it.  Measured in bf16: another order of the sums (other split
    # counts, the shared prefix apart or per row) moves results by up to 3.0e-3
    # and single values by 1.7e-2; rotations whose angles are evaluated in 32
    # or in 64 bits differ by 1.2e-4, single values by one step of the type
    # (7.8e-3).  The figures are four times that; fp16's steps are an eighth.
    scale = 1.0 if case["dtype"] == "bf16" else 0.125
    if case["kind"] == "rope":
        return {"rel": 5e-4 * scale, "max": 3.2e-2 * scale}
    return {"rel": 1.2e-2 * scale, "max": 7e-2 * scale}


# ------------------------------------------------------------------ exact --
def _attend(q, k_rows, v_rows):
    """q [Hq, D] on k/v rows [Hkv, L, D], in 64 bits."""
    hkv, group = k_rows.shape[0], q.shape[0] // k_rows.shape[0]
    out = []
    for h in range(hkv):
        qh = q[h * group : (h + 1) * group].double()
        kh, vh = k_rows[h].double().contiguous(), v_rows[h].double().contiguous()
        p = torch.softmax((kh @ qh.t().contiguous()).t() / math.sqrt(q.shape[-1]), dim=-1)
        out.append(p.contiguous() @ vh)
    return torch.cat(out)


def _rows(cache, table_row, length, block, dim_major=False):
    ids = table_row[: -(-length // block)].long()
    pages = cache[ids]  # [n, Hkv, block, D] or [n, Hkv, D, block]
    if dim_major:
        pages = pages.transpose(2, 3)
    return pages.transpose(0, 1).reshape(cache.shape[1], -1, pages.shape[-1])[:, :length]


def _rotate(x, positions, rotary_dim, base=10_000.0, table=True):
    """Split-half RoPE.  The API defines the angles by 32-bit frequencies and products; the frequencies
    are torch's where a table made by it is read, else the nearest 32-bit values."""
    steps = torch.arange(0, rotary_dim, 2, device=x.device, dtype=torch.float32)
    exponent = -steps / rotary_dim
    freq = torch.pow(base, exponent) if table else torch.pow(base, exponent.double()).float()
    angles = positions.float()[:, None] * freq[None, :]
    cos, sin = torch.cos(angles.double())[:, None], torch.sin(angles.double())[:, None]
    half = rotary_dim // 2
    lo, hi = x[..., :half].double(), x[..., half:rotary_dim].double()
    return torch.cat((lo * cos - hi * sin, hi * cos + lo * sin, x[..., rotary_dim:].double()), dim=-1)


def exact(case, seed):
    kind = case["kind"]
    state = prepare(case, seed)
    if kind == "rope":
        rotary, table = case["rotary_dim"], case["table"]
        k, v = state["k_cache"].double(), state["v_cache"].double()
        k[state["block_ids"], :, state["block_offsets"]] = _rotate(state["k"], state["positions"], rotary, table=table)
        v[state["block_ids"], :, state["block_offsets"]] = state["v"].double()
        return {"q": _rotate(state["q"], state["positions"], rotary, table=table), "k": k, "v": v}
    if kind == "engine":
        return _exact_engine(case, state)
    block, dim_major = case["block"], case.get("layout") == "dim_major"
    lens = state["lens"].tolist()
    if kind == "append":
        ids, off = state["slots"] // block, state["slots"] % block
        state["k"][ids, :, off], state["v"][ids, :, off] = state["new_k"], state["new_v"]
    out = torch.stack([_attend(state["q"][b], _rows(state["k"], state["tables"][b], n, block, dim_major),
                               _rows(state["v"], state["tables"][b], n, block, dim_major))
                       for b, n in enumerate(lens)])
    return {"out": out, "k": state["k"].double(), "v": state["v"].double()} if kind == "append" else out


def _exact_engine(case, state):
    cache, graph, engine = state["cache"], state["graph"], state["engine"]
    ctx, block = case["ctx"], case["block"]
    step = engine.begin_step(state["ids"])  # the new token's slots, as the step reserves them
    tables, ids, off, pos = (t.clone().long() for t in (step.block_tables, step.physical_block_ids,
                                                        step.block_offsets, step.positions))
    engine.abort_step(step)
    k, v = cache.k_cache, cache.v_cache
    out, rotated = [], []
    for layer in range(case["layers"]):
        # the rotated query and key are rounded to the cache's type before the attention, as the API's are
        q = _rotate(graph.q[layer], pos, 128).to(k.dtype)
        new_k = _rotate(graph.k[layer], pos, 128)
        rotated.append(new_k)
        k[layer][ids, :, off], v[layer][ids, :, off] = new_k.to(k.dtype), graph.v[layer]
        out.append(torch.stack([_attend(q[b], _rows(k[layer], tables[b], ctx + 1, block),
                                        _rows(v[layer], tables[b], ctx + 1, block))
                                for b in range(case["batch"])]))
    return {"out": torch.stack(out), "k": k.double(), "v": v.double()}
