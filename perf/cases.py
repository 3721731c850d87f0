"""Performance cases of the MLA serving path: what a program that serves a model with this
package has it do, through the package's public entry points.

Kinds (``case["kind"]``):
  step     GPU metadata + one batched decode step of a model (``build_metadata``,
           ``HipModel.step``), eager or replayed from a HIP graph
  forward  GPU metadata + one continuous-batching forward (``mla_model_forward``): decode rows
           beside prompt chunks
  prefill  one prompt through a session of the engine (``HipExecution.prefill``)
  score    every position's logits of whole sequences (``HipEngine.forward``)
  attend   decode attention over the paged cache (``decode_attention``)
  chunk    chunked-prefill attention over the paged cache (``prefill_attention``)
  ingest   GPU metadata + paged append, for a host that runs its own model code
           (``build_metadata``, ``append_latent``)

Lengths follow from the case's numbers alone; the seed draws the contents (weights, cache,
queries, tokens, page permutation).  Cached latents are kv_norm-ed, so N(0, 1).
"""
import ctypes
import math
import random

import numpy as np
import torch

import cpp_inference_train_engine_amd as mla
from cpp_inference_train_engine_amd.workloads import MLA36M

PAGE = 64


# ------------------------------------------------------------------------------- cases ----
def listed():
    return [
        # One user's chat turn: the smallest decode step, launches and latency.
        dict(name="step_1", kind="step", sessions=1, min_len=1040, max_len=1040, graph=False),
        # The benchmark's headline step: 64 ragged sessions, captured in a HIP graph.
        dict(name="step_64", kind="step", sessions=64, min_len=128, max_len=4096, graph=True),
        # A full server: 200 sessions decoding at once, eager launches.
        dict(name="step_200", kind="step", sessions=200, min_len=100, max_len=4200, graph=False),
        # A serving step: 61 running sessions and three prompt chunks beside them.
        dict(name="forward_mixed", kind="forward", decodes=61, chunks=3, chunk=319, min_len=64,
             max_len=2048),
        # Time to first token of a 1024-token prompt.
        dict(name="prefill_1024", kind="prefill", tokens=1024),
        # Scoring (perplexity): every position's logits of four sequences.
        dict(name="score_4x250", kind="score", batch=4, tokens=250),
        # One layer's decode attention of a busy server: log-normal lengths, a long tail.
        dict(name="attend_120", kind="attend", sessions=120, median=2048, max_len=16384, heads=8,
             kv=128, rope=16, page=PAGE, dtype="f16", placed=True),
        # One layer's attention of eight 512-token prompt chunks on cached contexts.
        dict(name="chunk_8x512", kind="chunk", sessions=8, chunk=512, max_ctx=2048, heads=8,
             kv=128, rope=16, page=PAGE, dtype="f16"),
        # The DeepSeek-like latent shape, long contexts: the largest calls.
        dict(name="attend_wide", kind="attend", sessions=256, median=19000, max_len=32768,
             heads=128, kv=512, rope=64, page=PAGE, dtype="bf16", placed=False),
        # Other architectures through the kernel-level entry points: decode ...
        dict(name="attend_other", kind="attend", sessions=32, median=1500, max_len=4096, heads=32,
             kv=256, rope=32, page=32, dtype="bf16", placed=False),
        # ... and prompt chunks.
        dict(name="chunk_other", kind="chunk", sessions=4, chunk=129, max_ctx=1000, heads=16,
             kv=64, rope=16, page=PAGE, dtype="f16"),
        # Metadata and append of a large batch: 500 sessions, 16 of them with a chunk.
        dict(name="ingest_500", kind="ingest", decodes=484, chunks=16, chunk=256, max_len=8192),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "step", "forward", "prefill", "score", "attend", "attend", "chunk",
                       "wide", "attend_other", "chunk_other", "ingest"])
    if kind == "step":
        lo = _log_int(rng, 1, 1500)
        return dict(kind="step", sessions=_log_int(rng, 1, 256), min_len=lo,
                    max_len=_log_int(rng, max(lo, 64), 4400), graph=rng.random() < 0.5)
    if kind == "forward":
        return dict(kind="forward", decodes=_log_int(rng, 1, 200), chunks=rng.randint(1, 6),
                    chunk=_log_int(rng, 5, 500), min_len=16, max_len=_log_int(rng, 64, 3500))
    if kind == "prefill":
        return dict(kind="prefill", tokens=_log_int(rng, 8, 4000))
    if kind == "score":
        return dict(kind="score", batch=rng.randint(1, 6), tokens=_log_int(rng, 8, 400))
    if kind == "attend":
        b = _log_int(rng, 1, 500)
        m = _log_int(rng, 16, 6000)
        return dict(kind="attend", sessions=b, median=m, max_len=_log_int(rng, m, 16384),
                    heads=rng.choice([8, 8, 16]), kv=128, rope=16, page=PAGE,
                    dtype=rng.choice(["f16", "bf16"]), placed=b <= 256 and rng.random() < 0.7)
    if kind == "chunk":
        return dict(kind="chunk", sessions=rng.randint(1, 12), chunk=_log_int(rng, 3, 700),
                    max_ctx=_log_int(rng, 16, 4000), heads=rng.choice([8, 8, 16]), kv=128, rope=16,
                    page=PAGE, dtype=rng.choice(["f16", "bf16"]))
    if kind == "wide":
        b = _log_int(rng, 4, 200)
        m = _log_int(rng, 200, 16000)
        return dict(kind="attend", sessions=b, median=m, max_len=_log_int(rng, m, 24000),
                    heads=rng.choice([32, 64, 128, 128]), kv=512, rope=64, page=PAGE,
                    dtype=rng.choice(["f16", "bf16", "bf16"]), placed=False)
    shape = dict(heads=rng.choice([4, 8, 12, 16, 20, 32]), kv=rng.choice([32, 64, 96, 256, 512]),
                 rope=rng.choice([8, 16, 32, 64]), page=rng.choice([16, 32, 64]),
                 dtype=rng.choice(["f16", "bf16"]))
    if kind == "attend_other":
        m = _log_int(rng, 16, 2000)
        return dict(kind="attend", sessions=_log_int(rng, 1, 64), median=m,
                    max_len=_log_int(rng, m, 4096), placed=False, **shape)
    if kind == "chunk_other":
        return dict(kind="chunk", sessions=rng.randint(1, 6), chunk=_log_int(rng, 3, 200),
                    max_ctx=_log_int(rng, 16, 1000), **shape)
    return dict(kind="ingest", decodes=_log_int(rng, 1, 1000), chunks=rng.randint(0, 16),
                chunk=_log_int(rng, 2, 512), max_len=_log_int(rng, 64, 16384))


# --------------------------------------------------------------------- shapes of a case ----
def _lengths(case):
    """(ctx, q): tokens already cached and tokens appended, per session."""
    rng = random.Random(repr(sorted((k, v) for k, v in case.items() if k != "name")))
    kind = case["kind"]
    if kind == "step":
        n = [rng.randint(case["min_len"], case["max_len"]) for _ in range(case["sessions"])]
        return [x - 1 for x in n], [1] * len(n)
    if kind == "attend":
        n = [min(case["max_len"], max(1, round(case["median"] * math.exp(rng.gauss(0, 0.7)))))
             for _ in range(case["sessions"])]
        return [x - 1 for x in n], [1] * len(n)
    if kind == "chunk":
        return ([rng.randint(0, case["max_ctx"]) for _ in range(case["sessions"])],
                [case["chunk"]] * case["sessions"])
    low = case.get("min_len", 1)
    ctx = [rng.randint(low, case["max_len"]) for _ in range(case["decodes"] + case["chunks"])]
    return ctx, [1] * case["decodes"] + [case["chunk"]] * case["chunks"]


def _pages_of(case, page):
    ctx, q = _lengths(case)
    return [-(-(c + n) // page) for c, n in zip(ctx, q)]


def _work_items(case, page, split, placed):
    ctx, q = _lengths(case)
    if placed:
        return mla.placed_work_slots(np.array(ctx), np.array(q), page, split, mla.xcd_count())
    return sum(-(-n // split) for n in _pages_of(case, page))


def _split(case):
    """Pages per work item, as a caller picks it: the page kernel's constant, or enough items
    to fill the GPU."""
    if case.get("kv", 128) == 128:
        return 4
    total = sum(_pages_of(case, case["page"]))
    return max(1, min(128, total // 512))


# ------------------------------------------------------------------------------- states ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _dtype(name):
    return torch.float16 if name == "f16" else torch.bfloat16


def _randn(gen, shape, dtype):
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        part = flat[i:i + (1 << 28)]
        part.copy_(torch.randn(part.numel(), generator=gen, device="cuda"))
    return out


def _batch(case, gen, page):
    """Device inputs of build_metadata: lengths and page lists at a random page permutation."""
    ctx, q = _lengths(case)
    need = _pages_of(case, page)
    total = sum(need)
    ids = torch.randperm(total, generator=gen, device="cuda").to(torch.int32)
    return dict(ctx=_ints(ctx), q=_ints(q), ids=ids, cu=_ints([0] + np.cumsum(need).tolist()),
                pages=total, max_pages=max(need), rows=sum(q))


def _tensors(cfg):
    """(name, rows, columns) of every parameter, in the order that a model takes them."""
    d, r, kv, h = cfg["d_model"], cfg["q_lora_rank"], cfg["kv_lora_rank"], cfg["n_heads"]
    nope, rope, dv, ff = (cfg["head_dim_nope"], cfg["head_dim_rope"], cfg["head_dim_value"],
                          cfg["d_ff"])
    out = [("embed", cfg["vocab_size"], d), ("final_norm", 1, d)]
    for l in range(cfg["n_layers"]):
        out += [(f"{l}.{n}", a, b) for n, a, b in (
            ("attn_norm", 1, d), ("w_dq", d, r), ("q_norm", 1, r), ("w_uq", r, h * (nope + rope)),
            ("w_dkv", d, kv + rope), ("kv_norm", 1, kv), ("w_uk", kv, h * nope),
            ("w_uv", kv, h * dv), ("w_o", h * dv, d), ("ffn_norm", 1, d), ("w_gate", d, ff),
            ("w_up", d, ff), ("w_down", ff, d))]
    return out


def _params(cfg, seed):
    """A checkpoint's parameters (fp16 values, as exported), fp32 on the GPU."""
    gen, parts = _gen(seed), []
    for name, a, b in _tensors(cfg):
        if name.endswith("norm"):
            p = 1 + 0.1 * torch.randn(a * b, generator=gen, device="cuda")
        else:
            scale = 0.02 / math.sqrt(2 * cfg["n_layers"]) if name[-3:] in ("w_o", "own") else 0.02
            p = scale * torch.randn(a * b, generator=gen, device="cuda")
        parts.append(p.half().float())
    return torch.cat(parts)


def _cache(cfg, gen, pages):
    rec = PAGE * (cfg["kv_lora_rank"] + cfg["head_dim_rope"])
    return _randn(gen, (cfg["n_layers"], pages, rec), torch.float16)


def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    if kind in ("prefill", "score"):
        cfg = MLA36M
        tokens = case["tokens"] * case.get("batch", 1)
        ids = torch.randint(0, cfg["vocab_size"], (tokens,), generator=gen, device="cuda")
        engine = mla.HipEngine(mla.ModelConfig.from_dict(cfg), _params(cfg, seed).cpu().numpy(),
                               max_sessions=8, max_rows=1024, num_pages=128)
        return dict(case=case, engine=engine, session=engine.session() if kind == "prefill" else
                    None, ids=ids.cpu().numpy().astype(np.uint16))
    if kind in ("step", "forward"):
        return _prepare_model(case, gen, seed)
    if kind == "ingest":
        cfg = MLA36M
        s = _batch(case, gen, PAGE)
        cache = mla.PagedLatentCache(1, s["pages"], PAGE, 128, 16)
        return dict(s, case=case, cache=cache, work=_work_items(case, PAGE, 4, False),
                    ckv=torch.randn((s["rows"], 128), generator=gen, device="cuda"),
                    krope=torch.randn((s["rows"], 16), generator=gen, device="cuda"))
    dt = _dtype(case["dtype"])
    page, kv, rope, heads = case["page"], case["kv"], case["rope"], case["heads"]
    s = _batch(case, gen, page)
    split, placed = _split(case), case.get("placed", False)
    work = _work_items(case, page, split, placed)
    s.update(case=case, cache=_randn(gen, (s["pages"], page * (kv + rope)), dt),
             ql=_randn(gen, (s["rows"], heads, kv), dt), qr=_randn(gen, (s["rows"], heads, rope), dt),
             out=torch.zeros((s["rows"], heads, kv), device="cuda"),
             lse=torch.zeros((s["rows"], heads), device="cuda"))
    s["meta"] = mla.build_metadata(s["ctx"], s["q"], s["cu"], s["ids"], page, s["max_pages"],
                                   s["pages"], split_pages=split, max_work=work,
                                   max_rows=s["rows"], placement=placed)
    s["meta"].read_info()
    if kind == "attend":
        s["ws"] = mla.decode_workspace(work, case["sessions"], heads, kv)
    return s


def _prepare_model(case, gen, seed):
    cfg = MLA36M
    s = _batch(case, gen, PAGE)
    ctx, q = _lengths(case)
    sessions = len(q)
    placed = sessions <= mla.PLACE_MAX_SESSIONS
    work = _work_items(case, PAGE, 4, placed)
    cache = _cache(cfg, gen, s["pages"])
    pos = [c + i for c, n in zip(ctx, q) for i in range(n)]
    s.update(case=case, work=work, placed=placed, cache=cache, sessions=sessions,
             pools=[cache[l] for l in range(cfg["n_layers"])], positions=_ints(pos),
             model=mla.HipModel(mla.ModelConfig.from_dict(cfg), _params(cfg, seed).cpu().numpy(),
                                max_batch=s["rows"]),
             tokens=torch.randint(0, cfg["vocab_size"], (s["rows"],), generator=gen,
                                  device="cuda").to(torch.int32),
             ws=mla.decode_workspace(work, sessions, cfg["n_heads"], cfg["kv_lora_rank"]),
             logits=torch.empty((sessions, cfg["vocab_size"]), device="cuda"),
             next=torch.empty(sessions, dtype=torch.int32, device="cuda"))
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _step(s)
    return s


# --------------------------------------------------------------------------------- runs ----
def _metadata(s):
    return mla.build_metadata(s["ctx"], s["q"], s["cu"], s["ids"], PAGE, s["max_pages"],
                              s["pages"], split_pages=4, max_work=s["work"], max_rows=s["rows"],
                              placement=s.get("placed", False))


def _step(s):
    rb = _metadata(s)
    s["model"].step(rb, s["tokens"], s["positions"], s["pools"], s["ws"], logits=s["logits"],
                    next_tokens=s["next"])


def _forward(s):
    rb, p = _metadata(s), mla.ptr
    pools = (ctypes.c_void_p * len(s["pools"]))(*[x.data_ptr() for x in s["pools"]])
    mla.check(mla.lib().mla_model_forward(
        s["model"]._h, mla.stream_handle(), s["rows"], p(s["tokens"]), p(s["positions"]),
        s["sessions"], s["case"]["chunk"], p(rb.cu_seqlens_q), p(rb.cu_seqlens_k),
        p(rb.page_table), rb.max_pages, rb.num_pool_pages, p(rb.slot_mapping), p(rb.num_splits),
        p(rb.cu_splits), p(rb.work_desc), p(rb.work_pages), p(rb.info), rb.max_work, pools,
        p(s["ws"]), s["ws"].numel(), p(s["logits"]), p(s["next"]),
        mla.DECODE_FUSED_MERGE if rb.placed else 0))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        s["graph"].replay() if "graph" in s else _step(s)
        return {"logits": s["logits"], "pages": s["cache"]}
    if kind == "forward":
        _forward(s)
        return {"logits": s["logits"], "pages": s["cache"]}
    if kind == "prefill":
        return {"logits": s["session"].prefill(s["ids"])}
    if kind == "score":
        return {"logits": s["engine"].forward(s["ids"], case["batch"], case["tokens"])}
    if kind == "ingest":
        rb = _metadata(s)
        mla.append_latent(s["cache"], 0, s["ckv"], s["krope"], rb.slot_mapping)
        return {"cu_q": rb.cu_seqlens_q, "cu_k": rb.cu_seqlens_k, "table": rb.page_table,
                "slots": rb.slot_mapping, "splits": rb.num_splits, "cu_splits": rb.cu_splits,
                "desc": rb.work_desc, "item_pages": rb.work_pages, "info": rb.info,
                "pages": s["cache"].pages.view(torch.int16)}
    code = mla.DTYPE_F16 if case["dtype"] == "f16" else mla.DTYPE_BF16
    args = dict(kv_rank=case["kv"], rope_dim=case["rope"], dtype=code, out=s["out"], lse=s["lse"])
    if kind == "attend":
        mla.decode_attention(s["meta"], s["cache"], s["ql"], s["qr"], _scale(case),
                             workspace=s["ws"], **args)
    else:
        mla.prefill_attention(s["meta"], s["cache"], s["ql"], s["qr"], _scale(case),
                              max_q_len=case["chunk"], **args)
    return {"out": s["out"], "lse": s["lse"]}


def _scale(case):
    return 1 / math.sqrt(case["kv"] / 2 + case["rope"])


# --------------------------------------------------------------------------------- work ----
def work(case):
    """Bytes: every input read once and every output written once; flops: the products."""
    kind = case["kind"]
    cfg = MLA36M
    if kind == "ingest":
        ctx, q = _lengths(case)
        pages, rows = sum(_pages_of(case, PAGE)), sum(q)
        items = _work_items(case, PAGE, 4, False)
        table = len(q) * max(_pages_of(case, PAGE))
        return {"bytes": rows * 144 * 6 + 4 * (pages + table + rows + 18 * items + 8 * len(q)),
                "flops": 0}
    if kind in ("prefill", "score"):
        ctx, q = [0] * case.get("batch", 1), [case["tokens"]] * case.get("batch", 1)
    else:
        ctx, q = _lengths(case)
    seen = sum(n * c + n * (n + 1) // 2 for c, n in zip(ctx, q))  # (row, key) pairs
    keys, rows = sum(ctx) + sum(q), sum(q)
    if kind in ("attend", "chunk"):
        kv, rope, heads = case["kv"], case["rope"], case["heads"]
        return {"bytes": keys * (kv + rope) * 2 + rows * heads * (6 * kv + 2 * rope + 4),
                "flops": 2 * seen * heads * (2 * kv + rope)}
    layers, kv, rope, heads = (cfg["n_layers"], cfg["kv_lora_rank"], cfg["head_dim_rope"],
                               cfg["n_heads"])
    weights = sum(a * b for _, a, b in _tensors(cfg))
    embed = cfg["vocab_size"] * cfg["d_model"]
    logits = rows if kind == "score" else len(q)
    return {"bytes": 2 * weights + layers * (keys + rows) * (kv + rope) * 2
            + 4 * logits * cfg["vocab_size"],
            "flops": 2 * (weights - embed) * rows + 2 * embed * logits
            + 2 * layers * seen * heads * (2 * kv + rope)}


def tolerance(case):
    kind = case["kind"]
    if kind == "ingest":
        return "exact"  # whole numbers, and rounding to 16 bits
    if kind in ("step", "forward", "prefill", "score"):
        return {"rel": 3.5e-3, "max": 3e-2}  # ten layers of fp16 operands: 8.5e-4 off 64 bits
    # fp16 probabilities are 1e-4 off 64 bits, bf16 ones (high and low parts) 1e-6
    return {"rel": 4e-4, "max": 1e-2} if case["dtype"] == "f16" else {"rel": 1e-5, "max": 2e-4}


# -------------------------------------------------------------------------------- exact ----
def _tiled(page, kv, rope):
    return page % 16 == 0 and kv % 32 == 0 and rope % 8 == 0


def _unpack(records, page, kv, rope):
    """Page records [n, page * (kv + rope)] as token rows in 64 bits: (latent, key)."""
    n = records.shape[0]
    lat, key = records[:, :page * kv], records[:, page * kv:]
    if _tiled(page, kv, rope):
        lat = lat.reshape(n, page // 16, kv // 32, 4, 16, 8).permute(0, 1, 4, 2, 3, 5)
        key = key.reshape(n, page // 16, rope // 8, 16, 8).permute(0, 1, 3, 2, 4)
    return lat.reshape(n * page, kv).double(), key.reshape(n * page, rope).double()


def _pack(lat, key, page):
    """The records that _unpack takes apart, in 64 bits."""
    n, kv, rope = lat.shape[0] // page, lat.shape[1], key.shape[1]
    if _tiled(page, kv, rope):
        lat = lat.reshape(n, page // 16, 16, kv // 32, 4, 8).permute(0, 1, 3, 4, 2, 5)
        key = key.reshape(n, page // 16, 16, rope // 8, 8).permute(0, 1, 3, 2, 4)
    return torch.cat([lat.reshape(n, page * kv), key.reshape(n, page * rope)], 1)


def _softmax_rows(scores, ctx):
    """(probabilities, log-sum-exp) of scores [q, heads, keys]; query i sees keys <= ctx + i."""
    q, _, keys = scores.shape
    late = torch.arange(keys, device="cuda")[None] > ctx + torch.arange(q, device="cuda")[:, None]
    scores = scores.masked_fill(late[:, None], -math.inf)
    lse = torch.logsumexp(scores, -1)
    return torch.exp(scores - lse[..., None]), lse


def _exact_attention(case, seed):
    s = prepare(case, seed)
    page, kv, rope, heads = case["page"], case["kv"], case["rope"], case["heads"]
    ctx, q = _lengths(case)
    cu, at = s["cu"].tolist(), 0
    out = torch.zeros((s["rows"], heads, kv), dtype=torch.float64, device="cuda")
    lse = torch.zeros((s["rows"], heads), dtype=torch.float64, device="cuda")
    for b, (c, n) in enumerate(zip(ctx, q)):
        lat, key = _unpack(s["cache"][s["ids"][cu[b]:cu[b + 1]].long()], page, kv, rope)
        lat, key = lat[:c + n], key[:c + n]
        ql, qr = s["ql"][at:at + n].double(), s["qr"][at:at + n].double()
        scores = (ql.view(n * heads, kv) @ lat.T + qr.view(n * heads, rope) @ key.T) * _scale(case)
        p, lse[at:at + n] = _softmax_rows(scores.view(n, heads, -1), c)
        out[at:at + n] = (p.view(n * heads, -1) @ lat).view(n, heads, kv)
        at += n
    return {"out": out, "lse": lse}


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope_rows(x, positions, theta):
    """RoPE of adjacent pairs of the last axis; x [rows, ..., rope]."""
    rope = x.shape[-1]
    freq = theta ** (-torch.arange(0, rope, 2, dtype=torch.float64, device="cuda") / rope)
    angle = positions.double()[:, None] * freq
    cos, sin = angle.cos(), angle.sin()
    if x.dim() == 3:
        cos, sin = cos[:, None], sin[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)


def _exact_rows(cfg, w, tokens, positions, ctx, q, cached, keep):
    """The final hidden rows of a forward; cached(l, b) gives session b's cached (latent, key)
    rows of layer l, and keep(l, latent, key) takes the rows that the forward appends."""
    h, nope, rope, dv = (cfg["n_heads"], cfg["head_dim_nope"], cfg["head_dim_rope"],
                         cfg["head_dim_value"])
    kv, eps, theta = cfg["kv_lora_rank"], cfg["norm_epsilon"], cfg["rope_theta"]
    rows = len(tokens)
    x = w["embed"][tokens.long()]
    for l in range(cfg["n_layers"]):
        p = lambda name: w[f"{l}.{name}"]  # noqa: E731
        xn = _rms(x, p("attn_norm"), eps)
        query = (_rms(xn @ p("w_dq"), p("q_norm"), eps) @ p("w_uq")).view(rows, h, nope + rope)
        qr = _rope_rows(query[..., nope:], positions, theta)
        down = xn @ p("w_dkv")
        lat = _rms(down[:, :kv], p("kv_norm"), eps)
        key = _rope_rows(down[:, kv:], positions, theta)
        keep(l, lat, key)
        ql = torch.einsum("rhn,khn->rhk", query[..., :nope], p("w_uk").view(kv, h, nope))
        mixed, at = torch.empty((rows, h, kv), dtype=torch.float64, device="cuda"), 0
        for b, (c, n) in enumerate(zip(ctx, q)):
            old = cached(l, b)
            cl = torch.cat([old[0], lat[at:at + n]])
            ck = torch.cat([old[1], key[at:at + n]])
            scores = ql[at:at + n].reshape(n * h, kv) @ cl.T + qr[at:at + n].reshape(n * h, rope) @ ck.T
            prob, _ = _softmax_rows(scores.view(n, h, -1) / math.sqrt(nope + rope), c)
            mixed[at:at + n] = (prob.view(n * h, -1) @ cl).view(n, h, kv)
            at += n
        value = torch.einsum("rhk,khd->rhd", mixed, p("w_uv").view(kv, h, dv))
        x = x + value.reshape(rows, h * dv) @ p("w_o")
        xn = _rms(x, p("ffn_norm"), eps)
        gate = xn @ p("w_gate")
        x = x + (gate * torch.sigmoid(gate) * (xn @ p("w_up"))) @ p("w_down")
    return _rms(x, w["final_norm"], eps)


def _weights(cfg, seed):
    flat, at, out = _params(cfg, seed).double(), 0, {}
    for name, a, b in _tensors(cfg):
        out[name] = flat[at:at + a * b].view(a, b) if a > 1 else flat[at:at + b]
        at += a * b
    return out


def _exact_model(case, seed):
    cfg, kind = MLA36M, case["kind"]
    w = _weights(cfg, seed)
    kv, rope = cfg["kv_lora_rank"], cfg["head_dim_rope"]
    empty = (torch.zeros((0, kv), dtype=torch.float64, device="cuda"),
             torch.zeros((0, rope), dtype=torch.float64, device="cuda"))
    if kind in ("prefill", "score"):
        n, batch = case["tokens"], case.get("batch", 1)
        ids = torch.randint(0, cfg["vocab_size"], (n * batch,), generator=_gen(seed),
                            device="cuda")
        x = _exact_rows(cfg, w, ids, torch.arange(n, device="cuda").repeat(batch), [0] * batch,
                        [n] * batch, lambda l, b: empty, lambda *a: None)
        return {"logits": (x if kind == "score" else x[-1]) @ w["embed"].T}
    ctx, q = _lengths(case)
    gen = _gen(seed)  # the draws of prepare, in its order
    s = _batch(case, gen, PAGE)
    cache = _cache(cfg, gen, s["pages"])
    tokens = torch.randint(0, cfg["vocab_size"], (s["rows"],), generator=gen, device="cuda")
    cu, ids = s["cu"].tolist(), s["ids"].long()
    pos = torch.tensor([c + i for c, n in zip(ctx, q) for i in range(n)], device="cuda")
    page_of = torch.cat([ids[cu[b] + (c + torch.arange(n, device="cuda")) // PAGE]
                         for b, (c, n) in enumerate(zip(ctx, q))])
    pages = torch.empty(cache.shape, dtype=torch.float64, device="cuda")

    def cached(l, b):
        lat, key = _unpack(cache[l][ids[cu[b]:cu[b + 1]]], PAGE, kv, rope)
        return lat[:ctx[b]], key[:ctx[b]]

    def keep(l, lat, key):
        rows, keys = _unpack(cache[l], PAGE, kv, rope)
        rows[page_of * PAGE + pos % PAGE] = lat
        keys[page_of * PAGE + pos % PAGE] = key
        pages[l] = _pack(rows, keys, PAGE)

    x = _exact_rows(cfg, w, tokens, pos, ctx, q, cached, keep)
    last = torch.tensor(np.cumsum(q) - 1, device="cuda")
    return {"logits": x[last] @ w["embed"].T, "pages": pages}


def exact(case, seed):
    if case["kind"] == "ingest":
        return None
    if case["kind"] in ("attend", "chunk"):
        return _exact_attention(case, seed)
    return _exact_model(case, seed)
