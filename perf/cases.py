"""The work a serving program hands to this package, as cases that can be timed.

Three kinds of calls, all through public entry points:

* ``decode``   one decode step of one attention layer: ``Attention`` stores the
               new K/V rows and attends over the block-paged cache;
* ``prefill``  the prompt rows of one attention layer, packed, or behind cached
               positions that are read through the block tables;
* ``model``    one step of the whole model (``DecodeStepRunner``, Qwen3-0.6B
               shape) up to the logits, from which a program samples: a decode step
               built from host lists, a decode step replayed from a HIP graph, or
               the prefill of new prompts.

Head counts, page size and lengths are those of ``workloads.py`` and the tests.
Lengths, pages and values follow from the case's sizes and the seed; the lengths
from the sizes alone, so that ``work`` is the same for every seed.
"""
import math

import numpy as np
import torch

from nanovllm_jax_amd import Attention, create_decode_context, create_prefill_context
from nanovllm_jax_amd.engine.decode_step import DecodeModelConfig, DecodeStepRunner
from nanovllm_jax_amd.layers.paged_attention import DecodeWorkspace, choose_split

HEAD_DIM = 128
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}


def _decode(name, batch, lo, hi, heads, kv_heads, dtype="bf16", spread="uniform", page=256,
            k_f32=True, own_workspace=True, host_split=False, q_gain=1.0):
    c = {"kind": "decode", "batch": batch, "lo": lo, "hi": hi, "spread": spread, "heads": heads,
         "kv_heads": kv_heads, "dtype": dtype, "page": page, "k_f32": k_f32,
         "own_workspace": own_workspace, "host_split": host_split, "q_gain": q_gain}
    return {"name": name, **c} if name else c


def _prefill(name, batch, lo, hi, heads, kv_heads, dtype="bf16", cached_lo=0, cached_hi=0,
             page=256, k_f32=False):
    c = {"kind": "prefill", "batch": batch, "lo": lo, "hi": hi, "cached_lo": cached_lo,
         "cached_hi": cached_hi, "spread": "uniform", "heads": heads, "kv_heads": kv_heads,
         "dtype": dtype, "page": page, "k_f32": k_f32}
    return {"name": name, **c} if name else c


def _model(name, step, batch, lo, hi, cached_lo=0, cached_hi=0):
    c = {"kind": "model", "step": step, "batch": batch, "lo": lo, "hi": hi,
         "cached_lo": cached_lo, "cached_hi": cached_hi, "spread": "uniform"}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one user at a prompt: a single sequence, the layer as it is constructed
        _decode("decode_one", 1, 700, 700, 16, 8, own_workspace=False),
        # a handful of short conversations (the Qwen3-0.6B shape of workload C1)
        _decode("decode_few", 8, 128, 2048, 16, 8),
        # a full batch at equal length, the Qwen3-8B shape (C2)
        _decode("decode_4k", 64, 4096, 4096, 32, 8),
        # few very long contexts, the Qwen3-32B shape with a sharp softmax (C4)
        _decode("decode_32k", 16, 32768, 32768, 64, 8, q_gain=4.0),
        # a server's mix of lengths over three orders of magnitude (C3)
        _decode("decode_mixed", 256, 16, 32768, 32, 8, spread="log"),
        # the first turn of one conversation; K comes in float32, as rotary embedding leaves it
        _prefill("prefill_one", 1, 700, 700, 16, 8, k_f32=True),
        # many short questions packed into one call
        _prefill("prefill_short", 128, 16, 300, 32, 8),
        # long prompts, the Qwen3-8B shape
        _prefill("prefill_4k", 8, 4096, 4096, 32, 8),
        # follow-up turns and chunked prompts behind a cached prefix, float16
        _prefill("prefill_cached", 16, 30, 600, 32, 8, dtype="f16", cached_lo=100, cached_hi=5000),
        # a few users' next tokens: metadata from host lists, an eager step
        _model("model_decode_few", "decode", 4, 100, 900),
        # a server's full batch replayed from a graph (C5)
        _model("model_decode_batch", "decode_graph", 128, 1024, 1024),
        # new prompts through the whole model
        _model("model_prefill", "prefill", 8, 100, 1000),
    ]


# The most a drawn case may ask for: what the largest listed case of its kind does.
_MAX_POSITIONS = 900_000            # decode: cached positions times kv_heads / 8
_MAX_PREFILL_FLOPS = 1.05e12        # prefill: 8 prompts of 4096 tokens, 32 heads
_MAX_MODEL_POSITIONS = 128 * 1024   # model decode
_MAX_MODEL_TOKENS = 4400            # model prefill


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "cached", "model"])
        dtype = rng.choice(["bf16", "bf16", "f16"])
        page = rng.choice([256, 256, 256, 64, 128])
        heads, kv_heads = rng.choice([(16, 8), (32, 8), (32, 8), (64, 8), (32, 32)])
        spread = rng.choice(["uniform", "log"])
        if kind == "decode":
            batch = _log_int(rng, 1, 256)
            hi = _log_int(rng, 100, 32768)
            lo = max(1, int(hi * rng.choice([1.0, rng.uniform(0.03, 0.95)])))
            case = _decode(None, batch, lo, hi, heads, kv_heads, dtype, spread, page,
                           k_f32=rng.random() < 0.5, own_workspace=rng.random() < 0.7,
                           host_split=rng.random() < 0.3)
            if int(_lengths(case).sum()) * kv_heads <= 8 * _MAX_POSITIONS:
                return case
        elif kind in ("prefill", "cached"):
            batch = _log_int(rng, 1, 200)
            hi = _log_int(rng, 16, 8192)
            lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
            cached = kind == "cached"
            cached_hi = _log_int(rng, 64, 8192) if cached else 0
            cached_lo = int(cached_hi * rng.uniform(0.0, 1.0))
            case = _prefill(None, batch, lo, hi, heads, kv_heads, dtype, cached_lo, cached_hi,
                            page, k_f32=rng.random() < 0.5)
            case["spread"] = spread
            keys = int((_lengths(case) + _cached(case)).sum())
            if work(case)["flops"] <= _MAX_PREFILL_FLOPS and keys * kv_heads <= 8 * _MAX_POSITIONS:
                return case
        else:
            step = rng.choice(["decode", "decode_graph", "prefill"])
            batch = _log_int(rng, 1, 128 if step != "prefill" else 16)
            hi = _log_int(rng, 20, 3000)
            lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
            cached_hi = rng.choice([0, rng.randint(64, 900)]) if step == "prefill" else 0
            case = _model(None, step, batch, lo, hi, cached_hi // 3, cached_hi)
            limit = _MAX_MODEL_TOKENS if step == "prefill" else _MAX_MODEL_POSITIONS
            if int(_lengths(case).sum()) <= limit:
                return case


# ---------------------------------------------------------------------------
# sizes
# ---------------------------------------------------------------------------
def _spread_ints(case, lo, hi, salt):
    rng = np.random.Generator(np.random.PCG64([case["batch"], case["lo"], case["hi"], salt]))
    if case["spread"] == "log" and lo > 0:
        x = np.exp(rng.uniform(math.log(lo), math.log(hi), size=case["batch"]))
    else:
        x = rng.uniform(lo, hi, size=case["batch"])
    return np.clip(np.rint(x), lo, hi).astype(np.int64)


def _lengths(case):
    """decode: positions of every sequence, the token being decoded included;
    prefill: new tokens of every prompt."""
    return _spread_ints(case, case["lo"], case["hi"], 1)


def _cached(case):
    """Positions of every prompt that are in the cache already."""
    if case["cached_hi"] == 0:
        return np.zeros(case["batch"], np.int64)
    return _spread_ints(case, case["cached_lo"], case["cached_hi"], 2)


def _pages(rng, lens, page):
    """Every sequence's pages, out of a pool a tenth larger than needed, in random order."""
    need = -(-lens // page)
    pool = int(need.sum() * 1.1) + 1
    ids = rng.permutation(pool)
    ends = np.cumsum(need)
    return pool, [ids[e - n:e].tolist() for n, e in zip(need, ends)]


def _table(rows):
    out = np.full((len(rows), max(len(r) for r in rows)), -1, np.int32)
    for i, r in enumerate(rows):
        out[i, :len(r)] = r
    return out


def _slots(rows, first, last, page):
    """Cache slot of positions [first[i], last[i]) of every sequence."""
    out = []
    for row, a, b in zip(rows, first, last):
        pos = np.arange(a, b)
        out.append(np.asarray(row, np.int64)[pos // page] * page + pos % page)
    return np.concatenate(out).astype(np.int32)


def _cumulative(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


# ---------------------------------------------------------------------------
# what is in hand before a call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rng = np.random.Generator(np.random.PCG64(seed))
    if case["kind"] == "decode":
        return _prepare_decode(case, rng, g, dev)
    if case["kind"] == "prefill":
        return _prepare_prefill(case, rng, g, dev)
    return _prepare_model(case, seed, rng, dev)


def _normal(g, dev, dtype, *shape):
    return torch.randn(shape, generator=g, device=dev, dtype=dtype)


def _layer(case, pool, dt, g, dev):
    attn = Attention(case["heads"], HEAD_DIM, HEAD_DIM ** -0.5, case["kv_heads"], case["page"])
    shape = (pool, case["page"], case["kv_heads"], HEAD_DIM)
    attn.set_kv_cache(_normal(g, dev, dt, *shape), _normal(g, dev, dt, *shape))
    return attn


def _prepare_decode(case, rng, g, dev):
    lens, page, dt = _lengths(case), case["page"], DTYPES[case["dtype"]]
    pool, rows = _pages(rng, lens, page)
    batch, heads, kv_heads = case["batch"], case["heads"], case["kv_heads"]
    attn = _layer(case, pool, dt, g, dev)
    table = _table(rows)
    if case["own_workspace"]:
        attn.workspace = DecodeWorkspace.for_shape(batch, heads, HEAD_DIM, table.shape[1], page,
                                                   kv_heads, dev)
    split = choose_split(lens.tolist(), kv_heads, heads) if case["host_split"] else 0
    context = create_decode_context(torch.from_numpy(lens.astype(np.int32)).to(dev),
                                    torch.from_numpy(_slots(rows, lens - 1, lens, page)).to(dev),
                                    torch.from_numpy(table).to(dev), split)
    q = (_normal(g, dev, torch.float32, batch, heads, HEAD_DIM) * case["q_gain"]).to(dt)
    k = _normal(g, dev, torch.float32 if case["k_f32"] else dt, batch, kv_heads, HEAD_DIM)
    v = _normal(g, dev, dt, batch, kv_heads, HEAD_DIM)
    return {"kind": "layer", "attn": attn, "q": q, "k": k, "v": v, "context": context}


def _prepare_prefill(case, rng, g, dev):
    new, cached, page, dt = _lengths(case), _cached(case), case["page"], DTYPES[case["dtype"]]
    total = new + cached
    pool, rows = _pages(rng, total, page)
    attn = _layer(case, pool, dt, g, dev)
    behind_prefix = case["cached_hi"] > 0
    context = create_prefill_context(
        torch.from_numpy(_cumulative(new)).to(dev), torch.from_numpy(_cumulative(total)).to(dev),
        int(new.max()), int(total.max()), torch.from_numpy(_slots(rows, cached, total, page)).to(dev),
        block_tables=torch.from_numpy(_table(rows)).to(dev) if behind_prefix else None)
    tokens = int(new.sum())
    q = _normal(g, dev, dt, tokens, case["heads"], HEAD_DIM)
    k = _normal(g, dev, torch.float32 if case["k_f32"] else dt, tokens, case["kv_heads"], HEAD_DIM)
    v = _normal(g, dev, dt, tokens, case["kv_heads"], HEAD_DIM)
    return {"kind": "layer", "attn": attn, "q": q, "k": k, "v": v, "context": context}


def _prepare_model(case, seed, rng, dev):
    lens, cached = _lengths(case), _cached(case)
    total = lens + cached
    page = DecodeModelConfig.block_size
    pool, rows = _pages(rng, total, page)
    cfg = DecodeModelConfig(num_kvcache_blocks=pool)
    runner = DecodeStepRunner(cfg, dev, seed=seed)
    state = {"kind": case["step"], "runner": runner, "rows": rows, "lens": lens.tolist()}
    if case["step"] == "prefill":
        # a token list starts with the cached tokens, as the filler expects
        state["tokens"] = [rng.integers(0, cfg.vocab_size, n).tolist() for n in total]
        state["cached"] = cached.tolist() if case["cached_hi"] > 0 else None
        return state
    state["last"] = rng.integers(0, cfg.vocab_size, case["batch"]).tolist()
    if case["step"] == "decode_graph":
        inputs = runner.make_inputs(state["last"], state["lens"], rows)
        side = torch.cuda.Stream(dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            runner.forward(*inputs)
        torch.cuda.current_stream(dev).wait_stream(side)
        torch.cuda.synchronize(dev)
        state["inputs"], state["graph"] = inputs, torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["logits"] = runner.forward(*inputs)
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "layer":
        attn = state["attn"]
        out = attn(state["q"], state["k"], state["v"], state["context"])
        return {"out": out, "k_cache": attn.k_cache, "v_cache": attn.v_cache}
    runner = state["runner"]
    if kind == "decode_graph":
        state["graph"].replay()
        logits = state["logits"]
    elif kind == "decode":
        logits = runner.forward(*runner.make_inputs(state["last"], state["lens"], state["rows"]))
    else:
        logits = runner.forward(*runner.make_prefill_inputs(state["tokens"], state["rows"],
                                                            state["cached"]))
    return {"logits": logits, "kv_cache": runner.kv_cache}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    lens = _lengths(case)
    if case["kind"] == "model":
        return _model_work(case, lens)
    heads, kv_heads, row = case["heads"], case["kv_heads"], case["kv_heads"] * HEAD_DIM
    if case["kind"] == "decode":
        new, keys_read, pairs = case["batch"], int(lens.sum()) - case["batch"], int(lens.sum())
    else:
        cached = _cached(case)
        new, keys_read = int(lens.sum()), int(cached.sum())
        pairs = int((lens * (lens + 1) // 2 + lens * cached).sum())
    k_bytes = 4 if case["k_f32"] else 2
    return {"bytes": keys_read * row * 4                        # cached keys and values
            + new * row * (k_bytes + 2 + 4)                     # new rows in, and into the cache
            + 2 * new * heads * HEAD_DIM * 2,                   # q and the output
            "flops": 4 * heads * HEAD_DIM * pairs}


def _model_work(case, lens):
    c = DecodeModelConfig()
    q_row, kv_row = c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim
    per_layer = (c.hidden_size * (q_row + 2 * kv_row) + q_row * c.hidden_size
                 + 3 * c.hidden_size * c.intermediate_size)
    head = c.hidden_size * c.vocab_size
    if case["step"] == "prefill":
        cached = _cached(case)
        tokens, keys_read = int(lens.sum()), int(cached.sum())
        pairs = int((lens * (lens + 1) // 2 + lens * cached).sum())
    else:
        tokens, keys_read, pairs = case["batch"], int(lens.sum()) - case["batch"], int(lens.sum())
    return {"bytes": 2 * (c.num_layers * per_layer + head)                  # weights, bf16
            + c.num_layers * 4 * kv_row * (keys_read + tokens)              # KV read, new rows written
            + 2 * case["batch"] * c.vocab_size,                             # logits
            "flops": 2 * tokens * c.num_layers * per_layer + 2 * case["batch"] * head
            + 4 * q_row * c.num_layers * pairs}


def tolerance(case):
    """The cache rows are copied or rounded once and have to be the same to well below
    these; attention outputs and logits are 16-bit results of 16-bit operands with
    float32 sums, logits after 28 layers of roundings."""
    if case["kind"] == "model":
        return {"rel": 2e-2}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
