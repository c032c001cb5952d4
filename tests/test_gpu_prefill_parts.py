"""Prefill behind a cached prefix where keys are cut into parts, through the layer and at the C entry
point: what the context says of the longest sequence, memory that is short, other streams, graphs
and threads, many sequences, values that are not finite."""
import functools
import threading
from types import SimpleNamespace

import numpy as np
import pytest

from helpers import torch_to_bits

pytestmark = pytest.mark.gpu


@functools.lru_cache(maxsize=6)
def _problem(new, cached, Hq, Hkv, bs, dtype, width, seed):
    import torch
    from oracle.paged_attention_oracle import paged_prefill_attention_ref, store_kv_to_cache_ref
    rng = np.random.Generator(np.random.PCG64(seed))
    total = [a + b for a, b in zip(new, cached)]
    pages = [-(-n // bs) for n in total]
    table = np.full((len(new), max(max(pages), width)), -1, np.int32)
    ids, at = rng.permutation(sum(pages) + 2), 0
    for i, n in enumerate(pages):
        table[i, :n] = ids[at:at + n]
        at += n
    slots = [np.zeros(0, np.int32)]
    for i, (a, b) in enumerate(zip(cached, total)):
        p = np.arange(a, b)
        slots.append((table[i, p // bs] * bs + p % bs).astype(np.int32))
    slots = np.concatenate(slots)
    cu_q, cu_k = (np.concatenate([[0], np.cumsum(n)]).astype(np.int32) for n in (new, total))
    draw = lambda *shape: torch.from_numpy(rng.standard_normal(shape, np.float32)).to(
        torch.bfloat16 if dtype == "bf16" else torch.float16)
    q, k, v = (draw(sum(new), h, 128) for h in (Hq, Hkv, Hkv))
    kc, vc = (draw(sum(pages) + 2, bs, Hkv, 128) for _ in range(2))
    flat = (-1, Hkv, 128)
    bits = [torch_to_bits(x) for x in (k, v, kc, vc)]
    wk, wv = store_kv_to_cache_ref(bits[0], bits[1], bits[2].reshape(flat), bits[3].reshape(flat),
                                   slots, negative_slots="skip")
    want = paged_prefill_attention_ref(torch_to_bits(q), wk.reshape(kc.shape), wv.reshape(vc.shape),
                                       table, cu_q, cu_k, 128 ** -0.5, return_f32=True, dtype=dtype)
    return (kc, vc), (q, k, v), (cu_q, cu_k, slots, table), want


def _call(new, cached, Hq=32, Hkv=8, bs=64, dtype="bf16", width=0, seed=1):
    """A layer, its q, k and v, the fields of a context, and the result of the oracle."""
    import torch
    from nanovllm_jax_amd import Attention
    caches, qkv, ints, want = _problem(tuple(new), tuple(cached), Hq, Hkv, bs, dtype, width, seed)
    dev = "cuda:0"
    attn = Attention(Hq, 128, 128 ** -0.5, Hkv, bs)
    attn.set_kv_cache(*(x.to(dev) for x in caches))
    names = ("cu_seqlens_q", "cu_seqlens_k", "slot_mapping", "block_tables")
    fields = dict(zip(names, (torch.from_numpy(x).to(dev) for x in ints)), is_prefill=True)
    return attn, [x.to(dev) for x in qkv], fields, want


def _check(out, want):
    """Probabilities and results are rounded to the 16-bit type, sums are not: a rounding each,
    and as much again for the oracle's."""
    import torch
    got = out.float().cpu().numpy()
    tol = 2.0 ** -6 if out.dtype == torch.bfloat16 else 2.0 ** -9
    assert np.abs(got - want).max() <= tol * np.abs(want).max()


def _parts(fields, Hq, Hkv, bs, max_keys):
    """Bytes of partials, 0 where keys are not cut."""
    from nanovllm_jax_amd import _lib
    table, cu = fields["block_tables"], fields["cu_seqlens_q"]
    return _lib.load().nvj_paged_prefill_split_workspace_bytes(
        int(cu[-1]), len(cu) - 1, Hq, Hkv, bs, table.shape[1], max_keys)


@pytest.fixture
def native_only(monkeypatch):
    """The general path is no way out."""
    from nanovllm_jax_amd.layers import attention

    def refused(*_):
        raise AssertionError("declined by the native call")
    monkeypatch.setattr(attention, "store_kv_to_cache", refused)


@pytest.mark.parametrize("paged", [True, False])
def test_context_without_the_longest_length(paged, native_only):
    """A context object of a caller's own need not have a field that no launch needs."""
    print(f"case context without max_seqlen_k paged={paged}", flush=True)
    attn, qkv, fields, want = _call([9, 33], [1500, 0] if paged else [0, 0])
    if not paged:
        fields.update(block_tables=None, cu_seqlens_k=fields["cu_seqlens_q"])
    _check(attn(*qkv, SimpleNamespace(**fields)), want)


@pytest.mark.parametrize("paged", [True, False])
@pytest.mark.parametrize("longest", [None, 1533.0, "on the host", "on the device", "numpy", -1,
                                     1 << 40, 1 << 70])
def test_longest_length_that_is_no_number_at_hand(longest, paged, native_only):
    """It is a hint: whatever stands there, the call is the ordinary one, and nothing is asked of a
    tensor, which would wait for the GPU (and cannot be, in a capture)."""
    print(f"case max_seqlen_k {longest} paged={paged}", flush=True)
    import torch
    from nanovllm_jax_amd import AttentionContext
    attn, qkv, fields, want = _call([9, 33], [1500, 0] if paged else [0, 0])
    if not paged:
        fields.update(block_tables=None, cu_seqlens_k=fields["cu_seqlens_q"])
    longest = {"on the host": torch.tensor(1533), "on the device": torch.tensor(1533).cuda(),
               "numpy": np.int64(1533)}.get(longest, longest)
    context = AttentionContext(max_seqlen_k=longest, **fields)
    attn(*qkv, AttentionContext(**fields))       # code objects are loaded
    torch.cuda.synchronize()
    torch.cuda.set_sync_debug_mode("error")
    try:
        out = attn(*qkv, context)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    _check(out, want)


@pytest.mark.parametrize("new,cached,Hq,Hkv", [([30], [5000], 32, 8), ([500], [4200], 32, 8)])
def test_partials_that_find_no_memory(new, cached, Hq, Hkv):
    """Without memory for partials a call is what it is where keys are not cut."""
    print(f"case no memory for partials {new} {cached}", flush=True)
    import torch
    from nanovllm_jax_amd import create_prefill_context, paged_prefill_attention
    attn, qkv, f, want = _call(new, cached, Hq, Hkv)
    context = create_prefill_context(f["cu_seqlens_q"], f["cu_seqlens_k"], max(new),
                                     new[0] + cached[0], f["slot_mapping"], f["block_tables"])
    need = _parts(f, Hq, Hkv, 64, context.max_seqlen_k)
    assert need > 4 << 20
    room, held = torch.empty_like(qkv[0]), []    # room for the result, and none for the partials
    torch.cuda.synchronize()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(need, dtype=torch.uint8, device="cuda:0"))
        del room
        out = attn(*qkv, context)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    del held
    whole = paged_prefill_attention(qkv[0], attn.k_cache, attn.v_cache, f["block_tables"],
                                    f["cu_seqlens_q"], f["cu_seqlens_k"], attn.scale)
    assert torch.equal(out, whole)
    _check(out, want)
    _check(attn(*qkv, context), want)            # and with memory again


def test_longest_length_not_known_means_whole():
    """Without a bound on the lengths keys stay whole, however wide the tables: the bits are those
    of every other way to this call, alone or in a batch."""
    print("case unknown longest length", flush=True)
    import torch
    from nanovllm_jax_amd import AttentionContext, paged_prefill_attention
    attn, qkv, fields, want = _call([30, 5], [3000, 100])
    assert _parts(fields, 32, 8, 64, 0) > 0
    out = attn(*qkv, AttentionContext(**fields))
    whole = paged_prefill_attention(qkv[0], attn.k_cache, attn.v_cache, fields["block_tables"],
                                    fields["cu_seqlens_q"], fields["cu_seqlens_k"], attn.scale)
    assert torch.equal(out, whole)
    _check(out, want)


LAYERS = [
    ([30], [5000], 32, 8, 64, 200),                            # tables much wider than their rows
    ([17, 1, 40], [2500, 0, 4000], 16, 8, 256, 0),
    ([9], [700], 28, 4, 64, 0),                                # three parts
    ([500], [4200], 32, 8, 64, 0),                             # two column groups a wave
    ([23, 0, 44, 37, 5, 31], [4300, 0, 100, 2000, 64, 4096], 64, 8, 64, 160),
]


def _context(f, new, cached):
    from nanovllm_jax_amd import create_prefill_context
    return create_prefill_context(f["cu_seqlens_q"], f["cu_seqlens_k"], max(new),
                                  max(a + b for a, b in zip(new, cached)), f["slot_mapping"],
                                  f["block_tables"])


@pytest.mark.parametrize("new,cached,Hq,Hkv,bs,width", LAYERS)
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_layer_call_in_parts(new, cached, Hq, Hkv, bs, width, dtype, native_only):
    """The layer's own call: the bound of its context, its partials, both workgroup forms."""
    print(f"case layer in parts {new} {cached} {Hq} / {Hkv} {dtype}", flush=True)
    import torch
    attn, qkv, f, want = _call(new, cached, Hq, Hkv, bs, dtype, width)
    context = _context(f, new, cached)
    assert _parts(f, Hq, Hkv, bs, context.max_seqlen_k) > 0
    out = attn(*qkv, context)
    _check(out, want)
    assert torch.equal(attn(*qkv, context), out)


@pytest.mark.parametrize("new,cached,Hq,Hkv,bs,width", LAYERS[:1] + LAYERS[3:])
def test_layer_call_in_parts_on_other_streams_and_in_graphs(new, cached, Hq, Hkv, bs, width):
    print(f"case parts elsewhere {new} {cached} {Hq} / {Hkv}", flush=True)
    import torch
    attn, qkv, f, want = _call(new, cached, Hq, Hkv, bs, "bf16", width)
    context = _context(f, new, cached)
    out = attn(*qkv, context)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        outs = [attn(*qkv, context) for _ in range(3)]
    torch.cuda.synchronize()
    assert all(torch.equal(x, out) for x in outs)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = attn(*qkv, context)
    for _ in range(3):
        captured.zero_()
        graph.replay()
        own = attn(*qkv, context)                # the program's own work in between
        torch.cuda.synchronize()
        assert torch.equal(captured, out) and torch.equal(own, out)
    _check(out, want)


def test_layer_calls_in_parts_of_several_threads():
    """Threads with a layer and a stream each: partials belong to a call."""
    print("case parts of several threads", flush=True)
    import torch
    calls = []
    for i, (new, cached, Hq, Hkv, bs, width) in enumerate(LAYERS):
        attn, qkv, f, _ = _call(new, cached, Hq, Hkv, bs, "bf16", width, seed=40 + i)
        context = _context(f, new, cached)
        calls.append((attn, qkv, context, attn(*qkv, context)))
    torch.cuda.synchronize()
    wrong = []

    def work(attn, qkv, context, want):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                outs = [attn(*qkv, context) for _ in range(30)]
                torch.cuda.current_stream().synchronize()
            wrong.extend(i for i, x in enumerate(outs) if not torch.equal(x, want))
        except Exception as e:                   # noqa: BLE001 (reported by the main thread)
            wrong.append(e)

    threads = [threading.Thread(target=work, args=c) for c in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def _launch(attn, q, f, max_keys, scale=128 ** -0.5, whole=False):
    """The attention of the layer's cache by the C entry points; the partials' memory has a guard of
    1 MB behind it and holds NaN before the launch."""
    import torch
    from nanovllm_jax_amd import _lib
    lib, out = _lib.load(), torch.full_like(q, 7.0)
    table, cu_q, cu_k = f["block_tables"], f["cu_seqlens_q"], f["cu_seqlens_k"]
    blocks, bs, Hkv, _ = attn.k_cache.shape
    sizes = (q.shape[0], len(cu_q) - 1, q.shape[1], Hkv)
    stream = torch.cuda.current_stream().cuda_stream
    ptrs = [x.data_ptr() for x in (q, attn.k_cache, attn.v_cache, table, cu_q, cu_k, out)]
    end = (float(scale), _lib.NVJ_DTYPE_BF16 if q.dtype == torch.bfloat16 else _lib.NVJ_DTYPE_F16)
    tail = (*sizes, 128, bs, table.shape[1], blocks)
    if whole:
        _lib.check(lib.nvj_paged_prefill_attention_launch(stream, *ptrs, *tail, *end), "whole")
        return out
    need = lib.nvj_paged_prefill_split_workspace_bytes(*sizes, bs, table.shape[1], max_keys)
    assert need > 0
    ws = torch.full((need + (1 << 20),), 0xFF, dtype=torch.uint8, device=q.device)
    _lib.check(lib.nvj_paged_prefill_split_launch(stream, *ptrs, ws.data_ptr(), need, *tail, max_keys,
                                                  *end), "parts")
    assert bool((ws[need:] == 0xFF).all())       # nothing is written behind what was asked for
    return out


@pytest.mark.parametrize("new,cached,Hq,Hkv,bs,width", LAYERS[:2] + LAYERS[3:])
@pytest.mark.parametrize("bound", ["none", "exact", "between", "below"])
def test_bound_on_the_keys_changes_the_parts_only(new, cached, Hq, Hkv, bs, width, bound):
    """0 (what the tables hold), the longest length, one in between, and one below the true lengths:
    other parts and other forms of workgroups, the same result."""
    print(f"case bound {bound} {new} {cached} {Hq} / {Hkv}", flush=True)
    attn, qkv, f, want = _call(new, cached, Hq, Hkv, bs, "bf16", width)
    attn(*qkv, _context(f, new, cached))         # (the rows of the call are in the cache now)
    longest = max(a + b for a, b in zip(new, cached))
    held = f["block_tables"].shape[1] * bs
    max_keys = {"none": 0, "exact": longest, "between": (longest + held) // 2,
                "below": 4128 if longest > 4128 and sum(new) > 100 else 2100}[bound]
    _check(_launch(attn, qkv[0], f, max_keys), want)


@pytest.mark.parametrize("batch,Hq,Hkv,long", [(63, 2, 1, 5), (100, 2, 1, 5), (180, 2, 1, 9)])
def test_parts_of_many_sequences(batch, Hq, Hkv, long):
    """One, two and four sequences to a lane of the lookup, which the merge does again: very uneven
    prefixes (longest tiles first) and alike ones, sequences without rows or without a prefix."""
    print(f"case parts of many sequences {batch}", flush=True)
    rng = np.random.Generator(np.random.PCG64(batch))
    for uneven in (True, False):
        new = rng.integers(0, 3, batch)
        new[[0, batch // 2, batch - 1]] = [0, 20, 1]
        cached = rng.integers(0, 90 if uneven else 700, batch)
        cached[rng.integers(0, batch, long)] = 8000 if uneven else 900
        cached[batch // 3] = 0
        attn, qkv, f, want = _call([int(x) for x in new], [int(x) for x in cached], Hq, Hkv, 32,
                                   "bf16", 8192 // 32)
        attn(*qkv, _context(f, new.tolist(), cached.tolist()))
        _check(_launch(attn, qkv[0], f, 8192), want)


def test_parts_with_values_that_are_not_finite():
    """A NaN or an infinity in a live key or value reaches the rows and heads that it reaches where
    keys stay whole, and no others; without a scale every key weighs the same."""
    print("case parts, not finite", flush=True)
    import torch
    new, cached, Hq, Hkv, bs = [60, 5], [3000, 700], 8, 4, 64
    for seed, (cache, value) in enumerate([("k_cache", float("nan")), ("k_cache", float("inf")),
                                           ("v_cache", float("nan")), ("v_cache", float("-inf"))]):
        attn, qkv, f, _ = _call(new, cached, Hq, Hkv, bs, seed=70 + seed)
        attn(*qkv, _context(f, new, cached))
        for position in (5, 1500, 3030):         # the first part, one between, among the new rows
            page = int(f["block_tables"][0, position // bs])
            row = getattr(attn, cache)[page, position % bs, position % Hkv]
            row[:: 1 if value != value else 128] = value
        parts, whole = _launch(attn, qkv[0], f, 0), _launch(attn, qkv[0], f, 0, whole=True)
        assert whole.isnan().any() or whole.isinf().any()
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(parts), kind(whole))
        live = whole.isfinite()
        # two roundings of the probabilities and of the result
        assert (parts - whole)[live].abs().max() <= 2.0 ** -6 * whole[live].abs().max()
    attn, qkv, f, _ = _call(new, cached, Hq, Hkv, bs, seed=80)
    attn(*qkv, _context(f, new, cached))
    flat = _launch(attn, qkv[0], f, 0, scale=0.0)
    same = _launch(attn, qkv[0], f, 0, scale=0.0, whole=True)
    assert (flat - same).abs().max() <= 2.0 ** -6 * same.abs().max()
