"""The native step, in both its forms (up to 16 rows, and more), against the same step
through library GEMMs and separate launches, at the edges of its row counts and row lengths,
within what two orders of bf16 roundings give (the products have tests of their own against
float64, test_gpu_linear.py); what it declines or refuses; and the QK norm / RoPE launch with
rows in place, strided and at odd offsets."""
import numpy as np
import pytest
import torch

from helpers import bits_to_torch, torch_to_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,hidden,inter,heads", [(1, 256, 256, 2), (4, 512, 768, 4),
                                                     (5, 1024, 3072, 16), (16, 1024, 512, 8),
                                                     (16, 2048, 2560, 24), (17, 512, 512, 4),
                                                     (33, 1024, 768, 6), (128, 256, 256, 2),
                                                     (129, 320, 448, 6), (300, 1024, 3072, 16),
                                                     (1100, 1024, 512, 8)])
@pytest.mark.parametrize("kind", ["decode", "packed", "paged"])
def test_native_step_equals_the_long_way(rows, hidden, inter, heads, kind, monkeypatch):
    print(f"case native step rows={rows} hidden={hidden} {kind}", flush=True)
    from nanovllm_jax_amd.engine import decode_step as ds
    cfg = ds.DecodeModelConfig(num_layers=2, hidden_size=hidden, num_heads=heads, num_kv_heads=2,
                               head_dim=128, intermediate_size=inter, vocab_size=1000,
                               max_position=2048, block_size=64, num_kvcache_blocks=2 * rows + 60)
    runner = ds.DecodeStepRunner(cfg, "cuda:0", seed=rows)
    rng = np.random.Generator(np.random.PCG64(rows))
    pages = rng.permutation(cfg.num_kvcache_blocks).tolist()
    if kind == "decode":
        lens = rng.integers(1, 100, rows).tolist()
    else:                                     # new rows: one long prompt and short ones
        lens = [rows] if rows < 5 else [rows - 3, 2, 1]
    cached = [37] * len(lens) if kind == "paged" else [0] * len(lens)
    tables = []
    for n, c in zip(lens, cached):
        tables.append([pages.pop() for _ in range(-(-(n + c) // cfg.block_size))])
    if kind == "decode":
        inputs = runner.make_inputs(rng.integers(0, 1000, rows).tolist(), lens, tables)
    else:
        toks = [rng.integers(0, 1000, n + c).tolist() for n, c in zip(lens, cached)]
        inputs = runner.make_prefill_inputs(toks, tables, cached if kind == "paged" else None)
    before = runner.kv_cache.clone()
    assert runner._native_forward(*inputs) is not None       # the path under test is taken
    runner.kv_cache.copy_(before)
    got = runner.forward(*inputs).float()
    kv = runner.kv_cache.clone()
    runner.kv_cache.copy_(before)
    monkeypatch.setattr(ds, "_NATIVE_STEP_ROWS", 0)
    want = runner.forward(*inputs).float()
    torch.cuda.synchronize()
    assert (got - want).abs().max().item() <= 0.02 * want.abs().max().item() + 0.02
    err = (kv.float() - runner.kv_cache.float()).abs()
    assert (err <= 0.03 + 0.03 * runner.kv_cache.float().abs()).all()


@pytest.mark.parametrize("offset,pad", [(0, 0), (2, 6), (4, 4)])
def test_qk_rows_in_place_and_unaligned(offset, pad):
    print(f"case qk rows offset={offset} pad={pad}", flush=True)
    from nanovllm_jax_amd import _lib
    from oracle.paged_attention_oracle import qk_norm_rope_store_ref
    T, hq, hkv, d = 7, 3, 2, 128
    rng = np.random.Generator(np.random.PCG64(offset + 1))
    width = (hq + 2 * hkv) * d
    dev = "cuda:0"
    buf = torch.randn(T, offset + width + pad, device=dev).to(torch.bfloat16)
    view = buf[:, offset:offset + width]
    pos = rng.integers(0, 60, T).astype(np.int32)
    slots = np.array([5, -1, 9, 0, 64, 3, 2], np.int32)
    cs = rng.standard_normal((60, d), dtype=np.float32)
    qw, kw = (rng.standard_normal(d, dtype=np.float32) for _ in range(2))
    kc = torch.zeros(16, hkv, d, dtype=torch.bfloat16, device=dev)
    vc = torch.zeros_like(kc)
    all_slots = np.arange(T, dtype=np.int32)               # every row stored: the packed rows
    qkv_bits = torch_to_bits(view.contiguous())
    zero = np.zeros((16, hkv, d), np.uint16)
    want_q, want_k, want_v = qk_norm_rope_store_ref(qkv_bits, pos, cs, qw, kw, 1e-6, zero, zero,
                                                    all_slots, hq, hkv)
    up = lambda a: torch.from_numpy(a).to(dev)
    t = [up(a) for a in (pos, cs, qw, kw, slots)]
    v_rows = torch.zeros(T, hkv * d, dtype=torch.bfloat16, device=dev)
    lib = _lib.load()
    k_part = view.data_ptr() + 2 * hq * d
    # (kv_row_stride is shared by k_out and v_out: V comes out in a second, cache-less call)
    for k_out, v_out, stride in ((None, v_rows.data_ptr(), hkv * d),
                                 (k_part, None, buf.stride(0))):
        _lib.check(lib.nvj_qk_norm_rope_rows_launch(
            torch.cuda.current_stream().cuda_stream, view.data_ptr(), buf.stride(0), t[0].data_ptr(),
            t[1].data_ptr(), 60, t[2].data_ptr(), t[3].data_ptr(), 1e-6, t[4].data_ptr(),
            kc.data_ptr(), vc.data_ptr(),
            view.data_ptr() if k_out else torch.empty(T * hq * d, dtype=torch.bfloat16,
                                                      device=dev).data_ptr(),
            buf.stride(0) if k_out else hq * d, k_out, v_out, stride, T, hq, hkv, d, 16), "rows")
    torch.cuda.synchronize()
    got = torch_to_bits(view.contiguous()).reshape(T, hq + 2 * hkv, d)
    assert np.array_equal(got[:, :hq], want_q.reshape(T, hq, d))
    assert np.array_equal(got[:, hq:hq + hkv], want_k[:T])
    assert np.array_equal(got[:, hq + hkv:], qkv_bits.reshape(T, -1, d)[:, hq + hkv:])
    assert np.array_equal(torch_to_bits(v_rows).reshape(T, hkv, d), want_v[:T])
    for i, s in enumerate(slots):
        if 0 <= s < 16:
            assert np.array_equal(torch_to_bits(kc)[s], want_k[i])
            assert np.array_equal(torch_to_bits(vc)[s], want_v[i])


@pytest.mark.parametrize("tokens,heads,clear", [(1, 1, 1), (3, 2, 257), (40, 8, 576)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_store_with_packed_copies_and_cleared_words(tokens, heads, clear, dtype):
    print(f"case store rows tokens={tokens} clear={clear} {dtype}", flush=True)
    from nanovllm_jax_amd import _lib, store_kv_to_cache
    dev, dt = "cuda:0", torch.bfloat16 if dtype == "bf16" else torch.float16
    code = _lib.NVJ_DTYPE_BF16 if dtype == "bf16" else _lib.NVJ_DTYPE_F16
    k = torch.randn(tokens, heads, 128, device=dev)
    v = torch.randn(tokens, heads, 128, device=dev).to(dt)
    slots = torch.randperm(64)[:tokens].to(torch.int32)
    slots[0] = -1
    slots = slots.to(dev)
    kc, vc, want_k, want_v = (torch.zeros(64, heads, 128, dtype=dt, device=dev) for _ in range(4))
    k_rows, v_rows = torch.zeros_like(v), torch.zeros_like(v)
    words = torch.full((clear + 1,), 7, dtype=torch.int32, device=dev)
    _lib.check(_lib.load().nvj_store_kvcache_rows_launch(
        torch.cuda.current_stream().cuda_stream, k.data_ptr(), v.data_ptr(), kc.data_ptr(),
        vc.data_ptr(), slots.data_ptr(), tokens, heads, 128, 64, _lib.NVJ_DTYPE_F32, code, code,
        k_rows.data_ptr(), v_rows.data_ptr(), words.data_ptr(), 4 * clear), "rows")
    store_kv_to_cache(k, v, want_k, want_v, slots)
    torch.cuda.synchronize()
    assert torch.equal(kc, want_k) and torch.equal(vc, want_v)
    assert torch.equal(k_rows, k.to(dt)) and torch.equal(v_rows, v)
    assert words.tolist() == [0] * clear + [7]


def _small_runner(seed=0, hidden=512, inter=768, heads=4, vocab=1000, layers=2, blocks=60, **kw):
    from nanovllm_jax_amd.engine import decode_step as ds
    cfg = ds.DecodeModelConfig(num_layers=layers, hidden_size=hidden, num_heads=heads,
                               num_kv_heads=2, head_dim=128, intermediate_size=inter,
                               vocab_size=vocab, max_position=512, block_size=64,
                               num_kvcache_blocks=blocks, **kw)
    return ds, ds.DecodeStepRunner(cfg, "cuda:0", seed=seed)


def _close(got, want):
    """Two orders of bf16 roundings of the same step (as in the comparison above)."""
    return (got - want).abs().max().item() <= 0.02 * want.abs().max().item() + 0.02


# rows of the few-row form, of the many-row form with few and with many sequences
@pytest.mark.parametrize("lens", [[0, 5, 9], [0, 30, 4], [0] + [2] * 20])
def test_native_step_first_sequence_without_new_tokens(lens, monkeypatch):
    print(f"case no new tokens {lens[:3]} of {len(lens)}", flush=True)
    ds, runner = _small_runner()
    cached = [40] + [0] * (len(lens) - 1)
    rng = np.random.Generator(np.random.PCG64(len(lens)))
    toks = [rng.integers(0, 1000, n + c).tolist() for n, c in zip(lens, cached)]
    ids, pos, ctx = runner.make_prefill_inputs(toks, [[i] for i in range(len(lens))], cached)
    assert ctx.last_token_indices[0].item() == -1
    before = runner.kv_cache.clone()
    got = runner._native_forward(ids, pos, ctx).float()
    runner.kv_cache.copy_(before)
    with monkeypatch.context() as m:
        m.setattr(ds, "_NATIVE_STEP_ROWS", 0)
        want = runner.forward(ids, pos, ctx).float()
    # index -1 is the last row, whatever sequence it belongs to, as host indexing has it
    assert torch.equal(got[0], got[-1]) and _close(got, want)
    # one that names no row shows, and harms no other
    bad = ctx.last_token_indices.clone()
    bad[0], bad[1] = int(ids.shape[0]), -int(ids.shape[0]) - 1
    ctx.last_token_indices = bad
    runner.kv_cache.copy_(before)
    out = runner._native_forward(ids, pos, ctx).float()
    assert out[:2].isnan().all() and torch.equal(out[2:], got[2:])


@pytest.mark.parametrize("what", ["host", "longer", "shorter", "int64", "strided", "2d"])
def test_native_step_takes_any_last_token_indices(what):
    """Logits of exactly the rows asked for, by any tensor that indexes rows."""
    print(f"case last token indices {what}", flush=True)
    ds, runner = _small_runner()
    ids, pos, ctx = runner.make_prefill_inputs([[1, 2, 3], [4, 5], [6, 7, 8, 9]], [[0], [1], [2]])
    want = runner.forward(ids, pos, ctx).float()
    last, rows = ctx.last_token_indices, [0, 1, 2]
    if what == "host":
        last = last.cpu()
    elif what == "longer":
        last, rows = torch.cat([last, last[:1]]), [0, 1, 2, 0]
    elif what == "shorter":
        last, rows = last[1:2], [1]
    elif what == "int64":
        last = last.long()
    elif what == "strided":
        last = last.repeat_interleave(2)[::2]
    else:
        last = last[None, :].expand(2, 3)
    ctx.last_token_indices = last
    got = runner.forward(ids, pos, ctx).float()
    assert (runner._native_forward(ids, pos, ctx) is not None) == (what in ("int64", "strided"))
    if what == "2d":
        assert got.shape == (2, 3, want.shape[1]) and torch.equal(got[0], got[1])
        got = got[0]
    assert got.shape == (len(rows), want.shape[1]) and _close(got, want[rows])


def _decode_inputs(runner, rows):
    return runner.make_inputs(list(range(rows)), [20 + i for i in range(rows)],
                              [[i] for i in range(rows)])


@pytest.mark.parametrize("rows", [3, 20, -3, -20])      # decode; new tokens of a packed prompt
def test_native_step_reads_the_model_on_every_step(rows, monkeypatch):
    """What changes between two steps changes the second: a layer's scale, the norms' eps,
    weights in place, and weights replaced by others."""
    print(f"case model read on every step rows={rows}", flush=True)
    ds, runner = _small_runner()
    inputs = _decode_inputs(runner, rows) if rows > 0 else \
        runner.make_prefill_inputs([list(range(-rows))], [[0]])
    first = runner.forward(*inputs).float()

    def both():
        got = runner.forward(*inputs).float()
        with monkeypatch.context() as m:
            m.setattr(ds, "_NATIVE_STEP_ROWS", 0)
            want = runner.forward(*inputs).float()
        assert _close(got, want)
        return got

    attn, lw = runner.attn, runner.layers
    attn[1].scale = 1.0             # one layer's alone: not a model for the native step
    assert runner._native_forward(*inputs) is None
    last = both()
    assert not torch.equal(last, first)
    for a in attn:
        a.scale = 1.0
    assert runner._native_forward(*inputs) is not None
    assert not torch.equal(both(), last)
    for a in attn:
        a.scale = 128 ** -0.5
    assert torch.equal(runner.forward(*inputs).float(), first)
    runner.cfg.rms_norm_eps = 100.0
    assert not torch.equal(both(), first)
    runner.cfg.rms_norm_eps = 1e-6
    kept = lw[1]["down"]
    lw[1]["down"] = torch.zeros_like(kept)
    assert not torch.equal(both(), first)
    lw[1]["down"] = kept
    for w in lw:                    # no norm of q and k
        w["q_norm"] = w["k_norm"] = None
    assert runner._native_forward(*inputs) is not None
    assert not torch.equal(both(), first)


@pytest.mark.parametrize("name,shape", [("qkv", (256, 512)), ("o", (512, 256)),
                                        ("gate_up", (512, 512)), ("down", (256, 768)),
                                        ("ln1", (256,)), ("ln2", (256,)), ("q_norm", (64,)),
                                        ("k_norm", (64,)), ("cos_sin", (512, 64)),
                                        ("final_norm", (256,))])
@pytest.mark.parametrize("kind", ["decode", "packed"])
def test_native_step_refuses_weights_of_another_shape(name, shape, kind):
    """A weight that was replaced by a smaller one is never read past its end: the native
    step declines, and the long way names the mistake."""
    print(f"case weight {name} {shape} {kind}", flush=True)
    _, runner = _small_runner()
    inputs = _decode_inputs(runner, 3) if kind == "decode" else \
        runner.make_prefill_inputs([[1, 2, 3], [4, 5]], [[0], [1]])
    assert runner._native_forward(*inputs) is not None
    at = runner.layers[1] if name in runner.layers[1] else runner.__dict__
    at[name] = torch.ones(shape, dtype=at[name].dtype, device="cuda:0")
    assert runner._native_forward(*inputs) is None
    with pytest.raises((RuntimeError, ValueError)):
        runner.forward(*inputs)


def test_native_step_declines_what_it_is_not_built_for():
    print("case weights of another type, layout or alignment", flush=True)
    _, runner = _small_runner()
    inputs = _decode_inputs(runner, 3)
    want = runner.forward(*inputs).float()
    for name, other in (("qkv", lambda t: t.t().contiguous().t()),                # strided
                        ("down", lambda t: torch.cat([t.new_zeros(1), t.flatten()])[1:]
                         .view(t.shape))):                                        # 2 bytes off
        kept = runner.layers[0][name]
        runner.layers[0][name] = other(kept)
        assert runner._native_forward(*inputs) is None
        assert _close(runner.forward(*inputs).float(), want)
        runner.layers[0][name] = kept
    runner.attn[0].block_size = 32
    assert runner._native_forward(*inputs) is None
    with pytest.raises(ValueError):
        runner.forward(*inputs)


@pytest.mark.parametrize("rows", [4, 20])
def test_token_ids_outside_the_vocabulary(rows):
    """Refused where the ids come from the host; on the device the sequence concerned, and
    no other, gets NaN logits."""
    print(f"case ids outside the vocabulary rows={rows}", flush=True)
    _, runner = _small_runner()
    lens, tables = [20 + i for i in range(rows)], [[i] for i in range(rows)]
    for bad in (1000, -1):
        with pytest.raises(ValueError):
            runner.make_inputs([0] * (rows - 1) + [bad], lens, tables)
        with pytest.raises(ValueError):
            runner.make_prefill_inputs([[1, bad]], [[0]])
    ids, pos, ctx = runner.make_inputs([999] * rows, lens, tables)
    want = runner.forward(ids, pos, ctx).float()
    assert not want.isnan().any()
    ids[1], ids[2] = 1000, -1
    got = runner._native_forward(ids, pos, ctx).float()
    keep = [i for i in range(rows) if i not in (1, 2)]
    assert got[1:3].isnan().all() and torch.equal(got[keep], want[keep])


def test_native_step_declines_a_workspace_of_another_device():
    print("case workspace on the host", flush=True)
    from nanovllm_jax_amd.layers.paged_attention import DecodeWorkspace
    _, runner = _small_runner()
    inputs = _decode_inputs(runner, 3)
    ws = DecodeWorkspace(1 << 20, "cpu")
    for a in runner.attn:
        a.workspace = ws
    assert runner._native_forward(*inputs) is None
    with pytest.raises(ValueError):
        runner.forward(*inputs)


def test_wide_models_take_the_library_products():
    print("case wide model", flush=True)
    _, runner = _small_runner(hidden=4096, inter=512, heads=2, layers=1)
    for rows, native in ((24, True), (25, False)):
        inputs = _decode_inputs(runner, rows)
        assert (runner._native_forward(*inputs) is not None) == native
        assert not runner.forward(*inputs).isnan().any()


def test_packed_prefill_refuses_offsets_of_another_length(monkeypatch):
    print("case cu_seqlens of another length", flush=True)
    ds, runner = _small_runner()
    for patch in (False, True):
        if patch:
            monkeypatch.setattr(ds, "_NATIVE_STEP_ROWS", 0)
        ids, pos, ctx = runner.make_prefill_inputs([[1, 2, 3], [4, 5]], [[0], [1]])
        ctx.cu_seqlens_k = ctx.cu_seqlens_k[:2]
        with pytest.raises(ValueError):
            runner.forward(ids, pos, ctx)


@pytest.mark.parametrize("rows", [4, 24])
@pytest.mark.parametrize("kind", ["decode", "packed", "paged"])
def test_native_step_with_slots_that_are_not_stored(rows, kind, monkeypatch):
    print(f"case skipped slots rows={rows} {kind}", flush=True)
    ds, runner = _small_runner()
    if kind == "decode":
        ids, pos, ctx = _decode_inputs(runner, rows)
    else:
        toks = [list(range(rows - 2)), [5, 6]]
        cached = [9, 0] if kind == "paged" else None
        if cached:
            toks[0] = [1] * 9 + toks[0]
        ids, pos, ctx = runner.make_prefill_inputs(toks, [[0], [1]], cached)
    slots = ctx.slot_mapping.clone()
    slots[1], slots[-1] = -1, 60 * 64                       # skipped, and out of the cache
    ctx.slot_mapping = slots
    before = runner.kv_cache.clone()
    got = runner._native_forward(ids, pos, ctx).float()
    kv = runner.kv_cache.clone()
    runner.kv_cache.copy_(before)
    monkeypatch.setattr(ds, "_NATIVE_STEP_ROWS", 0)
    want = runner.forward(ids, pos, ctx).float()
    assert _close(got, want)
    # rows written by both, and by neither
    flat = lambda t: t.view(2, 2, -1, 2, 128)
    written = torch.zeros(60 * 64, dtype=torch.bool, device="cuda:0")
    written[slots[(slots >= 0) & (slots < 60 * 64)].long()] = True
    for cache in (kv, runner.kv_cache):
        same = (flat(cache) == flat(before)).all(-1).all(-1)
        assert same[:, :, ~written].all() and not same[:, :, written].any()
    assert ((kv.float() - runner.kv_cache.float()).abs()
            <= 0.03 + 0.03 * runner.kv_cache.float().abs()).all()


@pytest.mark.parametrize("kind", ["decode", "packed"])
@pytest.mark.parametrize("native", [True, False])
def test_inputs_reach_a_step_on_another_stream(kind, native, monkeypatch):
    """Inputs made behind long work on one stream, and a step on another stream at once."""
    print(f"case inputs of another stream {kind} native={native}", flush=True)
    ds, runner = _small_runner()
    if not native:
        monkeypatch.setattr(ds, "_NATIVE_STEP_ROWS", 0)
    def make(first):
        if kind == "decode":
            return runner.make_inputs([first + i for i in range(20)], [20 + i for i in range(20)],
                                      [[i] for i in range(20)])
        return runner.make_prefill_inputs([[first + i for i in range(9)], [first, 8]], [[0], [1]])

    wants = [runner.forward(*make(first)) for first in (0, 500)]
    assert not torch.equal(*wants)
    side = torch.cuda.Stream()
    a = torch.randn(8192, 8192, device="cuda:0")
    side.wait_stream(torch.cuda.current_stream())
    torch.cuda.synchronize()
    for turn in range(6):     # in turn: memory that is used again holds the other inputs
        for _ in range(4):
            torch.mm(a, a)
        inputs = make(500 * (turn % 2))
        with torch.cuda.stream(side):
            got = runner.forward(*inputs)
        side.synchronize()
        assert torch.equal(got, wants[turn % 2])
        torch.cuda.synchronize()


def test_contexts_can_be_copied_and_pickled():
    print("case copies of a context", flush=True)
    import copy
    import dataclasses
    import pickle
    _, runner = _small_runner()
    ids, pos, ctx = _decode_inputs(runner, 3)
    want = runner.forward(ids, pos, ctx)
    for other in (copy.copy(ctx), copy.deepcopy(ctx), dataclasses.replace(ctx),
                  type(ctx)(**dataclasses.asdict(ctx)), pickle.loads(pickle.dumps(ctx))):
        assert torch.equal(runner.forward(ids, pos, other), want)


@pytest.mark.parametrize("rows,hidden,inter,heads,layers,wide_mb", [
    (3, 1024, 3072, 16, 8, 0), (3, 1024, 3072, 16, 8, 25), (16, 1024, 3072, 16, 8, 40),
    (4, 2048, 3072, 16, 4, 0), (16, 2048, 3072, 16, 4, 51), (5, 1024, 3072, 16, 1, 0),
    (17, 320, 34816, 6, 4, 0), (40, 2048, 4096, 24, 3, 0), (20, 2560, 9728, 16, 2, 0),
    (64, 1024, 3072, 16, 8, 0), (129, 320, 34816, 6, 4, 0), (200, 1024, 3072, 16, 8, 0)])
def test_weights_read_ahead(rows, hidden, inter, heads, layers, wide_mb, monkeypatch):
    """Which weights a launch reads ahead depends on the size of the model (200 MB of layers, all
    but one case here), the row count, the widths and, up to 16 rows, on the K and V that the
    block table holds: every set of them against the library's products.  Two orders of bf16
    roundings leave the logits of 28 layers of random weights 2-3 % apart."""
    print(f"case read ahead rows={rows} hidden={hidden} layers={layers} {wide_mb}", flush=True)
    from nanovllm_jax_amd.engine import decode_step as ds
    cfg = ds.DecodeModelConfig(num_layers=layers, hidden_size=hidden, num_heads=heads,
                               num_kv_heads=2, head_dim=128, intermediate_size=inter,
                               vocab_size=1000, max_position=64, block_size=64,
                               num_kvcache_blocks=rows)
    runner = ds.DecodeStepRunner(cfg, "cuda:0", seed=rows)
    inputs = runner.make_inputs([7 * i % 1000 for i in range(rows)],
                                [1 + 5 * i % 64 for i in range(rows)], [[i] for i in range(rows)])
    # 1 KB of K and V a position
    inputs[2].block_tables = torch.nn.functional.pad(
        inputs[2].block_tables, (0, (wide_mb << 20) // (rows * 64 * 1024)), value=-1).contiguous()
    runner.kv_cache.normal_()
    before = runner.kv_cache.clone()
    got = runner._native_forward(*inputs).float()
    runner.kv_cache.copy_(before)
    monkeypatch.setattr(ds, "_NATIVE_STEP_ROWS", 0)
    want = runner.forward(*inputs).float()
    torch.cuda.synchronize()
    assert (got - want).norm().item() <= 0.03 * want.norm().item()


@pytest.mark.parametrize("rows,hidden,inter,heads,layers,wide_mb", [
    (3, 1024, 3072, 16, 8, 0), (3, 1024, 3072, 16, 8, 25), (16, 1024, 3072, 16, 8, 40),
    (4, 2048, 3072, 16, 4, 0), (16, 2048, 3072, 16, 4, 51), (17, 320, 34816, 6, 4, 0),
    (40, 2048, 4096, 24, 3, 0), (20, 2560, 9728, 16, 2, 0), (64, 1024, 3072, 16, 8, 0),
    (129, 320, 34816, 6, 4, 0), (200, 1024, 3072, 16, 8, 0)])
@pytest.mark.parametrize("kind", ["decode", "packed"])
def test_reading_ahead_changes_no_bit(rows, hidden, inter, heads, layers, wide_mb, kind):
    """Layers of up to 200 MB are not read ahead, larger models are.  A layer in front whose
    output and down projections are zero adds nothing to the (bf16) embedding rows, so the same
    layers are run with it, beyond the line, and without it, below: the same logits and the
    same cache rows, bit for bit."""
    print(f"case no bit rows={rows} hidden={hidden} layers={layers} {wide_mb} {kind}", flush=True)
    from nanovllm_jax_amd.engine import decode_step as ds
    cfg = ds.DecodeModelConfig(num_layers=layers, hidden_size=hidden, num_heads=heads,
                               num_kv_heads=2, head_dim=128, intermediate_size=inter,
                               vocab_size=1000, max_position=256, block_size=64,
                               num_kvcache_blocks=rows + 4)
    runner = ds.DecodeStepRunner(cfg, "cuda:0", seed=rows + layers)
    weights = sum(runner.layers[0][n].nbytes for n in ("qkv", "o", "gate_up", "down"))
    assert (layers - 1) * weights <= 200 << 20 < layers * weights
    for name in ("o", "down"):
        runner.layers[0][name].zero_()
    ids = [7 * i % 1000 for i in range(rows)]
    if kind == "decode":
        inputs = runner.make_inputs(ids, [1 + 5 * i % 64 for i in range(rows)],
                                    [[i] for i in range(rows)])
        # 1 KB of K and V a position
        inputs[2].block_tables = torch.nn.functional.pad(
            inputs[2].block_tables, (0, (wide_mb << 20) // (rows * 64 * 1024)),
            value=-1).contiguous()
    else:
        inputs = runner.make_prefill_inputs([ids], [list(range(-(-rows // 64)))])
    before = runner.kv_cache.clone()
    with_it = runner._native_forward(*inputs)
    kv = runner.kv_cache.clone()
    runner.kv_cache.copy_(before)
    del runner.layers[0], runner.attn[0]
    for _ in range(2):            # (the second with whatever the caches hold by then)
        without = runner._native_forward(*inputs)
        torch.cuda.synchronize()
        assert not without.isnan().any() and torch.equal(with_it, without)
        assert torch.equal(kv[:, 1:].view(torch.int16), runner.kv_cache[:, 1:].view(torch.int16))
