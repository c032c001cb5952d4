"""GPU parity of the HIP variable-length causal prefill attention against the
CPU oracle (atol/rtol 1e-2, bf16 out, fp32 accumulate), through the C ABI."""
import numpy as np
import pytest

from helpers import assert_close_bf16, bits_to_torch, torch_to_bits

pytestmark = pytest.mark.gpu


def _problem(seed, lens_q, lens_k, Hq, Hkv, D=128, gain=1.0):
    from nanovllm_jax_amd.workloads import draw_bf16_bits
    rng = np.random.Generator(np.random.PCG64(seed))
    cu_q = np.concatenate([[0], np.cumsum(lens_q)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(lens_k)]).astype(np.int32)
    q = draw_bf16_bits(rng, (int(cu_q[-1]), Hq, D), gain)
    k = draw_bf16_bits(rng, (max(int(cu_k[-1]), 1), Hkv, D))
    v = draw_bf16_bits(rng, (max(int(cu_k[-1]), 1), Hkv, D))
    return q, k, v, cu_q, cu_k


def run_hip(q, k, v, cu_q, cu_k, scale):
    import torch
    from nanovllm_jax_amd import variable_length_attention_prefill
    dev = "cuda:0"
    out = variable_length_attention_prefill(
        bits_to_torch(q, dev), bits_to_torch(k, dev), bits_to_torch(v, dev),
        torch.from_numpy(cu_q).to(dev), torch.from_numpy(cu_k).to(dev), scale=scale)
    torch.cuda.synchronize()
    return torch_to_bits(out)


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (16, 8), (32, 8), (8, 1)])
def test_prefill_ragged_batch(Hq, Hkv):
    print(f"case prefill ragged Hq={Hq} Hkv={Hkv}", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    lens = [1, 31, 32, 33, 127, 128, 129, 300, 17]
    q, k, v, cu_q, cu_k = _problem(10 + Hq, lens, lens, Hq, Hkv)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    got = run_hip(q, k, v, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what=f"prefill Hq={Hq} Hkv={Hkv}")
    G = Hq // Hkv
    for i in range(len(lens)):                    # first row of a sequence == its first V row
        assert np.array_equal(got[cu_q[i]], np.repeat(v[cu_k[i]], G, axis=0))


@pytest.mark.parametrize("batch,Hq,Hkv", [(1, 7, 7), (63, 6, 2), (64, 10, 2), (127, 3, 3),
                                           (128, 12, 2), (129, 6, 2), (255, 5, 1), (256, 14, 2),
                                           (257, 6, 2), (512, 3, 1), (513, 6, 2)])
def test_prefill_finds_the_tiles_of_every_sequence(batch, Hq, Hkv):
    """Batches at the edges of what the lanes of a wave hold (one, two or four sequences each, then
    256 at a time), groups that are no power of two, empty sequences at both ends and beside each
    other."""
    print(f"case prefill lookup batch={batch} Hq={Hq} Hkv={Hkv}", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    rng = np.random.Generator(np.random.PCG64(900 + batch))
    lens = rng.integers(0, 20, size=batch)
    lens[rng.integers(0, batch, size=2)] = [140, 75]
    if batch > 1:
        lens[[0, 1, batch // 2, batch - 1]] = 0
    lens = [int(x) for x in lens]
    q, k, v, cu_q, cu_k = _problem(910 + batch, lens, lens, Hq, Hkv)
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, 128 ** -0.5)
    assert_close_bf16(run_hip(q, k, v, cu_q, cu_k, 128 ** -0.5), want, what=f"batch {batch}")


@pytest.mark.parametrize("lens,Hq,Hkv,dtype", [
    ([33, 1, 0, 64, 20, 5, 32, 17, 31, 15] * 15 + [129, 300, 65], 32, 8, "bf16"),  # three workgroups
    ([60, 16, 97, 1, 250] * 8, 32, 32, "f16"),                                     # to a CU
    ([3] * 150 + [160, 0], 16, 8, "bf16"),
    ([500, 433, 512, 0, 640, 1, 500, 700, 505], 16, 8, "bf16"),    # longest tiles first
    ([1000, 999, 97], 32, 8, "f16"),
])
def test_prefill_is_the_same_however_a_launch_is_cut(lens, Hq, Hkv, dtype):
    """Launches of many or uneven prompts have workgroups, rings and orders of their own; a row's
    sums are in the same order in all of them: bit for bit as every prompt by itself."""
    print(f"case prefill forms {len(lens)} prompts Hq={Hq} Hkv={Hkv} {dtype}", flush=True)
    import torch
    from nanovllm_jax_amd import variable_length_attention_prefill
    dev, dt = "cuda:0", {"bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    g = torch.Generator(device=dev)
    g.manual_seed(len(lens))
    T = sum(lens)
    q, k, v = (torch.randn(T, h, 128, generator=g, device=dev).to(dt) for h in (Hq, Hkv, Hkv))
    cu = lambda n: torch.from_numpy(np.concatenate([[0], np.cumsum(n)]).astype(np.int32)).to(dev)
    got = variable_length_attention_prefill(q, k, v, cu(lens), cu(lens))
    at = np.concatenate([[0], np.cumsum(lens)])
    for i, n in enumerate(lens):
        part = slice(int(at[i]), int(at[i + 1]))
        one = variable_length_attention_prefill(q[part], k[part], v[part], cu([n]), cu([n]))
        assert torch.equal(got[part], one), f"prompt {i} of {n} tokens"


@pytest.mark.parametrize("batch", [65, 130, 300, 600])
def test_prefill_batches_of_many_short_prompts(batch):
    """More sequences than the 64 a wave looks at together, and than the 256 whose
    lengths it fetches in one go, when it finds the sequence of a query tile: short
    prompts, empty ones and a few longer than a tile among them."""
    print(f"case prefill many prompts batch={batch}", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    rng = np.random.Generator(np.random.PCG64(700 + batch))
    lens = rng.integers(0, 41, size=batch)
    lens[rng.integers(0, batch, size=5)] = [129, 257, 128, 1, 300]
    lens[[0, 63, 64, batch - 1]] = [3, 130, 0, 131]
    lens = [int(x) for x in lens]
    q, k, v, cu_q, cu_k = _problem(710 + batch, lens, lens, 4, 2)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    got = run_hip(q, k, v, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what=f"prefill {batch} prompts")
    for i in range(batch):                        # first row of a sequence == its first V row
        if lens[i] > 0:
            assert np.array_equal(got[cu_q[i]], np.repeat(v[cu_k[i]], 2, axis=0)), i


@pytest.mark.parametrize("Hq,Hkv", [(6, 2), (5, 1), (24, 2), (16, 1), (4, 4)])
def test_prefill_column_groups_and_rows_of_one_buffer(Hq, Hkv):
    """Group sizes that do not divide the 8 column groups of a tile, lengths around the
    16 tokens of a column group, and q, k, v as parts of one projection buffer."""
    print(f"case prefill column groups Hq={Hq} Hkv={Hkv}", flush=True)
    import torch
    from nanovllm_jax_amd import _lib
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    lens = [15, 16, 17, 1, 0, 40, 113]
    q, k, v, cu_q, cu_k = _problem(90 + Hq, lens, lens, Hq, Hkv)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    T, dev = sum(lens), "cuda:0"
    buf = torch.cat([bits_to_torch(x, dev).reshape(T, -1) for x in (q, k, v)], 1).contiguous()
    out = torch.empty(T, Hq, 128, dtype=torch.bfloat16, device=dev)
    cq = torch.from_numpy(cu_q).to(dev)
    at = buf.data_ptr()
    _lib.check(_lib.load().nvj_prefill_attention_rows_launch(
        torch.cuda.current_stream().cuda_stream, at, buf.shape[1], at + 256 * Hq,
        at + 256 * (Hq + Hkv), buf.shape[1], cq.data_ptr(), cq.data_ptr(), out.data_ptr(), T,
        len(lens), Hq, Hkv, 128, scale, _lib.NVJ_DTYPE_BF16), "rows")
    torch.cuda.synchronize()
    assert_close_bf16(torch_to_bits(out), want, what=f"rows Hq={Hq} Hkv={Hkv}")
    assert np.array_equal(torch_to_bits(out), run_hip(q, k, v, cu_q, cu_k, scale))


def test_prefill_reference_smoke_lengths():
    """Sequence lengths of the reference's prefill smoke test
    (test_mosaic_kernels.py:90-159): 512, 768, 1024, 1536; Hq=32, Hkv=8, D=128."""
    print("case prefill reference smoke lengths", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    lens = [512, 768, 1024, 1536]
    q, k, v, cu_q, cu_k = _problem(20, lens, lens, 32, 8)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    got = run_hip(q, k, v, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what="prefill smoke lengths")


def test_prefill_unequal_q_and_k_lengths_and_empty_sequences():
    print("case prefill unequal lengths / empty", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    lens_q = [40, 0, 5, 200, 64]
    lens_k = [12, 7, 90, 200, 0]
    q, k, v, cu_q, cu_k = _problem(30, lens_q, lens_k, 16, 8)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    got = run_hip(q, k, v, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what="prefill unequal")
    assert not got[cu_q[4]:cu_q[5]].any()         # no keys at all -> zeros


def test_prefill_sharp_softmax_and_packing_invariance():
    print("case prefill sharp softmax / packing", flush=True)
    from oracle.paged_attention_oracle import variable_length_attention_prefill_ref
    lens = [257, 100]
    q, k, v, cu_q, cu_k = _problem(40, lens, lens, 16, 8, gain=4.0)
    scale = 128 ** -0.5
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, scale)
    got = run_hip(q, k, v, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what="prefill sharp")
    alone = run_hip(q[cu_q[1]:], k[cu_k[1]:], v[cu_k[1]:], np.array([0, 100], np.int32),
                    np.array([0, 100], np.int32), scale)
    assert np.array_equal(alone, got[cu_q[1]:])


def test_attention_layer_prefill_then_decode():
    """Attention.__call__ in prefill mode stores the prompt's K/V through
    slot_mapping and attends over the packed rows; a decode step over the same
    cache then equals the last prefill row recomputed (same keys, same query)."""
    print("case Attention prefill then decode", flush=True)
    import torch
    from nanovllm_jax_amd import Attention, create_decode_context, create_prefill_context
    from nanovllm_jax_amd.workloads import draw_bf16_bits
    from oracle.paged_attention_oracle import (store_kv_to_cache_ref,
                                               variable_length_attention_prefill_ref)
    Hq, Hkv, D, bs, NB = 16, 8, 128, 256, 8
    lens = [300, 77]
    q, k, v, cu_q, cu_k = _problem(50, lens, lens, Hq, Hkv)
    tables = [[3, 5], [6]]
    slots = np.concatenate([np.concatenate([np.arange(p * bs, p * bs + min(bs, n - j * bs))
                                            for j, p in enumerate(t)])
                            for t, n in zip(tables, lens)]).astype(np.int32)
    dev = "cuda:0"
    attn = Attention(Hq, D, D ** -0.5, Hkv, bs)
    kc = np.zeros((NB, bs, Hkv, D), np.uint16)
    attn.set_kv_cache(bits_to_torch(kc, dev), bits_to_torch(kc.copy(), dev))
    up = lambda a: torch.from_numpy(a).to(dev)
    ctx = create_prefill_context(up(cu_q), up(cu_k), max(lens), max(lens), up(slots))
    out = attn(bits_to_torch(q, dev), bits_to_torch(k, dev), bits_to_torch(v, dev), ctx)
    torch.cuda.synchronize()
    want = variable_length_attention_prefill_ref(q, k, v, cu_q, cu_k, D ** -0.5)
    assert_close_bf16(torch_to_bits(out), want, what="layer prefill")
    flat = (-1, Hkv, D)
    wk, wv = store_kv_to_cache_ref(k, v, kc.reshape(flat), kc.reshape(flat), slots, negative_slots="skip")
    assert np.array_equal(torch_to_bits(attn.k_cache).reshape(flat), wk)
    assert np.array_equal(torch_to_bits(attn.v_cache).reshape(flat), wv)
    # decode with the last prompt token as the query, its K/V already in the cache
    last = cu_q[1:] - 1
    bt = np.array([[3, 5], [6, -1]], np.int32)
    dctx = create_decode_context(up(np.array(lens, np.int32)),
                                 up(np.array([-1, -1], np.int32)), up(bt))
    dq = bits_to_torch(q[last], dev)
    dout = attn(dq, bits_to_torch(k[last], dev), bits_to_torch(v[last], dev), dctx)
    torch.cuda.synchronize()
    assert_close_bf16(torch_to_bits(dout), want[last], what="decode == last prefill row")


# ---- prefill behind a cached prefix: keys and values from the paged cache ----
def _paged_problem(seed, lens_k, lens_q, Hq, Hkv, bs, extra_pages=3):
    from nanovllm_jax_amd.workloads import draw_bf16_bits
    rng = np.random.Generator(np.random.PCG64(seed))
    D = 128
    B = len(lens_k)
    nblk = [-(-n // bs) for n in lens_k]
    NB = sum(nblk) + extra_pages
    kc, vc = draw_bf16_bits(rng, (NB, bs, Hkv, D)), draw_bf16_bits(rng, (NB, bs, Hkv, D))
    cu_q = np.concatenate([[0], np.cumsum(lens_q)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(lens_k)]).astype(np.int32)
    q = draw_bf16_bits(rng, (max(int(cu_q[-1]), 1), Hq, D), 2.0)[:int(cu_q[-1])]
    bt = np.full((B, max(max(nblk), 1) + 1), -1, np.int32)       # one padding column
    pages = rng.permutation(NB)
    used = 0
    for i, n in enumerate(nblk):
        bt[i, :n] = pages[used:used + n]
        used += n
    return q, kc, vc, bt, cu_q, cu_k


def run_hip_paged(q, kc, vc, bt, cu_q, cu_k, scale):
    import torch
    from nanovllm_jax_amd import paged_prefill_attention
    dev = "cuda:0"
    out = paged_prefill_attention(bits_to_torch(q, dev), bits_to_torch(kc, dev),
                                  bits_to_torch(vc, dev), torch.from_numpy(bt).to(dev),
                                  torch.from_numpy(cu_q).to(dev), torch.from_numpy(cu_k).to(dev),
                                  scale)
    torch.cuda.synchronize()
    return torch_to_bits(out)


@pytest.mark.parametrize("Hq,Hkv,bs", [(8, 2, 32), (16, 8, 64), (32, 8, 256), (4, 4, 96)])
def test_paged_prefill_behind_a_cached_prefix(Hq, Hkv, bs):
    """Prompt chunks of many lengths behind prefixes of many lengths (none, shorter
    and longer than a page, ending on and off page and tile boundaries), pages in
    random order, padding table entries, garbage in unused pages."""
    print(f"case paged prefill Hq={Hq} Hkv={Hkv} bs={bs}", flush=True)
    from oracle.paged_attention_oracle import paged_prefill_attention_ref
    lens_q = [1, 33, 128, 129, 40, 300, 5, 64]
    prefix = [0, 31, 32, 500, 257, 0, 700, 64]
    lens_k = [a + b for a, b in zip(lens_q, prefix)]
    q, kc, vc, bt, cu_q, cu_k = _paged_problem(70 + Hq + bs, lens_k, lens_q, Hq, Hkv, bs)
    scale = 128 ** -0.5
    want = paged_prefill_attention_ref(q, kc, vc, bt, cu_q, cu_k, scale)
    got = run_hip_paged(q, kc, vc, bt, cu_q, cu_k, scale)
    assert_close_bf16(got, want, what="paged prefill")
    # poison everything no live key sits on: the result must not move
    live = np.zeros(kc.shape[:2], bool)
    for i, n in enumerate(lens_k):
        for p in range(n):
            live[bt[i, p // bs], p % bs] = True
    kc2, vc2 = kc.copy(), vc.copy()
    kc2[~live] = 0x7FC0
    vc2[~live] = 0x7FC0                                           # NaN
    bt2 = np.where(bt < 0, 10 ** 6, bt).astype(np.int32)          # padding entries out of range
    got2 = run_hip_paged(q, kc2, vc2, bt2, cu_q, cu_k, scale)
    assert np.array_equal(got, got2), "something outside the live keys was read"


def test_paged_prefill_without_prefix_equals_packed_prefill_bit_for_bit():
    print("case paged prefill == packed prefill", flush=True)
    lens = [300, 77, 1, 129]
    Hq, Hkv, bs = 16, 8, 64
    q, kc, vc, bt, cu_q, cu_k = _paged_problem(81, lens, lens, Hq, Hkv, bs)
    # the packed rows are the live cache rows in sequence order
    k = np.concatenate([kc[bt[i, p // bs], p % bs][None] for i, n in enumerate(lens) for p in range(n)])
    v = np.concatenate([vc[bt[i, p // bs], p % bs][None] for i, n in enumerate(lens) for p in range(n)])
    scale = 0.11
    packed = run_hip(q, k, v, cu_q, cu_k, scale)
    paged = run_hip_paged(q, kc, vc, bt, cu_q, cu_k, scale)
    assert np.array_equal(packed, paged)


def test_attention_layer_prefill_with_cached_prefix():
    """Attention.__call__ with a prefill context that carries block_tables (the
    reference's filler sets them when a prefix is cached): the chunk's K/V rows are
    stored, then the chunk attends over prefix + chunk from the cache; a decode step
    with the chunk's last token as the query sees the same keys."""
    print("case Attention prefill behind a cached prefix", flush=True)
    import torch
    from nanovllm_jax_amd import Attention, create_decode_context, create_prefill_context
    from nanovllm_jax_amd.workloads import draw_bf16_bits
    from oracle.paged_attention_oracle import (paged_prefill_attention_ref,
                                               store_kv_to_cache_ref)
    Hq, Hkv, D, bs = 16, 8, 128, 64
    prefix, chunk = [100, 0, 64], [60, 130, 7]
    lens_k = [a + b for a, b in zip(prefix, chunk)]
    q, kc, vc, bt, cu_q, cu_k = _paged_problem(82, lens_k, chunk, Hq, Hkv, bs)
    rng = np.random.Generator(np.random.PCG64(83))
    k_new = draw_bf16_bits(rng, (int(cu_q[-1]), Hkv, D))
    v_new = draw_bf16_bits(rng, (int(cu_q[-1]), Hkv, D))
    slots = np.concatenate([bt[i, np.arange(prefix[i], lens_k[i]) // bs] * bs +
                            np.arange(prefix[i], lens_k[i]) % bs for i in range(3)]).astype(np.int32)
    dev = "cuda:0"
    up = lambda a: torch.from_numpy(a).to(dev)
    attn = Attention(Hq, D, D ** -0.5, Hkv, bs)
    attn.set_kv_cache(bits_to_torch(kc, dev), bits_to_torch(vc, dev))
    ctx = create_prefill_context(up(cu_q), up(cu_k), max(chunk), max(lens_k), up(slots),
                                 block_tables=up(bt))
    out = attn(bits_to_torch(q, dev), bits_to_torch(k_new, dev), bits_to_torch(v_new, dev), ctx)
    torch.cuda.synchronize()
    flat = (-1, Hkv, D)
    wk, wv = store_kv_to_cache_ref(k_new, v_new, kc.reshape(flat), vc.reshape(flat), slots,
                                   negative_slots="skip")
    assert np.array_equal(torch_to_bits(attn.k_cache).reshape(flat), wk)
    want = paged_prefill_attention_ref(q, wk.reshape(kc.shape), wv.reshape(vc.shape), bt, cu_q,
                                       cu_k, D ** -0.5)
    assert_close_bf16(torch_to_bits(out), want, what="layer prefill behind a prefix")
    last = cu_q[1:] - 1
    dctx = create_decode_context(up(np.array(lens_k, np.int32)), up(np.full(3, -1, np.int32)),
                                 up(bt))
    dout = attn(bits_to_torch(q[last], dev), bits_to_torch(k_new[last], dev),
                bits_to_torch(v_new[last], dev), dctx)
    torch.cuda.synchronize()
    assert_close_bf16(torch_to_bits(dout), want[last], what="decode == last chunk row")


@pytest.mark.parametrize("batch,Hq,Hkv", [(5, 8, 8), (70, 6, 2), (200, 8, 4)])
def test_paged_prefill_longest_tiles_first(batch, Hq, Hkv):
    """Cached prefixes of very different lengths: tiles are handed out by the keys they walk.
    Sequences without new tokens, without a prefix, and tiles that tie among them."""
    print(f"case paged prefill longest first batch={batch} Hq={Hq}", flush=True)
    import torch
    from nanovllm_jax_amd import paged_prefill_attention
    rng = np.random.Generator(np.random.PCG64(batch))
    new = rng.integers(1, 60, batch)
    cached = rng.integers(0, 300, batch)
    new[[0, 1, batch // 2]], cached[[0, 1, batch // 2]] = [17, 300, 0], [1500, 0, 900]
    total, page = new + cached, 32
    pages = -(-total // page)
    ids = rng.permutation(int(pages.sum()))
    table = np.full((batch, int(pages.max())), -1, np.int32)
    for i, e in enumerate(np.cumsum(pages)):
        table[i, :pages[i]] = ids[e - pages[i]:e]
    dev = "cuda:0"
    g = torch.Generator(device=dev)
    g.manual_seed(batch)
    kc, vc = (torch.randn(int(pages.sum()), page, Hkv, 128, generator=g, device=dev)
              .to(torch.bfloat16) for _ in range(2))
    q = torch.randn(int(new.sum()), Hq, 128, generator=g, device=dev).to(torch.bfloat16)
    cu = lambda n: torch.from_numpy(np.concatenate([[0], np.cumsum(n)]).astype(np.int32)).to(dev)
    got = paged_prefill_attention(q, kc, vc, torch.from_numpy(table).to(dev), cu(new), cu(total),
                                  128 ** -0.5)
    # every sequence on its own: one launch each, where there is nothing to order
    at = np.concatenate([[0], np.cumsum(new)])
    for i in range(batch):
        if new[i] == 0:
            continue
        one = paged_prefill_attention(q[at[i]:at[i + 1]].contiguous(), kc, vc,
                                      torch.from_numpy(table[i:i + 1].copy()).to(dev),
                                      cu(new[i:i + 1]), cu(total[i:i + 1]), 128 ** -0.5)
        assert torch.equal(got[at[i]:at[i + 1]], one), f"sequence {i}"


@pytest.mark.parametrize("batch,most,Hq,Hkv", [
    (72, 4, 28, 4), (70, 4, 28, 4),     # KV heads that do not fill the XCDs, around two rounds
    (169, 7, 6, 2), (61, 25, 32, 8),    # up to a block of tokens in the mean, some with two
    (140, 27, 32, 8), (165, 27, 32, 8), # the same at eight workgroups a CU and beyond
])
def test_paged_prefill_of_many_short_sequences(batch, most, Hq, Hkv):
    """Small or large workgroups: a sequence's bits are those it has alone."""
    print(f"case paged prefill, many short batch={batch} Hq={Hq}", flush=True)
    import torch
    from nanovllm_jax_amd import paged_prefill_attention
    rng = np.random.Generator(np.random.PCG64(batch))
    new = rng.integers(1, most + 1, batch)
    total = new + rng.integers(0, 200, batch)
    pages = -(-total // 32)
    ends = np.cumsum(pages)
    table = np.full((batch, int(pages.max())), -1, np.int32)
    for i, e in enumerate(ends):
        table[i, :pages[i]] = np.arange(e - pages[i], e)[::-1]
    dev = "cuda:0"
    g = torch.Generator(device=dev).manual_seed(batch)
    draw = lambda *shape: torch.randn(shape, generator=g, device=dev).to(torch.bfloat16)
    kc, vc = (draw(int(ends[-1]), 32, Hkv, 128) for _ in range(2))
    q = draw(int(new.sum()), Hq, 128)
    up = lambda x: torch.from_numpy(np.ascontiguousarray(x, np.int32)).to(dev)
    cu = lambda n: up(np.concatenate([[0], np.cumsum(n)]))
    got = paged_prefill_attention(q, kc, vc, up(table), cu(new), cu(total), 128 ** -0.5)
    at = np.concatenate([[0], np.cumsum(new)])
    for i in range(batch):
        one = paged_prefill_attention(q[at[i]:at[i + 1]].contiguous(), kc, vc, up(table[i:i + 1]),
                                      cu(new[i:i + 1]), cu(total[i:i + 1]), 128 ** -0.5)
        assert torch.equal(got[at[i]:at[i + 1]], one), f"sequence {i}"


@pytest.mark.parametrize("new,cached,Hq,Hkv,bs,splits", [
    ([1], [2000], 8, 8, 64, True),                    # one row, with parts for every ring of tiles
    ([30, 0, 17], [1500, 700, 31], 16, 8, 256, True),  # an empty sequence, tiles of one part
    ([5, 16, 40], [512, 480, 3000], 12, 2, 32, True),  # 16, 17 and 95 tiles, a group of 6
    ([100], [4097], 32, 2, 96, True),                 # a group of 16, pages that are no power of two
    ([300], [2000], 8, 4, 64, True),                  # parts that rows in front do not see
    ([20, 30, 9], [0, 5000, 1111], 4, 1, 64, True),   # no prefix beside a long one
    ([500], [4200], 32, 8, 256, True),                # larger workgroups in parts
    ([23, 0, 44, 37, 5, 31], [4300, 0, 100, 2000, 64, 4096], 64, 8, 64, True),   # ... tiles of one part
    ([400], [4100], 32, 32, 64, True),                # ... no group, three column groups in the last
    ([700], [1200], 64, 8, 64, False),                # enough workgroups without
    ([9], [256], 8, 2, 64, False),                    # nothing to cut
])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_paged_prefill_with_the_keys_in_parts(new, cached, Hq, Hkv, bs, splits, dtype):
    """Few rows behind long prefixes, their keys cut into parts and put together again, against
    the oracle and against the launch that walks all keys in one workgroup; nothing but live keys
    is read, and nothing is taken over from the workspace."""
    print(f"case keys in parts {new} {cached} Hq={Hq} Hkv={Hkv} bs={bs} {dtype}", flush=True)
    import torch
    from nanovllm_jax_amd import _lib
    from oracle.paged_attention_oracle import paged_prefill_attention_ref
    lens_k = [a + b for a, b in zip(new, cached)]
    q, kc, vc, bt, cu_q, cu_k = _paged_problem(60 + Hq + bs, lens_k, new, Hq, Hkv, bs)
    scale, dev, lib = 128 ** -0.5, "cuda:0", _lib.load()
    live = np.zeros(kc.shape[:2], bool)
    for i, n in enumerate(lens_k):
        live[bt[i, np.arange(n) // bs], np.arange(n) % bs] = True
    want = paged_prefill_attention_ref(q, kc, vc, bt, cu_q, cu_k, scale)
    kc[~live], vc[~live] = 0x7FC0, 0x7FC0             # NaN
    t = [bits_to_torch(x, dev) for x in (q, kc, vc)]
    if dtype == "f16":
        t = [x.half() for x in t]
    t += [torch.from_numpy(x).to(dev) for x in (bt, cu_q, cu_k)]
    sizes = (sum(new), len(new), Hq, Hkv)
    need = lib.nvj_paged_prefill_split_workspace_bytes(*sizes, bs, bt.shape[1], 0)
    assert (need > 0) == splits
    assert lib.nvj_paged_prefill_split_workspace_bytes(*sizes, bs, bt.shape[1], 512) == 0
    ws = torch.full((max(need, 16),), 0xFF, dtype=torch.uint8, device=dev)       # NaN
    stream = torch.cuda.current_stream().cuda_stream
    end = (scale, _lib.NVJ_DTYPE_BF16 if dtype == "bf16" else _lib.NVJ_DTYPE_F16)
    tail = (*sizes, 128, bs, bt.shape[1], kc.shape[0])
    out, whole = torch.full_like(t[0], 7.0), torch.empty_like(t[0])
    ptrs = [x.data_ptr() for x in t]
    if need:
        assert lib.nvj_paged_prefill_split_launch(stream, *ptrs, out.data_ptr(), ws.data_ptr(),
                                                  need - 1, *tail, 0, *end) == -4      # NVJ_ERR_WORKSPACE
    for _ in range(2):
        _lib.check(lib.nvj_paged_prefill_split_launch(stream, *ptrs, out.data_ptr(), ws.data_ptr(),
                                                      need, *tail, 0, *end), "split")
    _lib.check(lib.nvj_paged_prefill_attention_launch(stream, *ptrs, whole.data_ptr(), *tail, *end), "whole")
    torch.cuda.synchronize()
    if dtype == "bf16":
        assert_close_bf16(torch_to_bits(out), want, what="keys in parts")
    # each rounds its probabilities and its result to the 16-bit type
    tol = 2.0 ** -6 if dtype == "bf16" else 2.0 ** -9
    assert (out.float() - whole.float()).abs().max() <= tol * whole.float().abs().max()
    if not splits:
        assert torch.equal(out, whole)


@pytest.mark.parametrize("lens,Hq,Hkv,dtype,padding", [
    ([1], 8, 8, "bf16", 0),                       # one row: fewer pieces than threads
    ([0, 0, 0], 4, 2, "f16", 5),                  # rows that belong to no sequence only
    ([700], 16, 8, "bf16", 0),                    # the small workgroups
    ([3, 0, 130, 64, 17], 6, 2, "bf16", 9),       # rows behind the last offset are stored too
    ([250, 31, 0, 300] * 12, 32, 8, "f16", 0),    # shares of more than one batch
    ([90] * 60, 32, 8, "bf16", 1),                # 44 MB of output: past the L2s
    ([2100, 1], 8, 1, "bf16", 0),
    ([5, 9, 1] * 30, 32, 8, "f16", 3),            # shares of three or four rows of a head
    ([12, 0, 20] * 100, 32, 8, "bf16", 0),        # ... of six, over many rounds
    ([4, 1, 6] * 100, 64, 8, "bf16", 2),          # few tokens, many rounds: two launches
])
def test_prefill_with_the_store_in_the_launch(lens, Hq, Hkv, dtype, padding):
    """Caches and output bit for bit as the store's own launch and the attention's leave
    them, slots that are skipped or outside the caches among the rows."""
    print(f"case prefill with store Hq={Hq} Hkv={Hkv} {dtype} {len(lens)} prompts", flush=True)
    import torch
    from nanovllm_jax_amd import _lib
    lib, dev = _lib.load(), "cuda:0"
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}[dtype]
    code = {"bf16": _lib.NVJ_DTYPE_BF16, "f16": _lib.NVJ_DTYPE_F16}[dtype]
    g = torch.Generator(device=dev)
    g.manual_seed(len(lens) + Hq)
    rows, T = sum(lens), sum(lens) + padding
    q, k, v = (torch.randn(T, h, 128, generator=g, device=dev, dtype=dt) for h in (Hq, Hkv, Hkv))
    cu = torch.from_numpy(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)).to(dev)
    num_slots = T + 7
    slots = torch.randperm(num_slots, generator=g, device=dev)[:T].to(torch.int32)
    if T > 4:
        slots[T // 2], slots[T // 3], slots[1] = -1, num_slots, num_slots + 100
    caches = [torch.zeros(num_slots, Hkv, 128, dtype=dt, device=dev) for _ in range(4)]
    outs = [torch.zeros_like(q) for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.nvj_store_kvcache_launch(
        stream, k.data_ptr(), v.data_ptr(), caches[0].data_ptr(), caches[1].data_ptr(),
        slots.data_ptr(), T, Hkv, 128, num_slots, code, code, code), "store")
    _lib.check(lib.nvj_prefill_attention_launch(
        stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), cu.data_ptr(), cu.data_ptr(),
        outs[0].data_ptr(), T, len(lens), Hq, Hkv, 128, 128 ** -0.5, code), "attention")
    _lib.check(lib.nvj_prefill_attention_store_launch(
        stream, q.data_ptr(), k.data_ptr(), v.data_ptr(), cu.data_ptr(), cu.data_ptr(),
        outs[1].data_ptr(), slots.data_ptr(), caches[2].data_ptr(), caches[3].data_ptr(),
        num_slots, T, T, len(lens), Hq, Hkv, 128, 128 ** -0.5, code), "together")
    torch.cuda.synchronize()
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])
    assert torch.equal(outs[0][:rows], outs[1][:rows])
    assert not outs[1][rows:].any()               # rows of no sequence are left alone
    if rows > 0 and T > 4:
        want = k.double().cpu()
        live = (slots >= 0) & (slots < num_slots)
        assert torch.equal(caches[2][slots[live].long()].double().cpu(), want[live.cpu()])
