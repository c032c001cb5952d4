"""Prefill behind a cached prefix through the layer, where keys are cut into parts: what the
context says of the longest sequence, memory that is short, other streams, graphs and threads."""
from types import SimpleNamespace

import numpy as np
import pytest

from helpers import bits_to_torch, torch_to_bits

pytestmark = pytest.mark.gpu


def _call(new, cached, Hq=32, Hkv=8, bs=64, dtype="bf16", width=0, seed=1):
    """A layer, its q, k and v, the fields of a context, and the result of the oracle."""
    import torch
    from nanovllm_jax_amd import Attention
    from oracle.paged_attention_oracle import paged_prefill_attention_ref, store_kv_to_cache_ref
    rng = np.random.Generator(np.random.PCG64(seed))
    dev, total = "cuda:0", [a + b for a, b in zip(new, cached)]
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
    cu = lambda n: np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    draw = lambda *shape: torch.from_numpy(rng.standard_normal(shape, np.float32)).to(
        torch.bfloat16 if dtype == "bf16" else torch.float16)
    q, k, v = (draw(sum(new), h, 128) for h in (Hq, Hkv, Hkv))
    kc, vc = (draw(sum(pages) + 2, bs, Hkv, 128) for _ in range(2))
    flat = (-1, Hkv, 128)
    bits = [torch_to_bits(x) for x in (k, v, kc, vc)]
    wk, wv = store_kv_to_cache_ref(bits[0], bits[1], bits[2].reshape(flat), bits[3].reshape(flat),
                                   slots, negative_slots="skip")
    want = paged_prefill_attention_ref(torch_to_bits(q), wk.reshape(kc.shape), wv.reshape(vc.shape),
                                       table, cu(new), cu(total), 128 ** -0.5, return_f32=True,
                                       dtype=dtype)
    attn = Attention(Hq, 128, 128 ** -0.5, Hkv, bs)
    attn.set_kv_cache(kc.to(dev), vc.to(dev))
    up = lambda a: torch.from_numpy(a).to(dev)
    fields = dict(is_prefill=True, cu_seqlens_q=up(cu(new)), cu_seqlens_k=up(cu(total)),
                  slot_mapping=up(slots), block_tables=up(table))
    return attn, [x.to(dev) for x in (q, k, v)], fields, want


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
