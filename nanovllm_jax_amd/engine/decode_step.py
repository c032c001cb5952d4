"""Whole-model decode and prefill steps around the HIP attention path.

A step (embedding, per layer the projections, norms, RoPE, KV store and attention, the tied
LM head) is one native call where that is the faster way and the model is one it is built
for: ``nvj_decoder_step_launch``, all of it in kernels of this package.  Otherwise it goes
the long way: the same attention and element-wise launches with ``torch`` products
(hipBLASLt GEMMs) between them.  Greedy pick is ``torch`` in both.  Written from the
architecture the reference describes: ``models/qwen3.py:130-172`` (attention block: fused
QKV, per-head QK-RMSNorm when there is no QKV bias, RoPE, attention, output projection),
``:285-318`` (pre-norm decoder layer with fused residual), ``:366-393`` (stack
+ final norm), ``:472-491`` (tied LM head), ``layers/layernorm.py:31-79``,
``layers/rotary_embedding.py:13-37,50-106``, ``layers/activation.py:22-33``.
Cache allocation, wiring and the per-step metadata follow
``engine/model_runner.py:140-204, 225-246, 334-376``.

Weights are random (N(0, 0.02), bf16); greedy = argmax of the logits, the
temperature -> 0 limit of the reference's Gumbel-max sampler
(``layers/sampler.py:39-48``).
"""
from __future__ import annotations

import ctypes
from dataclasses import dataclass
from operator import itemgetter

import numpy as np
import torch
import torch.nn.functional as F

from .. import _lib
from ..layers.activation import silu_and_mul
from ..layers.attention import Attention
from ..layers.layernorm import rms_norm
from ..layers.paged_attention import (DecodeWorkspace, choose_split, paged_attention,
                                      paged_decode_workspace_bytes)
from ..layers.prefill_attention import packed_qkv_attention, paged_prefill_attention
from ..layers.qk_rope_store import qk_norm_rope_store
from ..utils.context import AttentionContext, create_decode_context, create_prefill_context

# A step is one native call (nvj_decoder_step_launch) up to this many token rows and where
# that is the faster way; otherwise, and for models the call is not built for, it is library
# GEMMs with the element-wise launches between them.
_NATIVE_STEP_ROWS = 1 << 18
_LAYER_WEIGHTS = itemgetter("qkv", "o", "gate_up", "down", "ln1", "ln2", "q_norm", "k_norm")

__all__ = ["DecodeModelConfig", "DecodeStepRunner", "prepare_block_tables", "prepare_decode",
           "prepare_prefill", "advance_decode"]


@dataclass
class DecodeModelConfig:
    """Qwen3-0.6B shape by default."""
    num_layers: int = 28
    hidden_size: int = 1024
    num_heads: int = 16
    num_kv_heads: int = 8
    head_dim: int = 128
    intermediate_size: int = 3072
    vocab_size: int = 151936
    rms_norm_eps: float = 1e-6
    rope_theta: float = 1e6
    max_position: int = 4096
    block_size: int = 256
    num_kvcache_blocks: int = 512


def _native_step_pays(tokens: int, hidden: int, q_width: int, kv_width: int,
                      intermediate: int) -> bool:
    """Whether the native step is at least as fast as library GEMMs for these sizes.

    It saves launches, the passes of the element-wise stages and host work per launch;
    the library's products are the faster ones where they are large.  Measured per layer,
    native against library (decode replayed from a graph, prefill eager), us:

    ========================  =====================================================
    hidden (intermediate)     rows: native / library
    ========================  =====================================================
    1024 (3072)               4: 37 / 59, 128: 46 / 64, 800: 72 / 161, 4400: 216 / 240,
                              8000: 348 / 339, 16000: 643 / 589
    2048 (6144)               4: 76 / 90, 64: 78 / 94, 200: 102 / 163, 600: 151 / 165,
                              1200: 203 / 199, 8000: 762 / 672
    2048 (11008)              48: 98 / 114, 96: 124 / 118, 200: 134 / 162, 600: 212 / 197
    2560 (9728)               4: 104 / 135, 24: 113 / 114, 64: 128 / 125, 96: 144 / 137,
                              1200: 368 / 344
    4096 (12288)              4: 143 / 149, 24: 156 / 158, 64: 174 / 162, 400: 304 / 261
    5120 (25600)              4: 286 / 326, 24: 317 / 356, 128: 497 / 439
    8192 (29568)              4: 455 / 423, 64: 499 / 484, 1200: 2042 / 1613
    ========================  =====================================================
    """
    products = tokens * (hidden * (2 * q_width + 2 * kv_width) + 3 * hidden * intermediate)
    if hidden <= 1024:
        return products <= 100e9
    if hidden <= 2048:
        return tokens <= 64 or (tokens > 128 and products <= 40e9)
    return hidden <= 5120 and tokens <= 24


class _Upload:
    """The stream the tensors of a context are being uploaded on, and an event behind them.
    Copies of the context share it; a pickled one is read back with its values in place."""
    __slots__ = ("stream", "event")

    def __init__(self, device):
        self.stream = torch.cuda.current_stream(device)
        self.event = self.stream.record_event()

    def __deepcopy__(self, memo):
        return self

    def __reduce__(self):
        self.event.synchronize()
        return type(None), ()


def prepare_block_tables(block_tables: list[list[int]]) -> np.ndarray:
    """Rows padded with -1 to the longest table (``engine/model_runner.py:225-246``)."""
    width = max(len(t) for t in block_tables)
    out = np.full((len(block_tables), width), -1, dtype=np.int32)
    for i, t in enumerate(block_tables):
        out[i, :len(t)] = t
    return out


def prepare_decode(last_tokens, seq_lens, block_tables, block_size):
    """Host filler of one decode step (``engine/model_runner.py:334-376``):
    ``positions = len - 1``, ``context_lens = len``,
    ``slot = block_table[-1] * block_size + last_block_num_tokens - 1``."""
    n = len(seq_lens)
    input_ids = np.asarray(last_tokens, dtype=np.int32)
    positions = np.empty(n, np.int32)
    context_lens = np.empty(n, np.int32)
    slot_mapping = np.empty(n, np.int32)
    for i, (length, table) in enumerate(zip(seq_lens, block_tables)):
        positions[i] = length - 1
        context_lens[i] = length
        last_block_tokens = length - (len(table) - 1) * block_size
        slot_mapping[i] = table[-1] * block_size + last_block_tokens - 1
    return input_ids, positions, context_lens, slot_mapping, prepare_block_tables(block_tables)


def prepare_prefill(token_lists, block_tables, block_size, num_cached_tokens=None):
    """Host filler of one prefill step (``engine/model_runner.py:248-332``): packed
    ``input_ids`` and ``positions`` of the tokens that are not cached yet,
    ``cu_seqlens_q`` over those, ``cu_seqlens_k`` over whole sequences, and per
    sequence the slots of the new tokens, page by page (:300-309).
    ``num_cached_tokens[i]`` leading tokens of sequence i already sit in the cache
    (0 everywhere by default); unlike the reference's block-granular prefix cache
    it may be any count.  Returns ``(input_ids, positions, cu_seqlens_q,
    cu_seqlens_k, slot_mapping, max_seqlen_q, max_seqlen_k)``."""
    lens = [len(t) for t in token_lists]
    cached = list(num_cached_tokens) if num_cached_tokens is not None else [0] * len(lens)
    new = [n - c for n, c in zip(lens, cached)]
    cu_q = np.zeros(len(lens) + 1, np.int32)
    cu_q[1:] = np.cumsum(new)
    cu_k = np.zeros(len(lens) + 1, np.int32)
    cu_k[1:] = np.cumsum(lens)
    input_ids = (np.concatenate([np.asarray(t[c:], np.int32) for t, c in zip(token_lists, cached)])
                 if lens else np.zeros(0, np.int32))
    positions = (np.concatenate([np.arange(c, n, dtype=np.int32) for n, c in zip(lens, cached)])
                 if lens else np.zeros(0, np.int32))
    slots = []
    for n, c, table in zip(lens, cached, block_tables):
        pos = np.arange(c, n)
        slots.append((np.asarray(table, np.int64)[pos // block_size] * block_size +
                      pos % block_size).astype(np.int32))
    slot_mapping = np.concatenate(slots) if slots else np.zeros(0, np.int32)
    return (input_ids, positions, cu_q, cu_k, slot_mapping, max(new) if new else 0,
            max(lens) if lens else 0)


def advance_decode(next_tokens, input_ids, positions, context: AttentionContext, block_size):
    """Advance the device-resident metadata of a decode batch by one step, in
    place: every active sequence grows by its ``next_tokens`` entry and
    ``input_ids / positions / context.context_lens / context.slot_mapping`` get
    the values ``prepare_decode`` would compute for the grown sequences
    (``engine/model_runner.py:334-376``), without a host round trip.
    ``context.block_tables`` must already hold the page a sequence is about to
    enter."""
    lib = _lib.load()
    bt = context.block_tables
    for name, t in (("next_tokens", next_tokens), ("input_ids", input_ids),
                    ("positions", positions), ("context_lens", context.context_lens),
                    ("slot_mapping", context.slot_mapping), ("block_tables", bt)):
        if not (isinstance(t, torch.Tensor) and t.is_cuda and t.is_contiguous()):
            raise ValueError(f"{name} must be a contiguous GPU tensor")
        if name != "next_tokens" and t.dtype != torch.int32:
            raise ValueError(f"{name} must be int32, got {t.dtype}")
    if next_tokens.dtype not in (torch.int32, torch.int64):
        raise ValueError("next_tokens must be int32 or int64")
    batch = input_ids.shape[0]
    for name, t in (("next_tokens", next_tokens), ("positions", positions),
                    ("context_lens", context.context_lens),
                    ("slot_mapping", context.slot_mapping)):
        if t.shape != (batch,):
            raise ValueError(f"{name} must have shape [{batch}]")
    if bt.dim() != 2 or bt.shape[0] != batch:
        raise ValueError("block_tables must be [batch, max_blocks]")
    with torch.cuda.device(input_ids.device):
        stream = torch.cuda.current_stream(input_ids.device).cuda_stream
        code = lib.nvj_advance_decode_launch(
            stream, next_tokens.data_ptr(), next_tokens.element_size(), input_ids.data_ptr(),
            positions.data_ptr(), context.context_lens.data_ptr(),
            context.slot_mapping.data_ptr(), bt.data_ptr(), batch, bt.shape[1], int(block_size))
    _lib.check(code, "nvj_advance_decode_launch")


class DecodeStepRunner:
    """Owns random weights, the KV cache ``[2, L, NB, bs, Hkv, D]`` bf16 and one
    ``Attention`` per layer; ``step`` runs one decode step for a batch."""

    def __init__(self, cfg: DecodeModelConfig, device="cuda:0", seed: int = 0,
                 fill_cache: bool = True, fused_qk_rope_store: bool = True,
                 fused_layer_glue: bool = True):
        self.cfg = cfg
        # True: RMSNorm (+ residual add) and SiLU-and-multiply as one HIP launch
        # each; False: the same stages as chains of torch kernels
        self.fused_layer_glue = fused_layer_glue
        # True: one HIP launch for QK-RMSNorm + RoPE + KV store; False: the
        # reference's op-by-op chain in torch followed by the plain store
        self.fused_qk_rope_store = fused_qk_rope_store
        self.device = torch.device(device)
        g = torch.Generator(device=self.device)
        g.manual_seed(seed)
        c = cfg

        def w(*shape):
            return (torch.randn(shape, generator=g, device=self.device, dtype=torch.float32)
                    * 0.02).to(torch.bfloat16)

        qkv_out = (c.num_heads + 2 * c.num_kv_heads) * c.head_dim
        self.embed = w(c.vocab_size, c.hidden_size)            # tied with the LM head
        self.layers = []
        for _ in range(c.num_layers):
            self.layers.append(dict(
                ln1=torch.ones(c.hidden_size, device=self.device),    # fp32, layernorm.py:29
                ln2=torch.ones(c.hidden_size, device=self.device),
                qkv=w(qkv_out, c.hidden_size),
                o=w(c.hidden_size, c.num_heads * c.head_dim),
                q_norm=torch.ones(c.head_dim, device=self.device),
                k_norm=torch.ones(c.head_dim, device=self.device),
                gate_up=w(2 * c.intermediate_size, c.hidden_size),
                down=w(c.hidden_size, c.intermediate_size)))
        self.final_norm = torch.ones(c.hidden_size, device=self.device)
        inv_freq = 1.0 / (c.rope_theta ** (torch.arange(0, c.head_dim, 2, dtype=torch.float32,
                                                        device=self.device) / c.head_dim))
        freqs = torch.outer(torch.arange(c.max_position, dtype=torch.float32,
                                         device=self.device), inv_freq)
        self.cos_sin = torch.cat([freqs.cos(), freqs.sin()], dim=-1)     # [max_pos, D] f32
        # KV cache, engine/model_runner.py:176,190
        shape = (2, c.num_layers, c.num_kvcache_blocks, c.block_size, c.num_kv_heads, c.head_dim)
        self.kv_cache = torch.zeros(shape, dtype=torch.bfloat16, device=self.device)
        if fill_cache:
            for layer in range(c.num_layers):
                for kv in range(2):
                    self.kv_cache[kv, layer] = torch.randn(
                        shape[2:], generator=g, device=self.device,
                        dtype=torch.float32).to(torch.bfloat16)
        self.attn = []
        for layer in range(c.num_layers):                        # _wire_kv_cache, :195-204
            a = Attention(c.num_heads, c.head_dim, c.head_dim ** -0.5, c.num_kv_heads,
                          c.block_size)
            a.set_kv_cache(self.kv_cache[0, layer], self.kv_cache[1, layer])
            self.attn.append(a)
        self._graph = None
        self._eager_ws = None
        self._eager_ws_shapes = set()

    # -- small torch pieces -------------------------------------------------
    def _rms(self, x, weight, residual=None):
        """RMSNorm, optionally fused with the residual add (layernorm.py:31-79).
        The HIP launch norms the unrounded fp32 sum as the reference does and
        updates the residual in place; the torch chain rounds the sum to the
        model dtype first (one bf16 rounding apart)."""
        if self.fused_layer_glue and x.dim() == 2:
            if residual is None:
                return rms_norm(x, weight, self.cfg.rms_norm_eps), x
            return rms_norm(x, weight, self.cfg.rms_norm_eps, residual, residual_out=residual)
        if residual is not None:
            x = (x.float() + residual.float()).to(x.dtype)
        return F.rms_norm(x, (x.shape[-1],), weight.to(x.dtype), self.cfg.rms_norm_eps), x

    def _silu_mul(self, gate_up):
        """SiLU(gate) * up of the fused projection (activation.py:22-33)."""
        if self.fused_layer_glue:
            return silu_and_mul(gate_up)
        gate, up = gate_up.chunk(2, dim=-1)
        return F.silu(gate) * up

    def _rope(self, x, cos, sin):
        """x bf16 [T, H, D]; result float32 like the reference's promotion
        (rotary_embedding.py:31-37)."""
        x1, x2 = x.chunk(2, dim=-1)
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], dim=-1)

    def _native(self):
        """The model as the native step wants it: ``(model, layers, the memory of
        layers)``, or None when it is not one that step is built for.  Everything the
        long way reads on a step is read here on every step too, shapes and types
        included."""
        c, n = self.cfg, min(len(self.layers), len(self.attn))
        if n == 0:
            return None
        scale, page = self.attn[0].scale, self.attn[0].block_size
        tensors = [self.embed, self.final_norm, self.cos_sin]
        for lw, a in zip(self.layers, self.attn):
            if a.scale != scale or a.block_size != page:
                return None
            tensors += _LAYER_WEIGHTS(lw)
            tensors += (a.k_cache, a.v_cache)
        found = _lib.load_host().decoder_layers(tensors, c.num_heads, c.num_kv_heads, c.head_dim,
                                                self.embed.device.index)
        if found is None or found[6] != page:
            return None
        layers, hidden, intermediate, vocab, max_position, num_blocks, _ = found
        model = _lib.DecoderModel(
            self.embed.data_ptr(), self.final_norm.data_ptr(), self.cos_sin.data_ptr(), n, hidden,
            c.num_heads, c.num_kv_heads, c.head_dim, intermediate, vocab, max_position, page,
            num_blocks, c.rms_norm_eps, scale)
        return model, ctypes.cast(layers, ctypes.POINTER(_lib.DecoderLayer)), layers

    def _native_forward(self, input_ids, positions, context: AttentionContext):
        """The whole step as one native call, or None when it has to go the long way."""
        tokens = input_ids.shape[0]
        sl, bt = context.slot_mapping, context.block_tables
        prefill = bool(context.is_prefill)
        ints = [input_ids, positions, sl]
        ints += [context.cu_seqlens_q, context.cu_seqlens_k] if prefill else [context.context_lens]
        ws0 = self.attn[0].workspace
        if not (0 < tokens <= _NATIVE_STEP_ROWS and self.fused_qk_rope_store
                and self.fused_layer_glue and (prefill or bt is not None)
                and (ws0 is None or isinstance(ws0, DecodeWorkspace))
                and all(a.workspace is ws0 for a in self.attn)):
            return None
        if bt is not None:
            ints.append(bt)
        for t in ints:
            if t is None or t.dtype != torch.int32 or not t.is_cuda or not t.is_contiguous() \
                    or t.device != self.embed.device:
                return None
        sequences = context.cu_seqlens_q.numel() - 1 if prefill else tokens
        if positions.shape != (tokens,) or sl.shape != (tokens,) or input_ids.dim() != 1 or \
                (bt is not None and (bt.dim() != 2 or bt.shape[0] != sequences
                                     or bt.shape[1] == 0)):
            return None
        if prefill:
            # any other count of rows, or indices from the host, as tensor indexing takes them
            last = context.last_token_indices
            offsets = (context.cu_seqlens_q.shape, context.cu_seqlens_k.shape)
            if offsets != ((sequences + 1,),) * 2 or sequences <= 0 or \
                    not isinstance(last, torch.Tensor) or last.shape != (sequences,) or \
                    last.dtype not in (torch.int32, torch.int64) or \
                    last.device != self.embed.device:
                return None
        elif context.context_lens.shape != (tokens,):
            return None
        built = self._native()
        if built is None:
            return None
        model, layers, _memory = built
        if not _native_step_pays(tokens, model.hidden, model.num_heads * model.head_dim,
                                 model.num_kv_heads * model.head_dim, model.intermediate):
            return None
        lib, dev = _lib.load(), self.embed.device
        need = lib.nvj_decoder_step_workspace_bytes(ctypes.byref(model), tokens, sequences)
        if need == 0:
            return None
        ws = None if prefill else ws0 or self._eager_workspace(context)
        if ws is not None and not ws.buffer.device == ws.counters.device == dev:
            return None
        b = _lib.DecoderBatch(num_tokens=tokens, num_sequences=sequences, is_prefill=int(prefill))
        b.input_ids, b.positions, b.slot_mapping = (input_ids.data_ptr(), positions.data_ptr(),
                                                    sl.data_ptr())
        if bt is not None:
            b.block_tables, b.max_blocks = bt.data_ptr(), bt.shape[1]
        if prefill:
            b.cu_seqlens_q, b.cu_seqlens_k = (context.cu_seqlens_q.data_ptr(),
                                              context.cu_seqlens_k.data_ptr())
            if last.dtype == torch.int64:
                last = last.clamp(-(1 << 31), (1 << 31) - 1).to(torch.int32)
            last = last.contiguous()
            b.last_token_indices = last.data_ptr()
        else:
            b.context_lens, b.chunk = context.context_lens.data_ptr(), int(context.decode_split)
            b.partials, b.partial_bytes = ws.buffer.data_ptr(), ws.buffer.numel()
            if b.chunk == 0:
                counters = ws._counters_for(4 * (1 + sequences * self.cfg.num_heads))
                b.counters, b.counter_bytes = counters.data_ptr(), counters.numel() * 4
                b.clear_counters = int(ws._clear_next)
        logits = torch.empty((sequences, model.vocab), dtype=torch.bfloat16, device=dev)
        b.logits = logits.data_ptr()
        scratch = torch.empty(need, dtype=torch.uint8, device=dev)
        with torch.cuda.device(dev):
            code = lib.nvj_decoder_step_launch(
                torch.cuda.current_stream(dev).cuda_stream, ctypes.byref(model), layers,
                ctypes.byref(b), scratch.data_ptr(), need)
        _lib.check(code, "nvj_decoder_step_launch")
        if b.clear_counters:
            ws._clear_next = False
        return logits

    def _wait_for_inputs(self, context: AttentionContext):
        """Inputs are uploaded without a wait, on the stream that was current then; another
        stream has to wait for them.  (A capture begins behind a device synchronisation.)"""
        here = torch.cuda.current_stream(self.device)
        if here != context.uploaded.stream and not torch.cuda.is_current_stream_capturing():
            here.wait_event(context.uploaded.event)

    def forward(self, input_ids, positions, context: AttentionContext):
        if context.uploaded is not None:
            self._wait_for_inputs(context)
        logits = self._native_forward(input_ids, positions, context)
        if logits is not None:
            return logits
        c = self.cfg
        h = F.embedding(input_ids.long(), self.embed)
        residual = None
        if not self.fused_qk_rope_store:
            cos, sin = self.cos_sin[positions.long()][:, None, :].chunk(2, dim=-1)
        qs, ks = c.num_heads * c.head_dim, c.num_kv_heads * c.head_dim
        for lw, attn in zip(self.layers, self.attn):
            if residual is None:
                h, residual = self._rms(h, lw["ln1"])
            else:
                h, residual = self._rms(h, lw["ln1"], residual)
            qkv = F.linear(h, lw["qkv"])
            if self.fused_qk_rope_store:
                packed = context.is_prefill and context.block_tables is None
                q = qk_norm_rope_store(qkv, positions, self.cos_sin, lw["q_norm"], lw["k_norm"],
                                       c.rms_norm_eps, attn.k_cache, attn.v_cache,
                                       context.slot_mapping, c.num_heads, c.num_kv_heads,
                                       c.head_dim, in_place=packed)
                if packed:
                    o = packed_qkv_attention(q, context.cu_seqlens_q, context.cu_seqlens_k,
                                             c.num_heads, c.num_kv_heads, c.head_dim, attn.scale)
                elif context.is_prefill:
                    # prompt rows behind a cached prefix: keys and values, the rows the
                    # fused launch just stored included, come from the paged cache
                    o = paged_prefill_attention(q, attn.k_cache, attn.v_cache,
                                                context.block_tables, context.cu_seqlens_q,
                                                context.cu_seqlens_k, attn.scale)
                else:
                    o = paged_attention(q, attn.k_cache, attn.v_cache, context.block_tables,
                                        context.context_lens, attn.scale, attn.block_size,
                                        chunk=context.decode_split,
                                        workspace=attn.workspace or
                                        self._eager_workspace(context))
                h = F.linear(o.reshape(-1, qs), lw["o"])
                h, residual = self._rms(h, lw["ln2"], residual)
                h = F.linear(self._silu_mul(F.linear(h, lw["gate_up"])), lw["down"])
                continue
            q, k, v = qkv.split([qs, ks, ks], dim=-1)
            q = q.reshape(-1, c.num_heads, c.head_dim)
            k = k.reshape(-1, c.num_kv_heads, c.head_dim)
            v = v.reshape(-1, c.num_kv_heads, c.head_dim).contiguous()
            q, _ = self._rms(q, lw["q_norm"])
            k, _ = self._rms(k, lw["k_norm"])
            q = self._rope(q, cos, sin)                 # f32
            k = self._rope(k, cos, sin).contiguous()    # f32, the store rounds it to bf16
            o = attn(q.to(torch.bfloat16).contiguous(), k, v, context)
            h = F.linear(o.reshape(-1, qs), lw["o"])
            h, residual = self._rms(h, lw["ln2"], residual)
            h = F.linear(self._silu_mul(F.linear(h, lw["gate_up"])), lw["down"])
        h, _ = self._rms(h, self.final_norm, residual)
        if context.is_prefill:                           # only the last token of each prompt
            h = h[context.last_token_indices.long()]     # (models/qwen3.py:472-491)
        return F.linear(h, self.embed)                   # logits [T or batch, vocab]

    # -- one decode step ------------------------------------------------------
    def make_inputs(self, last_tokens, seq_lens, block_tables):
        ids, pos, ctx, slots, bt = prepare_decode(last_tokens, seq_lens, block_tables,
                                                  self.cfg.block_size)
        self._check_ids(ids)
        # the lengths are host integers here, as in the reference's filler: pick the split
        split = choose_split(ctx, self.cfg.num_kv_heads, self.cfg.num_heads)
        d_ids, d_pos, d_ctx, d_slots, d_bt = self._upload(ids, pos, ctx, slots, bt)
        context = create_decode_context(d_ctx, d_slots, d_bt, split)
        context.uploaded = _Upload(self.device)
        return d_ids, d_pos, context

    def _check_ids(self, ids):
        """Host ids outside the vocabulary are an error here; ids that a caller writes
        into device tensors give rows of NaN."""
        if ids.size and int(ids.view(np.uint32).max()) >= self.embed.shape[0]:
            raise ValueError(f"token ids must be in [0, {self.embed.shape[0]})")

    def _upload(self, *arrays):
        """int32 host arrays as device tensors, in one copy that nobody waits for: they
        are laid out behind each other in a pinned block (which torch's host allocator
        hands out again only when the copy is done) and come back as views of one
        device block.  A copy from pageable memory, one per array, would wait each time
        for everything in front of it on the stream."""
        at, total = [], 0
        for a in arrays:
            at.append(total)
            total += -(-a.size // 64) * 64          # 256-byte pieces
        host = torch.empty(max(total, 1), dtype=torch.int32, pin_memory=True)
        flat = host.numpy()
        for a, o in zip(arrays, at):
            flat[o:o + a.size] = a.reshape(-1)
        block = torch.empty(max(total, 1), dtype=torch.int32, device=self.device)
        block.copy_(host, non_blocking=True)
        return [block[o:o + a.size].view(a.shape) for a, o in zip(arrays, at)]

    def make_prefill_inputs(self, token_lists, block_tables, num_cached_tokens=None):
        """Prefill inputs; with ``num_cached_tokens`` the context carries the block
        tables (as the reference's does when a prefix is cached,
        ``engine/model_runner.py:309-312``) and attention reads keys and values
        from the paged cache."""
        ids, pos, cu_q, cu_k, slots, max_q, max_k = prepare_prefill(
            token_lists, block_tables, self.cfg.block_size, num_cached_tokens)
        self._check_ids(ids)
        tables = ([prepare_block_tables(block_tables)] if num_cached_tokens is not None else [])
        d_ids, d_pos, d_cu_q, d_cu_k, d_slots, *bt = self._upload(ids, pos, cu_q, cu_k, slots,
                                                                  *tables)
        context = create_prefill_context(d_cu_q, d_cu_k, max_q, max_k, d_slots,
                                         block_tables=bt[0] if bt else None)
        context.uploaded = _Upload(self.device)     # (behind last_token_indices too)
        return d_ids, d_pos, context

    def step(self, input_ids, positions, context):
        """Eager decode step: logits -> greedy token ids [batch] int64."""
        return self.forward(input_ids, positions, context).argmax(dim=-1)

    def _eager_workspace(self, context):
        """The split workspace of the eager steps (one stream), grown on demand."""
        batch, max_blocks = context.block_tables.shape
        key = (batch, max_blocks, int(context.decode_split))
        if key not in self._eager_ws_shapes:
            ws = self._new_workspace(*key)
            if self._eager_ws is None or ws.buffer.numel() > self._eager_ws.buffer.numel():
                self._eager_ws = ws
            self._eager_ws_shapes.add(key)
        return self._eager_ws

    def _new_workspace(self, batch, max_blocks, decode_split):
        """A split workspace for all layers of one step (they run one after the
        other on one stream), large enough for the balanced split and for the
        split the context asks for; its counters are zero from the start."""
        c = self.cfg
        with torch.cuda.device(self.device):
            need = max(paged_decode_workspace_bytes(batch, c.num_heads, c.head_dim, max_blocks,
                                                    c.block_size, c.num_kv_heads, chunk)
                       for chunk in {0, int(decode_split)})
        return DecodeWorkspace(need, self.device)

    def _capture(self, input_ids, positions, context, body, warmups):
        """Record ``body()`` into a HIP graph.  The graph gets a split workspace of
        its own, which stays alive with the returned closure and is never handed
        to an eager call: a replay can then rely on counters that nothing but
        its own launches has touched, whatever eager steps (of any batch size)
        or further captures run in between."""
        batch, max_blocks = context.block_tables.shape
        graph_ws = self._new_workspace(batch, max_blocks, context.decode_split)
        eager_ws = [a.workspace for a in self.attn]
        for a in self.attn:
            a.workspace = graph_ws
        try:
            # warm every library handle on a side stream; a warm-up step writes the
            # K/V rows of the current step, which the captured step rewrites with
            # the same values, and does not touch the metadata
            s = torch.cuda.Stream(self.device)
            s.wait_stream(torch.cuda.current_stream(self.device))
            with torch.cuda.stream(s):
                for _ in range(warmups):
                    self.step(input_ids, positions, context)
            torch.cuda.current_stream(self.device).wait_stream(s)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = body()
        finally:
            for a, ws in zip(self.attn, eager_ws):
                a.workspace = ws
        self._graph = graph

        def replay():
            graph.replay()
            return out
        replay.workspace = graph_ws      # keeps it alive; also lets a caller check() it
        return replay

    def capture(self, input_ids, positions, context):
        """Capture the whole step in one HIP graph over static input buffers;
        returns ``replay() -> token ids`` (the inputs may be updated in place
        between replays)."""
        return self._capture(input_ids, positions, context,
                             lambda: self.step(input_ids, positions, context), 2)

    def capture_generation(self, input_ids, positions, context):
        """Capture step + metadata advance in one HIP graph: every replay decodes
        one token per sequence and leaves ``input_ids / positions / context``
        ready for the next replay, with nothing but block-table maintenance left
        to the host.  Returns ``replay() -> token ids of that step``."""
        def body():
            out = self.step(input_ids, positions, context)
            advance_decode(out, input_ids, positions, context, self.cfg.block_size)
            return out
        return self._capture(input_ids, positions, context, body, 1)
