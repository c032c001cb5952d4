"""ctypes binding of the C ABI declared in ``include/nvj_paged_attn.h``.

The library is loaded from ``nanovllm_jax_amd/_native/``; it is never built
here.  A missing library is an error: there is no CPU or PyTorch fallback for
this path.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
import threading

_LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_native",
                         "libnvj_paged_attn.so")

NVJ_ABI_VERSION = 3
NVJ_DTYPE_BF16 = 0
NVJ_DTYPE_F32 = 1
NVJ_DTYPE_F16 = 2

_c = ctypes


class DecoderModel(ctypes.Structure):
    """``nvj_decoder_model``."""
    _fields_ = [(n, _c.c_void_p) for n in ("embed", "final_norm", "cos_sin")] + [
        (n, _c.c_int32) for n in ("num_layers", "hidden", "num_heads", "num_kv_heads", "head_dim",
                                  "intermediate", "vocab", "max_position", "block_size",
                                  "num_blocks")] + [("eps", _c.c_float), ("scale", _c.c_float)]


class DecoderLayer(ctypes.Structure):
    """``nvj_decoder_layer``."""
    _fields_ = [(n, _c.c_void_p) for n in ("qkv", "o", "gate_up", "down", "ln1", "ln2", "q_norm",
                                           "k_norm", "k_cache", "v_cache")]


class DecoderBatch(ctypes.Structure):
    """``nvj_decoder_batch``."""
    _fields_ = [(n, _c.c_void_p) for n in (
        "input_ids", "positions", "slot_mapping", "context_lens", "block_tables", "cu_seqlens_q",
        "cu_seqlens_k", "last_token_indices")] + [
        ("partials", _c.c_void_p), ("partial_bytes", _c.c_size_t), ("counters", _c.c_void_p),
        ("counter_bytes", _c.c_size_t), ("logits", _c.c_void_p)] + [
        (n, _c.c_int32) for n in ("num_tokens", "num_sequences", "max_blocks", "chunk",
                                  "is_prefill", "clear_counters")]


# every symbol include/nvj_paged_attn.h declares: name -> (restype, argtypes)
SYMBOLS = {
    "nvj_error_string": (_c.c_char_p, [_c.c_int]),
    "nvj_abi_version": (_c.c_int, []),
    "nvj_store_kvcache_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_int32]),
    "nvj_store_kvcache_rows_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_size_t]),
    "nvj_paged_decode_default_chunk": (_c.c_int32, [_c.c_int32] * 4),
    "nvj_paged_decode_whole_sequence_workgroups": (_c.c_int32, [_c.c_int32] * 3),
    "nvj_paged_decode_workspace_bytes": (_c.c_size_t, [_c.c_int32] * 7),
    "nvj_paged_decode_counter_bytes": (_c.c_size_t, [_c.c_int32] * 3),
    "nvj_paged_decode_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p, _c.c_void_p, _c.c_size_t,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_int32, _c.c_float, _c.c_int32, _c.c_int32]),
    "nvj_paged_decode_launch_phases": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p, _c.c_void_p, _c.c_size_t,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_int32, _c.c_float, _c.c_int32, _c.c_int32, _c.c_uint32]),
    "nvj_paged_decode_launch_counters": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p, _c.c_void_p, _c.c_size_t, _c.c_void_p, _c.c_size_t,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_int32, _c.c_float, _c.c_int32, _c.c_uint32]),
    "nvj_paged_decode_store_takes": (_c.c_int32, [_c.c_int32] * 8),
    "nvj_paged_decode_store_launch": (_c.c_int, [_c.c_void_p] * 11 + [
        _c.c_size_t, _c.c_void_p, _c.c_size_t] + [_c.c_int32] * 7 + [_c.c_float] +
        [_c.c_int32] * 4),
    "nvj_paged_decode_counters_reset": (_c.c_int, [_c.c_void_p, _c.c_void_p, _c.c_size_t]),
    "nvj_paged_decode_library_counters": (_c.c_int, [_c.POINTER(_c.c_void_p),
                                                     _c.POINTER(_c.c_size_t)]),
    "nvj_paged_decode_null_stream_counters": (_c.c_int, [_c.POINTER(_c.c_void_p),
                                                         _c.POINTER(_c.c_size_t)]),
    "nvj_paged_decode_static_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_int32, _c.c_float, _c.c_int32]),
    "nvj_qk_norm_rope_store_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_void_p,
        _c.c_void_p, _c.c_float, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int64]),
    "nvj_qk_norm_rope_rows_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_void_p,
        _c.c_void_p, _c.c_float, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int64,
        _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_int64]),
    "nvj_advance_decode_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p, _c.c_int32, _c.c_int32, _c.c_int32]),
    "nvj_prefill_attention_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_float, _c.c_int32]),
    "nvj_prefill_attention_rows_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_void_p,
        _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32, _c.c_int32,
        _c.c_float, _c.c_int32]),
    "nvj_prefill_attention_store_launch": (_c.c_int, [
        _c.c_void_p] * 10 + [_c.c_int64] + [_c.c_int32] * 6 + [_c.c_float, _c.c_int32]),
    "nvj_paged_prefill_attention_launch": (_c.c_int, [
        _c.c_void_p] * 8 + [_c.c_int32] * 8 + [_c.c_float, _c.c_int32]),
    "nvj_paged_prefill_split_workspace_bytes": (_c.c_size_t, [_c.c_int32] * 7),
    "nvj_paged_prefill_split_launch": (_c.c_int, [
        _c.c_void_p] * 9 + [_c.c_size_t] + [_c.c_int32] * 9 + [_c.c_float, _c.c_int32]),
    "nvj_add_rms_norm_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_float, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_int32]),
    "nvj_silu_and_mul_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_int64, _c.c_void_p, _c.c_int32, _c.c_int32]),
    "nvj_linear_launch": (_c.c_int, [_c.c_void_p] * 4 + [_c.c_int32] * 5),
    "nvj_qkv_linear_launch": (_c.c_int, [
        _c.c_void_p, _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int32, _c.c_void_p, _c.c_void_p,
        _c.c_int32, _c.c_void_p, _c.c_void_p, _c.c_float, _c.c_void_p, _c.c_void_p, _c.c_void_p,
        _c.c_void_p, _c.c_void_p, _c.c_int32, _c.c_int32, _c.c_int64, _c.c_int32]),
    "nvj_decoder_step_workspace_bytes": (_c.c_size_t, [
        _c.POINTER(DecoderModel), _c.c_int32, _c.c_int32]),
    "nvj_decoder_step_launch": (_c.c_int, [
        _c.c_void_p, _c.POINTER(DecoderModel), _c.POINTER(DecoderLayer), _c.POINTER(DecoderBatch),
        _c.c_void_p, _c.c_size_t]),
}
NVJ_LINEAR_ROWS = 0
NVJ_LINEAR_SILU_MUL = 1
NVJ_LINEAR_CHAINS_4_1 = 2
NVJ_LINEAR_CHAINS_4_2 = 3
NVJ_LINEAR_CHAINS_2_4 = 4
NVJ_CHUNK_WHOLE_SEQUENCE = -1
NVJ_STATIC_SCRATCH_BYTES = 16 << 20
NVJ_ERR_SCRATCH_LIMIT = -7
NVJ_ERR_ALIGNMENT = -8
NVJ_PHASE_SPLITK = 1
NVJ_PHASE_COMBINE = 2
NVJ_PHASE_VALU_PRODUCTS = 4
NVJ_PHASE_CLEAR_COUNTERS = 8
NVJ_PHASE_LOADS_ONLY = 16
NVJ_PHASE_SHARED_ROWS = 32
NVJ_PHASE_SHORT_ROWS = 64

_lock = threading.Lock()
_lib = None


class NativeLibraryError(RuntimeError):
    """The HIP library is missing, stale or returned an error code."""


def lib_path() -> str:
    return _LIB_PATH


def load() -> ctypes.CDLL:
    """Load the shared library once and type every entry point."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(_LIB_PATH):
            raise NativeLibraryError(
                f"{_LIB_PATH} not found: build it with "
                "`python -c 'import __graft_entry__ as g; g.build()'` "
                "(there is no fallback for the paged-decode path)")
        lib = ctypes.CDLL(_LIB_PATH)
        for name, (restype, argtypes) in SYMBOLS.items():
            try:
                fn = getattr(lib, name)
            except AttributeError as e:
                raise NativeLibraryError(f"{_LIB_PATH} does not export {name}") from e
            fn.restype = restype
            fn.argtypes = argtypes
        got = lib.nvj_abi_version()
        if got != NVJ_ABI_VERSION:
            raise NativeLibraryError(
                f"{_LIB_PATH} has ABI version {got}, expected {NVJ_ABI_VERSION}: rebuild")
        _lib = lib
        return lib


_host = None


def load_host():
    """The native host side (``csrc/host/nvj_host.cpp``), loaded once; missing is an
    error, as for the library itself."""
    global _host
    if _host is not None:
        return _host
    load()
    with _lock:
        if _host is not None:
            return _host
        path = os.path.join(os.path.dirname(_LIB_PATH), "nvj_host.so")
        if not os.path.exists(path):
            raise NativeLibraryError(
                f"{path} not found: build it with `python -c 'import __graft_entry__ as g; "
                "g.build()'`")
        spec = importlib.util.spec_from_file_location("nvj_host", path)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        _host = module
    return _host


def check(code: int, what: str) -> None:
    if code != 0:
        msg = load().nvj_error_string(code).decode()
        raise NativeLibraryError(f"{what} failed: {msg} (code {code})")
