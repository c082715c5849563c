"""ctypes binding of libironcore_paged.so (the C ABI in include/ironcore_paged.h).

The library is loaded from ironcore_amd/lib/, built in-tree by
``python -m ironcore_amd.build``.  There is no fallback: if the library is
missing every paged operation raises.
"""
from __future__ import annotations

import ctypes
import importlib.util
from ctypes import c_char_p, c_float, c_int, c_int64, c_size_t, c_void_p
from pathlib import Path

import torch

LIB_PATH = Path(__file__).resolve().parent / "lib" / "libironcore_paged.so"
HOST_PATH = LIB_PATH.parent / "_host.so"

IC_OK = 0
IC_ERR_LAUNCH = -5
IC_DTYPE = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}

# Call descriptors, field by field as in the header (tests hold them to it).
_FIELDS = {
    "ic_step_linear_call": (
        ("out norm_out", c_void_p), ("out_stride norm_out_stride", c_int64), ("x", c_void_p), ("x_stride", c_int64),
        ("w bias", c_void_p), ("w_stride", c_int64), ("w2 bias2", c_void_p), ("w2_stride", c_int64),
        ("residual", c_void_p), ("residual_stride", c_int64), ("norm_weight norm_bias", c_void_p), ("m k n n2", c_int),
        ("norm act", c_int), ("eps", c_float), ("dtype tile_bytes splits", c_int), ("k_pool v_pool", c_void_p),
        ("pool_stride_block pool_stride_head pool_stride_token num_blocks", c_int64), ("hn gn hd block_size", c_int),
        ("slot_mapping positions cos_table sin_table", c_void_p), ("table_rows", c_int64), ("workspace", c_void_p),
        ("workspace_bytes", c_size_t)),
    "ic_step_layer": (
        ("input_norm_weight input_norm_bias q_weight q_bias kv_weight kv_bias proj_weight proj_bias", c_void_p),
        ("post_norm_weight post_norm_bias up_weight up_bias down_weight down_bias k_pool v_pool", c_void_p),
        ("input_norm post_norm", c_int), ("input_norm_eps post_norm_eps", c_float)),
    "ic_step_stack_call": (
        ("layers x out norm_out norm_weight norm_bias", c_void_p), ("num_layers m d f hn gn hd act norm", c_int), ("eps", c_float),
        ("pool_stride_block pool_stride_head pool_stride_token num_blocks", c_int64), ("block_tables", c_void_p),
        ("block_table_stride", c_int64), ("context_lens slot_mapping positions cos_table sin_table", c_void_p),
        ("table_rows", c_int64), ("block_size max_context_len", c_int), ("scale", c_float), ("dtype workgroups draw", c_int),
        ("workspace", c_void_p), ("workspace_bytes", c_size_t), ("status", c_void_p), ("max_polls", c_int)),
    "ic_append_call": (
        ("k_new v_new", c_void_p), ("new_stride_token", c_int64), ("k_pool v_pool", c_void_p),
        ("pool_stride_block pool_stride_head pool_stride_token num_blocks", c_int64), ("slot_mapping", c_void_p),
        ("n_tokens", c_int64), ("gn hd block_size dtype", c_int), ("positions cos_table sin_table", c_void_p),
        ("table_rows", c_int64), ("zero_out", c_void_p), ("zero_stride_bytes", c_int64), ("rows", c_void_p),
        ("n_rows", c_int64), ("bounds", c_void_p), ("zero_row_bytes n_seqs row_pitch", c_int)),
    "ic_prefill_call": (
        ("out", c_void_p), ("out_stride_token", c_int64), ("q", c_void_p), ("q_stride_token", c_int64), ("k_pool v_pool", c_void_p),
        ("pool_stride_block pool_stride_head pool_stride_token", c_int64), ("block_tables", c_void_p),
        ("block_table_stride", c_int64), ("context_lens cu_seqlens_q", c_void_p),
        ("n_seqs max_chunk_len hn gn hd block_size", c_int), ("num_blocks", c_int64), ("scale", c_float),
        ("causal dtype uniform_context", c_int), ("row_pitch", c_int64), ("rows", c_void_p), ("n_rows q_rows", c_int64),
        ("positions cos_table sin_table", c_void_p), ("table_rows", c_int64), ("mask_bits mask_lists", c_void_p),
        ("mask_plane_seq mask_plane_head", c_int)),
    "ic_decode_append_call": (
        ("out", c_void_p), ("out_stride_seq", c_int64), ("q", c_void_p), ("q_stride_seq", c_int64), ("k_new v_new", c_void_p),
        ("new_stride_token", c_int64), ("k_pool v_pool", c_void_p),
        ("pool_stride_block pool_stride_head pool_stride_token num_blocks", c_int64), ("block_tables", c_void_p),
        ("block_table_stride", c_int64), ("context_lens slot_mapping positions cos_table sin_table", c_void_p),
        ("table_rows", c_int64), ("n_seqs hn gn hd block_size max_context_len", c_int), ("scale", c_float),
        ("dtype", c_int)),
}
STRUCTS = {name: type(name, (ctypes.Structure,), {"_fields_": [(n, t) for names, t in rows for n in names.split()]})
           for name, rows in _FIELDS.items()}

# name -> (restype, argtypes); mirrors include/ironcore_paged.h one to one.
SIGNATURES = {
    "ic_version": (c_int, []),
    "ic_error_string": (c_char_p, [c_int]),
    "ic_mfma_probe": (c_int64, [c_int, c_void_p, c_void_p]),
    "ic_decode_occupancy_queries": (c_int64, []),
    "ic_kv_append": (c_int, [
        c_void_p, c_void_p, c_int64,            # k_new, v_new, new_stride_token
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides: block, head, token
        c_void_p, c_int64,                      # slot_mapping, n_tokens
        c_int, c_int, c_int, c_int64,           # gn, hd, block_size, num_blocks
        c_int, c_void_p]),                      # dtype, stream
    "ic_rope_kv_append": (c_int, [
        c_void_p, c_int64, c_int,               # q, q_stride_token, hn
        c_void_p, c_void_p, c_int64,            # k_new, v_new, new_stride_token
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_void_p,                     # slot_mapping, positions
        c_void_p, c_void_p, c_int64,            # cos_table, sin_table, table_rows
        c_int64, c_int, c_int, c_int,           # n_tokens, gn, hd, block_size
        c_int64, c_int, c_void_p]),             # num_blocks, dtype, stream
    "ic_rope_kv_append_to": (c_int, [
        c_void_p, c_int64,                      # q_out, q_out_stride_token
        c_void_p, c_int64, c_int,               # q, q_stride_token, hn
        c_void_p, c_void_p, c_int64,            # k_new, v_new, new_stride_token
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_void_p,                     # slot_mapping, positions
        c_void_p, c_void_p, c_int64,            # cos_table, sin_table, table_rows
        c_int64, c_int, c_int, c_int,           # n_tokens, gn, hd, block_size
        c_int64, c_int, c_void_p]),             # num_blocks, dtype, stream
    "ic_paged_decode_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int]),
    "ic_paged_decode": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p,            # block_tables, stride, context_lens
        c_int, c_int, c_int, c_int, c_int,      # n_seqs, hn, gn, hd, block_size
        c_int64, c_int, c_float,                # num_blocks, max_context_len, scale
        c_int, c_void_p, c_size_t,              # min_chunk_tokens, workspace, workspace_bytes
        c_int, c_void_p]),                      # dtype, stream
    "ic_paged_decode_shared_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "ic_paged_decode_shared": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p,            # block_tables, stride, context_lens
        c_int, c_int, c_int, c_int, c_int,      # n_seqs, hn, gn, hd, block_size
        c_int64, c_int, c_float,                # num_blocks, max_context_len, scale
        c_int, c_int, c_void_p,                 # min_chunk_tokens, cohort_size, cohort_shared_blocks
        c_void_p, c_size_t,                     # workspace, workspace_bytes
        c_int, c_void_p]),                      # dtype, stream
    "ic_paged_decode_static_scratch_bytes": (c_size_t, [c_int, c_int, c_int, c_int]),
    "ic_paged_decode_static": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p,            # block_tables, stride, context_lens
        c_int, c_int, c_int, c_int, c_int,      # n_seqs, hn, gn, hd, block_size
        c_int64, c_int, c_float,                # num_blocks, max_context_len, scale
        c_int, c_int, c_void_p]),               # min_chunk_tokens, dtype, stream
    "ic_paged_prefill": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p, c_void_p,  # block_tables, stride, context_lens, cu_seqlens_q
        c_int, c_int,                           # n_seqs, max_chunk_len
        c_int, c_int, c_int, c_int,             # hn, gn, hd, block_size
        c_int64, c_float, c_int,                # num_blocks, scale, causal
        c_int, c_void_p]),                      # dtype, stream
    "ic_linear_rows_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "ic_linear_rows": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, x, x_stride
        c_void_p, c_int64, c_void_p,            # w, w_stride, bias
        c_int, c_int, c_int, c_int,             # m, n, k, splits
        c_void_p, c_size_t, c_int, c_void_p]),  # workspace, workspace_bytes, dtype, stream
    "ic_step_linear_workspace_bytes": (c_size_t, [c_void_p]),   # call descriptor
    "ic_step_linear": (c_int, [c_void_p, c_void_p]),    # call descriptor, stream
    "ic_step_stack_workspace_bytes": (c_size_t, [c_void_p]),   # call descriptor
    "ic_step_stack": (c_int, [c_void_p, c_void_p]),     # call descriptor, stream
    "ic_step_status": (c_void_p, []),
    "ic_append_chunks": (c_int, [c_void_p, c_void_p]),   # call descriptor, stream
    "ic_paged_decode_append": (c_int, [c_void_p, c_void_p]),   # call descriptor, stream
    "ic_greedy_workspace_bytes": (c_size_t, [c_int, c_int]),   # rows, n
    "ic_greedy": (c_int, [c_void_p, c_void_p]),         # call descriptor, stream
    "ic_advance": (c_int, [c_void_p, c_void_p]),        # call descriptor, stream
    "ic_mask_pack": (c_int, [
        c_void_p, c_int64, c_int64, c_int64,    # mask, strides: seq, head, row
        c_int, c_int, c_int, c_int,             # n_seqs, heads, rows, keys
        c_void_p, c_void_p, c_void_p, c_void_p]),   # bits, lists, flags, stream
    "ic_paged_prefill_ex": (c_int, [c_void_p, c_void_p]),   # call descriptor, stream
    "ic_zero_unlisted_rows": (c_int, [
        c_void_p, c_int64, c_int, c_void_p, c_int64,   # out, stride, row_bytes, rows, n_rows
        c_void_p, c_int, c_int, c_void_p]),             # bounds, n_seqs, row_pitch, stream
    "ic_paged_prefill_masked": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p, c_void_p,  # block_tables, stride, context_lens, cu_seqlens_q
        c_int, c_int,                           # n_seqs, max_chunk_len
        c_int, c_int, c_int, c_int,             # hn, gn, hd, block_size
        c_int64, c_float,                       # num_blocks, scale
        c_void_p, c_int64, c_int64, c_int64,    # mask, strides: seq, head, row
        c_int64, c_int, c_void_p]),             # mask_keys, dtype, stream
    "ic_paged_decode_masked": (c_int, [
        c_void_p, c_int64, c_void_p, c_int64,   # out, out_stride, q, q_stride
        c_void_p, c_void_p,                     # k_pool, v_pool
        c_int64, c_int64, c_int64,              # pool strides
        c_void_p, c_int64, c_void_p,            # block_tables, stride, context_lens
        c_int, c_int, c_int, c_int, c_int,      # n_seqs, hn, gn, hd, block_size
        c_int64, c_int, c_float,                # num_blocks, max_context_len, scale
        c_int,                                  # min_chunk_tokens
        c_void_p, c_int64, c_int64,             # key_mask, strides: seq, head
        c_void_p, c_size_t,                     # workspace, workspace_bytes
        c_int, c_void_p]),                      # dtype, stream
}


class PagedLibraryError(RuntimeError):
    """A C-ABI call returned a negative IC_ERR_* code."""

    def __init__(self, func: str, code: int, message: str):
        super().__init__(f"{func} failed with code {code}: {message}")
        self.func = func
        self.code = code


_lib = None


def load() -> ctypes.CDLL:
    """Load the shared library (once) and declare every prototype."""
    global _lib
    if _lib is not None:
        return _lib
    if not LIB_PATH.exists():
        raise RuntimeError(
            f"{LIB_PATH} is missing: build it with `python -m ironcore_amd.build` "
            "(there is no non-HIP fallback for the paged-attention path)")
    lib = ctypes.CDLL(str(LIB_PATH))
    for name, (restype, argtypes) in SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype = restype
        fn.argtypes = argtypes
    _lib = lib
    return lib


_host = None


def host():
    """The native call path (csrc/host_binding.cpp): each of its functions does
    the whole call for ordinary arguments, or returns None / False and leaves
    them to the Python wrapper, which handles or refuses the rest."""
    global _host
    if _host is None:
        if not HOST_PATH.exists():
            raise RuntimeError(f"{HOST_PATH} is missing: build it with `python -m ironcore_amd.build`")
        load()
        spec = importlib.util.spec_from_file_location("_host", HOST_PATH)
        _host = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(_host)
    return _host


def here(t: torch.Tensor):
    """(device index, stream) for a tensor on the current GPU, else None."""
    if not t.is_cuda:
        return None
    device = t.get_device()
    if device != torch._C._cuda_getDevice():
        return None
    return device, torch._C._cuda_getCurrentRawStream(device)


def check(func: str, code: int) -> None:
    if code != IC_OK:
        msg = load().ic_error_string(code).decode()
        raise PagedLibraryError(func, code, msg)


def dtype_code(dtype: torch.dtype) -> int:
    try:
        return IC_DTYPE[dtype]
    except KeyError:
        raise TypeError(f"paged attention supports bf16/fp16/fp32 tensors, got {dtype}") from None


def current_stream_ptr(device: torch.device) -> int:
    return torch.cuda.current_stream(device).cuda_stream
