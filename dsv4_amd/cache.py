"""Paged-KV cache writer: new latent KV rows -> the paged cache the forward
reads, through the same block tables.

The reference builds its paged caches on the host in its tests
(sparse_attn_sharedkv_tilelang/golden.py:315-408): row ``pos`` of batch ``b``
is stored in physical block ``block_table[b, pos // block_size]`` at offset
``pos % block_size``; ``-1`` marks an unused table entry. This module writes
rows into that layout on the GPU with ``sas_cache_write_v1``, either as a
bf16/fp16 copy or quantised into the 656-byte fp8 rows of
:mod:`dsv4_amd.paged` (``quantize_kv_fp8``'s format and rounding, bit for bit).
"""

from __future__ import annotations

import ctypes as C
import struct
from typing import Optional

import torch

from . import _lib

_DT = {torch.bfloat16: _lib.SAS_DT_BF16, torch.float16: _lib.SAS_DT_FP16}
FP8_ROW_BYTES = 656
# the current stream as a hipStream_t value, without a Stream object
_raw = getattr(torch._C, "_cuda_getCurrentRawStream", None)


class PreparedCacheWrite:
    """Arguments of one cache write, validated once; :meth:`launch` runs the
    kernel on the current (or given) stream without host syncs."""

    def __init__(self, args: _lib.SasCacheWriteArgs, keep: list, device):
        self.args = args
        self._keep = keep
        self.device = device
        # the int32 / contiguous conversions were enqueued on this stream
        self._prep_stream = torch.cuda.current_stream(device)

    def launch(self, stream: Optional[torch.cuda.Stream] = None) -> None:
        st = stream if stream is not None else torch.cuda.current_stream(self.device)
        if st != self._prep_stream:
            # order the launch after the conversions, and keep every bound
            # tensor's memory from being reused by the caching allocator on
            # its own stream while the kernel on `st` may still touch it
            ev = torch.cuda.Event()
            ev.record(self._prep_stream)
            st.wait_event(ev)
            for t in self._keep:
                t.record_stream(st)
        _lib.check(_lib.lib().sas_cache_write_v1(C.byref(self.args), C.c_void_p(st.cuda_stream)),
                   "write_kv_cache")


def _i32(t: torch.Tensor) -> torch.Tensor:
    return t if t.dtype is torch.int32 and t.is_contiguous() else t.to(torch.int32).contiguous()


def _bind(kv, cache, block_table, seq_ids, positions):
    """Validate and convert: (launch arguments in SasCacheWriteArgs' order,
    the tensors they point into, device)."""
    if kv.dim() != 2:
        raise ValueError(f"kv must be [N, D], got {tuple(kv.shape)}")
    if kv.dtype not in _DT:
        raise ValueError(f"kv dtype must be bf16 or fp16, got {kv.dtype}")
    if cache.dim() != 4 or cache.shape[2] != 1:
        raise ValueError(f"cache must be [num_blocks, block_size, 1, row], got {tuple(cache.shape)}")
    N, D = kv.shape
    fp8 = cache.dtype == torch.uint8
    if fp8:
        if cache.shape[-1] != FP8_ROW_BYTES or kv.dtype != torch.bfloat16 or D != 576:
            raise ValueError("fp8 cache rows need uint8 [..., 656] and bf16 kv with D = 576")
    elif cache.dtype != kv.dtype or cache.shape[-1] != D:
        raise ValueError("cache must hold rows of kv's dtype and width, or uint8 fp8 rows")
    if block_table.dim() != 2:
        raise ValueError("block_table must be [B, max_blocks]")
    if seq_ids.shape != (N,) or positions.shape != (N,):
        name, t = ("seq_ids", seq_ids) if seq_ids.shape != (N,) else ("positions", positions)
        raise ValueError(f"{name} must be [N] = [{N}], got {tuple(t.shape)}")
    dev = kv.device
    if cache.device != dev or block_table.device != dev or seq_ids.device != dev or positions.device != dev:
        raise ValueError("all tensors must be on kv's device")
    if kv.stride(1) != 1 or not cache.is_contiguous():
        raise ValueError("kv rows and cache must be contiguous")
    bt, sid, pos = _i32(block_table), _i32(seq_ids), _i32(positions)
    nb, bs = cache.shape[0], cache.shape[1]
    return ((kv.data_ptr(), sid.data_ptr(), pos.data_ptr(), bt.data_ptr(), cache.data_ptr(), N, bt.shape[0], D,
             kv.stride(0), bt.shape[1], bs, nb, _DT[kv.dtype],
             _lib.SAS_DT_FP8_E4M3_ROW656 if fp8 else _DT[kv.dtype]), (kv, cache, bt, sid, pos), dev)


def prepare_kv_cache_write(kv: torch.Tensor, cache: torch.Tensor, block_table: torch.Tensor,
                           seq_ids: torch.Tensor, positions: torch.Tensor) -> PreparedCacheWrite:
    """Validate the arguments of :func:`write_kv_cache` and bind them."""
    args, keep, dev = _bind(kv, cache, block_table, seq_ids, positions)
    return PreparedCacheWrite(_lib.SasCacheWriteArgs(*args), list(keep), dev)


# SasCacheWriteArgs as packed bytes (five pointers, seven int64, two int32):
# filling the ctypes structure field by field took a third of a small call
_ARGS = struct.Struct("@5Q7q2i")
assert _ARGS.size == C.sizeof(_lib.SasCacheWriteArgs)
_write_raw = None


def _write_bytes():
    """sas_cache_write_v1 taking its arguments as packed bytes."""
    global _write_raw
    if _write_raw is None:
        f = _lib.lib()["sas_cache_write_v1"]   # a function object of its own: other argument types
        f.argtypes = [C.c_char_p, C.c_void_p]
        f.restype = C.c_int
        _write_raw = f
    return _write_raw


def write_kv_cache(kv: torch.Tensor, cache: torch.Tensor, block_table: torch.Tensor,
                   seq_ids: torch.Tensor, positions: torch.Tensor,
                   stream: Optional[torch.cuda.Stream] = None) -> None:
    """Scatter ``kv [N, D]`` into ``cache`` on the GPU (no host sync).

    ``cache`` is ``[num_blocks, block_size, 1, D]`` in ``kv``'s dtype (rows
    copied) or uint8 ``[num_blocks, block_size, 1, 656]`` (bf16 ``kv`` with
    D = 576, quantised to fp8 rows). ``seq_ids`` / ``positions`` (int32
    ``[N]``) give each row's batch and logical position; rows whose position
    is negative, or whose block-table entry is -1 or missing, are skipped.
    The rows of one call must go to distinct cache rows.
    """
    if stream is not None or not kv.is_cuda:
        prepare_kv_cache_write(kv, cache, block_table, seq_ids, positions).launch(stream)
        return
    # on the current stream, as any conversion made by _bind
    args, keep, dev = _bind(kv, cache, block_table, seq_ids, positions)
    rc = _write_bytes()(_ARGS.pack(*args), torch.cuda.current_stream(dev).cuda_stream if _raw is None else _raw(dev.index))
    if rc:
        _lib.check(rc, "write_kv_cache")
