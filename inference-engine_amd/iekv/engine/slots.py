"""Slot-level KV access on either side of the handoff, through libiekv.

``write_slots`` is the prefill side: it scatters a step's new K/V rows into the
pool by slot, as the reference's ``write_kv`` does (ie/kernels/reference.py:45-51,
ie/kernels/torch_backend.py:13-16). ``gather_rows`` is the decode side: it reads a
sequence's context back through its block table, as ``gather_context`` does
(ie/kernels/reference.py:54-63, ie/kernels/torch_backend.py:19-24). Slot
``r`` is row ``r`` of a layer's ``[N*bs, H, D]`` array, so both address the same
bytes the handoff moves.

``write_slots_layers`` and ``gather_rows_arrays`` do the same for many layers or
arrays in one launch: a forward pass's KV writes for every layer at once, and
a sequence's context in every layer's K and V cache at once.
"""
from __future__ import annotations

from array import array as _ints

import numpy as np
import torch

from .. import _native
from .pools import KVPool, current_stream_handle


# Longest host slot list the library carries in its launches' arguments (IEKV_INLINE_IDS
# tokens each): two launches. Longer lists are uploaded once.
HOST_SLOTS_MAX = 2 * _native.INLINE_IDS

# Longest host block table the library carries in its launches' arguments (512 entries each):
# four launches. A longer one is uploaded and gathered in one: each launch more drains and
# fills the GPU again. Host table / uploaded, whole call on MI355X, us: 1,024 blocks of 8
# arrays of 8 KiB tiles 29 / 47, of 48 of 4 KiB 71 / 68; 2,048 53 / 66 and 152 / 140, of 64 of
# 32 KiB 1,357 / 1,386; 4,096 103 / 105, 294 / 271 and 2,732 / 2,806; 8,192 of 8 arrays
# 239 / 223, of 48 of 2 KiB 363 / 307 (row by row, uploaded, 240 and 317).
HOST_TABLE_MAX = 2048

_TYPES = {torch.float32: _native.IEKV_TYPE_F32, torch.float16: _native.IEKV_TYPE_F16,
          torch.bfloat16: _native.IEKV_TYPE_BF16, torch.float8_e4m3fn: _native.IEKV_TYPE_E4M3}
# (row type, cache type) pairs iekv_write_slots_cast rounds on the way.
_CASTS = {(torch.float32, torch.float16), (torch.float32, torch.bfloat16),
          (torch.float32, torch.float8_e4m3fn), (torch.float16, torch.float8_e4m3fn),
          (torch.bfloat16, torch.float8_e4m3fn)}


def _capturing(device: torch.device) -> bool:
    """Whether the device's current stream is under capture. An upload made there would be
    replayed from its pinned source long after that was freed."""
    with torch.cuda.device(device):
        return torch.cuda.is_current_stream_capturing()


def _slots(pool: KVPool, slots):
    """The slots of a call as the library takes them, and the entry point that does: a
    device int64 tensor, or a short host list as an int64 array that the library checks
    and carries in its launch. Host slots outside the pool raise IndexError."""
    if isinstance(slots, torch.Tensor):
        t = slots.to(device=pool.device, dtype=torch.int64)
        return t.contiguous(), "iekv_write_slots_cast"
    rows = pool.num_blocks * pool.block_size
    try:
        host = _ints("q", slots if type(slots) in (list, tuple) else list(slots))
    except (TypeError, OverflowError):      # not 64-bit integers
        bad = [s for s in slots if not 0 <= int(s) < rows]
        if bad:
            raise IndexError(f"slot {bad[0]} out of range for a pool of {rows} slots")
        t = torch.as_tensor(slots, dtype=torch.int64, device=pool.device)
        return t.contiguous(), "iekv_write_slots_cast"
    if len(host) <= HOST_SLOTS_MAX:
        return host, "iekv_write_slots_cast_ids"
    checked = np.frombuffer(host, dtype=np.int64)
    if checked.min() < 0 or checked.max() >= rows:
        bad = checked[(checked < 0) | (checked >= rows)][0]
        raise IndexError(f"slot {bad} out of range for a pool of {rows} slots")
    if _capturing(pool.device):
        raise RuntimeError(f"a list of {len(host)} slots is uploaded, which a stream under "
                           f"capture cannot do: pass a device tensor, or at most "
                           f"{HOST_SLOTS_MAX} slots")
    t = torch.from_numpy(checked).pin_memory().to(pool.device, non_blocking=True)
    return t, "iekv_write_slots_cast"


def _rows(pool: KVPool, k: torch.Tensor, v: torch.Tensor):
    """K and V rows as the library reads them, and the types of the rows and the cache:
    contiguous rows in a wider type that it can round itself as they are, others cast
    first (the cast also makes them contiguous)."""
    if k.dtype != pool.dtype and k.dtype == v.dtype and (k.dtype, pool.dtype) in _CASTS and \
            k.device == v.device == pool.device and not (k.is_neg() or v.is_neg()) and \
            k.is_contiguous() and v.is_contiguous():
        return k, v, _TYPES[k.dtype], _TYPES[pool.dtype]
    return (_in_cache_type(pool, k), _in_cache_type(pool, v), _native.IEKV_TYPE_BYTES,
            _native.IEKV_TYPE_BYTES)


def _in_cache_type(pool: KVPool, t: torch.Tensor) -> torch.Tensor:
    return t.to(device=pool.device, dtype=pool.dtype).contiguous()


def _write(pool: KVPool, first_layer: int, n_layers: int, n: int, k: torch.Tensor,
           v: torch.Tensor, slots) -> None:
    if isinstance(slots, torch.Tensor) and k.dtype == pool.dtype:
        # A step's writes of a model that computes in the cache's type: no more host work
        # than the call needs.
        where = slots.to(device=pool.device, dtype=torch.int64).contiguous()
        kc, vc = _in_cache_type(pool, k), _in_cache_type(pool, v)
        stride = kc.numel() // n_layers * kc.element_size() if n_layers > 1 else 0
        _native.call("iekv_write_slots_layers", pool.native.handle, first_layer, n_layers,
                     pool.block_size, kc.data_ptr(), vc.data_ptr(), stride, where.data_ptr(), n,
                     current_stream_handle(pool.device))
        return
    where, fn = _slots(pool, slots)
    kc, vc, row_type, cache_type = _rows(pool, k, v)
    stride = kc.numel() // n_layers * kc.element_size() if n_layers > 1 else 0
    _native.call(fn, pool.native.handle, first_layer, n_layers, pool.block_size, kc.data_ptr(),
                 vc.data_ptr(), stride, _address(where), n, row_type, cache_type,
                 current_stream_handle(pool.device))


def write_slots(pool: KVPool, layer: int, k: torch.Tensor, v: torch.Tensor, slots) -> None:
    """Scatter rows ``k[i]``, ``v[i]`` ([n, H, D]) into slot ``slots[i]`` of ``layer``.

    The rows are cast to the cache dtype (as ``index_copy_`` of
    ``k.to(cache dtype)`` does), on their way where the library has the cast;
    slots are range-checked on the host when given as a list.
    """
    n = k.shape[0]
    if v.shape[0] != n or len(slots) != n:
        raise ValueError(f"{len(slots)} slots for {n} K rows and {v.shape[0]} V rows")
    if tuple(k.shape[1:]) != pool.tile_shape[1:] or tuple(v.shape[1:]) != pool.tile_shape[1:]:
        raise ValueError(f"rows of shape {tuple(k.shape[1:])} do not fit a pool of "
                         f"{pool.tile_shape[1:]}")
    if not 0 <= layer < pool.num_layers:
        raise IndexError(f"layer {layer} out of range for {pool.num_layers} layers")
    _write(pool, layer, 1, n, k, v, slots)


def _context_table(pool: KVPool, block_table, context_len: int):
    """The table entries a context uses, and the entry point that takes them: a device
    int32 tensor as it is, host ids as an int32 array the library checks and carries in
    its launches (no upload), long ones checked and uploaded. IndexError for a table too
    short for the context."""
    needed = -(-context_len // pool.block_size)
    if isinstance(block_table, torch.Tensor):
        table = block_table.to(dtype=torch.int32)
        if table.numel() < needed:
            raise IndexError(f"context of {context_len} needs {needed} blocks, table has "
                             f"{table.numel()}")
        return table[:needed].to(pool.device).contiguous(), "iekv_gather_rows_arrays"
    if needed > len(block_table):
        raise IndexError(f"context of {context_len} needs {needed} blocks, table has "
                         f"{len(block_table)}")
    if needed > HOST_TABLE_MAX and not _capturing(pool.device):
        return pool.block_ids(block_table[:needed], what="context block"), \
            "iekv_gather_rows_arrays"
    used = list(block_table[:needed])
    try:
        return _ints("i", used), "iekv_gather_rows_arrays_ids"
    except (TypeError, OverflowError):      # not 32-bit integers: refused as elsewhere
        ids = pool.host_ids(used, what="context block")
        return _ints("i", ids.tolist()), "iekv_gather_rows_arrays_ids"


def _address(table) -> int:
    return table.data_ptr() if isinstance(table, torch.Tensor) else table.buffer_info()[0]


def gather_rows(pool: KVPool, array: int, block_table, context_len: int) -> torch.Tensor:
    """Rows ``0..context_len-1`` of a sequence in array ``array`` (K of layer l is l, V is L+l).

    Returns a new ``[context_len, H, D]`` tensor of the cache dtype. Raises
    IndexError when the table is too short for ``context_len`` (as the
    reference does) or holds a block outside the pool.
    """
    table, fn = _context_table(pool, block_table, context_len)
    out = torch.empty((context_len, *pool.tile_shape[1:]), dtype=pool.dtype, device=pool.device)
    _native.call(fn, pool.native.handle, array, 1, pool.block_size, _address(table),
                 context_len, out.data_ptr(), out.numel() * out.element_size(),
                 current_stream_handle(pool.device))
    return out


def write_slots_layers(pool: KVPool, k: torch.Tensor, v: torch.Tensor, slots,
                       first_layer: int = 0) -> None:
    """Scatter ``k[l, i]``, ``v[l, i]`` ([n_layers, n, H, D]) into slot ``slots[i]`` of
    layer ``first_layer + l``, every layer in one launch (rows cast to the cache dtype)."""
    if k.dim() != 4 or k.shape != v.shape:
        raise ValueError(f"K rows {tuple(k.shape)} and V rows {tuple(v.shape)} must both be "
                         "[n_layers, n, H, D]")
    n_layers, n = k.shape[0], k.shape[1]
    if len(slots) != n:
        raise ValueError(f"{len(slots)} slots for {n} rows per layer")
    if tuple(k.shape[2:]) != pool.tile_shape[1:]:
        raise ValueError(f"rows of shape {tuple(k.shape[2:])} do not fit a pool of "
                         f"{pool.tile_shape[1:]}")
    if first_layer < 0 or first_layer + n_layers > pool.num_layers:
        raise IndexError(f"layers {first_layer}..{first_layer + n_layers - 1} out of range for "
                         f"{pool.num_layers} layers")
    _write(pool, first_layer, n_layers, n, k, v, slots)


def gather_rows_arrays(pool: KVPool, block_table, context_len: int, first_array: int = 0,
                       n_arrays: int | None = None) -> torch.Tensor:
    """Rows ``0..context_len-1`` of a sequence in arrays ``first_array ..`` (all 2L by
    default: K of layers 0..L-1, then V), in one launch; a new
    ``[n_arrays, context_len, H, D]`` tensor of the cache dtype."""
    n_arrays = pool.n_arrays - first_array if n_arrays is None else n_arrays
    if first_array < 0 or n_arrays <= 0 or first_array + n_arrays > pool.n_arrays:
        raise IndexError(f"arrays {first_array}..{first_array + n_arrays - 1} out of range for "
                         f"{pool.n_arrays} arrays")
    table, fn = _context_table(pool, block_table, context_len)
    out = torch.empty((n_arrays, context_len, *pool.tile_shape[1:]), dtype=pool.dtype,
                      device=pool.device)
    _native.call(fn, pool.native.handle, first_array, n_arrays, pool.block_size,
                 _address(table), context_len, out.data_ptr(),
                 out.numel() * out.element_size(), current_stream_handle(pool.device))
    return out
