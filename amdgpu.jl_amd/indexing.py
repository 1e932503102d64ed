"""Host mirror of ``Base.findall(::AnyROCArray{Bool})`` (src/kernels/indexing.jl:8-36).

``findall`` is the one-pass form: count the true entries (a U8 -> Int64 reduction), fetch the count,
allocate, then one stream-compaction pass (``rk_findall``).  ``findall_two_pass`` keeps the reference's
own structure -- Int64 cumsum of the flattened mask, scalar fetch of its last entry, scatter kernel -- on
the native scan and ``rk_findall_scatter``."""
from __future__ import annotations

import numpy as np
import torch

from . import _lib as L
from .accumulate import accumulate
from .array import ROCArray, device, fill_slot, give_slot, note_waiting_call, stream_ptr, take_slot, workspace
from .mapreduce import count


def _empty(nd: int) -> ROCArray:
    return ROCArray(dims=(0,) if nd == 1 else (nd, 0), dtype=np.int64)


def findall(*args) -> ROCArray:
    """1-based indices of the true entries, in column-major order: an Int64 vector for vectors, an
    Int64 ``(N, count)`` array of CartesianIndex columns for N-d arrays (``keytype(bools)``).
    ``findall(pred, A)`` is ``findall(pred.(A))`` (benchmarked in perf/array.jl:39-42)."""
    if len(args) == 2 and callable(args[0]):
        from .broadcast import lazy, materialize
        bools = materialize(args[0](lazy(args[1])))
    else:
        (bools,) = args
    if bools.dtype != np.bool_:
        raise L.UnsupportedError(L.RK_ERR_UNSUPPORTED, "findall needs a Bool array")
    n, nd = len(bools), bools.ndim
    if n == 0:
        return _empty(nd)
    total = int(count(bools))                                # indexing.jl:12 (the scalar fetch)
    ys = ROCArray(dims=(total,) if nd == 1 else (nd, total), dtype=np.int64)
    if total > 0:
        shape = L.shape_array(bools.dims)
        ws, ws_bytes = workspace(L.lib.rk_workspace_bytes(L.RK_KIND_FINDALL, L.RK_U8, nd, shape, 0))
        note_waiting_call()
        L.check(L.lib.rk_findall(bools.ptr, nd, shape, ys.ptr, None, ws, ws_bytes, stream_ptr()), "rk_findall")
    return ys


def findall_two_pass(bools: ROCArray) -> ROCArray:
    """The reference's sequence of kernels: cumsum (indexing.jl:10), count fetch (:12), scatter (:16-31)."""
    if bools.dtype != np.bool_:
        raise L.UnsupportedError(L.RK_ERR_UNSUPPORTED, "findall needs a Bool array")
    n, nd = len(bools), bools.ndim
    if n == 0:
        return _empty(nd)
    indices = accumulate("add", bools.reshape(n))
    total = int(indices.view_range(n, n).item())
    ys = ROCArray(dims=(total,) if nd == 1 else (nd, total), dtype=np.int64)
    if total > 0:
        st = L.lib.rk_findall_scatter(bools.ptr, indices.ptr, ys.ptr, nd, L.shape_array(bools.dims), stream_ptr())
        L.check(st, "rk_findall_scatter")
    return ys


def _select(x: ROCArray, mask: ROCArray) -> ROCArray:
    """``x[mask]`` with a mask of x's shape: count, allocate, then one streaming pass that moves the selected elements
    (no index array in between)."""
    n = len(x)
    if n == 0:
        return ROCArray(dims=(0,), dtype=x.dtype)
    nbytes = int(L.lib.rk_mask_bits_tmp_bytes(n))
    tmp = torch.empty(nbytes, dtype=torch.uint8, device=device())
    ws, ws_bytes = workspace()
    slot = take_slot()
    fill_slot(slot, L.lib.rk_mask_count_bits, "rk_mask_count_bits", (mask.ptr, n, slot[0], tmp.data_ptr(), nbytes, ws, ws_bytes), words=1)
    total = int(slot[1][:8].view(np.int64)[0])
    give_slot(slot)
    y = ROCArray(dims=(total,), dtype=x.dtype)
    if total > 0:
        L.check(L.lib.rk_mask_select_bits(n, x.ptr, y.ptr, x.dtype.itemsize, total, tmp.data_ptr(), nbytes, stream_ptr()), "rk_mask_select_bits")
    return y


def getindex_mask(x: ROCArray, mask: ROCArray) -> ROCArray:
    """``x[mask]`` for a mask of x's shape, or ``x[:, ..., :, mask]`` for a Bool vector along the last dim
    (test/hip_rocarray/indexing.jl:5-18).  The first moves the selected elements in one pass over the mask; for the second
    ``Base.to_index`` turns the mask into ``findall(mask)`` (indexing.jl:1) and the selected slices are gathered."""
    if mask.dtype != np.bool_:
        raise L.UnsupportedError(L.RK_ERR_UNSUPPORTED, "logical indexing needs a Bool mask")
    if mask.dims == x.dims:
        return _select(x, mask)
    elif mask.ndim == 1 and x.ndim >= 1 and mask.dims[0] == x.dims[-1]:
        lead = x.dims[:-1]
        inner, nsrc = int(np.prod(lead, dtype=np.int64)), x.dims[-1]
        idx = findall(mask)
    else:
        raise IndexError(f"BoundsError: mask {mask.dims} against array {x.dims}")       # Base.checkbounds
    n = len(idx)
    y = ROCArray(dims=lead + (n,), dtype=x.dtype)
    if n > 0 and inner > 0:
        L.check(L.lib.rk_gather_slices(x.ptr, idx.ptr, y.ptr, x.dtype.itemsize, inner, n, nsrc, stream_ptr()), "rk_gather_slices")
    return y
