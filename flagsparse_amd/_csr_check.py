"""The structural checks of index arrays and their narrowing, in one device pass whose results the
host waits for (csrc/check.hip)."""

import ctypes

import torch

from . import _abi

_BITS = {torch.int32: 32, torch.int64: 64}


def _capturing():
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("index arrays cannot be checked while a graph is captured (the host "
                           "waits for the result): prepare the matrix before the capture")


def _pinned():
    """Pinned words for one call (from torch's cache of pinned blocks; given back with the
    tensor, by when every word has been stored)."""
    return torch.empty(int(_abi.lib().fsp_check_pinned_len()), dtype=torch.int64, pin_memory=True)


def csr_check(indices, indptr, ptr_bits=None, classes=()):
    """([first, last, decreases, longest row, min column, max column] as Python ints, the columns
    as int32, the row pointers at ``ptr_bits``) of contiguous 1-D device arrays (columns int32 or
    int64; row pointers of another type are converted first).  ``classes`` (uneven, block, chunk):
    two more ints, the rows of more than ``uneven`` and at most ``block`` entries and the entries in
    rows of more than ``chunk``.

    The two arrays are the arguments themselves where they already have that width (or where
    ``ptr_bits`` is None); the column bounds are meaningless without entries.  Copies are made
    before the checks are known: they are only good once the caller has looked at them.
    """
    L = _abi.lib()
    dev = indices.device
    if indptr.device != dev:
        raise RuntimeError(f"indices and indptr are on different devices: {dev} and "
                           f"{indptr.device}")
    _capturing()
    if indptr.dtype not in _BITS:
        indptr = indptr.to(torch.int64)
    nnz, n_rows = indices.numel(), indptr.numel() - 1
    idx_bits, have_bits = _BITS[indices.dtype], _BITS[indptr.dtype]
    idx32 = torch.empty(nnz, dtype=torch.int32, device=dev) if idx_bits == 64 else indices
    ptr = indptr
    if ptr_bits is not None and ptr_bits != have_bits:
        ptr = torch.empty(n_rows + 1, dtype=torch.int32 if ptr_bits == 32 else torch.int64,
                          device=dev)
    pinned = _pinned()
    out = (ctypes.c_int64 * (6 + (2 if classes else 0)))()
    call = L.fsp_csr_check_rows if classes else L.fsp_csr_check
    _abi.check(
        call(indices.data_ptr() if nnz else None, idx_bits, nnz, indptr.data_ptr(), have_bits,
             n_rows, idx32.data_ptr() if idx32 is not indices and nnz else None,
             None if ptr is indptr else ptr.data_ptr(), ptr_bits or have_bits, *classes,
             pinned.data_ptr(), ctypes.addressof(out), _abi.raw_stream(dev)),
        "fsp_csr_check")
    return list(out), idx32, ptr


def coo_check(row, col):
    """([min row, max row, min column, max column, decreases of the rows] as Python ints, the rows
    and the columns as int32) of contiguous, non-empty 1-D int32 / int64 device arrays of one
    length.  Arrays that are int32 already are returned themselves; see csr_check."""
    L = _abi.lib()
    dev, nnz = row.device, row.numel()
    if col.device != dev:
        raise RuntimeError(f"row and col are on different devices: {dev} and {col.device}")
    _capturing()
    row32 = row if row.dtype == torch.int32 else torch.empty(nnz, dtype=torch.int32, device=dev)
    col32 = col if col.dtype == torch.int32 else torch.empty(nnz, dtype=torch.int32, device=dev)
    pinned = _pinned()
    out = (ctypes.c_int64 * 5)()
    _abi.check(
        L.fsp_coo_check(row.data_ptr(), _BITS[row.dtype], col.data_ptr(), _BITS[col.dtype], nnz,
                        None if row32 is row else row32.data_ptr(),
                        None if col32 is col else col32.data_ptr(), pinned.data_ptr(),
                        ctypes.addressof(out), _abi.raw_stream(dev)), "fsp_coo_check")
    return list(out), row32, col32
