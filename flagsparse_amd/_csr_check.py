"""The structural checks of a CSR matrix and the narrowing of its index arrays, in one device
pass and one host synchronisation (fsp_csr_check in csrc/check.hip)."""

import torch

from . import _abi


def csr_check(indices, indptr, ptr_bits=None):
    """((first, last, decreases, longest row, min column, max column) as Python ints, the columns
    as int32, the row pointers at ``ptr_bits``) of contiguous 1-D device arrays (columns int32 or
    int64; row pointers of another type are converted first).

    The two arrays are the arguments themselves where they already have that width (or where
    ``ptr_bits`` is None); the column bounds are meaningless without entries.  Copies are made
    before the checks are known: they are only good once the caller has looked at them.
    """
    L = _abi.lib()
    dev = indices.device
    if indptr.device != dev:
        raise RuntimeError(f"indices and indptr are on different devices: {dev} and "
                           f"{indptr.device}")
    if indptr.dtype not in (torch.int32, torch.int64):
        indptr = indptr.to(torch.int64)
    nnz, n_rows = int(indices.numel()), int(indptr.numel()) - 1
    idx_bits = 32 if indices.dtype == torch.int32 else 64
    have_bits = 32 if indptr.dtype == torch.int32 else 64
    idx32 = torch.empty(nnz, dtype=torch.int32, device=dev) if idx_bits == 64 else None
    ptr = None
    if ptr_bits is not None and ptr_bits != have_bits:
        ptr = torch.empty(n_rows + 1, dtype=torch.int32 if ptr_bits == 32 else torch.int64,
                          device=dev)
    scratch = torch.empty(int(L.fsp_csr_check_partial_len()) + 6, dtype=torch.int64, device=dev)
    out = scratch[-6:]
    _abi.check(
        L.fsp_csr_check(indices.data_ptr() if nnz else None, idx_bits, nnz, indptr.data_ptr(),
                        have_bits, n_rows, idx32.data_ptr() if idx32 is not None and nnz else None,
                        None if ptr is None else ptr.data_ptr(), ptr_bits or have_bits,
                        scratch.data_ptr(), out.data_ptr(), _abi.raw_stream(dev)),
        "fsp_csr_check")
    return out.tolist(), indices if idx32 is None else idx32, indptr if ptr is None else ptr
