"""COO entries in row order and their CSR row pointers, for products that need each row's
entries together but not their order inside the row (csrc/coo_sort.hip)."""

import torch

from . import _abi, _common


def _bits(t):
    return 32 if t.dtype == torch.int32 else 64


def rows_in_order(data, row, col, max_row):
    """(data, row, col) of contiguous float32 / float64 COO arrays in row order, indices int32; a
    row's entries keep their input order.  Every row must lie in [0, max_row]."""
    L = _abi.lib()
    nnz, dev = int(data.numel()), data.device
    if nnz > L.fsp_coo_sort_max_nnz() or data.dtype not in _common.KERNEL_VALUE_DTYPES:
        order = torch.sort(row, stable=True).indices
        return data[order], row[order].to(torch.int32), col[order].to(torch.int32)
    code = _abi.dtype_code(data.dtype)
    index = torch.empty((2, (nnz + 3) // 4 * 4), dtype=torch.int32, device=dev)
    out = torch.empty_like(data)
    scratch = torch.empty(int(L.fsp_coo_sort_scratch(code, nnz, max_row)), dtype=torch.uint8,
                          device=dev)
    _abi.check(
        L.fsp_coo_sort_rows(code, row.data_ptr(), _bits(row), col.data_ptr(), _bits(col),
                            data.data_ptr(), nnz, max_row, index[0].data_ptr(),
                            index[1].data_ptr(), out.data_ptr(), scratch.data_ptr(),
                            _abi.raw_stream(dev)), "fsp_coo_sort_rows")
    return out, index[0, :nnz], index[1, :nnz]


def row_pointers(row, n_rows):
    """CSR row pointers of ``row`` (contiguous, non-decreasing, inside [0, n_rows)), at the width
    the kernels read."""
    nnz = int(row.numel())
    bits = 32 if nnz <= _common.ROWPTR32_MAX_NNZ else 64
    ptr = torch.empty(n_rows + 1, dtype=torch.int32 if bits == 32 else torch.int64,
                      device=row.device)
    _abi.check(_abi.lib().fsp_coo_rowptr(row.data_ptr() if nnz else None, _bits(row), nnz, n_rows,
                                         ptr.data_ptr(), bits, _abi.raw_stream(row.device)),
               "fsp_coo_rowptr")
    return ptr
