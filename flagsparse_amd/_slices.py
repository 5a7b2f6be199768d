"""Slices of equal work for SpMM and SDDMM (csrc/slices.hip): their boundaries, and the launch
order in which the long rows of a skewed matrix share what they read of the dense operand."""

import torch

from . import _abi

_L2_BYTES = 4 << 20  # one XCD's L2
# A launch holds fewer than 2^32 threads, so this many workgroups of 256 at most, a slice each.  More
# are not refused by the runtime: it launches the number modulo 2^32, and rows stay unwritten.
MAX_SLICES = (2**32 - 1) // 256


def ordered(longest_row, items, dense_bytes, gathered_bytes, one_call):
    """Whether the slices should run in column order where they lie inside one row: rows long
    enough to hold several slices, a dense operand larger than an L2, and enough read of it that
    the order is worth its three launches (14 us on MI355X; it saves 30 to 45 % of the time that
    gathered_bytes take at 7.5 TB/s: 384 MB of a one-off SDDMM 68 -> 47 us)."""
    return (longest_row is not None and longest_row >= 4 * items and dense_bytes > _L2_BYTES
            and gathered_bytes > ((256 if one_call else 32) << 20))


def build(rowptr, n_rows, nnz, items, keep, what, cols=None, n_cols=0):
    """(boundaries, order) of slices of ``items`` rows + entries, made on the current stream; with
    ``cols`` in column order, else None.  what: the product, for the message."""
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError(f"an {what} must run once before it is captured into a graph "
                           "(the first call of this width builds its slices)")
    L = _abi.lib()
    dev = rowptr.device
    stream = _abi.raw_stream(dev)
    n = int(L.fsp_slice_count(n_rows, nnz, items))
    table = torch.empty(2 * (n + 1), dtype=torch.int64, device=dev)
    _abi.check(L.fsp_slice_table(rowptr.data_ptr(), 32 if rowptr.dtype == torch.int32 else 64,
                                 n_rows, nnz, items, keep, table.data_ptr(), stream),
               "fsp_slice_table")
    if cols is None or nnz == 0:
        return table, None
    order = torch.empty(n + int(L.fsp_slice_order_scratch(n)), dtype=torch.int32, device=dev)
    _abi.check(L.fsp_slice_order(table.data_ptr(), n, cols.data_ptr(), n_cols, order.data_ptr(),
                                 order[n:].data_ptr(), stream), "fsp_slice_order")
    return table, order[:n]


def pieces(rowptr, table):
    """(``table`` with the first piece of a cut row in each slice behind it, the number of pieces):
    for sums that take room only where rows are cut.  Waits for the device."""
    n = table.numel() // 2 - 1
    both = torch.empty(2 * (n + 1) + n // 2 + 1, dtype=torch.int64, device=table.device)
    both[:2 * (n + 1)].copy_(table)
    _abi.check(_abi.lib().fsp_slice_pieces(rowptr.data_ptr(),
                                           32 if rowptr.dtype == torch.int32 else 64, n,
                                           both.data_ptr(), _abi.raw_stream(table.device)),
               "fsp_slice_pieces")
    return both, int(both[2 * (n + 1):].view(torch.int32)[n])
