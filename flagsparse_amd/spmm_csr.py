"""CSR SpMM C = A @ B on gfx950, behind the reference's entry points.

Public API and error behaviour mirror ``src/flagsparse/sparse_operations/spmm_csr.py``:
``flagsparse_spmm_csr`` (:1057-1126, base "ALG1" path, float32 computed in float64),
``prepare_spmm_csr_opt`` (:480-522) and ``flagsparse_spmm_csr_opt`` (:1129-1183, native
precision), the validation metrics (:6-90, :1186-1192) and the benchmark cases
(:1195-1562).

Two kernels, both with G lanes sharing each B row by 16-byte loads along N:
``spmm_rowblock_kernel`` (flagsparse_amd/csrc/spmm.hip) for prepared matrices whose rows are all
short (at most 128 entries), one row per lane group over a planned table, or so long that the
order of additions shows (over 8192; ``spmm_ragged_kernel`` where N is odd and over 16); ``spmm_slices_kernel``
(csrc/spmm_slices.hip) for everything else: slices of equal work found by a search in the row
pointers, the pieces of a cut row added in slice order (deterministic).
"""

import time

import torch

from . import _abi, _common, _slices
from ._common import (
    SUPPORTED_INDEX_DTYPES,
    SUPPORTED_VALUE_DTYPES,
    _INDEX_LIMIT_INT32,
    _aligned,
    _benchmark_cuda_op,
    _is_complex_dtype,
    _require_kernel_dtype,
    _tolerance_for_dtype,
)
from ._csr_check import csr_check
from ._plan import StreamOrder, build_row_block_plan_device
from .synthetic import build_random_csr, build_random_dense

SUPPORTED_SPMM_VALUE_DTYPES = SUPPORTED_VALUE_DTYPES

XCD_REMAP = 1
# The row-block plan is built in windows of SPMM_PLAN_WINDOW_BLOCKS x the block row cap (each
# window's last block may be short).  Windows of one block's rows cut a block after every
# row-cap rows even when the entry cap ended the one before.  Measured on MI355X, cfg5's matrix
# prepared: fp32 N=16 380 / 329 / 327 us with windows of 1 / 4 / 16 blocks, N=64 663 / 663 / 662
# (the planner takes longer on wide windows: one thread each).
SPMM_PLAN_WINDOW_BLOCKS = 4
# A one-off COO matrix's longest row is not known.  Up to this many values its slices get room for
# the pieces of cut rows unseen; beyond it (32 MB of float64) the row pointers are looked at first
# (25 us with its host wait, on products of milliseconds).
_SUMS_UNSEEN = 1 << 22
# Room for the pieces of cut rows, two for every slice, is taken without a count up to this many bytes.
# One row over the longest uncut length is enough for it, and it grows with N: 1M rows of 32 entries
# with one of 300, N = 256, would take 1.06 GB for three pieces.  Beyond the limit the pieces are
# counted, once per matrix and slice size (two launches and a host wait: 0.1 ms of a 4.8 ms product
# without a prepared object there).
_SUMS_ROOM = 256 << 20
# Rows longer than this go to the part path (several lane groups per row).
_SPMM_ROW_SPLIT_THRESHOLD = 128


# ------------------------------------------------------------------------------------------
# Validation metrics (spmm_csr.py:6-90)
# ------------------------------------------------------------------------------------------


def _spmm_relative_threshold(value_dtype):
    if value_dtype == torch.float16:
        return 5e-3
    if value_dtype == torch.bfloat16:
        return 1e-2
    if value_dtype in (torch.float32, torch.complex64):
        return 1e-6
    if value_dtype in (torch.float64, torch.complex128):
        return 1e-12
    return 1e-6


def _spmm_coo_reference_tolerance(value_dtype):
    if value_dtype == torch.float16:
        return 2e-3, 2e-3
    if value_dtype == torch.bfloat16:
        return 1e-1, 1e-1
    if value_dtype in (torch.float32, torch.complex64):
        return 1e-4, 1e-2
    if value_dtype in (torch.float64, torch.complex128):
        return 1e-12, 1e-10
    return 1e-6, 1e-5


def _spmm_error_metrics(candidate, reference):
    if candidate.shape != reference.shape:
        raise ValueError(
            f"candidate and reference must have the same shape, got {candidate.shape} vs "
            f"{reference.shape}")
    if candidate.numel() == 0:
        return {"max_abs_error": 0.0, "max_relative_error": 0.0, "sum_relative_error": 0.0,
                "reference_max_magnitude": 0.0, "reference_sum_magnitude": 0.0}
    if _is_complex_dtype(reference.dtype):
        reference_compare = torch.abs(reference)
        abs_diff = torch.abs(torch.abs(candidate) - reference_compare)
    else:
        reference_compare = torch.abs(reference)
        abs_diff = torch.abs(candidate - reference)
    max_abs_error = float(torch.max(abs_diff).item())
    reference_max_magnitude = float(torch.max(reference_compare).item())
    sum_abs_error = float(torch.sum(abs_diff).item())
    reference_sum_magnitude = float(torch.sum(reference_compare).item())
    if reference_max_magnitude == 0.0:
        max_relative_error = 0.0 if max_abs_error == 0.0 else float("inf")
    else:
        max_relative_error = max_abs_error / reference_max_magnitude
    if reference_sum_magnitude == 0.0:
        sum_relative_error = 0.0 if sum_abs_error == 0.0 else float("inf")
    else:
        sum_relative_error = sum_abs_error / reference_sum_magnitude
    return {"max_abs_error": max_abs_error, "max_relative_error": max_relative_error,
            "sum_relative_error": sum_relative_error,
            "reference_max_magnitude": reference_max_magnitude,
            "reference_sum_magnitude": reference_sum_magnitude}


def _spmm_validation_metrics(candidate, reference):
    metrics = _spmm_error_metrics(candidate, reference)
    threshold = _spmm_relative_threshold(reference.dtype)
    atol, rtol = _tolerance_for_dtype(reference.dtype)
    metrics.update({
        "relative_threshold": threshold,
        "matches_threshold": metrics["max_relative_error"] <= threshold,
        "strict_allclose_match": torch.allclose(candidate, reference, atol=atol, rtol=rtol),
    })
    return metrics


def _spmm_opt_reference_error(candidate, reference, value_dtype):
    atol, rtol = _spmm_coo_reference_tolerance(value_dtype)
    if candidate.numel() == 0:
        return 0.0
    diff = torch.abs(candidate - reference)
    denom = atol + rtol * torch.abs(reference)
    return float(torch.max(diff / denom).item())


# ------------------------------------------------------------------------------------------
# Validation and launch configuration
# ------------------------------------------------------------------------------------------


def _check_spmm_csr_matrix(data, indices, indptr, shape, ptr_bits):
    """The checks of spmm_csr.py:197-255 (same order and exceptions): (data, int32 columns, row
    pointers of ``ptr_bits``, n_rows, n_cols, longest row)."""
    if len(shape) != 2:
        raise ValueError("shape must be a 2-tuple: (n_rows, n_cols)")
    if data.ndim != 1 or indices.ndim != 1 or indptr.ndim != 1:
        raise ValueError("data, indices, and indptr must be 1D tensors")
    n_rows, n_cols = int(shape[0]), int(shape[1])
    if n_rows < 0 or n_cols < 0:
        raise ValueError("shape dimensions must be non-negative")
    if indptr.numel() != n_rows + 1:
        raise ValueError(f"indptr length must be n_rows+1={n_rows + 1}, got {indptr.numel()}")
    if data.numel() != indices.numel():
        raise ValueError("data and indices must have the same length (nnz)")
    if not all(t.is_cuda for t in (data, indices, indptr)):
        raise ValueError("data, indices, and indptr must be CUDA tensors")
    if not all(t.device == data.device for t in (indices, indptr)):
        raise ValueError("data, indices, and indptr must be on the same CUDA device")
    if data.dtype not in SUPPORTED_SPMM_VALUE_DTYPES:
        raise TypeError(
            "data dtype must be one of: float16, bfloat16, float32, float64, complex64, complex128"
        )
    if indices.dtype not in SUPPORTED_INDEX_DTYPES:
        raise TypeError("indices dtype must be torch.int32 or torch.int64")
    if indptr.dtype not in SUPPORTED_INDEX_DTYPES:
        raise TypeError("indptr dtype must be torch.int32 or torch.int64")

    nnz = data.numel()
    data, indices, indptr = data.contiguous(), indices.contiguous(), indptr.contiguous()
    # one pass over the index arrays, one host synchronisation
    (first, last, decreases, max_row_nnz, min_col, max_col), kernel_indices, kernel_ptr = \
        csr_check(indices, indptr, ptr_bits)
    if first != 0:
        raise ValueError("indptr[0] must be 0")
    if last != nnz:
        raise ValueError(f"indptr[-1] must equal nnz={nnz}, got {last}")
    if decreases:
        raise ValueError("indptr must be nondecreasing")
    if nnz > 0:
        if min_col < 0 or max_col >= n_cols:
            raise IndexError("indices out of range for n_cols")
        if max_col > _INDEX_LIMIT_INT32:
            raise ValueError(
                "column indices exceed the int32 range supported by the Triton kernel")
    return data, kernel_indices, kernel_ptr, n_rows, n_cols, int(max_row_nnz)


def _prepare_spmm_csr_matrix(data, indices, indptr, shape):
    """spmm_csr.py:197-255 (same checks, order and exceptions), row pointers as int64."""
    data, kernel_indices, kernel_indptr, n_rows, n_cols, max_row_nnz = \
        _check_spmm_csr_matrix(data, indices, indptr, shape, 64)
    row_lengths = (kernel_indptr[1:] - kernel_indptr[:-1] if n_rows > 0
                   else kernel_indptr.new_empty((0,)))
    return data, kernel_indices, kernel_indptr, n_rows, n_cols, row_lengths, max_row_nnz


def _prepare_spmm_csr_inputs(data, indices, indptr, B, shape):
    """spmm_csr.py:258-281, row pointers at the width the kernels read."""
    if B.ndim != 2:
        raise ValueError("B must be a 2D dense tensor")
    data, kernel_indices, kernel_indptr, n_rows, n_cols, max_row_nnz = \
        _check_spmm_csr_matrix(data, indices, indptr, shape,
                               32 if data.numel() <= _common.ROWPTR32_MAX_NNZ else 64)
    if B.shape[0] != n_cols:
        raise ValueError(f"B.shape[0] must be n_cols={n_cols}, got {B.shape[0]}")
    if not B.is_cuda:
        raise ValueError("B must be a CUDA tensor")
    if B.device != data.device:
        raise ValueError("B must be on the same CUDA device as the sparse matrix")
    if B.dtype != data.dtype:
        raise TypeError("B dtype must match data dtype")
    B = B.contiguous()
    return (data, kernel_indices, kernel_indptr, B, n_rows, n_cols, int(B.shape[1]),
            max_row_nnz)


def _select_spmm_alg1_warp_and_factor(n_dense_cols):
    """spmm_csr.py:284-296."""
    if n_dense_cols > 64:
        return 32, 4
    if n_dense_cols > 32:
        return 32, 2
    if n_dense_cols > 16:
        return 32, 1
    if n_dense_cols > 8:
        return 16, 1
    if n_dense_cols > 4:
        return 8, 1
    return 4, 1


def _resolve_spmm_alg1_launch_config(n_dense_cols, max_row_nnz, block_n=None, block_nnz=None,
                                     max_segments=None):
    """spmm_csr.py:299-334 (ValueError when max_segments cannot cover the longest row)."""
    warp_size, factor = _select_spmm_alg1_warp_and_factor(n_dense_cols)
    if block_n is None:
        block_n = warp_size * factor
    if block_nnz is None:
        block_nnz = warp_size
    if block_n <= 0 or block_nnz <= 0:
        raise ValueError("block_n and block_nnz must be positive when provided")
    if max_segments is not None and max_segments <= 0:
        raise ValueError("max_segments must be positive when provided")
    required_segments = -(-max_row_nnz // block_nnz) if max_row_nnz > 0 else 0
    if max_segments is not None and required_segments > int(max_segments):
        raise ValueError(
            "row nnz requires more CSR segments than the explicit max_segments override allows: "
            f"required {required_segments}, provided {int(max_segments)}")
    return {
        "block_n": int(block_n),
        "block_nnz": int(block_nnz),
        "max_segments": (None if max_segments is None else int(max_segments)),
        "required_segments": int(required_segments),
        "warp_size": int(warp_size),
        "factor": int(factor),
        "max_row_nnz": int(max_row_nnz),
        "auto_max_segments": max_segments is None,
    }


def _next_pow2(v):
    p = 1
    while p < v:
        p <<= 1
    return p


def _spmm_lane_shape(n_dense_cols, dtype, B, C, tile_cols=None):
    """(lanes per B row G, elements per lane vec) for the gfx950 kernel.

    vec: 16-byte loads (4 fp32 / 2 fp64) when N and both base pointers allow it, else 2 or 1.
    G: enough lanes to cover min(N, tile_cols) columns, a power of two <= 64.  The kernel's
    column tile is G * vec, so with narrower lanes (odd N, unaligned B or C) a tile of more
    than 64 * vec columns is launched as tiles of 64 * vec.
    """
    vmax = 4 if dtype == torch.float32 else 2
    aligned = B.data_ptr() % 16 == 0 and C.data_ptr() % 16 == 0
    vec = 1
    for v in (vmax, 2):
        if aligned and n_dense_cols % v == 0:
            vec = v
            break
    width = n_dense_cols if tile_cols is None else max(1, min(n_dense_cols, int(tile_cols)))
    lanes = min(64, _next_pow2(max(1, -(-width // vec))))
    return lanes, vec


def _spmm_slice_lanes(n_dense_cols, dtype, tile_cols=None):
    """(lanes per B row G, elements per lane vec) for the sliced kernel: 16-byte loads for every
    N that holds one (any alignment), single elements for N = 3 (measured on MI355X, fp32, 15M
    entries: 75.6 us against 76.4 with pairs)."""
    vec = 4 if dtype == torch.float32 else 2
    if n_dense_cols < vec:
        vec = 2 if n_dense_cols == 2 else 1
    width = n_dense_cols if tile_cols is None else max(1, min(n_dense_cols, int(tile_cols)))
    return min(64, _next_pow2(-(-width // vec))), vec


def _spmm_slice_shape(lanes, positions, by_column=False):
    """(rows + entries per slice, longest row never cut).  A slice should give each of a
    workgroup's 256 / lanes groups several entries, and the matrix enough slices to fill the
    256 CUs.  Measured on MI355X with 128 / 256 / 512 / 1024 positions: 16 lanes (fp32 N=64, 33.5M
    entries) 781 / 670 / 661 / 701 us; 64 lanes (N=256, 4M) 557 / 564 / - / -; 8 lanes (N=32,
    1.2M) 29.8 / 22.0 / 19.7 / 19.2; the same with 80k entries 5.2 / 5.3 / 6.3 / 6.9, hence the
    limit by size.  Slices that run by column are shorter, so that more rows hold several (a power
    law, 128 / 256 / 512 positions: N=128, 32 lanes 190 / 200 / - us; N=47, 16 lanes 151 / 125 /
    127; 4 lanes, N=16, 512 / 1024 / 1536: 120 / 123 / 131)."""
    if by_column:
        items = {64: 128, 32: 128, 16: 256}.get(lanes, 512)
    else:
        items = {64: 128, 32: 256, 16: 512, 8: 1024}.get(lanes, 1536)
    while items > 64 and positions < 1024 * items:
        items = max(64, items >> 1)
    while items < 1536 and positions > _slices.MAX_SLICES * items:
        items = min(1536, items << 1)
    return items, 256 if items >= 128 else 128


# Sums of more than this many products depend visibly on the order of addition: in float32 two
# orders differ by up to 4.6e-5 of the result's root mean square (200k rows of power-law lengths,
# N = 47), against 1e-6 below.  Prepared products on such rows keep the order of the row-block
# kernel, 128-entry parts added one after another, bit for bit, and change only the launch order
# of the parts (slices would take 57 / 122 / 214 us where that takes 60 / 130 / 233: fp32, N = 16 / 47
# / 128).
_SPMM_SUMS_KEPT = 8192


def _parts_by_column(desc, cols, n_cols, rowptr, chunk):
    """The descriptor table in launch order: row blocks as they are, then the parts of long rows
    by the first column they hold, each XCD a contiguous eighth of either.  Parts of different
    rows over the same columns then read the same rows of B while they are in that XCD's L2.
    Measured on MI355X, us, in row order / in this order: 200k rows of power-law lengths, fp32
    N=16 89 / 60, N=47 231 / 130, N=128 382 / 233; fp64 N=33 287 / 176, N=64 379 / 256.  Ordered
    by 256 column bins in three launches (csrc/slices.hip): a full sort and gathers by torch took
    0.34 ms more of a matrix's first product (N=47: 815 / 479 us) for the same 195 us after it."""
    L = _abi.lib()
    n, dev = int(desc.shape[0]), desc.device
    out = torch.empty_like(desc)
    scratch = torch.empty(int(L.fsp_slice_order_scratch(n)), dtype=torch.int32, device=dev)
    _abi.check(L.fsp_part_order(desc.data_ptr(), n, rowptr.data_ptr(),
                                32 if rowptr.dtype == torch.int32 else 64, chunk, cols.data_ptr(),
                                n_cols, out.data_ptr(), scratch.data_ptr(), _abi.raw_stream(dev)),
               "fsp_part_order")
    return out


class _SpmmKernelCsr:
    """Kernel-facing CSR arrays (aligned, int32 offsets when they fit), their row-block plans per
    G and their slices.  max_row_nnz: the longest row, where known; one_shot: the object serves
    one call, so nothing is planned."""

    __slots__ = ("data", "cols", "rowptr", "rowptr_bits", "nnz", "n_rows", "_plans", "_args",
                 "_keep", "_order", "max_row_nnz", "one_shot", "_tables", "_shared")

    def __init__(self, data, cols, indptr, max_row_nnz=None, one_shot=False):
        self.max_row_nnz = max_row_nnz
        self.one_shot = one_shot
        self.data = _aligned(data)
        self.cols = _aligned(cols)
        self.nnz = int(data.numel())
        self.n_rows = int(indptr.numel()) - 1
        if self.nnz <= _common.ROWPTR32_MAX_NNZ:
            self.rowptr, self.rowptr_bits = indptr.to(torch.int32), 32
        else:
            self.rowptr, self.rowptr_bits = indptr.to(torch.int64).contiguous(), 64
        self._tables = {}
        # what products of several widths share: ("pieces", slice size), ("sums", length, dtype),
        # ("row order", lanes), and ("name", N), the kernel of that width's latest bound call
        self._shared = {}
        self._plans = {}  # by lanes and whether in column order
        self._args = {} if one_shot else _abi.Calls()
        self._keep = [self.data, self.cols, self.rowptr]  # what a launch reads or writes
        self._order = StreamOrder(self.data.device)

    def kernel_name(self, n_dense_cols=None):
        """The kernel that the latest product of this width ran; without a width, or before a
        product of it, the kernel of the matrix's layout for whole vectors."""
        layout = "spmm_rowblock_kernel" if self._plans or not self.sliced() else "spmm_slices_kernel"
        return self._shared.get(("name", n_dense_cols), layout)

    def describe(self):
        plans = {f"{lanes} by column" if by_column else lanes:
                 {"descriptors": p.n_desc, "split_rows": p.n_split_rows}
                 for (lanes, by_column), p in self._plans.items()}
        return {"layout": "rowblock" if self._plans or not self.sliced() else "slices",
                "plans": plans,
                "slices": {k[0]: int(t[0].numel()) // 2 - 1 for k, t in self._tables.items()}}

    def sliced(self):
        """Whether products run on slices whatever their N.  Row blocks are kept where they are
        the faster: prepared, every row one group's work (and, in _run_spmm, N, B and C whole
        vectors).  Measured on MI355X, row blocks / slices: fp32 N=16, 100k rows of 0 to 32
        entries 18.4 / 20.8 us; N=33, 3M entries 80.6 / 53.0; a power law, N=128 457 / 316, N=47
        326 / 214.  Short rows with a few of more than 128 entries are the faster on row blocks too
        (300k rows of 0 to 60 and 300 of 400, fp32 N=16 53 / 81), but sums are more exact on slices
        (there 1.2e-7 / 6.7e-8 of the result).  A matrix used once has no plan to use.  A prepared
        one with rows of more than _SPMM_SUMS_KEPT entries keeps the row blocks' order of additions
        (see there)."""
        if self.one_shot or self.max_row_nnz is None:
            return True
        return _SPMM_ROW_SPLIT_THRESHOLD < self.max_row_nnz <= _SPMM_SUMS_KEPT

    def slices(self, items, keep, n_cols, by_column):
        """The slices' boundaries and launch order (built on the current stream, once)."""
        key = (items, keep, by_column)
        t = self._tables.get(key)
        if t is None:
            t = _slices.build(self.rowptr, self.n_rows, self.nnz, items, keep, "SpMM",
                              self.cols if by_column else None, n_cols)
            self._tables[key] = t
        return t

    def piece_slots(self, items, table, n_dense_cols, dtype):
        """(the table to launch with, room for the pieces of cut rows, the kind of cut): a slot for
        either end of every slice, or, where that is too much, for each piece.  Calls are ordered
        (StreamOrder), so those of one size share it."""
        length, cut = (table.numel() - 2) * n_dense_cols, 1
        if length * dtype.itemsize > _SUMS_ROOM and (
                ("pieces", items) in self._shared
                or not torch.cuda.is_current_stream_capturing()):  # the count is waited for
            counted = self._shared.get(("pieces", items))
            if counted is None:
                counted = self._shared["pieces", items] = _slices.pieces(self.rowptr, table)
            table, n = counted
            if n == 0:
                return table, None, 0
            length, cut = n * n_dense_cols, _abi.FSP_CUT_PIECES
        sums = self._shared.get(("sums", length, dtype))
        if sums is None:
            sums = torch.empty(length, dtype=dtype, device=table.device)
            self._shared["sums", length, dtype] = sums
        return table, sums, cut

    def plan(self, lanes, row_bytes=0, n_cols=0):
        """The row-block plan for ``lanes``, in the launch order that suits rows of B of
        ``row_bytes`` (widths of several sizes can share a lane count)."""
        ngrp = 256 // lanes
        cap = _abi.caps()["spmm_block_nnz"]
        threshold = min(_SPMM_ROW_SPLIT_THRESHOLD, cap)
        chunk = min(cap, max(threshold, 16 * ngrp))
        by_column = _slices.ordered(self.max_row_nnz, chunk, n_cols * row_bytes,
                                    self.nnz * row_bytes, False)
        p = self._plans.get((lanes, by_column))
        if p is None:
            p = self._shared.get(("row order", lanes))
            if p is None:
                p = self._shared["row order", lanes] = build_row_block_plan_device(
                    self.rowptr, cap, ngrp, threshold, chunk,
                    window_rows=SPMM_PLAN_WINDOW_BLOCKS * ngrp)
            if by_column:
                if torch.cuda.is_current_stream_capturing():
                    return p  # the order would only be written by a replay; the sums are the same
                p = p.in_order(_parts_by_column(p.desc, self.cols, n_cols, self.rowptr, chunk))
            self._plans[lanes, by_column] = p
        return p


# A B of more than half this many bytes is read in column tiles: the widest power of two of
# columns narrower than B whose slice is at most this many bytes (the kernel walks the tiles in
# launch order, so one tile's rows of B are gathered at a time and stay in the 256 MiB MALL for
# longer).  Measured on MI355X, cfg5's matrix: fp32 N=256 (B of 1 GiB) 3.34 -> 2.86 ms with
# tiles of 128 columns (64: 3.01, 32: 2.92); fp64 N=256 6.69 -> 5.82 ms (64); B of 512 MiB:
# fp64 N=64 1437 -> 1372 us (32; 16: 1466), fp32 N=128 1416 -> 1350 us (64; 32: 1490); B of
# 256 MiB is fastest untiled (fp32 N=64 662 vs 710 us with 32; fp64 N=32 689 vs 770 with 16).
SPMM_B_TILE_BYTES = 512 << 20


def _auto_tile_cols(B):
    """Column tile for a large B (None: no tiling), by the rule above."""
    rows, n, v = int(B.shape[0]), int(B.shape[1]), B.element_size()
    if 2 * rows * n * v <= SPMM_B_TILE_BYTES:
        return None
    t = _next_pow2(n)
    while t > 4 and (t >= n or rows * t * v > SPMM_B_TILE_BYTES):
        t >>= 1
    return t if t < n else None


def _bind_sliced(kc, B, acc_f64, lanes, vec):
    n_dense_cols, n_cols, positions = int(B.shape[1]), int(B.shape[0]), kc.n_rows + kc.nnz
    row_bytes = min(n_dense_cols, lanes * vec) * B.element_size()  # of one column tile
    items, keep = _spmm_slice_shape(lanes, positions, True)
    by_column = _slices.ordered(kc.max_row_nnz, items, n_cols * row_bytes, kc.nnz * row_bytes,
                                kc.one_shot)
    if not by_column:
        items, keep = _spmm_slice_shape(lanes, positions)
    table, order = kc.slices(items, keep, n_cols, by_column)
    length = (table.numel() - 2) * n_dense_cols
    if kc.max_row_nnz is None and length > _SUMS_UNSEEN:
        kc.max_row_nnz = int((kc.rowptr[1:] - kc.rowptr[:-1]).max())
    sums, cut = None, 0
    if kc.max_row_nnz is None or kc.max_row_nnz > keep:
        dtype = torch.float64 if acc_f64 else B.dtype
        if kc.one_shot and 8 * length <= _SUMS_ROOM:  # (piece_slots' first answer)
            sums, cut = torch.empty(length, dtype=dtype, device=table.device), 1
        else:
            table, sums, cut = kc.piece_slots((items, keep), table, n_dense_cols, dtype)
    if not kc.one_shot:
        kc._shared["name", n_dense_cols] = "spmm_slices_kernel"
    kc._keep.extend((table, order, sums))
    return _abi.bind(
        "spmm_sliced", _abi.dtype_code(B.dtype), 1 if acc_f64 else 0, kc.data.data_ptr(),
        kc.cols.data_ptr(), kc.rowptr.data_ptr(), kc.rowptr_bits, kc.n_rows, kc.nnz,
        n_dense_cols, table.data_ptr(), None if order is None else order.data_ptr(), items, keep,
        None if sums is None else sums.data_ptr(), cut, lanes, vec, XCD_REMAP)


def _bind_row_blocks(kc, B, acc_f64, lanes, vec):
    n_dense_cols = int(B.shape[1])
    plan = kc.plan(lanes, min(n_dense_cols, lanes * vec) * B.element_size(), int(B.shape[0]))
    if plan.n_desc > _slices.MAX_SLICES:
        return None  # more workgroups than a launch holds (four rows each with 64 lanes)
    partials = plan.workspace(n_dense_cols)
    groups, group_base, split_rows = plan.split_groups()
    p = lambda t: t.data_ptr() if t.numel() else None  # noqa: E731
    # launch_spmm's rule (csrc/spmm.hip)
    ragged = (vec == 1 and lanes >= 32 and n_dense_cols * B.element_size() >= 16
              and (not acc_f64 or B.dtype == torch.float64))
    kc._shared["name", n_dense_cols] = "spmm_ragged_kernel" if ragged else "spmm_rowblock_kernel"
    kc._keep.extend((partials, plan.desc, groups, group_base, split_rows))
    return _abi.bind(
        "spmm_csr", _abi.dtype_code(B.dtype), 1 if acc_f64 else 0, p(kc.data), p(kc.cols),
        p(kc.rowptr), kc.rowptr_bits, kc.n_rows, kc.nnz, n_dense_cols, p(plan.desc), plan.n_desc,
        plan.chunk, lanes, vec, p(partials), p(groups), p(group_base), p(split_rows),
        int(groups.shape[0]), 0 if plan.by_column else XCD_REMAP)


def _run_spmm(kc, B, C, acc_f64, tile_cols=None):
    """C[n_rows, N] = A @ B (B, C contiguous row-major) on slices or row blocks (kc.sliced).
    Without an explicit tile (the reference's block_n), a B over SPMM_B_TILE_BYTES is tiled by
    columns."""
    n_dense_cols = B.shape[1]
    if kc.n_rows == 0 or n_dense_cols == 0:
        return C
    if tile_cols is None and 2 * B.numel() * B.element_size() > SPMM_B_TILE_BYTES:
        tile_cols = _auto_tile_cols(B)
    b, c = B.data_ptr(), C.data_ptr()
    stream = kc._order.stream(C.device, kc._keep)
    # what a launch is bound to follows from the matrix and these
    key = (n_dense_cols, B.dtype, bool(acc_f64), tile_cols, (b | c) & 15 == 0)
    bound = kc._args.get(key)
    if bound is None:
        slice_lanes, slice_vec = _spmm_slice_lanes(n_dense_cols, B.dtype, tile_cols)
        lanes, vec = _spmm_lane_shape(n_dense_cols, B.dtype, B, C, tile_cols)
        kept = not kc.one_shot and (kc.max_row_nnz or 0) > _SPMM_SUMS_KEPT
        # the row-block kernel's loads need aligned vectors
        bound = None
        if not (kc.sliced() or (vec < slice_vec and not kept)):
            bound = _bind_row_blocks(kc, B, acc_f64, lanes, vec)
        if bound is None:
            bound = _bind_sliced(kc, B, acc_f64, slice_lanes, slice_vec)
        kc._args[key] = bound
    _abi.run(bound, b, c, stream)
    return C


def _out_ok_direct(out, inputs):
    if out is None or not out.is_contiguous() or out.data_ptr() % 16:
        return False
    base = out.untyped_storage().data_ptr()
    return all(t.untyped_storage().data_ptr() != base for t in inputs)


# ------------------------------------------------------------------------------------------
# Opt path: prepared object and entry point
# ------------------------------------------------------------------------------------------

_SPMM_OPT_BUCKET_SPECS = (
    {"max_row_nnz": 32, "kind": "batched", "batch_rows": 8, "block_nnz": 32},
    {"max_row_nnz": 128, "kind": "batched", "batch_rows": 4, "block_nnz": 64},
    {"max_row_nnz": 512, "kind": "vector", "batch_rows": 1, "block_nnz": 128},
    {"max_row_nnz": 2048, "kind": "vector", "batch_rows": 1, "block_nnz": 128},
    {"max_row_nnz": None, "kind": "split", "batch_rows": 1, "block_nnz": 256},
)
_SPMM_OPT_LONG_ROW_THRESHOLD = 2048


class PreparedCsrSpmmOpt:
    """Cached CSR metadata for repeated SpMM-opt calls (spmm_csr.py:337-392).

    ``row_buckets`` and the ``long_*`` split attributes reproduce the reference's metadata on
    first access (spmm_csr.py:417-477); the gfx950 kernel runs from its own descriptor plan.
    """

    __slots__ = (
        "data",
        "kernel_indices",
        "kernel_indptr",
        "shape",
        "n_rows",
        "n_cols",
        "row_lengths",
        "max_row_nnz",
        "supports_opt",
        "long_row_fallback_only",
        "_ref_meta",
        "_kernel",
    )

    def __init__(self, data, kernel_indices, kernel_indptr, shape, n_rows, n_cols, row_lengths,
                 max_row_nnz):
        self.data = data
        self.kernel_indices = kernel_indices
        self.kernel_indptr = kernel_indptr
        self.shape = (int(shape[0]), int(shape[1]))
        self.n_rows = int(n_rows)
        self.n_cols = int(n_cols)
        self.row_lengths = row_lengths
        self.max_row_nnz = int(max_row_nnz)
        self.supports_opt = data.dtype in (torch.float32, torch.float64)
        self.long_row_fallback_only = False
        self._ref_meta = None
        self._kernel = None

    def _kernel_csr(self, one_shot=False):
        if self._kernel is None:
            self._kernel = _SpmmKernelCsr(self.data, self.kernel_indices, self.kernel_indptr,
                                          self.max_row_nnz, one_shot)
        return self._kernel

    def _reference_metadata(self):
        if self._ref_meta is None:
            device = self.data.device
            row_index_dtype = (torch.int32 if self.row_lengths.numel() - 1 <= _INDEX_LIMIT_INT32
                               else torch.int64)
            buckets = []
            lower = 0
            long_rows = torch.empty((0,), dtype=row_index_dtype, device=device)
            for spec in _SPMM_OPT_BUCKET_SPECS:
                upper = spec["max_row_nnz"]
                if upper is None:
                    mask = self.row_lengths > lower
                elif lower == 0:
                    mask = self.row_lengths <= upper
                else:
                    mask = (self.row_lengths > lower) & (self.row_lengths <= upper)
                rows = torch.nonzero(mask, as_tuple=False).flatten().to(row_index_dtype)
                if rows.numel():
                    buckets.append({"kind": spec["kind"], "rows": rows,
                                    "batch_rows": spec["batch_rows"],
                                    "block_nnz": spec["block_nnz"]})
                    if spec["kind"] == "split":
                        long_rows = rows
                if upper is not None:
                    lower = upper
            part_rows, starts, ends, ptr = [], [], [], [0]
            if long_rows.numel():
                ip = self.kernel_indptr.to(torch.int64).cpu().tolist()
                for r in long_rows.to(torch.int64).cpu().tolist():
                    cur, end = ip[r], ip[r + 1]
                    while cur < end:
                        part_rows.append(r)
                        starts.append(cur)
                        cur = min(cur + 256, end)
                        ends.append(cur)
                    ptr.append(len(part_rows))
            self._ref_meta = {
                "row_buckets": buckets,
                "long_row_ids": long_rows,
                "long_part_rows": torch.tensor(part_rows, dtype=long_rows.dtype, device=device),
                "long_part_starts": torch.tensor(starts, dtype=torch.int64, device=device),
                "long_part_ends": torch.tensor(ends, dtype=torch.int64, device=device),
                "long_row_part_ptr": torch.tensor(ptr, dtype=torch.int64, device=device),
            }
        return self._ref_meta

    @property
    def row_buckets(self):
        return self._reference_metadata()["row_buckets"]

    @property
    def long_row_ids(self):
        return self._reference_metadata()["long_row_ids"]

    @property
    def long_part_rows(self):
        return self._reference_metadata()["long_part_rows"]

    @property
    def long_part_starts(self):
        return self._reference_metadata()["long_part_starts"]

    @property
    def long_part_ends(self):
        return self._reference_metadata()["long_part_ends"]

    @property
    def long_row_part_ptr(self):
        return self._reference_metadata()["long_row_part_ptr"]


def prepare_spmm_csr_opt(data, indices, indptr, shape):
    """spmm_csr.py:480-522: validation and narrowing; plans and slices are built by the first call
    of each width."""
    return _prepare_spmm_csr_opt(data, indices, indptr, shape, False)


def _prepare_spmm_csr_opt(data, indices, indptr, shape, one_shot):
    """prepare_spmm_csr_opt; one_shot: for a single call, so nothing is planned."""
    (data, kernel_indices, kernel_indptr, n_rows, n_cols, row_lengths,
     max_row_nnz) = _prepare_spmm_csr_matrix(data, indices, indptr, shape)
    prepared = PreparedCsrSpmmOpt(data, kernel_indices, kernel_indptr, shape, n_rows, n_cols,
                                  row_lengths, max_row_nnz)
    if prepared.supports_opt and n_rows > 0:
        prepared._kernel_csr(one_shot)
    return prepared


def _triton_spmm_csr_impl_opt_prepared(prepared, B):
    """spmm_csr.py:1033-1055 checks, then one gfx950 launch (native-precision accumulation)."""
    if not prepared.supports_opt:
        raise TypeError("spmm opt only supports float32 and float64")
    if not B.is_cuda:
        raise ValueError("B must be a CUDA tensor")
    if B.device != prepared.data.device:
        raise ValueError("B must be on the same CUDA device as the sparse matrix")
    if B.dtype != prepared.data.dtype:
        raise TypeError("B dtype must match sparse matrix dtype")
    if B.shape[0] != prepared.n_cols:
        raise ValueError(f"B.shape[0] must be n_cols={prepared.n_cols}, got {B.shape[0]}")
    if B.ndim != 2:
        raise ValueError("B must be a 2D dense tensor")
    return B.contiguous()


def flagsparse_spmm_csr_opt(data=None, indices=None, indptr=None, B=None, shape=None,
                            prepared=None, out=None, return_time=False):
    """CSR SpMM-opt: native float32/float64 path for CSR @ dense (spmm_csr.py:1129-1183)."""
    if prepared is not None and not isinstance(prepared, PreparedCsrSpmmOpt):
        raise TypeError("prepared must be a PreparedCsrSpmmOpt instance")
    if prepared is None:
        if any(arg is None for arg in (data, indices, indptr, shape)):
            raise ValueError(
                "data, indices, indptr, and shape are required when prepared is not provided")
        prepared = _prepare_spmm_csr_opt(data, indices, indptr, shape, True)
    elif shape is not None:
        resolved_shape = (int(shape[0]), int(shape[1]))
        if resolved_shape != prepared.shape:
            raise ValueError(
                f"shape {resolved_shape} does not match prepared.shape {prepared.shape}")
    if B is None:
        raise ValueError("B is required")
    if not prepared.supports_opt:
        raise TypeError("flagsparse_spmm_csr_opt only supports float32 and float64")
    if not B.is_cuda:
        raise ValueError("B must be a CUDA tensor")
    if B.device != prepared.data.device:
        raise ValueError("B must be on the same CUDA device as sparse matrix data")
    if out is not None:
        if not out.is_cuda:
            raise ValueError("out must be a CUDA tensor")
        if out.device != prepared.data.device:
            raise ValueError("out must be on the same CUDA device as sparse matrix data")
        if out.shape != (prepared.n_rows, int(B.shape[1])) or out.dtype != prepared.data.dtype:
            raise ValueError("out shape/dtype must match result")
    t0 = None
    if return_time:
        torch.cuda.synchronize()
        t0 = time.perf_counter()
    B = _triton_spmm_csr_impl_opt_prepared(prepared, B)
    n_dense_cols = int(B.shape[1])
    direct = _out_ok_direct(out, (B, prepared.data))
    C = out if direct else torch.empty((prepared.n_rows, n_dense_cols), dtype=B.dtype,
                                       device=B.device)
    _run_spmm(prepared._kernel_csr(), B, C, acc_f64=B.dtype == torch.float64)
    elapsed_ms = None
    if return_time:
        torch.cuda.synchronize()
        elapsed_ms = (time.perf_counter() - t0) * 1000.0
    if out is not None and not direct:
        out.copy_(C)
        C = out
    if return_time:
        return C, elapsed_ms
    return C


# ------------------------------------------------------------------------------------------
# Base (ALG1) path
# ------------------------------------------------------------------------------------------


def flagsparse_spmm_csr(data, indices, indptr, B, shape, block_n=None, block_nnz=None,
                        max_segments=None, out=None, return_time=False):
    """CSR SpMM C = A @ B (spmm_csr.py:1057-1126).

    float32 is accumulated in float64 and rounded once, as in the reference.  ``block_n``
    sets the column tile of a workgroup; ``block_nnz`` / ``max_segments`` are validated with
    the reference's ALG1 rules (ValueError when max_segments cannot cover the longest row).
    """
    if block_n is not None and block_n <= 0:
        raise ValueError("block_n must be positive when provided")
    if block_nnz is not None and block_nnz <= 0:
        raise ValueError("block_nnz must be positive when provided")
    if max_segments is not None and max_segments <= 0:
        raise ValueError("max_segments must be positive when provided")
    (data, kernel_indices, kernel_indptr, B, n_rows, _n_cols, n_dense_cols,
     max_row_nnz) = _prepare_spmm_csr_inputs(data, indices, indptr, B, shape)
    launch = _resolve_spmm_alg1_launch_config(n_dense_cols, max_row_nnz, block_n=block_n,
                                              block_nnz=block_nnz, max_segments=max_segments)
    if out is not None:
        if not out.is_cuda:
            raise ValueError("out must be a CUDA tensor")
        if out.device != data.device:
            raise ValueError("out must be on the same CUDA device as the inputs")
        if out.shape != (n_rows, n_dense_cols) or out.dtype != data.dtype:
            raise ValueError("out shape/dtype must match result")
    dtype = data.dtype
    t0 = None
    if return_time:
        torch.cuda.synchronize()
        t0 = time.perf_counter()
    if n_rows == 0 or n_dense_cols == 0 or B.shape[0] == 0:
        C = torch.zeros((n_rows, n_dense_cols), dtype=dtype, device=data.device)
        direct = False
    else:
        _require_kernel_dtype(dtype, "flagsparse_spmm_csr")
        kc = _SpmmKernelCsr(data, kernel_indices, kernel_indptr, max_row_nnz, one_shot=True)
        direct = _out_ok_direct(out, (B, data))
        C = out if direct else torch.empty((n_rows, n_dense_cols), dtype=dtype,
                                           device=data.device)
        tile = launch["block_n"] if block_n is not None else None
        _run_spmm(kc, B, C, acc_f64=True, tile_cols=tile)
    elapsed_ms = None
    if return_time:
        torch.cuda.synchronize()
        elapsed_ms = (time.perf_counter() - t0) * 1000.0
    if out is not None and not direct:
        out.copy_(C)
        C = out
    if return_time:
        return C, elapsed_ms
    return C


# ------------------------------------------------------------------------------------------
# Benchmark cases (spmm_csr.py:1195-1562): same result dictionaries; the "triton_*" keys
# name the flagsparse kernel as in the reference, cuSPARSE/CuPy is reported unavailable.
# ------------------------------------------------------------------------------------------


def _torch_sparse_reference(data, indices, indptr, B, shape):
    indptr64 = indptr.to(torch.int64)
    indices64 = indices.to(torch.int64)
    ref_dtype = torch.float64 if data.dtype == torch.float32 else data.dtype
    csr_ref = torch.sparse_csr_tensor(indptr64, indices64, data.to(ref_dtype), size=shape,
                                      device=data.device)
    return torch.sparse.mm(csr_ref, B.to(ref_dtype)).to(data.dtype)


def benchmark_spmm_opt_case(n_rows=4096, n_cols=4096, nnz=65536, n_dense_cols=32,
                            value_dtype=torch.float32, index_dtype=torch.int32, warmup=20,
                            iters=200, run_cusparse=True, seed=0):
    """Base vs opt SpMM against one high-precision torch.sparse reference."""
    if value_dtype not in (torch.float32, torch.float64):
        raise TypeError("benchmark_spmm_opt_case only supports float32 and float64")
    device = torch.device("cuda")
    data, indices, indptr = build_random_csr(n_rows, n_cols, nnz, value_dtype, index_dtype,
                                             device, seed=seed)
    B = build_random_dense((n_cols, n_dense_cols), value_dtype, device, seed=seed)
    shape = (n_rows, n_cols)
    prepared = prepare_spmm_csr_opt(data, indices, indptr, shape)

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    base_values = flagsparse_spmm_csr(data, indices, indptr, B, shape)
    torch.cuda.synchronize()
    base_first_call_ms = (time.perf_counter() - t0) * 1000.0
    base_values, base_ms = _benchmark_cuda_op(
        lambda: flagsparse_spmm_csr(data, indices, indptr, B, shape), warmup=warmup, iters=iters)

    torch.cuda.synchronize()
    t0 = time.perf_counter()
    opt_values = flagsparse_spmm_csr_opt(B=B, prepared=prepared)
    torch.cuda.synchronize()
    opt_first_call_ms = (time.perf_counter() - t0) * 1000.0
    opt_values, opt_ms = _benchmark_cuda_op(
        lambda: flagsparse_spmm_csr_opt(B=B, prepared=prepared), warmup=warmup, iters=iters)

    ref = _torch_sparse_reference(data, indices, indptr, B, shape)
    pt_ms = None
    try:
        pt_sparse = torch.sparse_csr_tensor(indptr.to(torch.int64), indices.to(torch.int64),
                                            data, size=shape, device=device)
        _, pt_ms = _benchmark_cuda_op(lambda: torch.sparse.mm(pt_sparse, B), warmup=warmup,
                                      iters=iters)
    except Exception:
        pt_ms = None
    err_base = _spmm_opt_reference_error(base_values, ref, value_dtype)
    err_opt = _spmm_opt_reference_error(opt_values, ref, value_dtype)
    return {
        "parameters": {"n_rows": n_rows, "n_cols": n_cols, "nnz": nnz,
                       "n_dense_cols": n_dense_cols, "value_dtype": str(value_dtype),
                       "index_dtype": str(index_dtype)},
        "performance": {
            "base_ms": base_ms, "base_first_call_ms": base_first_call_ms, "opt_ms": opt_ms,
            "opt_first_call_ms": opt_first_call_ms, "pt_ms": pt_ms, "cu_ms": None,
            "opt_vs_base": (base_ms / opt_ms if opt_ms and opt_ms > 0 else None),
            "opt_vs_pt": (pt_ms / opt_ms if pt_ms is not None and opt_ms > 0 else None),
            "opt_vs_cu": None,
        },
        "verification": {"err_base": err_base, "err_opt": err_opt, "base_ok": err_base <= 1.0,
                         "opt_ok": err_opt <= 1.0,
                         "status": ("PASS" if err_opt <= 1.0 else "FAIL")},
        "backend_status": {"long_row_fallback_used": bool(prepared.long_row_fallback_only),
                           "flagsparse_internal_route": "gfx950-rowblock"},
        "samples": {"base": base_values, "opt": opt_values, "reference": ref},
    }


def benchmark_spmm_case(n_rows=4096, n_cols=4096, nnz=65536, n_dense_cols=32,
                        value_dtype=torch.float32, index_dtype=torch.int32, warmup=20, iters=200,
                        block_n=None, block_nnz=None, max_segments=None, run_cusparse=True,
                        seed=0):
    """flagsparse SpMM vs torch.sparse.mm (CuPy/cuSPARSE is not part of this build)."""
    device = torch.device("cuda")
    data, indices, indptr = build_random_csr(n_rows, n_cols, nnz, value_dtype, index_dtype,
                                             device, seed=seed)
    B = build_random_dense((n_cols, n_dense_cols), value_dtype, device, seed=seed)
    shape = (n_rows, n_cols)
    max_row_nnz = int(torch.max(indptr[1:] - indptr[:-1]).item()) if n_rows > 0 else 0
    launch = _resolve_spmm_alg1_launch_config(n_dense_cols, max_row_nnz, block_n=block_n,
                                              block_nnz=block_nnz, max_segments=max_segments)
    kwargs = {"data": data, "indices": indices, "indptr": indptr, "B": B, "shape": shape,
              "block_n": launch["block_n"], "block_nnz": launch["block_nnz"],
              "max_segments": launch["max_segments"], "return_time": False}
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    _ = flagsparse_spmm_csr(**kwargs)
    torch.cuda.synchronize()
    first_call_ms = (time.perf_counter() - t0) * 1000.0
    triton_C, triton_ms = _benchmark_cuda_op(lambda: flagsparse_spmm_csr(**kwargs),
                                             warmup=warmup, iters=iters)
    pytorch_reason = None
    pytorch_ms = None
    expected = _torch_sparse_reference(data, indices, indptr, B, shape)
    pytorch_values = expected
    try:
        csr_pt = torch.sparse_csr_tensor(indptr.to(torch.int64), indices.to(torch.int64), data,
                                         size=shape, device=device)
        pytorch_values, pytorch_ms = _benchmark_cuda_op(lambda: torch.sparse.mm(csr_pt, B),
                                                        warmup=warmup, iters=iters)
    except Exception as exc:
        pytorch_reason = str(exc)
    metrics = _spmm_validation_metrics(triton_C, expected)
    threshold = _spmm_relative_threshold(value_dtype)
    return {
        "parameters": {
            "format": "csr", "n_rows": n_rows, "n_cols": n_cols, "nnz": nnz,
            "n_dense_cols": n_dense_cols, "value_dtype": str(value_dtype),
            "index_dtype": str(index_dtype), "warmup": warmup, "iters": iters,
            "block_n": launch["block_n"], "block_nnz": launch["block_nnz"],
            "max_segments": launch["max_segments"],
            "required_segments": launch["required_segments"],
            "alg1_warp_size": launch["warp_size"], "alg1_factor": launch["factor"],
            "auto_max_segments": launch["auto_max_segments"], "run_cusparse": run_cusparse,
        },
        "performance": {
            "pytorch_ms": pytorch_ms, "triton_ms": triton_ms,
            "triton_first_call_ms": first_call_ms, "cusparse_ms": None,
            "triton_speedup_vs_pytorch": (pytorch_ms / triton_ms
                                          if pytorch_ms is not None and triton_ms > 0 else None),
            "triton_speedup_vs_cusparse": None,
        },
        "verification": {
            "triton_match_reference": metrics["strict_allclose_match"],
            "triton_match_pytorch": metrics["strict_allclose_match"],
            "triton_max_error": metrics["max_abs_error"],
            "triton_max_abs_error": metrics["max_abs_error"],
            "triton_max_relative_error": metrics["max_relative_error"],
            "triton_sum_relative_error": metrics["sum_relative_error"],
            "triton_relative_threshold": metrics["relative_threshold"],
            "triton_strict_allclose_match": metrics["strict_allclose_match"],
            "pytorch_match_reference": True, "pytorch_max_error": 0.0,
            "pytorch_max_abs_error": 0.0, "pytorch_max_relative_error": 0.0,
            "pytorch_sum_relative_error": 0.0, "pytorch_relative_threshold": threshold,
            "cusparse_match_reference": None, "cusparse_match_pytorch": None,
            "cusparse_max_error": None, "cusparse_max_abs_error": None,
            "cusparse_max_relative_error": None, "cusparse_sum_relative_error": None,
            "cusparse_relative_threshold": threshold, "cusparse_strict_allclose_match": None,
        },
        "backend_status": {
            "pytorch_unavailable_reason": pytorch_reason, "pytorch_sparse_format": "CSR",
            "cusparse_unavailable_reason": "CuPy/cuSPARSE is not part of the MI355X build",
            "flagsparse_internal_route": "gfx950-rowblock",
        },
        "samples": {"pytorch": pytorch_values, "triton": triton_C, "reference": expected,
                    "cusparse": None},
    }


def comprehensive_spmm_test(n_rows=4096, n_cols=4096, nnz=65536, n_dense_cols=32,
                            dtype=torch.float32, index_dtype=torch.int32, warmup=20, iters=200,
                            block_n=None, block_nnz=None, max_segments=None, run_cusparse=True):
    """Full SpMM benchmark entry for one configuration (spmm_csr.py:1534-1562)."""
    return benchmark_spmm_case(n_rows=n_rows, n_cols=n_cols, nnz=nnz, n_dense_cols=n_dense_cols,
                               value_dtype=dtype, index_dtype=index_dtype, warmup=warmup,
                               iters=iters, block_n=block_n, block_nnz=block_nnz,
                               max_segments=max_segments, run_cusparse=run_cusparse)
