"""The rules that pick slice sizes and launch orders (no GPU)."""

import copy
import pickle

import numpy as np
import pytest
import torch

from flagsparse_amd import _abi, _slices, _spmv_layouts, sddmm_csr, spmm_csr


@pytest.mark.parametrize("n,dtype,tile,want", [
    (1, torch.float32, None, (1, 1)), (2, torch.float32, None, (1, 2)),
    (3, torch.float32, None, (4, 1)), (4, torch.float32, None, (1, 4)),
    (5, torch.float32, None, (2, 4)), (47, torch.float32, None, (16, 4)),
    (300, torch.float32, None, (64, 4)), (255, torch.float32, 128, (32, 4)),
    (1, torch.float64, None, (1, 1)), (3, torch.float64, None, (2, 2)),
    (100, torch.float64, None, (64, 2)), (7, torch.float32, 1, (1, 4)),
])
def test_spmm_slice_lanes(n, dtype, tile, want):
    lanes, vec = spmm_csr._spmm_slice_lanes(n, dtype, tile)
    assert (lanes, vec) == want and vec <= n


@pytest.mark.parametrize("by_column", [False, True])
def test_spmm_slice_shape_limits(by_column):
    for lanes in (1, 2, 4, 8, 16, 32, 64):
        for positions in (1, 1000, 10**6, 10**9):
            items, keep = spmm_csr._spmm_slice_shape(lanes, positions, by_column)
            # the kernel stages at most 2 * 1024 entries and cuts rows longer than keep
            assert 64 <= items and items + keep + 6 <= 2048 and 128 <= keep <= 2 * items


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_sddmm_slice_lanes(dtype):
    vmax = 4 if dtype == torch.float32 else 2
    for K in range(1, 1500):
        lanes, vec = sddmm_csr._sddmm_slice_lanes(K, dtype)
        assert vec <= K and vec == (vmax if K >= vmax else min(K, 2))
        assert K <= 4 * lanes * vec or lanes == 64
        assert 64 <= sddmm_csr._sddmm_slice_items(lanes, 1 << 40) <= 2048


def test_ordered_rule():
    big = 1 << 30
    assert _slices.ordered(5000, 256, big, big, True)
    assert not _slices.ordered(None, 256, big, big, True)     # longest row unknown
    assert not _slices.ordered(1000, 256, big, big, True)     # no row holds several slices
    assert not _slices.ordered(5000, 256, 4 << 20, big, True)  # fits an L2
    assert not _slices.ordered(5000, 256, big, 200 << 20, True)
    assert _slices.ordered(5000, 256, big, 200 << 20, False)


def _stencil(side):
    i = torch.arange(side * side)
    r, c = i // side, i % side
    valid = torch.stack([r > 0, c > 0, r >= 0, c < side - 1, r < side - 1], 1)
    cols = (i[:, None] + torch.tensor([-side, -1, 0, 1, side])[None, :])[valid]
    return valid.sum(1), cols, side * side


def _random(lengths, n_cols):
    gen = torch.Generator().manual_seed(1)
    lengths = torch.as_tensor(lengths)
    return lengths, torch.randint(0, n_cols, (int(lengths.sum()),), generator=gen), n_cols


def _with_rows(matrix, rows, length):
    """``rows`` rows of ``length`` spread-out entries in the middle of a matrix."""
    lengths, cols, n_cols = matrix
    half = lengths.numel() // 2
    entries = int(lengths[:half].sum())
    _, more, _ = _random([length] * rows, n_cols)
    return (torch.cat([lengths[:half], torch.full((rows,), length), lengths[half:]]),
            torch.cat([cols[:entries], more, cols[entries:]]), n_cols)


_ZIPF = torch.as_tensor(np.minimum(np.random.default_rng(2).zipf(1.8, 40000), 9000))


@pytest.mark.parametrize("matrix,want", [
    # local or alike rows with a few long ones keep the row blocks and their launch order
    (_with_rows(_stencil(300), 1, 1100), False), (_with_rows(_stencil(300), 1, 20000), False),
    (_with_rows(_random([12] * 40000, 40000), 1, 1100), False),
    (_with_rows(_random([12] * 40000, 40000), 20, 2000), False),
    # no row longer than a block
    (_with_rows(_random([2] * 40000, 40000), 2000, 400), False),
    # rows of very different lengths side by side
    (_random(_ZIPF, 40000), True),
    (_with_rows(_with_rows(_random([6] * 40000, 40000), 60, 400), 1, 3000), True),
    # a large share in rows cut into chunks; spread-out columns with one of those
    (_with_rows(_stencil(300), 20, 5000), True),
    (_with_rows(_random([12] * 40000, 40000), 1, 5000), True),
])
def test_prepared_spmv_layout_rule(matrix, want):
    lengths, cols, n_cols = matrix
    rowptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(torch.int32)
    cols = cols.to(torch.int32)
    uneven, block, chunk = _spmv_layouts.row_class_bounds(lengths.numel(), cols.numel())
    assert _spmv_layouts.slices_pay(
        cols, rowptr, n_cols, int(lengths.max()),
        int(((lengths > uneven) & (lengths <= block)).sum()),
        int(lengths[lengths > chunk].sum())) == want


def test_copies_start_without_calls():
    calls = _abi.Calls(base=("buffer", 4096))
    assert dict(calls) and not copy.deepcopy({"a": calls})["a"]
    assert not copy.copy(calls) and not pickle.loads(pickle.dumps(calls))


@pytest.mark.parametrize("by_column", [False, True])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16, 32, 64])
def test_spmm_slices_fit_a_launch(lanes, by_column):
    for positions in (1 << 31, (1 << 31) + (1 << 25), 10**10, 1 << 34, _slices.MAX_SLICES * 128,
                      _slices.MAX_SLICES * 128 + 1):
        items, keep = spmm_csr._spmm_slice_shape(lanes, positions, by_column)
        assert -(-positions // items) <= _slices.MAX_SLICES and items + keep + 6 <= 2048


def test_spmv_slices_fit_a_launch(monkeypatch):
    lengths, cols, n_cols = _random([12] * 2000, 2000)
    rowptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    built = []
    monkeypatch.setattr(_spmv_layouts, "SliceLayout", lambda *a, **k: built.append("slices"))
    monkeypatch.setattr(_spmv_layouts, "RowBlockLayout", lambda *a, **k: built.append("rowblock"))
    data, cols = torch.ones(cols.numel()), cols.to(torch.int32)
    for limit in (_slices.MAX_SLICES, 10):  # the matrix has 35 slices
        monkeypatch.setattr(_slices, "MAX_SLICES", limit)
        _spmv_layouts.build_layout(data, cols, rowptr, n_cols, one_shot=True)
        _spmv_layouts.build_layout(data, cols, rowptr, n_cols, max_row_nnz=5000,
                                   row_classes=[0, cols.numel()])
    assert built == ["slices", "slices", "rowblock", "rowblock"]
