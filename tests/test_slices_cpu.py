"""The rules that pick slice sizes and launch orders (no GPU)."""

import pytest
import torch

from flagsparse_amd import _slices, sddmm_csr, spmm_csr


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
