"""The largest matrix that 32-bit row pointers reach, 2^31 - 1 entries: the last quads of entries end
at the type's limit, and no kernel's index arithmetic may run past it.  All values are 1, so every
row's sum is its length, exactly."""

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _common, _spmv_layouts

pytestmark = pytest.mark.gpu

NNZ = 2**31 - 1
COLS = 1024


@pytest.fixture(scope="module")
def entries(dev):
    """(values, columns): 17 GB, shared by the tests of this file."""
    assert NNZ == _common.ROWPTR32_MAX_NNZ
    cols = torch.arange(NNZ, dtype=torch.int32, device=dev).bitwise_and_(COLS - 1)
    yield torch.ones(NNZ, device=dev), cols
    torch.cuda.synchronize()
    torch.cuda.empty_cache()


def _matrix(entries, length, dev):
    """Rows of ``length`` entries, the last one short of one."""
    n = (NNZ + 1) // length
    ptr = (torch.arange(n + 1, dtype=torch.int64, device=dev) * length).clamp_(max=NNZ)
    want = torch.full((n,), float(length), device=dev)
    want[-1] -= 1
    return entries[0], entries[1], ptr.to(torch.int32), (n, COLS), want


def test_spmv_last_entries(dev, entries, monkeypatch):
    x = torch.ones(COLS, device=dev)
    for length in (64, 16384):  # whole rows to a block; rows cut into chunks and slices
        data, cols, ptr, shape, want = _matrix(entries, length, dev)
        for opt in (False, True):
            print(f"spmv one call, rows of {length}, opt={opt}", flush=True)
            y = fs.flagsparse_spmv_csr(data, cols, ptr, x, shape, use_opt=opt)
            assert torch.equal(y, want)
        print(f"spmv row blocks, rows of {length}", flush=True)
        monkeypatch.setattr(_spmv_layouts, "FORCE", "rowblock")
        p = fs.prepare_spmv_csr(data, cols, ptr, shape)
        assert p._kernel(False).kind == "rowblock" and p._kernel(False).rowptr_bits == 32
        assert torch.equal(fs.flagsparse_spmv_csr(x=x, prepared=p), want)
        monkeypatch.undo()
        del p


@pytest.mark.parametrize("length,n", [(64, 4), (16384, 4), (16384, 47)])
def test_spmm_last_entries(dev, entries, length, n):
    data, cols, ptr, shape, want = _matrix(entries, length, dev)
    B = torch.ones(COLS, n, device=dev)
    print(f"spmm one call, rows of {length}, N={n}", flush=True)
    C = fs.flagsparse_spmm_csr_opt(data, cols, ptr, B, shape)
    assert torch.equal(C, want[:, None].expand_as(C))
    print(f"spmm row blocks, rows of {length}, N={n}", flush=True)
    p = fs.prepare_spmm_csr_opt(data, cols, ptr, shape)
    C = fs.flagsparse_spmm_csr_opt(B=B, prepared=p)
    assert p._kernel_csr()._plans and p._kernel_csr().rowptr_bits == 32
    assert torch.equal(C, want[:, None].expand_as(C))


def test_spmm_many_slices(dev, entries):
    # 64 lanes take the smallest slices: 2^31 rows + entries of them must still fit one launch (a
    # larger grid runs modulo 2^32 threads, and leaves rows unwritten)
    data, cols, ptr, shape, want = _matrix(entries, 64, dev)
    C = fs.flagsparse_spmm_csr_opt(data, cols, ptr, torch.ones(COLS, 256, device=dev), shape)
    for k in range(0, shape[0], 1 << 22):
        part = C[k:k + (1 << 22)]
        assert torch.equal(part, want[k:k + (1 << 22), None].expand_as(part))
