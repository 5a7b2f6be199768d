"""The radix sort by row and the row pointers of COO calls (csrc/coo_sort.hip) against torch's
stable sort, at the sizes where they can go wrong: tile edges, one to four passes, digits that no
entry or every entry has, all index and value types; and the calls that use them."""

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _common, spmv_coo, synthetic
from flagsparse_amd._coo_order import row_pointers, rows_in_order
from flagsparse_amd._csr_check import coo_check
from oracle import oracle

pytestmark = pytest.mark.gpu

TILE = 2048  # entries of a tile below 2^20 entries, 4096 from there on; 32 tiles need no scan


@pytest.mark.parametrize("nnz", [1, 63, 64, TILE - 1, TILE, TILE + 1, 5 * TILE + 17, 32 * TILE,
                                 32 * TILE + 1, (1 << 20) - 1, 1 << 20])
@pytest.mark.parametrize("max_row", [1, 255, 511, 512, 70000, 262143, 262144, (1 << 27) + 5,
                                     2**31 - 2])
def test_rows_in_order(dev, nnz, max_row):
    row = synthetic.randint(4, nnz, nnz, max_row + 1, "cpu")
    row[nnz // 2] = max_row
    kinds = [(torch.int32, torch.int32, torch.float32), (torch.int64, torch.int64, torch.float64),
             (torch.int32, torch.int64, torch.float64), (torch.int64, torch.int32, torch.float32)]
    for rt, ct, vt in kinds if nnz < 2 * TILE else kinds[1:3]:
        col = torch.arange(nnz, dtype=ct)  # the input position: shows the order inside a row
        val = torch.arange(nnz, dtype=vt)
        print(f"sort nnz={nnz} max_row={max_row} {rt} {ct} {vt}", flush=True)
        v, r, c = rows_in_order(val.to(dev), row.to(rt).to(dev), col.to(dev), max_row)
        want = torch.sort(row, stable=True)
        assert r.dtype == c.dtype == torch.int32 and v.dtype == vt
        assert torch.equal(r.cpu().to(torch.int64), want.values)
        assert torch.equal(c.cpu().to(torch.int64), want.indices)
        assert torch.equal(v.cpu(), val[want.indices])


@pytest.mark.parametrize("rows", [[5] * 9000, list(range(9000)), list(range(8999, -1, -1)),
                                  [0, 8999] * 4500, [7] * 4096 + [3] * 4096 + [8000] * 5])
def test_rows_in_order_patterns(dev, rows):
    row = torch.tensor(rows)
    col = torch.arange(row.numel(), dtype=torch.int32)
    _, r, c = rows_in_order(col.to(dev).to(torch.float32), row.to(dev), col.to(dev), 8999)
    want = torch.sort(row, stable=True)
    assert torch.equal(r.cpu().to(torch.int64), want.values)
    assert torch.equal(c.cpu().to(torch.int64), want.indices)


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("bits64", [False, True])
def test_row_pointers(dev, monkeypatch, dtype, bits64):
    if bits64:
        monkeypatch.setattr(_common, "ROWPTR32_MAX_NNZ", 0)
    for n_rows, nnz in ((1, 1), (5, 0), (1000, 3), (300, 5000), (70001, 100000)):
        row = torch.sort(synthetic.randint(5, n_rows, nnz, n_rows, "cpu")).values
        ptr = row_pointers(row.to(dtype).to(dev), n_rows)
        assert ptr.dtype == (torch.int64 if bits64 and nnz else torch.int32)
        want = torch.searchsorted(row, torch.arange(n_rows + 1))
        assert torch.equal(ptr.cpu().to(torch.int64), want)


@pytest.mark.parametrize("n_rows", [(1 << 17) - 1, 1 << 17, (1 << 17) + 1, (1 << 17) + 255])
@pytest.mark.parametrize("lengths", [
    [1], [65], [0] * 255 + [300], [64] * 256, [64] * 255 + [65], [3] + [0] * 1000, [0] * 511 + [2000],
    [16384, 0, 1] + [0] * 997, [16385] + [0] * 255 + [3], [5] * 254 + [20000, 7, 0, 0, 2],
    [150000] + [0] * 200000],
    ids=lambda v: f"{len(v)}rows_{sum(v)}")
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_row_pointers_blocks(dev, n_rows, lengths, dtype):
    """Around the rows from which the entries are read once, around 256 pointers and 64 * 256
    entries of a workgroup, and multiples of the 65 parts that a search step cuts its range into;
    ``lengths`` is repeated over the rows."""
    n = torch.tensor((lengths * (n_rows // len(lengths) + 1))[:n_rows])
    n[-1] += max(0, n_rows - int(n.sum()))  # as many entries as rows, or more
    row = torch.repeat_interleave(torch.arange(n_rows), n).to(dtype)
    want = torch.cat([torch.zeros(1, dtype=torch.int64), n.cumsum(0)])
    assert torch.equal(row_pointers(row.to(dev), n_rows).cpu().to(torch.int64), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
@pytest.mark.parametrize("order", ["sorted", "rows", "any"])
def test_coo_calls(dev, dtype, index, order):
    # row-ordered rows with unordered columns, unordered entries with repeats, empty rows
    n_rows, n_cols, nnz = 3001, 2003, 20011
    data, row, col = synthetic.build_random_coo(n_rows, n_cols, nnz, dtype, index, "cpu", seed=9)
    row[row % 7 == 3] = 5
    if order != "any":
        perm = torch.sort(row.to(torch.int64) * (n_cols if order == "sorted" else 1)
                          + (col if order == "sorted" else 0), stable=True).indices
        data, row, col = data[perm], row[perm], col[perm]
    d, r, c = (t.to(dev) for t in (data, row, col))
    x = synthetic.uniform_values(9, 3, n_cols, dtype, "cpu")
    bound = oracle.REL_L2_BOUND[str(dtype)[6:]]
    print(f"coo calls {dtype} {index} {order}", flush=True)
    y = fs.flagsparse_spmv_coo(d, r, c, x.to(dev), (n_rows, n_cols))
    ref = oracle.spmv_coo(row, col, data, x, n_rows)
    assert oracle.rel_l2(y, ref) <= bound
    assert torch.equal(y, fs.flagsparse_spmv_coo(d, r, c, x.to(dev), (n_rows, n_cols)))
    p = fs.prepare_spmv_coo(d, r, c, (n_rows, n_cols))
    assert oracle.rel_l2(fs.flagsparse_spmv_coo(x=x.to(dev), prepared=p), ref) <= bound
    for N in (1, 5, 24):
        B = synthetic.dense_uniform(n_cols, N, dtype, seed=N, device="cpu")
        C = fs.flagsparse_spmm_coo(d, r, c, B.to(dev), (n_rows, n_cols))
        assert oracle.rel_l2(C, oracle.spmm_coo(row, col, data, B, n_rows)) <= bound
        assert torch.equal(C, fs.flagsparse_spmm_coo(d, r, c, B.to(dev), (n_rows, n_cols)))


def test_coo_one_call_routes(dev):
    # many more rows than entries, other index types and no entries go the prepared way
    data, row, col = synthetic.build_random_coo(100, 50, 400, torch.float32, torch.int64, dev, 3)
    one = spmv_coo._prepare_one_call
    assert one(data, row, col, (100, 50), True)._layout.kind == "slices"
    assert one(data, row, col, ((1 << 26) + 1, 50), True)._layout.kind == "rowblock"
    assert one(data, row.to(torch.int16), col, (100, 50), True)._layout.kind == "rowblock"
    assert one(data[:0], row[:0], col[:0], (100, 50), True)._layout is None
    assert not one(data, row, col, (100, 50), False).use_seg_kernel
    x = torch.ones(50, device=dev)
    want = fs.flagsparse_spmv_coo(data, row, col, x, (100, 50))
    got = fs.flagsparse_spmv_coo(data, row.to(torch.int16), col.to(torch.int16), x, (100, 50))
    torch.testing.assert_close(got, want)
    for bad, exc in (((row - 1, col), "row indices"), ((row, col + 50), "col indices")):
        with pytest.raises(IndexError, match=exc):
            fs.flagsparse_spmv_coo(data, *bad, x, (100, 50))


@pytest.mark.parametrize("nnz", [1, 3, 4, 1023, 1024, 1025, 2047, 70001, 5000003])
@pytest.mark.parametrize("rt", [torch.int32, torch.int64])
@pytest.mark.parametrize("ct", [torch.int32, torch.int64])
def test_coo_check(dev, nnz, rt, ct):
    row = synthetic.randint(6, 1, nnz, 50001, "cpu") - 7
    col = synthetic.randint(6, 2, nnz, 90001, "cpu")
    for order in ("any", "sorted", "one"):
        r = row if order == "any" else torch.sort(row).values
        if order == "one" and nnz > 1:  # a single decrease, across a quad or workgroup step
            r[-1] = r[0] - 1
        want = [int(r.min()), int(r.max()), int(col.min()), int(col.max()),
                int((r[1:] < r[:-1]).sum())]
        for shift in (0, 1):
            rd = torch.cat([r.new_zeros(shift), r]).to(rt).to(dev)[shift:]
            cd = torch.cat([col.new_zeros(shift), col]).to(ct).to(dev)[shift:]
            stats, r32, c32 = coo_check(rd, cd)
            assert stats == want, (order, shift)
            assert r32.dtype == c32.dtype == torch.int32
            assert torch.equal(r32.cpu().to(torch.int64), r)
            assert torch.equal(c32.cpu().to(torch.int64), col)


def test_checks_wait_for_queued_work(dev):
    # indices still being written by earlier work of the stream, longer than the host watches for
    row = torch.zeros(40000, dtype=torch.int64, device=dev)
    big = torch.randn(4096, 4096, device=dev)
    for _ in range(2):
        out = big
        for _ in range(12):
            out = out @ big * 1e-3
        row.copy_(torch.arange(40000, device=dev) + (out[0, 0] * 0).to(torch.int64))
        stats, r32, _ = coo_check(row, row)
        assert stats == [0, 39999, 0, 39999, 0]
        assert torch.equal(r32.to(torch.int64), torch.arange(40000, device=dev))
        row.zero_()


def test_checks_refuse_capture(dev):
    row = torch.zeros(10, dtype=torch.int32, device=dev)
    data = torch.ones(10, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="captured"):
        with torch.cuda.graph(g):
            fs.flagsparse_spmv_coo(data, row, row, data, (10, 10))
    torch.cuda.synchronize()
    assert float(fs.flagsparse_spmv_coo(data, row, row, data, (10, 10))[0]) == 10.0
