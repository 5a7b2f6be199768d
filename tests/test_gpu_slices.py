"""Sliced CSR SpMV (csrc/slices.hip: a matrix used once) and the one-pass CSR checks
(csrc/check.hip) against the fp64 oracle and torch, at the sizes where they can go wrong: rows at
the longest uncut length and beyond it, rows crossing several slices, runs of empty rows wider
than a slice, row starts on slice boundaries, unaligned arrays."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _abi, _common, synthetic
from flagsparse_amd._csr_check import csr_check
from flagsparse_amd._spmv_layouts import SliceLayout
from oracle import oracle

pytestmark = pytest.mark.gpu

KEEP, ITEMS = 256, 760  # fsp_spmv_slice_keep() and the positions of a slice
LENGTHS = {
    "empty": [0] * 5000,
    "one_entry": [0] * 2000 + [1] + [0] * 3000,
    "one_row": [20000],
    "at_keep": [KEEP, KEEP + 1, KEEP - 1, 0, 3] * 40,
    "crossing": [5, 4000, 0, 0, 1, 761, 7, 759, 760, 0, 100000, 2] + [0] * 2000 + [3000] * 5,
    "boundary": [ITEMS - 1] * 9 + [0] * ITEMS + [ITEMS - 1, 1, ITEMS * 3 - 1, 0],
    "short": [1, 0, 2, 5] * 3000,
    "mixed": [900] + [1] * 100 + [255] * 3 + [0] * 900 + [600, 1, 600],
}


def _csr(lengths, n_cols, seed, dtype):
    ip = torch.zeros(len(lengths) + 1, dtype=torch.int64)
    ip[1:] = torch.cumsum(torch.as_tensor(lengths), 0)
    nnz = int(ip[-1])
    cols = synthetic.randint(seed, 1, nnz, n_cols, "cpu")
    return synthetic.uniform_values(seed, 2, nnz, dtype, "cpu"), cols, ip


@pytest.mark.parametrize("name", sorted(LENGTHS))
@pytest.mark.parametrize("dtype,opt", [(torch.float32, False), (torch.float32, True),
                                       (torch.float64, False)])
@pytest.mark.parametrize("bits64", [False, True])
def test_sliced_spmv(dev, monkeypatch, name, dtype, opt, bits64):
    if bits64:  # the 64-bit row pointers of matrices past 2^31 entries, on a small one
        monkeypatch.setattr(_common, "ROWPTR32_MAX_NNZ", 0)
    lengths = LENGTHS[name]
    vals, cols, ip = _csr(lengths, 3001, 5, dtype)
    x = synthetic.uniform_values(5, 3, 3001, dtype, "cpu")
    shape = (len(lengths), 3001)
    assert _abi.lib().fsp_spmv_slice_keep() == KEEP
    print(f"sliced spmv {name} {dtype} opt={opt} bits64={bits64}", flush=True)
    args = [vals.to(dev), cols.to(dev), ip.to(dev), x.to(dev)]
    y = fs.flagsparse_spmv_csr(*args, shape, use_opt=opt)
    ref = oracle.spmv_csr(ip, cols, vals, x)
    assert oracle.rel_l2(y, ref) <= oracle.REL_L2_BOUND[str(dtype)[6:]]
    if dtype == torch.float32 and not opt:  # one rounding of an fp64 sum
        np.testing.assert_allclose(y.cpu().numpy(), ref, rtol=1.2e-7, atol=1e-12)
    assert torch.equal(y, fs.flagsparse_spmv_csr(*args, shape, use_opt=opt))
    # arrays that start between 16-byte boundaries
    if vals.numel():
        off = [torch.cat([t[:1], t])[1:] for t in args[:2]]
        assert torch.equal(y, fs.flagsparse_spmv_csr(*off, args[2], args[3], shape, use_opt=opt))
    # the prepared row-block path agrees to rounding
    p = fs.prepare_spmv_csr(*args[:3], shape)
    tol = 1e-5 if dtype == torch.float32 else 1e-12
    assert oracle.rel_l2(fs.flagsparse_spmv_csr(x=args[3], prepared=p, use_opt=opt), ref) <= tol


@pytest.mark.parametrize("name,kind", [("crossing", "slices"), ("mixed", "rowblock"),
                                       ("one_row", "slices"), ("short", "rowblock")])
def test_prepared_layout(dev, name, kind):
    # rows longer than a row block: the prepared matrix runs on slices whose table it keeps
    vals, cols, ip = _csr(LENGTHS[name], 3001, 8, torch.float32)
    shape = (len(LENGTHS[name]), 3001)
    p = fs.prepare_spmv_csr(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    assert p._kernel(False).kind == kind
    for k in range(3):
        x = synthetic.uniform_values(9 + k, 3, 3001, torch.float32, "cpu")
        y = fs.flagsparse_spmv_csr(x=x.to(dev), prepared=p)
        assert oracle.rel_l2(y, oracle.spmv_csr(ip, cols, vals, x)) <= 1e-5
    one = fs.flagsparse_spmv_csr(vals.to(dev), cols.to(dev), ip.to(dev), x.to(dev), shape)
    if kind == "slices":
        assert torch.equal(one, y)


def test_prepare_leaves_nothing_queued(dev):
    """A prepared matrix's narrowed copies may be read on any stream, by what orders nothing
    (rows truncated later, the row lengths), so prepare waits for the stream that wrote them."""
    d, c, ip = (t.to(dev) for t in _csr([5000] + [12] * 300000, 100000, 5, torch.float32))
    torch.cuda.synchronize()
    side = torch.cuda.Stream(dev)
    with torch.cuda.stream(side):
        prepared = fs.prepare_spmv_csr(d, c, ip, (300001, 100000))
        done = side.query()
    assert done
    assert prepared._kernel(False).kind == "slices"


def test_sliced_spmv_nonfinite(dev):
    # an infinity and a NaN of x reach the rows that name them and no others
    vals, cols, ip = _csr(LENGTHS["crossing"], 3001, 6, torch.float32)
    x = synthetic.uniform_values(6, 3, 3001, torch.float32, "cpu")
    x[0], x[17] = float("inf"), float("nan")
    shape = (len(LENGTHS["crossing"]), 3001)
    y = fs.flagsparse_spmv_csr(vals.to(dev), cols.to(dev), ip.to(dev), x.to(dev), shape)
    lay = SliceLayout(vals.to(dev), cols.to(torch.int32).to(dev), ip.to(dev))
    assert lay.cut_rows  # an unknown longest row
    y2 = torch.empty_like(y)
    lay.launch(x.to(dev), y2, True)
    ref = oracle.spmv_csr(ip, cols, vals, x)
    for got in (y.cpu().numpy(), y2.cpu().numpy()):
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
        np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))


@pytest.mark.parametrize("idx", [torch.int32, torch.int64])
@pytest.mark.parametrize("ptr", [torch.int32, torch.int64])
@pytest.mark.parametrize("n_rows,nnz", [(0, 0), (1, 0), (7, 1), (3000, 4099), (500, 3000001)])
def test_csr_check(dev, idx, ptr, n_rows, nnz):
    cols = synthetic.randint(3, 1, nnz, 70001, "cpu") - (1 if nnz > 5 else 0)
    cuts = torch.sort(synthetic.randint(3, 2, max(n_rows - 1, 0), nnz + 1, "cpu")).values
    ip = torch.cat([torch.zeros(1, dtype=torch.int64), cuts,
                    torch.full((min(n_rows, 1),), nnz, dtype=torch.int64)])
    if n_rows > 600:
        ip[5], ip[900] = ip[6] + 1, -4  # decreases
    want = [int(ip[0]), int(ip[-1]), int((ip[1:] < ip[:-1]).sum()),
            max(int((ip[1:] - ip[:-1]).max()), 0) if n_rows else 0]
    for shift in (0, 1):  # arrays on and off 16-byte boundaries
        c = torch.cat([cols.new_zeros(shift), cols]).to(idx).to(dev)[shift:]
        p = torch.cat([ip.new_zeros(shift), ip]).to(ptr).to(dev)[shift:]
        for bits in (None, 32, 64):
            stats, c32, q = csr_check(c, p, bits)
            assert stats[:4] == want
            if nnz:
                assert stats[4:] == [int(cols.min()), int(cols.max())]
            assert c32.dtype == torch.int32 and torch.equal(c32.cpu().to(torch.int64), cols)
            assert q.dtype == (ptr if bits is None else torch.int32 if bits == 32
                               else torch.int64)
            assert torch.equal(q.cpu().to(torch.int64), ip)


def test_one_call_errors(dev):
    # each fault is refused with its own exception before anything is gathered
    vals, cols, ip = _csr([3, 0, 4, 2], 10, 7, torch.float32)
    x = torch.zeros(10, device=dev)
    cases = [(ValueError, "start at zero", cols, ip + 1), (ValueError, "equal nnz", cols, ip * 2),
             (ValueError, "non-decreasing", cols, torch.tensor([0, 5, 3, 7, 9])),
             (IndexError, "out of range", cols + 10, ip), (IndexError, "out of range", cols - 10, ip)]
    for kind, text, c, p in cases:
        y = torch.full((4,), 7.0, device=dev)
        with pytest.raises(kind, match=text):
            fs.flagsparse_spmv_csr(vals.to(dev), c.to(dev), p.to(dev), x, (4, 10), out=y)
        assert bool((y == 7.0).all())


@pytest.mark.parametrize("ptr", [torch.int32, torch.int64])
@pytest.mark.parametrize("n_rows", [0, 1, 2047, 2048, 300001])
def test_csr_check_row_classes(dev, ptr, n_rows):
    lengths = synthetic.randint(4, n_rows, n_rows, 40, "cpu") ** 2
    ip = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = torch.zeros(int(ip[-1]), dtype=torch.int32)
    stats, _, _ = csr_check(cols.to(dev), ip.to(ptr).to(dev), 32, (100, 1000, 1200))
    plain, _, _ = csr_check(cols.to(dev), ip.to(ptr).to(dev), 32)
    assert stats[:6] == plain and len(plain) == 6
    assert stats[6:] == [int(((lengths > 100) & (lengths <= 1000)).sum()),
                         int(lengths[lengths > 1200].sum())]


@pytest.mark.parametrize("long_row", [1100, 20000])
def test_stencil_with_a_dense_row_keeps_its_band_order(dev, long_row):
    side = 700
    i = torch.arange(side * side)
    r, c = i // side, i % side
    valid = torch.stack([r > 0, c > 0, r >= 0, c < side - 1, r < side - 1], 1)
    cols = (i[:, None] + torch.tensor([-side, -1, 0, 1, side])[None, :])[valid]
    more = torch.arange(long_row) * (side * side // long_row)
    lengths = torch.cat([valid.sum(1), torch.tensor([long_row])])
    ip = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = torch.cat([cols, more])
    vals = synthetic.uniform_values(5, 2, cols.numel(), torch.float64, "cpu")
    x = synthetic.uniform_values(5, 3, side * side, torch.float64, "cpu")
    p = fs.prepare_spmv_csr(vals.to(dev), cols.to(dev), ip.to(dev), (ip.numel() - 1, side * side))
    assert p._kernel(False).kind == "rowblock" and p._kernel(False).band_offset is not None
    y = fs.flagsparse_spmv_csr(x=x.to(dev), prepared=p)
    assert oracle.rel_l2(y, oracle.spmv_csr(ip, cols, vals, x)) <= 1e-12
