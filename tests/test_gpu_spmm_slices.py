"""SpMM over slices (csrc/spmm_slices.hip) against the fp64 oracle where it can go wrong: widths
that are no whole number of vectors, column tiles, unaligned B and C, rows at the longest uncut
length and beyond, rows crossing many slices, one row for a whole slice, runs of empty rows,
64-bit row pointers, infinities outside a row's columns; and the rule that picks it."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _common, _slices, spmm_csr, synthetic
from oracle import oracle

pytestmark = pytest.mark.gpu

LENGTHS = {
    "empty": [0] * 700,
    "one_row": [9000],
    "short": [1, 0, 2, 5, 33, 3] * 200,
    "at_keep": [255, 256, 257, 0, 127, 128, 129] * 12,
    "crossing": [5, 4000, 0, 0, 1, 61, 7, 64, 65] + [0] * 1500 + [3000] * 3 + [2] * 90,
    "uniform60": [60] * 300,
}


def _case(name, n_cols, N, dtype, dev, seed=3):
    lengths = LENGTHS[name]
    ip = torch.zeros(len(lengths) + 1, dtype=torch.int64)
    ip[1:] = torch.cumsum(torch.as_tensor(lengths), 0)
    nnz = int(ip[-1])
    cols = synthetic.randint(seed, 1, nnz, n_cols, "cpu")
    vals = synthetic.uniform_values(seed, 2, nnz, dtype, "cpu")
    B = synthetic.dense_uniform(n_cols, N, dtype, seed=seed, device="cpu")
    return vals, cols, ip, B, (len(lengths), n_cols)


def _run(vals, cols, ip, B, shape, dev, acc_f64, tile=None, one_shot=True):
    lengths = ip[1:] - ip[:-1]
    kc = spmm_csr._SpmmKernelCsr(vals.to(dev), cols.to(torch.int32).to(dev), ip.to(dev),
                                 int(lengths.max()), one_shot=one_shot)
    C = torch.full((shape[0], B.shape[1]), float("nan"), dtype=B.dtype, device=dev)
    spmm_csr._run_spmm(kc, B.to(dev), C, acc_f64, tile)
    return C, kc


@pytest.mark.parametrize("name", sorted(LENGTHS))
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 7, 16, 33, 47, 64, 130, 257])
@pytest.mark.parametrize("dtype,acc", [(torch.float32, False), (torch.float32, True),
                                       (torch.float64, True)])
def test_sliced_spmm(dev, name, N, dtype, acc):
    vals, cols, ip, B, shape = _case(name, 901, N, dtype, dev)
    print(f"sliced spmm {name} N={N} {dtype} acc64={acc}", flush=True)
    C, kc = _run(vals, cols, ip, B, shape, dev, acc)
    assert kc._tables and not kc._plans
    ref = oracle.spmm_csr(ip, cols, vals, B)
    assert oracle.rel_l2(C, ref) <= oracle.REL_L2_BOUND[str(dtype)[6:]]
    if dtype == torch.float32 and acc:  # one rounding of an fp64 sum
        np.testing.assert_allclose(C.cpu().numpy(), ref, rtol=1.2e-7, atol=1e-12)
    again = torch.empty_like(C)
    spmm_csr._run_spmm(kc, B.to(dev), again, acc)
    assert torch.equal(C, again)


@pytest.mark.parametrize("N,tile", [(130, 32), (33, 8), (257, 64), (70, 1)])
def test_sliced_spmm_tiles_and_alignment(dev, N, tile):
    vals, cols, ip, B, shape = _case("crossing", 901, N, torch.float32, dev)
    C, _ = _run(vals, cols, ip, B, shape, dev, False)
    Ct, _ = _run(vals, cols, ip, B, shape, dev, False, tile)
    ref = oracle.spmm_csr(ip, cols, vals, B)
    assert oracle.rel_l2(Ct, ref) <= 1e-5 and oracle.rel_l2(C, ref) <= 1e-5
    # B one element past a 16-byte boundary: same sums
    flat = torch.empty(B.numel() + 1, device=dev)
    Bu = flat[1:].view(B.shape)
    Bu.copy_(B)
    p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    assert torch.equal(fs.flagsparse_spmm_csr_opt(B=Bu, prepared=p), C)


def test_sliced_spmm_rowptr64(dev, monkeypatch):
    vals, cols, ip, B, shape = _case("crossing", 901, 20, torch.float64, dev)
    C, _ = _run(vals, cols, ip, B, shape, dev, True)
    monkeypatch.setattr(_common, "ROWPTR32_MAX_NNZ", 0)
    C64, kc = _run(vals, cols, ip, B, shape, dev, True)
    assert kc.rowptr_bits == 64 and torch.equal(C, C64)


def test_sliced_spmm_nonfinite(dev):
    # the masked loads of a row's last entries read B's first row; nothing of it may show
    vals, cols, ip, B, shape = _case("short", 901, 47, torch.float32, dev)
    B[0], B[5, 3] = float("inf"), float("nan")
    C, _ = _run(vals, cols, ip, B, shape, dev, False)
    ref = oracle.spmm_csr(ip, cols, vals, B)
    np.testing.assert_array_equal(np.isnan(C.cpu().numpy()), np.isnan(ref))
    np.testing.assert_array_equal(np.isfinite(C.cpu().numpy()), np.isfinite(ref))


def test_spmm_route(dev):
    # row blocks: prepared, short rows, whole aligned vectors; else slices
    for name, N, blocks in (("short", 16, True), ("short", 15, False), ("at_keep", 16, False)):
        vals, cols, ip, B, shape = _case(name, 901, N, torch.float32, dev)
        p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
        C = fs.flagsparse_spmm_csr_opt(B=B.to(dev), prepared=p)
        kc = p._kernel_csr()
        assert bool(kc._plans) == blocks and bool(kc._tables) == (not blocks)
        Cs, _ = _run(vals, cols, ip, B, shape, dev, False)  # the other route
        ref = oracle.spmm_csr(ip, cols, vals, B)
        assert oracle.rel_l2(C, ref) <= 1e-5 and oracle.rel_l2(Cs, ref) <= 1e-5


def test_spmm_capture_needs_a_first_call(dev):
    vals, cols, ip, B, shape = _case("at_keep", 901, 8, torch.float32, dev)
    p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    Bd = B.to(dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with pytest.raises(RuntimeError, match="once before"):
        with torch.cuda.graph(g):
            fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p)
    torch.cuda.synchronize()
    ref = oracle.spmm_csr(ip, cols, vals, B)
    assert oracle.rel_l2(fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p), ref) <= 1e-5


@pytest.mark.parametrize("name", sorted(set(LENGTHS) - {"empty"}))
def test_slices_by_column(dev, monkeypatch, name):
    # any launch order gives the same sums; the order is a permutation with the slices inside one
    # row last, by column within each XCD's part
    vals, cols, ip, B, shape = _case(name, 901, 20, torch.float32, dev)
    C, _ = _run(vals, cols, ip, B, shape, dev, False)
    shape_of = spmm_csr._spmm_slice_shape
    monkeypatch.setattr(spmm_csr._slices, "ordered", lambda *a: True)
    monkeypatch.setattr(spmm_csr, "_spmm_slice_shape", lambda l, p, by=False: shape_of(l, p))
    Co, kc = _run(vals, cols, ip, B, shape, dev, False)
    assert torch.equal(C, Co)
    (table, order), = kc._tables.values()
    t, o = table.view(-1, 2).cpu(), order.cpu().to(torch.int64)
    n = t.shape[0] - 1
    assert torch.equal(torch.sort(o).values, torch.arange(n))
    inside = (t[:-1, 0] == t[1:, 0]) & (t[1:, 1] > t[:-1, 1])
    others = int((~inside).sum())
    assert not bool(inside[o[:others]].any()) and bool(inside[o[others:]].all())
    k = cols[t[o[others:], 1]] * 255 // shape[1]
    for x in range(8):  # slots 8 apart are one XCD's, in column bins that rise
        assert bool((k[x::8][1:] >= k[x::8][:-1]).all())


def test_unknown_longest_row(dev, monkeypatch):
    # a one-off COO matrix: room for cut rows' pieces is only taken unseen while it is small
    for name, cut in (("crossing", True), ("short", False)):
        vals, cols, ip, B, shape = _case(name, 901, 24, torch.float32, dev)
        row = torch.repeat_interleave(torch.arange(shape[0]), ip[1:] - ip[:-1])
        args = [t.to(dev) for t in (vals, row, cols, B)]
        C = fs.flagsparse_spmm_coo(*args, shape)
        monkeypatch.setattr(spmm_csr, "_SUMS_UNSEEN", 0)
        assert torch.equal(fs.flagsparse_spmm_coo(*args, shape), C)
        kc = spmm_csr._SpmmKernelCsr(args[0], args[2].to(torch.int32), ip.to(dev), one_shot=True)
        spmm_csr._run_spmm(kc, args[3], torch.empty_like(C), True)
        assert (kc.max_row_nnz > 256) == cut and (kc._keep[-1] is not None) == cut
        monkeypatch.undo()
        assert oracle.rel_l2(C, oracle.spmm_csr(ip, cols, vals, B)) <= 1e-5


def _row_block_kernel(n, dtype, aligned=True):
    """The kernel of a prepared matrix with rows over 8192 entries: vectors of any alignment from 32
    lanes of single elements on, which N takes that is no whole number of pairs or not aligned."""
    single = n % 2 == 1 or not aligned
    return "spmm_ragged_kernel" if single and n > 16 else "spmm_rowblock_kernel"


@pytest.mark.parametrize("n,wide", [(17, 2), (31, 2), (33, 4), (47, 4), (101, 4), (130, 4)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_odd_widths_keep_their_order_of_additions(dev, n, wide, dtype):
    """spmm_ragged_kernel adds as spmm_rowblock_kernel does, bit for bit: the first n columns of a
    wider B, whose whole vectors take as many lanes and so as many groups and the same plan, come out
    the same.  Rows over 8192 entries, short ones, single and several parts; 130 columns from B off a
    vector's alignment, in three tiles."""
    lengths = torch.tensor([3, 0, 9000, 127, 128, 129, 40, 250, 700] * 20 + [20000, 1])
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = synthetic.randint(7, 1, int(ptr[-1]), 3000, "cpu").to(torch.int32)
    data = synthetic.uniform_values(7, 2, cols.numel(), dtype, "cpu")
    p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), (lengths.numel(), 3000))
    # 2 * 16 or 4 * 16 lanes of 16 bytes: 32 or 64 lanes
    N = max(n, (64 if wide == 4 else 32) * (16 // dtype.itemsize))
    Bw = synthetic.dense_uniform(3000, N, dtype, seed=5, device=dev)
    want = fs.flagsparse_spmm_csr_opt(B=Bw, prepared=p)[:, :n]
    kc = p._kernel_csr()
    assert kc.kernel_name(N) == "spmm_rowblock_kernel"
    room = torch.empty(3000 * n + 1, dtype=dtype, device=dev)
    B = room[n == 130:][:3000 * n].view(3000, n)
    B.copy_(Bw[:, :n])
    got = fs.flagsparse_spmm_csr_opt(B=B, prepared=p)
    if N != n:
        assert kc.kernel_name(n) == "spmm_ragged_kernel"
    assert {k[0] for k in kc._plans} == {32 if wide == 2 else 64}  # one plan for both
    assert torch.equal(got, want)
    ref = oracle.spmm_csr(ptr, cols, data, B.cpu())
    assert oracle.rel_l2(got, ref) <= oracle.REL_L2_BOUND[str(dtype)[6:]]


@pytest.mark.parametrize("n", [1, 16, 47, 64])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_long_rows_keep_their_order_of_additions(dev, monkeypatch, n, dtype):
    """Over 8192 entries in a row: row blocks, whose parts in column order give the same bits as in
    row order."""
    lengths = torch.tensor([3, 0, 9000, 127, 128, 129, 40] * 20 + [20000, 1])
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = torch.cat([torch.sort(synthetic.randint(7, k, int(m), 60000, "cpu")).values
                      for k, m in enumerate(lengths)]).to(torch.int32)
    data = (torch.arange(cols.numel()) % 17 - 8).to(dtype) / 7
    B = ((torch.arange(60000 * n) % 1013).to(dtype) / 1013 - 0.5).reshape(60000, n)
    shape = (lengths.numel(), 60000)
    out = []
    for order in (True, False):
        monkeypatch.setattr(_slices, "ordered", lambda *a: order)
        p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), shape)
        out.append(fs.flagsparse_spmm_csr_opt(B=B.to(dev), prepared=p).cpu())
        assert p._kernel_csr().kernel_name() == "spmm_rowblock_kernel"
        assert p._kernel_csr().kernel_name(n) == _row_block_kernel(n, dtype)
        assert all(q.by_column == order for q in p._kernel_csr()._plans.values())
    assert torch.equal(out[0], out[1])
    ref = oracle.spmm_csr(ptr, cols, data, B)
    assert oracle.rel_l2(out[0], ref) <= oracle.REL_L2_BOUND[str(dtype)[6:]]


@pytest.mark.parametrize("ptr", [torch.int32, torch.int64])
@pytest.mark.parametrize("lengths", [[9000], [3, 0, 5], [3, 9000, 0, 300] * 9 + [1],
                                     [1] * 40 + [2000] * 1100])
def test_part_order(dev, ptr, lengths):
    """A permutation of the plan's descriptors: the row blocks first, then the parts, by column
    within each XCD's share."""
    lengths = torch.tensor(lengths)
    rowptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(ptr).to(dev)
    nnz, n_cols = int(lengths.sum()), 40000
    cols = synthetic.randint(3, 1, nnz, n_cols, "cpu").to(torch.int32)
    plan = spmm_csr.build_row_block_plan_device(rowptr, 1024, 16, 128, 256, window_rows=256)
    out = spmm_csr._parts_by_column(plan.desc, cols.to(dev), n_cols, rowptr, 256).cpu().long()
    desc = plan.desc.cpu().long()
    key = lambda t: (t[:, 0] << 32) + (t[:, 1] << 1) + (t[:, 2] > 0)  # noqa: E731
    assert torch.equal(key(out).sort().values, key(desc).sort().values)
    part = out[:, 2] > 0
    n = int((~part).sum())
    assert not bool(part[:n].any()) and bool(part[n:].all())
    first = rowptr.cpu().long()[out[n:, 0]] + out[n:, 1] * 256
    k = cols[first].long() * 255 // n_cols
    for x in range(8):
        assert bool((k[x::8][1:] >= k[x::8][:-1]).all())


@pytest.mark.parametrize("n", [1, 3, 16, 17, 31, 33, 47, 64, 65, 101, 128, 129])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("offset, longest", [(0, 128), (1, 128), (0, 250)])
def test_parts_of_every_length(dev, monkeypatch, n, dtype, offset, longest):
    """Rows over 8192 entries whose last parts leave every remainder to the rows of B requested
    together; single columns in a last tile, B off a vector's alignment, blocks of more entries
    than the odd widths' kernel stages (rows of over 128 uncut).  Whole numbers with sums below
    2^24, so the result is exact in any order."""
    monkeypatch.setattr(spmm_csr, "_SPMM_ROW_SPLIT_THRESHOLD", longest)
    tails = [1, 2, 3, 4, 5, 12, 15, 16, 17, 31, 32, 33, 60, 61, 63, 64, 65, 100, 127, 128]
    lengths = torch.tensor([1024 * 9 + t for t in tails] + [129, 192, 200, 0, 7, 1, 2] + [250] * 9)
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = synthetic.randint(5, 1, int(ptr[-1]), 3000, "cpu").to(torch.int32)
    data = (torch.arange(cols.numel()) % 13 - 6).to(dtype)
    B = (torch.arange(3000 * n) % 101 - 50).to(dtype).reshape(3000, n)
    room = torch.empty(3000 * n + offset, dtype=dtype, device=dev)
    Bd = room[offset:].view(3000, n)
    Bd.copy_(B)
    p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), (lengths.numel(), 3000))
    out = fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p).cpu()
    assert p._kernel_csr().kernel_name() == "spmm_rowblock_kernel"
    assert p._kernel_csr().kernel_name(n) == _row_block_kernel(n, dtype, offset == 0)
    ref = oracle.spmm_csr(ptr, cols, data, B)
    assert torch.equal(out.double(), torch.as_tensor(ref).double())


def _shared(kc, kind):
    return [v for k, v in kc._shared.items() if k[0] == kind]


@pytest.mark.parametrize("name", sorted(set(LENGTHS) - {"empty"}))
@pytest.mark.parametrize("N,dtype,acc", [(3, torch.float32, False), (47, torch.float32, True),
                                         (130, torch.float64, True)])
def test_room_for_cut_rows_only(dev, monkeypatch, name, N, dtype, acc):
    """Where a slot for both ends of every slice is too much room: a slot for each piece of a cut
    row, counted, and the same bits."""
    vals, cols, ip, B, shape = _case(name, 901, N, dtype, dev)
    C, plain = _run(vals, cols, ip, B, shape, dev, acc)
    monkeypatch.setattr(spmm_csr, "_SUMS_ROOM", 0)
    for one_shot in (True, False):
        Cp, kc = _run(vals, cols, ip, B, shape, dev, acc, one_shot=one_shot)
        if kc._tables:
            assert torch.equal(C, Cp)
        elif name != "one_row":
            continue  # short rows, prepared: row blocks
    (table, _), = plain._tables.values()
    t = table.view(-1, 2).cpu()
    inside = ip[t[1:-1, 0]] < t[1:-1, 1]  # boundaries inside a row: a piece before each, and
    rows = t[1:-1, 0][inside]             # one after the row's last
    want = int(inside.sum()) + int(torch.unique(rows).numel())
    _, kc = _run(vals, cols, ip, B, shape, dev, acc)
    cut = int((ip[1:] - ip[:-1]).max()) > next(iter(plain._tables))[1]
    sums = kc._keep[-1]
    assert (0 if sums is None else sums.numel()) == (want * N if cut else 0)
    if cut:
        (counted, n), = _shared(kc, "pieces")
        assert n == want and sums.numel() < plain._keep[-1].numel()


def test_room_is_shared(dev):
    # one width with B aligned and not, and again: one workspace
    vals, cols, ip, B, shape = _case("at_keep", 901, 130, torch.float32, dev)
    p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    flat = torch.empty(B.numel() + 1, device=dev)
    Bu = flat[1:].view(B.shape)
    Bu.copy_(B)
    outs = [fs.flagsparse_spmm_csr_opt(B=b, prepared=p) for b in (B.to(dev), Bu, B.to(dev))]
    assert len(p._kernel_csr()._args) == 2 and len(_shared(p._kernel_csr(), "sums")) == 1
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


def test_room_at_size(dev):
    """A million rows with one that is cut, N = 256: three pieces take their own room, not 1 GB."""
    n = 1_000_000
    lengths = torch.full((n,), 32, dtype=torch.int64)
    lengths[777] = 300
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = torch.arange(int(ptr[-1]), dtype=torch.int32) % 1000
    data = torch.ones(cols.numel())
    p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), (n, 1000))
    C = fs.flagsparse_spmm_csr_opt(B=torch.ones(1000, 256, device=dev), prepared=p)
    assert torch.equal(C, lengths.float().to(dev)[:, None].expand_as(C))
    (sums,) = _shared(p._kernel_csr(), "sums")
    assert 2 * 256 <= sums.numel() <= 5 * 256


def test_room_of_a_new_width_while_capturing(dev, monkeypatch):
    # a width first used in a capture, on slices that exist: nothing is counted (a host wait)
    vals, cols, ip, B, shape = _case("at_keep", 901, 33, torch.float32, dev)
    p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    fs.flagsparse_spmm_csr_opt(B=torch.ones(901, 36, device=dev), prepared=p)
    monkeypatch.setattr(spmm_csr, "_SUMS_ROOM", 0)
    Bd = B.to(dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        C = fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p)
    for _ in range(3):
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert oracle.rel_l2(C, oracle.spmm_csr(ip, cols, vals, B)) <= 1e-5
    assert torch.equal(fs.flagsparse_spmm_csr_opt(B=Bd.clone(), prepared=p), C)


@pytest.mark.parametrize("widths", [(47, 256), (256, 47)])
def test_launch_order_follows_the_width(dev, widths):
    """Two widths of one lane count, of which the wider B does not fit an L2: each has the launch
    order of its own size, whichever comes first, on one plan."""
    lengths = torch.tensor([40, 9000, 3, 128] * 12)
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = synthetic.randint(7, 1, int(ptr[-1]), 10000, "cpu").to(torch.int32)
    data = synthetic.uniform_values(7, 2, cols.numel(), torch.float32, "cpu")
    shape = (lengths.numel(), 10000)
    p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), shape)
    kc = p._kernel_csr()
    for n in widths:
        B = synthetic.dense_uniform(10000, n, torch.float32, seed=n, device="cpu")
        out = fs.flagsparse_spmm_csr_opt(B=B.to(dev), prepared=p)
        assert oracle.rel_l2(out, oracle.spmm_csr(ptr, cols, data, B)) <= 1e-5
    assert set(kc._plans) == {(64, False), (64, True)} and len(_shared(kc, "row order")) == 1
    assert kc._plans[64, True].by_column and not kc._plans[64, False].by_column
    assert kc._plans[64, True]._workspaces is kc._plans[64, False]._workspaces
    assert len(kc.describe()["plans"]) == 2


def test_launch_order_is_not_built_in_a_capture(dev):
    lengths = torch.tensor([40, 9000, 3, 128] * 12)
    ptr = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)])
    cols = synthetic.randint(7, 1, int(ptr[-1]), 10000, "cpu").to(torch.int32)
    data = synthetic.uniform_values(7, 2, cols.numel(), torch.float32, "cpu")
    p = fs.prepare_spmm_csr_opt(data.to(dev), cols.to(dev), ptr.to(dev), (48, 10000))
    fs.flagsparse_spmm_csr_opt(B=torch.ones(10000, 47, device=dev), prepared=p)  # row order
    B = synthetic.dense_uniform(10000, 256, torch.float32, seed=3, device="cpu")
    Bd = B.to(dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        C = fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p)
    assert set(p._kernel_csr()._plans) == {(64, False)}
    eager = fs.flagsparse_spmm_csr_opt(B=Bd, prepared=p)  # before any replay
    ref = oracle.spmm_csr(ptr, cols, data, B)
    assert oracle.rel_l2(eager, ref) <= 1e-5
    for _ in range(3):
        C.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(C, eager)


def test_more_row_blocks_than_a_launch_holds(dev, monkeypatch):
    # the prepared product runs on slices instead (here with a limit that 1200 rows reach)
    vals, cols, ip, B, shape = _case("short", 901, 16, torch.float32, dev)
    p = fs.prepare_spmm_csr_opt(vals.to(dev), cols.to(dev), ip.to(dev), shape)
    monkeypatch.setattr(_slices, "MAX_SLICES", 12)
    C = fs.flagsparse_spmm_csr_opt(B=B.to(dev), prepared=p)
    assert p._kernel_csr()._tables
    assert oracle.rel_l2(C, oracle.spmm_csr(ip, cols, vals, B)) <= 1e-5
