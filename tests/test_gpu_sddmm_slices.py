"""SDDMM over slices (csrc/sddmm_slices.hip) against the fp64 oracle where it can go wrong: K that
is no whole number of vectors, every lane count, rows crossing slices and lane groups, runs of
empty rows, unaligned x and y, accumulation variants, infinities that a masked element must not
let through; and a prepared pattern first used on another stream."""

import numpy as np
import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _common, sddmm_csr, synthetic
from oracle import oracle

pytestmark = pytest.mark.gpu

LENGTHS = {
    "one_row": [5003],
    "one_entry": [0] * 300 + [1] + [0] * 500,
    "short": [1, 0, 2, 5, 33, 3] * 300,
    "crossing": [5, 3000, 0, 0, 1, 61, 7, 64, 65] + [0] * 1500 + [700] * 3 + [2] * 90,
}


def _case(name, n_cols, K, dtype, dev, seed=4):
    lengths = LENGTHS[name]
    ip = torch.zeros(len(lengths) + 1, dtype=torch.int64)
    ip[1:] = torch.cumsum(torch.as_tensor(lengths), 0)
    nnz = int(ip[-1])
    cols = synthetic.randint(seed, 1, nnz, n_cols, "cpu").to(torch.int32)
    data = synthetic.uniform_values(seed, 2, nnz, dtype, "cpu")
    x = synthetic.dense_uniform(len(lengths), K, dtype, seed=seed, device="cpu")
    y = synthetic.dense_uniform(n_cols, K, dtype, seed=seed + 1, device="cpu")
    return ip, cols, data, x, y, (len(lengths), n_cols)


@pytest.mark.parametrize("name", sorted(LENGTHS))
@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 7, 16, 31, 32, 33, 50, 64, 65, 127, 250, 257, 511])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_sliced_sddmm(dev, name, K, dtype):
    ip, cols, data, x, y, shape = _case(name, 503, K, dtype, dev)
    print(f"sliced sddmm {name} K={K} {dtype}", flush=True)
    bound = oracle.REL_L2_BOUND[str(dtype)[6:]]
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=K)
    out = fs.flagsparse_sddmm_csr(x=x.to(dev), y=y.to(dev), prepared=p)
    assert p._tables  # the sliced kernel ran
    assert oracle.rel_l2(out, oracle.sddmm_csr(ip, cols, x, y)) <= bound
    one = fs.flagsparse_sddmm_csr(data=data.to(dev), indices=cols.to(dev),
                                  indptr=ip.to(torch.int32).to(dev), x=x.to(dev), y=y.to(dev),
                                  shape=shape, alpha=0.5, beta=2.0)
    assert oracle.rel_l2(one, oracle.sddmm_csr(ip, cols, x, y, data, alpha=0.5,
                                               beta=2.0)) <= bound
    again = fs.flagsparse_sddmm_csr(x=x.to(dev), y=y.to(dev), prepared=p)
    assert torch.equal(out, again)


@pytest.mark.parametrize("variant", ["acc64", "acc64_out64"])
@pytest.mark.parametrize("K", [3, 33, 64])
def test_sliced_sddmm_variants(dev, variant, K):
    ip, cols, data, x, y, shape = _case("crossing", 503, K, torch.float32, dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=K)
    out, meta = sddmm_csr._run_sddmm_prepared(p, x.to(dev), y.to(dev), data.to(dev), 1.0, 0.5,
                                              None, variant=variant)
    ref = oracle.sddmm_csr(ip, cols, x, y, data, alpha=1.0, beta=0.5)
    assert meta["fallback_used"] is False and p._tables
    # fp64 sums of fp32 products: exact to fp64 rounding, then one fp32 rounding unless out64
    assert oracle.rel_l2(out, ref) <= (1e-12 if variant == "acc64_out64" else 6e-8)


def test_sliced_sddmm_rowptr64_and_alignment(dev, monkeypatch):
    ip, cols, data, x, y, shape = _case("crossing", 503, 33, torch.float32, dev)

    def run(xx, yy):
        p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=33)
        return fs.flagsparse_sddmm_csr(x=xx, y=yy, prepared=p), p

    out, _ = run(x.to(dev), y.to(dev))
    shifted = []
    for t in (x, y):  # rows that start one element past a 16-byte boundary
        flat = torch.empty(t.numel() + 1, device=dev)
        flat[1:].copy_(t.reshape(-1))
        shifted.append(flat[1:].view(t.shape))
    assert torch.equal(run(*shifted)[0], out)
    monkeypatch.setattr(_common, "ROWPTR32_MAX_NNZ", 0)
    out64, p = run(x.to(dev), y.to(dev))
    assert p._kernel_ptr.dtype == torch.int64 and torch.equal(out64, out)


@pytest.mark.parametrize("K", [5, 33, 50])
def test_sliced_sddmm_nonfinite(dev, K):
    # y's first row (read by masked positions) and single elements next to a row's end
    ip, cols, data, x, y, shape = _case("short", 503, K, torch.float32, dev)
    y[0], y[7, K - 1], y[9, K - 2] = float("inf"), float("nan"), float("inf")
    out = fs.flagsparse_sddmm_csr(indices=cols.to(dev), indptr=ip.to(dev), x=x.to(dev),
                                  y=y.to(dev), shape=shape).cpu().numpy()
    ref = oracle.sddmm_csr(ip, cols, x, y)
    np.testing.assert_array_equal(np.isnan(out), np.isnan(ref))
    np.testing.assert_array_equal(np.isfinite(out), np.isfinite(ref))


def test_sddmm_two_streams(dev):
    ip, cols, data, x, y, shape = _case("crossing", 503, 40, torch.float32, dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=40)
    xd, yd = x.to(dev), y.to(dev)
    torch.cuda.synchronize()
    outs = []
    for _ in range(3):
        for s in (torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)):
            with torch.cuda.stream(s):
                outs.append(fs.flagsparse_sddmm_csr(x=xd, y=yd, prepared=p))
    torch.cuda.synchronize()
    ref = oracle.sddmm_csr(ip, cols, x, y)
    assert all(oracle.rel_l2(o, ref) <= 1e-5 for o in outs)


def test_sddmm_row_ids(dev):
    # made when asked for (the kernel of very wide K and callers that read the attribute)
    ip, cols, data, x, y, shape = _case("short", 503, 4, torch.float32, dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape)
    want = torch.repeat_interleave(torch.arange(shape[0], dtype=torch.int32), ip[1:] - ip[:-1])
    assert p.row_ids.dtype == torch.int32 and torch.equal(p.row_ids.cpu(), want)
    K = 2051  # past four steps of 64 lanes: one lane group per entry
    x = synthetic.dense_uniform(shape[0], K, torch.float32, seed=5, device="cpu")
    y = synthetic.dense_uniform(503, K, torch.float32, seed=6, device="cpu")
    q = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape)
    out = fs.flagsparse_sddmm_csr(x=x.to(dev), y=y.to(dev), prepared=q)
    assert not q._tables
    assert oracle.rel_l2(out, oracle.sddmm_csr(ip, cols, x, y)) <= 1e-5


@pytest.mark.parametrize("name", sorted(LENGTHS))
def test_sliced_sddmm_by_column(dev, monkeypatch, name):
    ip, cols, data, x, y, shape = _case(name, 503, 40, torch.float64, dev)
    args = dict(x=x.to(dev), y=y.to(dev))
    out = fs.flagsparse_sddmm_csr(
        prepared=fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape), **args)
    monkeypatch.setattr(sddmm_csr._slices, "ordered", lambda *a: True)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape)
    assert torch.equal(fs.flagsparse_sddmm_csr(prepared=p, **args), out)
    (_, order), = p._tables.values()
    assert torch.equal(torch.sort(order.cpu()).values.to(torch.int64),
                       torch.arange(order.numel()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_wide_sddmm_two_streams(dev, dtype):
    # the kernel of very wide K reads the row ids, which the first call makes on its own stream
    ip, cols, data, x, y, shape = _case("crossing", 503, 2051, dtype, dev)
    xd, yd = x.to(dev), y.to(dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=2051)
    outs = []
    for _ in range(2):
        for s in (torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)):
            with torch.cuda.stream(s):
                outs.append(fs.flagsparse_sddmm_csr(x=xd, y=yd, prepared=p))
    torch.cuda.synchronize()
    assert not p._tables
    ref = oracle.sddmm_csr(ip, cols, x, y)
    assert all(oracle.rel_l2(o, ref) <= oracle.REL_L2_BOUND[str(dtype)[6:]] for o in outs)


@pytest.mark.parametrize("K", [40, 2051])  # the sliced kernel, the flat one
def test_sddmm_keeps_its_arrays_from_other_streams(dev, monkeypatch, K):
    """A prepared pattern dropped after a call on another stream: the memory of its arrays is not
    given out while that stream is busy."""
    ip, cols, data, x, y, shape = _case("crossing", 503, K, torch.float32, dev)
    if K == 40:
        monkeypatch.setattr(sddmm_csr._slices, "ordered", lambda *a: True)
    xd, yd, mat = x.to(dev), y.to(dev), torch.ones(8192, 8192, device=dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=K)
    fs.flagsparse_sddmm_csr(x=xd, y=yd, prepared=p)  # its arrays belong to this stream
    side = torch.cuda.Stream(device=dev)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):  # about 10 ms each
            mat = mat @ mat
        out = fs.flagsparse_sddmm_csr(x=xd, y=yd, prepared=p)
    (launch,) = p._shapes.values()
    arrays = [t for t in launch.arrays if t is not None]
    assert len(arrays) == (4 if K == 40 else 2)
    sizes = [t.untyped_storage().nbytes() for t in arrays]
    held = {t.untyped_storage().data_ptr() for t in arrays}
    del p, launch, arrays
    taken = [torch.empty(n, dtype=torch.uint8, device=dev) for n in sizes * 4]
    busy = not side.query()
    assert not held & {t.untyped_storage().data_ptr() for t in taken}
    assert busy  # else the allocator was free to give them out
    torch.cuda.synchronize()
    assert oracle.rel_l2(out, oracle.sddmm_csr(ip, cols, x, y)) <= 1e-5


@pytest.mark.parametrize("K", [4, 8, 16, 64, 128])
def test_sliced_sddmm_order_of_additions(dev, K):
    """float32, bit for bit: a vector's four products in a chain of fused multiply-adds, a lane's
    vectors and then the lanes added in a tree.  The chain rounds one product of a vector where pairs
    would round two.  (The oracle's fused step rounds an extended-precision sum, which differs from a
    fused float32 step only where that sum lies half-way between two floats to 2^-63.)"""
    ip, cols, _, x, y, shape = _case("crossing", 503, K, torch.float32, dev)
    p = fs.prepare_sddmm_csr(cols.to(dev), ip.to(dev), shape, k_hint=K)
    out = fs.flagsparse_sddmm_csr(x=x.to(dev), y=y.to(dev), prepared=p).cpu().numpy()
    lanes, vec = sddmm_csr._sddmm_slice_lanes(K, torch.float32)
    steps = K // (lanes * vec)
    assert vec == 4 and K == steps * lanes * vec and steps in (1, 2, 4)
    row = torch.repeat_interleave(torch.arange(shape[0]), ip[1:] - ip[:-1])
    X = x[row].numpy().reshape(-1, steps, lanes, 4).astype(np.longdouble)
    Y = y[cols.long()].numpy().reshape(-1, steps, lanes, 4).astype(np.longdouble)
    v = np.zeros(X.shape[:3], dtype=np.float32)
    for j in range(4):
        v = (X[..., j] * Y[..., j] + v).astype(np.float32)
    for axis in (1, 2):
        while v.shape[axis] > 1:
            a, b = (np.take(v, range(k, v.shape[axis], 2), axis) for k in (0, 1))
            v = a + b
    np.testing.assert_array_equal(out, v[:, 0, 0])
