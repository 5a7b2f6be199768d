"""A copy of a prepared object works on its own arrays: the calls that the original converted once
hold addresses, which a copy must not take over."""

import copy

import pytest
import torch

import flagsparse_amd as fs
from flagsparse_amd import _spmv_layouts, synthetic
from oracle import oracle

pytestmark = pytest.mark.gpu


def _csr(dev, lengths, n_cols):
    ip = torch.cat([torch.zeros(1, dtype=torch.int64), torch.as_tensor(lengths).cumsum(0)])
    cols = synthetic.randint(5, 1, int(ip[-1]), n_cols, "cpu").to(torch.int32)
    vals = synthetic.uniform_values(5, 2, cols.numel(), torch.float32, "cpu")
    return vals, cols, ip, [t.to(dev) for t in (vals, cols, ip)], (len(lengths), n_cols)


def _spoil(obj, done):
    """Zeroes every device tensor the original holds, wherever it keeps it."""
    if id(obj) in done:
        return
    done.add(id(obj))
    if isinstance(obj, torch.Tensor):
        if obj.is_cuda:
            obj.zero_()
    elif isinstance(obj, dict):
        for v in obj.values():
            _spoil(v, done)
    elif isinstance(obj, (list, tuple)):
        for v in obj:
            _spoil(v, done)
    elif type(obj).__module__.startswith("flagsparse_amd"):
        names = list(getattr(obj, "__dict__", ()))
        for c in type(obj).__mro__:
            names += getattr(c, "__slots__", ())
        for n in names:
            _spoil(getattr(obj, n, None), done)


@pytest.mark.parametrize("layout", ["rowblock", "slices", "xstage", "xcs-hybrid"])
def test_copied_spmv(dev, monkeypatch, layout):
    lengths = [3, 0, 40, 5000, 17] * 400
    vals, cols, ip, args, shape = _csr(dev, lengths, 50000)
    if layout != "slices":
        monkeypatch.setattr(_spmv_layouts, "FORCE", layout)
    p = fs.prepare_spmv_csr(*args, shape)
    assert p._kernel(False).kind == layout
    x = synthetic.uniform_values(5, 3, shape[1], torch.float32, "cpu")
    xd = x.to(dev)
    y = fs.flagsparse_spmv_csr(x=xd, prepared=p)
    q = copy.deepcopy(p)
    _spoil(p, set())
    assert torch.equal(fs.flagsparse_spmv_csr(x=xd, prepared=q), y)
    assert oracle.rel_l2(y, oracle.spmv_csr(ip, cols, vals, x)) <= 1e-5


@pytest.mark.parametrize("lengths", [[3, 0, 40, 300, 17] * 400, [3, 0, 40, 17] * 400,
                                     [3, 9000, 40, 17] * 10])
def test_copied_spmm_and_sddmm(dev, lengths):
    vals, cols, ip, args, shape = _csr(dev, lengths, 5000)
    B = synthetic.dense_uniform(5000, 48, torch.float32, seed=5, device="cpu").to(dev)
    X = synthetic.dense_uniform(shape[0], 48, torch.float32, seed=6, device="cpu").to(dev)
    p = fs.prepare_spmm_csr_opt(*args, shape)
    C = fs.flagsparse_spmm_csr_opt(B=B, prepared=p)
    q = copy.deepcopy(p)
    _spoil(p, set())
    assert torch.equal(fs.flagsparse_spmm_csr_opt(B=B, prepared=q), C)
    _, _, _, args, shape = _csr(dev, lengths, 5000)
    s = fs.prepare_sddmm_csr(args[1], args[2], shape, k_hint=48)
    out = fs.flagsparse_sddmm_csr(x=X, y=B, prepared=s)
    t = copy.deepcopy(s)
    _spoil(s, set())
    assert torch.equal(fs.flagsparse_sddmm_csr(x=X, y=B, prepared=t), out)
