"""What a prepared SDDMM pattern keeps between calls is complete before it is kept: later calls may
come from other streams, which nothing orders after the one that built it (no GPU: the stream is a
recorder)."""

import copy
import pickle

import pytest
import torch

from flagsparse_amd import _slices, sddmm_csr


class _Stream:
    """Stands in for the current stream: notes what the object held at each wait."""

    def __init__(self, prepared):
        self.prepared = prepared
        self.held = []

    def synchronize(self):
        p = self.prepared
        self.held.append((p._row_ids, p._kernel_ptr, dict(p._tables)))


@pytest.fixture
def prepared(monkeypatch):
    indptr = torch.tensor([0, 2, 2, 5], dtype=torch.int64)
    p = sddmm_csr.SDDMMPrepared(torch.tensor([0, 1, 0, 2, 3], dtype=torch.int32), indptr, (3, 4),
                                None, 64, 4)
    stream = _Stream(p)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: stream)
    monkeypatch.setattr(_slices, "build", lambda *a: ("table", "order"))
    return p, stream


def test_row_ids_wait_before_they_are_kept(prepared):
    p, stream = prepared
    assert p.row_ids.tolist() == [0, 0, 2, 2, 2]
    assert stream.held == [(None, None, {})]  # one wait, and nothing was kept before it
    assert p.row_ids is p.row_ids and len(stream.held) == 1


def test_slices_wait_before_they_are_kept(prepared):
    p, stream = prepared
    assert p.slices(64, False) == ("table", "order")
    assert stream.held == [(None, None, {})]
    assert p._kernel_ptr.dtype == torch.int32
    p.slices(64, False)
    assert len(stream.held) == 1


def test_one_call_waits_for_nothing(prepared):
    p, stream = prepared
    p._one_call = True
    p.row_ids, p.slices(64, False)
    assert stream.held == []


def test_copied_launch_is_marked_nowhere():
    table = torch.arange(4)
    launch = sddmm_csr._Launch((8, 4, 256, table, table, None), (table, None))
    launch.streams.add(17)
    for other in (copy.deepcopy(launch), pickle.loads(pickle.dumps(launch))):
        assert other.streams == set() and other.sliced[:3] == (8, 4, 256)
        assert other.arrays[0] is other.sliced[3] and torch.equal(other.arrays[0], table)
        assert other.arrays[0].data_ptr() != table.data_ptr()
