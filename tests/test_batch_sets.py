"""Joining and parting particle sets of one device for a batch, on CPU
tensors: every field of every set comes back, in memory of the set's own, and
the device has finished the work of all streams on both sides."""
import numpy as np
import pytest
import torch

import xtrack_amd as xt
from xtrack_amd.batch import BatchTracker

COUNTS = (5, 0, 300, 1)


def _sets():
    out = []
    for k, n in enumerate(COUNTS):
        rng = np.random.default_rng(k)
        p = xt.Particles(p0c=7e12, x=rng.normal(0, 1, n))
        p._arrays['px'][:] = np.resize([-0.0, np.nan, np.inf, 5e-324], n)
        p._arrays['_rng_s1'][:] = rng.integers(0, 2 ** 32, n, dtype=np.uint32)
        p._arrays['at_turn'][:] = 2 ** 62 + k
        p._arrays = {nn: torch.from_numpy(vv.copy()) for nn, vv in p._arrays.items()}
        p._device = torch.device('cpu')
        out.append(p)
    return out


def _bytes(t):
    return t.contiguous().view(torch.uint8).numpy().tobytes() if t.numel() else b''


@pytest.fixture
def batch(monkeypatch):
    calls = []
    monkeypatch.setattr(torch.cuda, 'synchronize', lambda *a: calls.append('sync'))
    cat = torch.cat
    monkeypatch.setattr(torch, 'cat', lambda *a, **k: calls.append('join') or cat(*a, **k))
    b = BatchTracker.__new__(BatchTracker)
    b.device, b.lines, b.calls = torch.device('cpu'), [None] * len(COUNTS), calls
    return b


def test_sets_keep_their_values_and_own_their_memory(batch):
    sets, want = _sets(), _sets()
    big, starts = batch._concat(sets)
    for nn in big._arrays:
        assert big._arrays[nn].dtype == want[0]._arrays[nn].dtype
        assert _bytes(big._arrays[nn]) == b''.join(_bytes(p._arrays[nn]) for p in want)
        assert big._arrays[nn].is_contiguous()
    before = [p._arrays['x'] for p in sets]
    batch._split(big, starts, sets)
    storages = {}
    for k, (p, w) in enumerate(zip(sets, want)):
        assert list(p._arrays) == list(w._arrays)
        # a set's arrays are new ones, as after a copy through the host
        assert p._capacity == 0 or p._arrays['x'].data_ptr() != before[k].data_ptr()
        held = {}
        for nn, vv in p._arrays.items():
            assert vv.dtype == w._arrays[nn].dtype and vv.is_contiguous()
            assert _bytes(vv) == _bytes(w._arrays[nn])
            s = vv.untyped_storage()
            held[s.data_ptr()] = s.nbytes()
        assert sum(held.values()) <= sum(v.numel() * v.element_size()
                                         for v in w._arrays.values())
        for ptr in held:
            if held[ptr]:
                assert storages.setdefault(ptr, k) == k


def test_work_of_other_streams_is_complete(batch):
    """The sets may have been written, and may be read next, on any stream."""
    sets = _sets()
    big, starts = batch._concat(sets)
    assert batch.calls[0] == 'sync' and 'join' in batch.calls
    batch.calls.clear()
    batch._split(big, starts, sets)
    assert batch.calls[-1:] == ['sync']
