"""Joining and parting particle sets of one device for a batch, on CPU
tensors: the device has finished the work of all streams on both sides."""
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


@pytest.fixture
def batch(monkeypatch):
    calls = []
    monkeypatch.setattr(torch.cuda, 'synchronize', lambda *a: calls.append('sync'))
    cat = torch.cat
    monkeypatch.setattr(torch, 'cat', lambda *a, **k: calls.append('join') or cat(*a, **k))
    b = BatchTracker.__new__(BatchTracker)
    b.device, b.lines, b.calls = torch.device('cpu'), [None] * len(COUNTS), calls
    return b


def test_work_of_other_streams_is_complete(batch):
    """The sets may have been written, and may be read next, on any stream."""
    sets = _sets()
    big, starts = batch._concat(sets)
    assert batch.calls[0] == 'sync' and 'join' in batch.calls
    batch.calls.clear()
    batch._split(big, starts, sets)
    assert batch.calls[-1:] == ['sync']
