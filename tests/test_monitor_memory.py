"""Records made in device memory are zero before any stream can write to
them (on the CPU: the fill's stream is waited for)."""
import numpy as np
import torch

from xtrack_amd import monitor
from xtrack_amd.particles import per_particle_vars


def test_records_are_filled_when_the_monitor_is_made(monkeypatch):
    calls = []

    class Stream:
        def synchronize(self):
            calls.append('wait')

    zeros = torch.zeros
    monkeypatch.setattr(monitor, '_is_device_context', lambda ctx: True)
    monkeypatch.setattr(monitor, '_device_of', lambda ctx: torch.device('cpu'))
    monkeypatch.setattr(torch, 'zeros', lambda *a, **k: calls.append('fill') or zeros(*a, **k))
    monkeypatch.setattr(torch.cuda, 'current_stream', lambda dev=None: Stream())
    mon = monitor.ParticlesMonitor(start_at_turn=0, stop_at_turn=5, num_particles=7,
                                   _context='cuda:0', auto_to_numpy=False)
    assert calls == ['fill', 'wait']
    for tt, nn in per_particle_vars:
        vv = mon.data._arrays[nn]
        assert vv.numpy().dtype == np.dtype(tt) and len(vv) == 35
        assert not vv.numpy().any()
