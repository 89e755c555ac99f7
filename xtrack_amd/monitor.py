"""Turn-by-turn particle monitor with the record layout of the reference
``ParticlesMonitor`` (xtrack/monitors/particles_monitor.py:12-104,
particles_monitor.h:13-77): one record per (particle id, turn) holding every
per-particle field, read back as ``monitor.<field>`` arrays of shape
(n_particles, n_turns)."""
import numpy as np

from .particles import Particles, _device_of, _is_device_context, per_particle_vars


def _zero_particles(n_records, device=None):
    """n_records zero records, made where they are written: on the host, or
    in one fill on the device (its fields are parts of one buffer)."""
    out = Particles.__new__(Particles)
    n = out._capacity = int(n_records)
    out._device = None
    if device is not None and _is_device_context(device):
        import torch
        out._device = _device_of(device)
        buf = torch.zeros(n * sum(np.dtype(tt).itemsize for tt, _ in per_particle_vars),
                          dtype=torch.uint8, device=out._device)
        # the records may be written on another stream than the fill's
        torch.cuda.current_stream(out._device).synchronize()
        out._arrays, at = {}, 0
        # the 8-byte fields come first, so every field is aligned
        for tt, nn in per_particle_vars:
            size = n * np.dtype(tt).itemsize
            out._arrays[nn] = buf[at:at + size].view(getattr(torch, np.dtype(tt).name))
            at += size
    else:
        out._arrays = {nn: np.zeros(n, dtype=tt) for tt, nn in per_particle_vars}
    out.q0, out.mass0, out.t_sim = 1.0, 0.0, 0.0
    out.start_at_turn = 0
    out.start_tracking_at_element = -1
    return out


class ParticlesMonitor:
    def __init__(self, start_at_turn=0, stop_at_turn=None, n_repetitions=None,
                 repetition_period=None, num_particles=None, particle_id_range=None,
                 auto_to_numpy=True, _context=None):
        if particle_id_range is not None:
            assert num_particles is None
            part_id_start, part_id_end = particle_id_range
        else:
            assert num_particles is not None
            part_id_start, part_id_end = 0, num_particles
        n_part_ids = int(part_id_end) - int(part_id_start)
        assert n_part_ids >= 0
        n_turns = int(stop_at_turn) - int(start_at_turn)
        if repetition_period is None:
            assert n_repetitions is None
            repetition_period = -1
            n_repetitions = 1
        self.start_at_turn = int(start_at_turn)
        self.stop_at_turn = int(stop_at_turn)
        self.part_id_start = int(part_id_start)
        self.part_id_end = int(part_id_end)
        self.ebe_mode = 0
        self.n_repetitions = int(n_repetitions)
        self.repetition_period = int(repetition_period)
        self.n_records = n_turns * n_part_ids * self.n_repetitions
        self.auto_to_numpy = auto_to_numpy
        self.data = _zero_particles(max(self.n_records, 1), device=_context)

    def _field(self, name):
        vv = self.data._host_array(name) if self.auto_to_numpy else self.data._arrays[name]
        vv = vv[:self.n_records]
        n_cols = self.stop_at_turn - self.start_at_turn
        if self.n_repetitions == 1:
            return vv.reshape(self.n_records // n_cols, n_cols)
        n_rows = self.n_records // n_cols // self.n_repetitions
        return vv.reshape(self.n_repetitions, n_rows, n_cols)

    def __getattr__(self, name):
        if name in ('data', '__setstate__') or name.startswith('__'):
            raise AttributeError(name)
        if name in self.data._arrays:
            return self._field(name)
        if name == 'pzeta':
            return self._field('ptau') / self._field('beta0')
        raise AttributeError(name)
