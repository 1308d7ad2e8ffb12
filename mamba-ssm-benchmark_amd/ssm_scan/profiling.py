"""Optional per-launch timing of the engine's entry points with HIP events.

Inside ``with KernelTimer() as t:`` every launch of a scan, a linear scan or a discretization is
bracketed by two events recorded on the stream the kernels are enqueued on (torch's current
stream), right around the C-ABI call: operand checks, casts and allocations come before the first.
``t.times_ms()`` gives each entry point's device time per launch.  Outside a timer nothing is
recorded and launches are not touched.
"""

import torch

_active = None


class KernelTimer:
    def __init__(self):
        self.records = {}

    def __enter__(self):
        global _active
        self._prev = _active
        _active = self
        return self

    def __exit__(self, *exc):
        global _active
        _active = self._prev
        return False

    def begin(self, name):
        """Records the start of one launch of `name`; returns the event to record at its end."""
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        self.records.setdefault(name, []).append((start, end))
        start.record()
        return end

    def times_ms(self):
        torch.cuda.synchronize()
        return {k: [s.elapsed_time(e) for s, e in v] for k, v in self.records.items()}


def active():
    """The timer in effect, or None."""
    return _active
