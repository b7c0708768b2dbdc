"""HIP-event region timing on the launching stream.

The MI355X counterpart of the reference's per-block CUDA-event timing
(workers/ditserve/models/wan/block.py:555-578, `block_cuda_ms`): a region
records a start and an end event on the current stream around the launches it
encloses, so the measured duration is GPU time of exactly those kernels.
Disabled profilers cost nothing; nothing here synchronises until summary().
"""
import collections
import functools

import torch


class _Region:
    """A region that is not timed: a context manager, or a decorator, whose function is
    timed or not as the profiler stands at each call."""

    def __init__(self, profiler, name):
        self._profiler, self._name = profiler, name

    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False

    def __call__(self, fn):
        @functools.wraps(fn)
        def inside(*args, **kwargs):
            with self._profiler.region(self._name):
                return fn(*args, **kwargs)
        return inside


class _TimedRegion(_Region):
    def __enter__(self):
        self._start = torch.cuda.Event(enable_timing=True)
        self._end = torch.cuda.Event(enable_timing=True)
        self._start.record()

    def __exit__(self, *exc):
        self._end.record()
        self._profiler._events[self._name].append((self._start, self._end))
        return False


class EventProfiler:
    """`only`: names of the regions to time (None: all).  Each timed region costs
    two event records on the stream, which matters on short steps."""

    def __init__(self, enabled=True, only=None):
        self.enabled = enabled
        self.only = None if only is None else frozenset(only)
        self._events = collections.defaultdict(list)
        self._idle = {}

    def region(self, name):
        """Context manager (or decorator) timing the launches inside it as `name`."""
        if self.enabled and (self.only is None or name in self.only):
            return _TimedRegion(self, name)
        idle = self._idle.get(name)  # stateless: one per name, for the first few hundred names
        if idle is None:
            idle = _Region(self, name)
            if len(self._idle) < 256:
                self._idle[name] = idle
        return idle

    def reset(self):
        self._events.clear()

    def summary(self):
        """{region: {"count", "total_ms", "avg_ms"}} — synchronises."""
        torch.cuda.synchronize()
        out = {}
        for name, pairs in self._events.items():
            times = [s.elapsed_time(e) for s, e in pairs]
            out[name] = {"count": len(times), "total_ms": sum(times), "avg_ms": sum(times) / len(times)}
        return out


NULL = EventProfiler(enabled=False)
