"""optimus.profilers — the hot path's timing hook, same name and tag scheme as the reference
(optimus/profilers.py:99-119): record_pcl_function("a--b--c") starts/stops the nested timers
"a", "a--b", "a--b--c" on optimus.globals.profiler and is a no-op when that is None.

The reference marks events with a SYCL profiling tag on the XPU queue
(pytorch_xpu_extensions/pcl.xpu.profiler/csrc/profiler/profile.dp.cpp:36-42); here an event is a
HIP event recorded on PyTorch's current stream, so nothing synchronises until `summary()`.
"""
from contextlib import ContextDecorator

import torch

import optimus.globals


class record_pcl_function(ContextDecorator):
    """record_pcl_function(full_name, tag, exclude_from_trace, key, ignore): the nested timers run inside the scope."""
    __slots__ = ("args", "names")

    def __init__(self, full_name, tag=None, exclude_from_trace=False, key="", ignore=False):
        self.args = (full_name, tag, exclude_from_trace, key, ignore)
        self.names = None

    def _recreate_cm(self):
        return type(self)(*self.args)      # (as a decorator: a scope of its own for every call)

    def __enter__(self):
        profiler = optimus.globals.profiler
        if profiler is None or self.args[4]:
            return
        full_name, tag, exclude_from_trace, key, _ = self.args
        tokens = full_name.split("--")
        names = ["--".join(tokens[0:i + 1]) for i in range(len(tokens))]
        self.names = (profiler, names)
        try:
            for name in names:
                if name not in profiler.timers:
                    profiler.register_timer(name, tag=tag, exclude_from_trace=exclude_from_trace)
                profiler.start(name, key=key)
        except BaseException:
            self.__exit__(None, None, None)
            raise

    def __exit__(self, *exception):
        if self.names is not None:
            (profiler, names), self.names = self.names, None
            for name in names:
                profiler.stop(name)
        return False


class PclProfiler:
    """Hierarchical stream timers: start/stop record HIP events; summary() resolves them."""

    def __init__(self, process="GPU", rank=0, world_size=1):
        self.process = process
        self.rank = rank
        self.world_size = world_size
        self.timers = {}

    def register_timer(self, name, tag=None, exclude_from_trace=False):
        self.timers[name] = {"tag": tag, "exclude_from_trace": exclude_from_trace, "open": None,
                             "pairs": []}

    def start(self, name, key=""):
        ev = torch.cuda.Event(enable_timing=True)
        ev.record()
        self.timers[name]["open"] = ev

    def stop(self, name):
        t = self.timers[name]
        ev = torch.cuda.Event(enable_timing=True)
        ev.record()
        t["pairs"].append((t["open"], ev))
        t["open"] = None

    def summary(self, reset=True):
        """-> {name: (calls, total_ms)}; synchronises the device once."""
        torch.cuda.synchronize()
        out = {}
        for name, t in self.timers.items():
            out[name] = (len(t["pairs"]), sum(a.elapsed_time(b) for a, b in t["pairs"]))
            if reset:
                t["pairs"] = []
        return out
