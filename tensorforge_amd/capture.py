"""HIP graph capture with Python's cyclic collector held off.

A collection that happens to run inside a capture may free device objects that
only a reference cycle kept alive.  The destructor of a torch CUDAGraph waits
for the device on ROCm, a wait the runtime refuses while a stream is being
captured, and a destructor that fails ends the process.
"""

from __future__ import annotations

import gc
import threading
from collections.abc import Iterator
from contextlib import contextmanager
from typing import Any

import torch

_LOCK = threading.Lock()
_HOLDERS = 0
_RESUME = False


@contextmanager
def collector_held() -> Iterator[None]:
    """No automatic collection inside the block.  The collector is the
    process's, so overlapping blocks (several threads) share one hold: the
    first turns it off, the last turns it on again if it was on."""

    global _HOLDERS, _RESUME
    with _LOCK:
        if _HOLDERS == 0:
            _RESUME = gc.isenabled()
            gc.disable()
        _HOLDERS += 1
    try:
        yield
    finally:
        with _LOCK:
            _HOLDERS -= 1
            if _HOLDERS == 0 and _RESUME:
                gc.enable()


@contextmanager
def graph_capture(graph: torch.cuda.CUDAGraph, **options: Any) -> Iterator[None]:
    """``torch.cuda.graph(graph, **options)`` with the collector held."""

    with collector_held(), torch.cuda.graph(graph, **options):
        yield
