"""What a captured decode graph needs of the host (no GPU): an executor and its
buckets go with their last reference, and no cyclic collection runs inside a
capture -- it could destroy another executor's graph there, whose destructor
waits for the device and ends the process when that is refused."""

from __future__ import annotations

import contextlib
import gc
import threading
import weakref

import pytest
import torch

from tensorforge_amd import decode
from tensorforge_amd.cache import PagedKVCache, PagedKVCacheConfig
from tensorforge_amd.capture import collector_held, graph_capture
from tensorforge_amd.decode import BucketedDecodeExecutor, DecodeGraphBucket, DecoderWeights, small_config


@pytest.fixture
def host_executor(monkeypatch):
    """An executor over host tensors (nothing of it can run)."""

    zeros = torch.zeros

    def pageable(*args, pin_memory=False, **options):
        return zeros(*args, **options)

    monkeypatch.setattr(torch, "zeros", pageable)
    monkeypatch.setattr(decode, "linear_rows_supported", lambda x, weight: True)
    config = small_config()
    weights = DecoderWeights.random(config, seed=0, dtype=torch.float16, device="cpu")
    cache = PagedKVCache(PagedKVCacheConfig(
        num_layers=config.num_hidden_layers, num_blocks=8, block_size=16,
        num_kv_heads=config.num_key_value_heads, head_dim=config.head_dim, max_sequences=3,
        max_sequence_length=64, dtype=torch.float16, device=torch.device("cpu")))
    return lambda **options: BucketedDecodeExecutor(weights, cache, batch_buckets=(2,),
                                                    context_buckets=(64,), **options)


@pytest.mark.parametrize("fuse_norms", [True, False])
def test_executor_and_buckets_go_with_their_last_reference(host_executor, fuse_norms):
    executor = host_executor(fuse_norms=fuse_norms)
    bucket, fallback = executor.bucket(1, 32), executor._fallback_bucket(3, 64)
    assert bucket.fused_norms == fallback.fused_norms == fuse_norms
    alive = [weakref.ref(executor), weakref.ref(bucket), weakref.ref(fallback)]
    with collector_held():  # reference counts alone
        del executor, bucket, fallback
        assert [ref() for ref in alive] == [None] * 3


@pytest.mark.parametrize("fails", [False, True])
def test_decode_capture_holds_the_collector(monkeypatch, fails):
    seen = []

    class Stream:
        def __init__(self, *args):
            pass

        def wait_stream(self, other):
            pass

    class Graph:
        def replay(self):
            seen.append(("replay", gc.isenabled()))

    bucket = object.__new__(DecodeGraphBucket)
    bucket.graph, bucket._graph, bucket._metrics = True, None, None
    bucket.device, bucket.token_state = torch.device("cpu"), torch.zeros(1, dtype=torch.long)
    bucket.next_tokens = bucket.token_state

    def forward():
        seen.append(("forward", gc.isenabled()))
        if fails and len(seen) == 2:
            raise RuntimeError("capture failed")

    bucket._forward = forward
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: Stream())
    monkeypatch.setattr(torch.cuda, "Stream", Stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda stream: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "graph", lambda graph, **options: contextlib.nullcontext())
    assert gc.isenabled()
    if fails:
        with pytest.raises(RuntimeError, match="capture failed"):
            bucket.execute()
        assert seen == [("forward", True), ("forward", False)]
    else:
        bucket.execute()
        assert seen == [("forward", True), ("forward", False), ("replay", True)]
    assert gc.isenabled()


def test_overlapping_holds_restore_the_collector_once(monkeypatch):
    monkeypatch.setattr(torch.cuda, "graph", lambda graph, **options: contextlib.nullcontext())
    inside, leave = threading.Event(), threading.Event()

    def other():
        with graph_capture(None):
            inside.set()
            assert leave.wait(30)

    thread = threading.Thread(target=other)
    with collector_held():
        thread.start()
        assert inside.wait(30)
    assert not gc.isenabled()  # the other capture still runs
    leave.set()
    thread.join()
    assert gc.isenabled()
    gc.disable()
    try:
        with graph_capture(None):
            assert not gc.isenabled()
        assert not gc.isenabled()  # as the caller had it
    finally:
        gc.enable()
