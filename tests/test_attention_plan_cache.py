"""The plans that attention calls keep by size (no GPU): a plan filled while
another thread has fixed a partition size, or from arguments of another type,
must not stay under a key that later calls read."""

from __future__ import annotations

import pytest

from tensorforge_amd.kernels import set_attention_split_size
from tensorforge_amd.kernels.attention import _plan_for, attention_plan


@pytest.fixture(autouse=True)
def empty_cache():
    _plan_for.cache_clear()
    previous = set_attention_split_size(None)
    yield
    set_attention_split_size(previous)
    _plan_for.cache_clear()


@pytest.mark.parametrize("key", [None, 64, 512])
@pytest.mark.parametrize("other", [None, 64, 1024])
def test_kept_plan_follows_its_key(key, other):
    sizes = (2048, 4, 4, 2048)
    set_attention_split_size(key)
    want = attention_plan(*sizes, "auto", 1024, head_dim=64, element_bytes=2)
    set_attention_split_size(other)  # as another thread may between the read and the fill
    plan, flags = _plan_for(key, False, *sizes, "auto", 1024, 64, 2)
    assert plan == want and flags == want.flags


def test_kept_plan_follows_its_argument_types():
    first, _ = _plan_for(None, False, 2048.0, 4, 4, 2048, "auto", 1024, 64, 2)
    plan, _ = _plan_for(None, False, 2048, 4, 4, 2048, "auto", 1024, 64, 2)
    assert plan is not first and type(plan.split_size) is int and type(plan.num_splits) is int
