"""Prefill attention's launch limits (no GPU: every call is refused before it
touches a pointer)."""

from __future__ import annotations

import pytest

from tensorforge_amd import _native

FAKE = 0x1000
UNSUPPORTED = 2  # TF_ERROR_UNSUPPORTED


@pytest.mark.parametrize(("tiles", "query_heads", "kv_heads", "head_dim", "heads_per_wave"), [
    # tiles x head groups x 256 threads: 2^32 and its multiples, then just past the limit.
    (1 << 24, 16, 16, 64, 1),
    (1 << 27, 32, 4, 64, 1),
    (1 << 24, 1, 1, 128, 1),
    ((1 << 22) + 1, 32, 4, 64, 8),
    ((1 << 23) + 1, 32, 4, 32, 0),
])
def test_a_grid_past_the_launch_limit_is_refused(tiles, query_heads, kv_heads, head_dim, heads_per_wave):
    launch, width = _native.launch(), query_heads * head_dim
    status = launch.tf_prefill_attention(
        FAKE, width, FAKE, kv_heads * head_dim, FAKE, kv_heads * head_dim, FAKE, width, FAKE, tiles,
        query_heads, kv_heads, head_dim, 1.0, heads_per_wave, _native.TF_DTYPE_BFLOAT16, None)
    assert status == UNSUPPORTED
    assert b"grid too large" in _native.library().tf_last_error()
