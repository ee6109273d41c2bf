"""The generic decode-attention kernel at the sizes where its tiling can go
wrong, against the fp64 restatement below and the CPU oracle: head_dims that
are not a multiple of its vectors, caches that do not start on one, groups
above 16 heads, pages that straddle its 16-token tiles and 1024-token page
windows, absent pages and non-finite values behind masked tokens.

Bar: fp32 storage within 4e-6 of the largest output (fp32 products and sums
over at most 1,100 tokens; measured <= 6e-7); bf16/fp16 within one rounding
of the output, 2^-8 / 2^-11 relative, plus that."""

from __future__ import annotations

import pytest
import torch

from tensorforge_amd.kernels import PagedAttentionWorkspace, paged_gqa_decode_attention
from tensorforge_amd.workloads import make_decode_attention_case

pytestmark = pytest.mark.gpu

ROUNDING = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _reference64(case) -> torch.Tensor:
    query = case.query.double()
    out = torch.zeros_like(query)
    group = query.shape[1] // case.key_cache.shape[2]
    page = case.key_cache.shape[1]
    for row, length in enumerate(case.lengths):
        tokens = [t for t in range(length)
                  if 0 <= int(case.block_tables[row, t // page]) < case.key_cache.shape[0]]
        if not tokens:
            continue
        pages = torch.tensor([int(case.block_tables[row, t // page]) for t in tokens])
        offsets = torch.tensor([t % page for t in tokens])
        keys = case.key_cache[pages, offsets].double().repeat_interleave(group, dim=1)
        values = case.value_cache[pages, offsets].double().repeat_interleave(group, dim=1)
        scores = torch.einsum("hd,thd->ht", query[row], keys) * case.scale
        out[row] = torch.einsum("ht,thd->hd", torch.softmax(scores, dim=-1), values)
    return out


def _check(got: torch.Tensor, want: torch.Tensor, dtype: torch.dtype, what: str) -> None:
    off = (got.cpu().double() - want).abs()
    bar = 4e-6 * float(want.abs().max()) + ROUNDING[dtype] * want.abs()
    assert bool((off <= bar).all()), f"{what}: off by {float((off - bar).max()):.3g} more than the bar"


@pytest.mark.parametrize("path", ["one_pass", "split_kv"])
@pytest.mark.parametrize(("dtype", "query_heads", "kv_heads", "head_dim", "page", "lengths"), [
    (torch.float32, 32, 4, 64, 16, [1, 15, 16, 17, 64, 65, 0, 1024, 1025]),
    (torch.float32, 8, 2, 32, 16, [63, 1040, 5]),
    (torch.float32, 16, 2, 128, 5, [1029, 37, 128]),
    (torch.float32, 4, 2, 256, 1, [1030, 3]),
    (torch.float32, 6, 2, 30, 3, [333, 16]),
    (torch.float32, 34, 2, 12, 7, [520, 1]),
    (torch.float32, 64, 1, 128, 16, [300, 48]),
    (torch.bfloat16, 32, 4, 80, 16, [511, 512, 9]),
    (torch.float16, 40, 2, 192, 24, [700, 24]),
    (torch.bfloat16, 128, 2, 64, 16, [129, 1100]),
    (torch.float16, 2, 2, 1, 16, [50]),
    (torch.bfloat16, 32, 2, 256, 9, [260]),
])
def test_generic_attention_edges(device, path, dtype, query_heads, kv_heads, head_dim, page, lengths):
    case = make_decode_attention_case(lengths, query_heads=query_heads, kv_heads=kv_heads,
                                      head_dim=head_dim, block_size=page, dtype=dtype, seed=head_dim + page)
    gpu = case.to(device)
    got = paged_gqa_decode_attention(gpu.query, gpu.key_cache, gpu.value_cache, gpu.block_tables,
                                     gpu.context_lengths, scale=case.scale, attention_path=path,
                                     max_context_length=max(lengths))
    _check(got, _reference64(case), dtype, f"{path} D={head_dim} page={page}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_generic_attention_of_caches_off_the_vector_boundary(device, dtype):
    """Contiguous caches and queries that start one element past a 16-byte
    boundary take the element-wise loads."""

    case = make_decode_attention_case([200, 77], query_heads=4, kv_heads=2, head_dim=96, block_size=16,
                                      dtype=dtype, seed=3)

    def shifted(tensor: torch.Tensor) -> torch.Tensor:
        room = torch.empty(tensor.numel() + 1, dtype=tensor.dtype, device=device)
        view = room[1:].view(tensor.shape)
        view.copy_(tensor)
        return view

    query, key_cache, value_cache = (shifted(t) for t in (case.query, case.key_cache, case.value_cache))
    got = paged_gqa_decode_attention(query, key_cache, value_cache, case.block_tables.to(device),
                                     case.context_lengths.to(device), scale=case.scale, max_context_length=208)
    _check(got, _reference64(case), dtype, "shifted caches")


def test_generic_attention_skips_absent_pages_and_what_lies_behind_them(device):
    """Absent pages (a leading one, and every page of a tile) add nothing,
    whatever the unmapped pages and the tails of mapped ones hold."""

    case = make_decode_attention_case([300, 40], query_heads=8, kv_heads=2, head_dim=64, block_size=16,
                                      dtype=torch.float32, seed=9, extra_pages=1)
    case.block_tables[0, 0] = -1
    case.block_tables[0, 4] = case.key_cache.shape[0]
    case.block_tables[1, 1] = -1
    tail = int(case.block_tables[0, 18])  # 300 = 18 pages of 16 and 12 tokens
    case.key_cache[tail, 12:] = float("inf")
    case.value_cache[tail, 12:] = float("nan")
    gpu = case.to(device)
    workspace = PagedAttentionWorkspace.allocate(batch_capacity=2, query_heads=8, head_dim=64,
                                                 max_context_length=2048, device=device)
    for path in ("one_pass", "split_kv"):
        got = paged_gqa_decode_attention(gpu.query, gpu.key_cache, gpu.value_cache, gpu.block_tables,
                                         gpu.context_lengths, scale=case.scale, attention_path=path,
                                         max_context_length=304, workspace=workspace)
        _check(got, _reference64(case), torch.float32, path)


def test_generic_attention_of_long_rows_keeps_every_token(device):
    """At lengths where the matrix-core kernel would take partitions sized on
    the device, this one takes fixed partitions that cover the context."""

    case = make_decode_attention_case([8200, 8192, 31], query_heads=4, kv_heads=2, head_dim=32, block_size=16,
                                      dtype=torch.float32, seed=4)
    gpu = case.to(device)
    got = paged_gqa_decode_attention(gpu.query, gpu.key_cache, gpu.value_cache, gpu.block_tables,
                                     gpu.context_lengths, scale=case.scale, max_context_length=8208)
    _check(got, _reference64(case), torch.float32, "8200 tokens")
