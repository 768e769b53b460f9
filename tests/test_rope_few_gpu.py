"""The few-rows form of the RoPE + scatter kernel and the row count where the other one takes
over (GPU): byte-exact against the oracle on both sides of it, with cos/sin caches that take
16-byte loads and ones that do not."""
from __future__ import annotations

import pytest
import torch

from test_rope_gpu import assert_equivalent, fixture

pytestmark = pytest.mark.gpu


# 8 query and 2 KV heads of 128: 112 bf16 or 224 fp32 work items a row, one pass of 256
# threads; 32 and 8 heads: 448 or 896, two or four passes.  2048 workgroups are the limit.
@pytest.mark.parametrize("dtype,heads,rows", [
    (torch.bfloat16, (8, 2), 1), (torch.bfloat16, (8, 2), 2048), (torch.bfloat16, (8, 2), 2049),
    (torch.bfloat16, (32, 8), 1024), (torch.bfloat16, (32, 8), 1025),
    (torch.float32, (32, 8), 512), (torch.float32, (32, 8), 513)])
@pytest.mark.parametrize("cache_dtype", [torch.float32, torch.bfloat16])
def test_both_sides_of_the_row_limit(dtype, heads, rows, cache_dtype):
    args = fixture(dtype, rows=rows, q_heads=heads[0], kv_heads=heads[1], pages=9, cache_dtype=cache_dtype)
    assert_equivalent(args)


@pytest.mark.parametrize("cache_dtype", [torch.float32, torch.bfloat16])
def test_cache_rows_without_vector_loads(cache_dtype):
    args = list(fixture(cache_dtype=cache_dtype, cache_rank=2))
    cache = args[4]
    odd = torch.empty((cache.shape[0], cache.shape[1] + 1), dtype=cache.dtype, device=cache.device)
    odd[:, 1:] = cache
    args[4] = odd[:, 1:]   # rows start off 16-byte alignment
    assert_equivalent(tuple(args))
