"""Edges of the FP32 kernel's tiles, row blocks and key cuts (GPU).

The kernel works on blocks of 32 score rows and tiles of 32 keys, four waves to a block, and
cuts the keys of small batches over several workgroups.  Row counts, prefixes and head sizes
on both sides of those edges are compared with the fp64 oracle in every operand type, with
FP32 output.  Bound: each output is a convex combination of V entries of magnitude below 6,
and the sums run over at most 2100 keys and 512 dimensions in fp32, so 512 * 2^-24 * 6 =
1.8e-4 bounds the score error's effect at the worst and 1e-5 is what random signs leave of it
(sqrt(512) instead of 512).
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from gpu_helpers import errors, oracle_rows
from jetspec_amd import _lib, packed_tree_attention, read_and_clear_status
from jetspec_amd.paged_backend import _fp32_template, _launch_fp32
from test_fp32_kernel_gpu import make_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUND = 1e-5

# (prefixes, node counts, KV heads, query heads per KV head, head size, page)
SHAPES = [
    ((0, 31, 32, 33), (1, 1, 8, 9), 1, 4, 128, 16),        # one row block and one more row; empty prefix
    ((2047, 1, 300), (7, 30, 11), 2, 3, 96, 48),           # a cut prefix, blocks that end inside a node
    ((1023, 1025), (64, 63), 8, 12, 80, 16),               # the exact-size instance with a partial 64-dim pair
    ((513,), (33,), 1, 33, 112, 256),                      # more query heads than a block has rows
    ((200, 90), (20, 5), 2, 4, 72, 16),                    # element loads in 16 bits (72 is no multiple of 16)
    ((257, 64), (12, 40), 1, 5, 192, 32),                  # two register slabs
    ((129,), (17,), 1, 3, 500, 16),                        # the widest instance, ragged head size
    ((40, 7), (3, 2), 1, 2, 1, 5),                         # one dimension, odd page
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"D{s[4]}G{s[3]}")
def test_tile_edges(shape, dtype):
    prefixes, counts, kv_heads, groups, dim, block = shape
    q, k, v, meta, *_ = make_case(prefixes, counts, kv_heads=kv_heads, groups=groups, head_dim=dim, block=block,
                                  dtype=dtype, seed=dim + groups)
    scale = dim ** -0.5
    template = _fp32_template(meta, k, v, groups, q.device)
    out = torch.empty(q.shape, dtype=torch.float32, device=DEV)
    _launch_fp32(template, q, out, scale, torch.cuda.current_stream().cuda_stream)
    whole = torch.empty_like(out)   # the entry without a workspace: no cut
    args = _lib.TreeAttentionFp32Args.from_buffer_copy(template)
    args.q, args.q_stride_row, args.q_stride_head = q.data_ptr(), q.stride(0), q.stride(1)
    args.out, args.out_stride_row, args.out_stride_head = whole.data_ptr(), whole.stride(0), whole.stride(1)
    args.out_dtype, args.scale = _lib.TV_F32, scale
    assert _lib.library().tv_tree_attention_fp32(ctypes.byref(args), torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    expect = oracle_rows(q, k, v, meta, scale, list(range(meta.num_requests)))
    for name, got in (("cut", out), ("whole", whole)):
        error, _ = errors(got, expect)
        print(f"[D{dim} G{groups} {dtype} {name}] max-abs {error:.2e}", flush=True)
        assert error <= BOUND, name
    assert read_and_clear_status(DEV) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_values_that_are_not_finite_reach_only_the_rows_that_see_them(dtype, value):
    """A tree node's V with a NaN or an infinity: rows that cannot see the node keep their finite
    results, to the bit; rows that see it take the value as a sum over their keys would, and keep
    the other dimensions (added in another order: within two roundings of the output type)."""
    q, k, v, meta, slots, masks = make_case((70, 33), (40, 9), head_dim=96, dtype=dtype, seed=5)
    node, dim = 11, 37
    clean = packed_tree_attention(q, k, v, meta, 96 ** -0.5, 4)
    v.view(-1, *v.shape[2:])[slots[0][node], 1, dim] = value
    out = packed_tree_attention(q, k, v, meta, 96 ** -0.5, 4)
    torch.cuda.synchronize()
    sees = torch.zeros(out.shape[0], dtype=torch.bool, device=DEV)
    sees[:40] = masks[0][:, node]
    assert sees.any() and not sees.all()
    assert torch.equal(out[~sees], clean[~sees]) and torch.equal(out[:, :4], clean[:, :4])
    touched = torch.zeros_like(out, dtype=torch.bool)
    touched[sees, 4:, dim] = True   # query heads 4 to 7 read KV head 1
    torch.testing.assert_close(out[~touched], clean[~touched], rtol=2 * torch.finfo(dtype).eps, atol=1e-6)
    hit = out[touched].float()
    assert (torch.isnan(hit) if value != value else hit == value).all()
    assert read_and_clear_status(DEV) == 0
