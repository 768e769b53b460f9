"""Extreme scores through the FP32 kernel (GPU): additive masks of the type's lowest value, and
small probabilities beside a dominant one, against fp64."""
from __future__ import annotations

from dataclasses import replace

import numpy as np
import pytest
import torch

from jetspec_amd import packed_tree_attention, read_and_clear_status
from test_fp32_kernel_gpu import make_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
LOWEST = float(np.finfo(np.float32).min)


def attend(q, k, v, meta, slots, bias, scale, groups):
    """One request in fp64 on the host; `bias` [n, n], key j of the tree visible to rows i >= j."""
    n, prefix, block = meta.node_counts_host[0], meta.prefix_lengths[0], meta.block_size
    pos = np.arange(prefix)
    table = np.asarray(meta.block_tables_host[0], dtype=np.int64)
    index = np.concatenate([table[pos // block] * block + pos % block if prefix else pos, slots[0].cpu().numpy()])
    index = torch.as_tensor(index)
    out = torch.empty(q.shape, dtype=torch.float64)
    hidden = torch.ones(n, n).triu(1).bool() | (bias == float("-inf"))
    for h in range(q.shape[1]):
        keys = k.cpu().view(-1, *k.shape[2:])[index, h // groups].double()
        values = v.cpu().view(-1, *v.shape[2:])[index, h // groups].double()
        score = q[:, h].cpu().double() @ keys.T.contiguous() * scale
        score[:, prefix:] += bias.double()
        score[:, prefix:][hidden] = float("-inf")
        out[:, h] = torch.softmax(score, -1) @ values
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prefix,nodes", [(0, 37), (45, 37), (0, 700), (600, 50)])
def test_lowest_value_masks(prefix, nodes, dtype):
    """A mask of torch.finfo(float32).min instead of -inf: it hides a key beside any other, and a row
    whose every visible key carries it is the mean of those keys, as in torch's softmax.  Masks of
    two very low values keep their order.  Bound: test_fp32_tiles_gpu.py's for the scores and sums."""
    q, k, v, meta, slots, masks = make_case((prefix,), (nodes,), kv_heads=1, groups=3, head_dim=96, dtype=dtype, seed=7)
    bias = torch.where(masks[0].cpu(), 0.0, LOWEST)
    bias[5:9] = LOWEST                     # rows that see no tree key otherwise
    bias[nodes // 2:nodes // 2 + 3] = LOWEST
    bias[11], bias[11, 4] = -3.0e38, -2.5e38
    bias[12], bias[12, :2] = float("-inf"), LOWEST
    biased = replace(meta, qq_bias=bias.reshape(-1).to(DEV))
    out = packed_tree_attention(q, k, v, biased, 96 ** -0.5, 3, output_dtype=torch.float32)
    expect = attend(q, k, v, meta, slots, bias, 96 ** -0.5, 3)
    error = (out.cpu().double() - expect).abs().max().item()
    print(f"[lowest P{prefix} n{nodes} {dtype}] max-abs {error:.2e}", flush=True)
    assert error <= 1e-5
    assert read_and_clear_status(DEV) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("octaves", [10, 14, 16, 18, 20])
def test_small_probabilities_beside_a_dominant_one(octaves, dtype):
    """One key at the maximum with V = 0 and 8191 keys of one lower score with V = 1: the output is the
    sum of the small probabilities alone, all rounded alike, so its relative error is theirs.
    Bound: 2^-19 is the rounding of one held to 2^-39 of the reference at 2^-20 of it; the fp32
    score (below 16 in log2 units, 2^-20 there), exponential and sums add at most as much."""
    q, k, v, meta, *_ = make_case((8150,), (42,), kv_heads=1, groups=3, head_dim=96, dtype=dtype, seed=3)
    k.zero_(), v.fill_(1.0), q.zero_()
    q[..., 0] = 1.0
    top = meta.block_tables_host[0][0]   # position 3
    k[top, 3, 0, 0], v[top, 3] = 1.0, 0.0
    worst = 0.0
    for step in range(8):   # probabilities over one octave: the rounding of some is near the worst
        scale = (octaves + step / 8) * float(np.log(2.0))
        out = packed_tree_attention(q, k, v, meta, scale, 3, output_dtype=torch.float32)
        keys = (meta.prefix_lengths[0] + 1 + torch.tensor(
            [int((meta.qq_bias[i * 42:i * 42 + 42] == 0).sum()) - 1 for i in range(42)])).double()
        small = (keys - 1) * np.exp(-np.float64(np.float32(scale)))
        expect = (small / (1.0 + small)).view(-1, 1, 1)
        worst = max(worst, ((out.cpu().double() - expect) / expect).abs().max().item())
    print(f"[octaves {octaves} {dtype}] relative {worst:.2e}", flush=True)
    assert worst <= 2.0 ** -18
    assert read_and_clear_status(DEV) == 0
