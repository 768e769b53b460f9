"""The FP32 kernel's two forms around the length where they meet (GPU): a wave per packed row for
short requests, matrix instructions above.  Both against the fp64 oracle (bound as in
test_fp32_tiles_gpu.py), and the form must follow the live lengths alone: a launch that knows
them on the host, one that does not and a replayed graph give the same bits."""
from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from gpu_helpers import errors, oracle_rows
from jetspec_amd import packed_tree_attention, paged_tree_attention, read_and_clear_status
from jetspec_amd.paged_backend import _fp32_template, _launch_fp32
from test_fp32_kernel_gpu import FIELDS, make_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUND = 1e-5


@pytest.mark.parametrize("dtype,dim,groups,block", [
    (torch.float32, 128, 1, 256), (torch.float32, 64, 4, 16), (torch.float32, 40, 3, 16), (torch.float32, 200, 2, 256),
    (torch.float32, 500, 1, 16), (torch.bfloat16, 96, 1, 16), (torch.bfloat16, 72, 4, 48), (torch.float16, 80, 2, 16),
    (torch.float16, 1, 2, 5)])
@pytest.mark.parametrize("keys", [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 193, 255, 256, 257])
def test_both_sides_of_the_row_form(keys, dtype, dim, groups, block):
    """The longest request has `keys` keys; a few-row and a many-row batch of each."""
    for counts in ([1, 1], [min(keys, 23), min(keys, 40)]):
        prefixes = [max(0, keys - counts[0]), max(0, keys // 2 - counts[1])]
        q, k, v, meta, *_ = make_case(prefixes, counts, groups=groups, head_dim=dim, block=block, dtype=dtype,
                                      seed=keys + dim)
        out = packed_tree_attention(q, k, v, meta, dim ** -0.5, groups, output_dtype=torch.float32)
        unknown = torch.empty_like(out)   # the lengths read on the device
        _launch_fp32(_fp32_template(meta, k, v, groups, q.device), q, unknown, dim ** -0.5,
                     torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        error, _ = errors(out, oracle_rows(q, k, v, meta, dim ** -0.5, [0, 1]))
        assert error <= BOUND, (counts, error)
        assert torch.equal(out, unknown), counts
        assert read_and_clear_status(DEV) == 0


def test_a_replayed_graph_takes_the_live_lengths_form():
    """Rounds on both sides of the row form's limit (128 keys here) through one captured launch."""
    rounds = [((100, 3, 60), (12, 6, 9)), ((117, 40, 0), (12, 6, 9)), ((20, 119, 30), (9, 6, 12)),
              ((20, 123, 30), (9, 6, 12)), ((3, 900, 5), (6, 12, 9)), ((1, 2, 3), (9, 12, 6))]
    cases = [make_case(p, c, head_dim=128, dtype=torch.float32, seed=70 + i) for i, (p, c) in enumerate(rounds)]
    pages = max(int(c[1].shape[0]) for c in cases)
    k = torch.randn((pages, 256, 2, 128), device=DEV)
    v = torch.randn_like(k)
    first = cases[0][3]
    # The bias is sized for the largest of the rounds' trees.
    sizes = {"qq_bias": max(c[3].qq_bias.numel() for c in cases)}
    tensors = {name: torch.zeros(sizes.get(name, getattr(first, name).numel()), dtype=getattr(first, name).dtype,
                                 device=DEV) for name in FIELDS if name != "block_tables"}
    tensors["block_tables"] = torch.full((3, 4), -1, dtype=torch.int32, device=DEV)
    staged = replace(first, **{**tensors, "qq_bias": tensors["qq_bias"]})
    q_in = torch.empty_like(cases[0][0])
    graph = None
    for index, (q, _, _, meta, *_) in enumerate(cases):
        for name in FIELDS:
            dst, src = getattr(staged, name), getattr(meta, name)
            if name == "block_tables":
                dst[:, :src.shape[1]].copy_(src)
            else:
                dst[:src.numel()].copy_(src)
        q_in.copy_(q)
        if graph is None:
            captured = torch.empty_like(q)
            template = _fp32_template(staged, k, v, 4, q.device)
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.current_stream())
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                _launch_fp32(template, q_in, captured, 0.125, torch.cuda.current_stream().cuda_stream, 1)
        graph.replay()
        torch.cuda.synchronize()
        eager = packed_tree_attention(q, k, v, meta, 0.125, 4)
        error, _ = errors(eager, oracle_rows(q, k, v, meta, 0.125, [0, 1, 2]))
        assert error <= BOUND, index
        assert torch.equal(captured, eager), index
        torch.randn(1 << 20, device=DEV).sum().item()   # eager work between replays
    assert read_and_clear_status(DEV) == 0


@pytest.mark.parametrize("prefix", [7, 300])
def test_slot_addressed_entry(prefix):
    """The legacy entry's prefixes, in either form."""
    n, groups, dim = 19, 2, 48
    q, k, v, meta, slots, masks = make_case((prefix,), (n,), groups=groups, head_dim=dim, dtype=torch.float32, seed=2)
    pos = torch.arange(prefix)
    table = torch.tensor(meta.block_tables_host[0], dtype=torch.int64)
    logical = torch.cat([(table[pos // 256] * 256 + pos % 256).to(DEV), slots[0]])[None]
    bias = torch.where(masks[0], 0.0, float("-inf"))
    out = paged_tree_attention(q, k, v, None, None, torch.tensor([prefix + n], device=DEV), bias, dim ** -0.5, groups, 256,
                               logical)
    torch.cuda.synchronize()
    error, _ = errors(out, oracle_rows(q, k, v, meta, dim ** -0.5, [0]))
    assert error <= BOUND and read_and_clear_status(DEV) == 0
