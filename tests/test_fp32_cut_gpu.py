"""Batches at the edges of the FP32 kernel's key cut (GPU), against the fp64 oracle: the last request
count that is cut and the first that is not, one request far longer than the rest, the most
chunks a block takes, and a request without nodes among live metadata.  Bound: as in
test_fp32_tiles_gpu.py."""
from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from gpu_helpers import errors, oracle_rows
from jetspec_amd import packed_tree_attention, read_and_clear_status
from test_fp32_kernel_gpu import make_case

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOUND = 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("label,prefixes,counts,groups", [
    ("64 requests", [40 + 3 * i for i in range(63)] + [2500], [1 + i % 9 for i in range(64)], 4),
    ("65 requests", [40 + 3 * i for i in range(64)] + [2500], [1 + i % 9 for i in range(65)], 4),
    ("full row blocks", [6000] + [30] * 63, [36] * 64, 7),
    ("16 chunks", [9001], [2], 3)])
def test_edges_of_the_cut(label, prefixes, counts, groups, dtype):
    q, k, v, meta, *_ = make_case(prefixes, counts, kv_heads=1, groups=groups, head_dim=96, dtype=dtype, block=16,
                                  seed=len(prefixes))
    out = packed_tree_attention(q, k, v, meta, 96 ** -0.5, groups, output_dtype=torch.float32)
    torch.cuda.synchronize()
    error, _ = errors(out, oracle_rows(q, k, v, meta, 96 ** -0.5, list(range(len(prefixes))), rows_per_request=3))
    print(f"[{label} {dtype}] max-abs {error:.2e}", flush=True)
    assert error <= BOUND
    assert read_and_clear_status(DEV) == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("requests", [63, 64, 65])
def test_whole_keys_of_more_blocks_than_the_chip_takes_at_once(requests, dtype):
    """Short enough not to be cut, long enough for the matrix form: listed up to 64 requests, by
    number above."""
    q, k, v, meta, *_ = make_case([150 + i for i in range(requests)], [1 + i % 13 for i in range(requests)], kv_heads=8,
                                  groups=4, head_dim=80, dtype=dtype, block=16, seed=requests)
    out = packed_tree_attention(q, k, v, meta, 80 ** -0.5, 4, output_dtype=torch.float32)
    torch.cuda.synchronize()
    error, _ = errors(out, oracle_rows(q, k, v, meta, 80 ** -0.5, list(range(requests)), rows_per_request=2))
    assert error <= BOUND
    assert read_and_clear_status(DEV) == 0


def test_a_request_without_nodes_among_live_metadata():
    """Its rows are left alone, the others' are right."""
    q, k, v, meta, *_ = make_case((700, 900, 1200), (9, 12, 30), head_dim=96, dtype=torch.float32, seed=4)
    live = replace(meta, node_counts=meta.node_counts.clone())
    live.node_counts[1] = 0
    out = packed_tree_attention(q, k, v, live, 96 ** -0.5, 4)
    torch.cuda.synchronize()
    error, _ = errors(out, oracle_rows(q, k, v, meta, 96 ** -0.5, [0, 2]))
    assert error <= BOUND
    assert read_and_clear_status(DEV) == 0


def test_without_memory_for_the_workspace_the_keys_stay_whole(monkeypatch):
    q, k, v, meta, *_ = make_case((900, 1500), (9, 30), head_dim=96, dtype=torch.float32, seed=6)
    real = torch.empty

    def full(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.OutOfMemoryError("no memory")
        return real(*args, **kw)

    monkeypatch.setattr(torch, "empty", full)
    out = packed_tree_attention(q, k, v, meta, 96 ** -0.5, 4)
    monkeypatch.undo()
    torch.cuda.synchronize()
    error, _ = errors(out, oracle_rows(q, k, v, meta, 96 ** -0.5, [0, 1]))
    assert error <= BOUND
    assert read_and_clear_status(DEV) == 0
