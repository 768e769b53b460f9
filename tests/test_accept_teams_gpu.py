"""The team form of the output cut at its edges (GPU): paths around 16, 32 and 64 nodes, batches
around one pass and around 256 requests, against the oracle's host walk and cut.  Tokens and indices: every comparison is exact."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from jetspec_amd import accept_batch_device, greedy_argmax, read_and_clear_status, truncate_accepted, workloads
from test_accept_gpu import DEV, expected_cuts, random_batch

pytestmark = pytest.mark.gpu
VOCAB = 64


@pytest.mark.parametrize("index_dtype", [torch.int64, torch.int32])
@pytest.mark.parametrize("max_depth,sizes", [
    (0, [1, 5, 64]), (14, [16, 15, 17]), (15, [16, 64] * 32), (15, [1, 64, 65] * 22), (16, [18, 40] * 16 + [17]),
    (31, [64, 65, 128, 129] * 8), (32, [40] * 17), (63, [64, 70, 255, 256] * 5), (64, [66, 80, 257]),
    (15, [4] * 256), (15, [4] * 257), (12, [256, 257, 300])])
def test_walk_and_cut_equal_the_oracle(max_depth, sizes, index_dtype):
    print(f"[teams] max_depth={max_depth} requests={len(sizes)} {index_dtype}", flush=True)
    rng = np.random.default_rng(1000 * max_depth + len(sizes))
    trees, offsets = random_batch(rng, sizes, vocab=VOCAB)
    for tree in trees[::2]:   # every other request a chain, so that paths reach the depth limit
        tree.host_parents = workloads.chain_parents(tree.num_nodes)
        tree.host_depths = workloads.depths_of(tree.host_parents)
        tree.child_maps = oracle.child_maps(tree.host_token_ids, tree.host_parents)
    logits = torch.randn(offsets[-1], VOCAB)
    for tree, lo in zip(trees, offsets):
        for node, children in enumerate(tree.child_maps):
            if children and rng.random() < 0.98:
                logits[lo + node, int(rng.choice(list(children)))] += 20.0
    packed = [torch.tensor([x for tree in trees for x in getattr(tree, name)], dtype=index_dtype, device=DEV)
              for name in ("host_token_ids", "host_parents", "host_depths")]
    cu = torch.tensor(offsets, dtype=torch.int32, device=DEV)
    status = torch.zeros(1, dtype=torch.int32, device=DEV)
    greedy, paths, lengths, corrections = accept_batch_device(logits.to(DEV), *packed, cu, max_depth, status=status)
    greedy, host_paths = greedy.tolist(), paths.cpu()
    for i, tree in enumerate(trees):
        want = oracle.accept_walk(greedy[offsets[i]:offsets[i + 1]], tree.host_token_ids, tree.host_depths,
                                  tree.child_maps, max_depth)
        nodes = len(want["path"])
        assert host_paths[i].tolist() == want["path"] + [-1] * (max_depth + 1 - nodes), i
        assert int(lengths[i]) == nodes - 1 and int(corrections[i]) == want["correction"], i
    assert int(status) == 0

    budgets = torch.tensor(rng.integers(1, max_depth + 4, size=len(sizes)), dtype=torch.int32)
    ignore = torch.tensor(rng.random(len(sizes)) < 0.3)
    for count in (0, 1, 8, 9):   # up to 8 ids go with the launch, more are uploaded
        eos = {int(x) for x in rng.choice(VOCAB, size=count, replace=False)}
        limits, emitted, commit_paths, commit_offsets = truncate_accepted(
            paths, lengths, corrections, packed[0], cu, budgets.to(DEV), ignore.to(DEV), eos)
        cuts = expected_cuts(trees, host_paths, lengths.cpu(), corrections.cpu(), budgets.tolist(), ignore.tolist(), eos)
        assert limits.tolist() == [c["limit"] for c in cuts]
        assert emitted.tolist() == [c["emitted"] + [-1] * (max_depth + 1 - c["limit"]) for c in cuts]
        starts = np.concatenate([[0], np.cumsum([c["limit"] for c in cuts])]).tolist()
        assert commit_offsets.tolist() == starts
        assert commit_paths[:starts[-1]].tolist() == [x for c in cuts for x in c["path"]]
    assert read_and_clear_status(DEV) == 0


def test_bad_requests_beside_good_ones():
    """A length or a path node out of range and a spent budget cut their request to nothing, not its neighbours."""
    width, requests = 16, 70
    paths = torch.arange(width, dtype=torch.int32).repeat(requests, 1)
    lengths = torch.full((requests,), 5, dtype=torch.int32)
    budgets = torch.full((requests,), 40, dtype=torch.int32)
    lengths[1], lengths[3], paths[5, 4], paths[6, 0], budgets[69] = -1, width, 16, -1, 0
    paths[7, 6:] = -7   # past the path's end: not read
    tokens = torch.arange(requests * width)
    cu = torch.arange(0, (requests + 1) * width, width, dtype=torch.int32)
    limits, emitted, commit_paths, commit_offsets = truncate_accepted(
        paths.to(DEV), lengths.to(DEV), torch.full((requests,), 9999, device=DEV), tokens.to(DEV), cu.to(DEV),
        budgets.to(DEV), torch.zeros(requests, dtype=torch.bool, device=DEV), [])
    bad = {1, 3, 5, 6, 69}
    assert limits.tolist() == [0 if r in bad else 6 for r in range(requests)]
    want = [[-1] * width if r in bad else [r * width + j for j in range(1, 6)] + [9999] + [-1] * 10
            for r in range(requests)]
    assert emitted.tolist() == want
    assert commit_offsets.tolist() == np.concatenate([[0], np.cumsum(limits.tolist())]).tolist()
    assert commit_paths[:int(commit_offsets[-1])].tolist() == list(range(6)) * (requests - len(bad))
    assert read_and_clear_status(DEV) == 4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [1, 3, 7, 8, 9, 15, 2055, 50257])
def test_argmax_of_rows_off_the_vector_boundary(dtype, vocab):
    """Rows that start at every element offset from 16 bytes: the maximum, a tie and a NaN at the
    first element, around the first vector unit and at the end, as torch.argmax has them."""
    backing = torch.randn(16, vocab + 9, generator=torch.Generator(device=DEV).manual_seed(vocab), device=DEV).to(dtype)
    marks = sorted({m for m in (0, 1, 2, 3, 4, 5, 6, 7, 8, 9, vocab // 2, vocab - 2, vocab - 1) if 0 <= m < vocab})
    for start in range(9):
        rows = backing[:, start:start + vocab]
        for mark in marks:
            case = rows.clone()
            case[0, mark] = 50.0
            case[1, mark] = case[1, marks[-1]] = 50.0
            case[2, mark] = float("nan")
            case[3, mark], case[3, marks[0]] = float("nan"), float("inf")
            case[4] = float("-inf")
            rows_at = torch.empty_like(backing)[:, start:start + vocab]
            rows_at.copy_(case)
            assert torch.equal(greedy_argmax(rows_at), rows_at.argmax(-1)), (start, mark)
