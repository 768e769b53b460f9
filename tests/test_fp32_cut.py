"""How the FP32 kernel cuts the keys of a batch, on the host: the query runs the kernel's own
search over host lengths.  The cut must fit the rounds that the row blocks alone take, since a
part-filled round more would double the launch, and be the shortest that does."""
from __future__ import annotations

import ctypes
import random

import pytest

from jetspec_amd import _lib

BLOCK, TILE, WAVES, MAX_SPLITS = 32, 32, 4, 16
MIN_CHUNK = {_lib.TV_F32: 8, _lib.TV_BF16: 16}


def cut(prefixes, nodes, q_heads, kv_heads, head_dim, dtype):
    lib, n = _lib.library(), len(prefixes)
    keys, workgroups = ctypes.c_int32(), ctypes.c_int32()
    _lib.check(lib.tv_tree_attention_fp32_chunk_keys((ctypes.c_int32 * n)(*prefixes), (ctypes.c_int32 * n)(*nodes), n,
                                                     q_heads, kv_heads, head_dim, dtype, ctypes.byref(keys),
                                                     ctypes.byref(workgroups)), "chunk_keys")
    return keys.value, workgroups.value


def expected(prefixes, nodes, q_heads, kv_heads, head_dim, dtype):
    """The shortest chunk that fits, by trying every one."""
    groups = q_heads // kv_heads
    blocks = [-(-t * groups // BLOCK) for t in nodes]
    tiles = [-(-(p + t) // TILE) if t else 0 for p, t in zip(prefixes, nodes)]
    units, slots = sum(blocks) * kv_heads, 512 if head_dim <= 128 else 256
    limit = slots * max(1, -(-units // slots))

    def count(target):
        return sum(b * -(-t // target) for b, t in zip(blocks, tiles)) * kv_heads

    workspace = _lib.library().tv_tree_attention_fp32_workspace_bytes(sum(nodes), len(nodes), q_heads, kv_heads, head_dim)
    if workspace == 0:
        return 0, units
    rows = sum(nodes) * groups // BLOCK + len(nodes) + 1
    splits = max(1, min(MAX_SPLITS, 4096 // (rows * kv_heads)))
    target = max(MIN_CHUNK[dtype], -(-max(tiles) // splits))
    target = -(-target // WAVES) * WAVES
    while count(target) > limit and target < max(tiles):
        target += WAVES
    return target * TILE, count(target)


def batches():
    rng = random.Random(5)
    yield [20000] * 64, [73] * 64, 7, 1, 128, _lib.TV_BF16              # 1024 row blocks: two rounds
    yield [300 + 800 * i for i in range(64)], [36] * 64, 7, 1, 128, _lib.TV_F32   # 512 row blocks: no place to cut into
    yield [48000] + [40] * 63, [36] * 64, 7, 1, 128, _lib.TV_BF16       # ... one request far longer
    yield [50000], [1], 4, 1, 64, _lib.TV_F32                           # the most chunks a block takes
    yield [900, 500, 70], [5, 0, 9], 8, 2, 96, _lib.TV_BF16             # a request without nodes
    for _ in range(300):
        n, kv, groups = rng.choice([1, 3, 8, 40, 63, 64]), rng.choice([1, 2, 8]), rng.choice([1, 3, 4, 7, 12])
        top = rng.choice([100, 3000, 60000])
        yield ([rng.randint(0, top) for _ in range(n)], [rng.randint(1, 64) for _ in range(n)], kv * groups, kv,
               rng.choice([64, 96, 128, 192]), rng.choice(list(MIN_CHUNK)))


def test_the_cut_is_the_shortest_that_fits_the_row_blocks_rounds():
    cuts = 0
    for batch in batches():
        assert cut(*batch) == expected(*batch), batch
        cuts += cut(*batch)[0] > 0
    assert cuts > 150


def test_batches_beyond_64_requests_are_not_cut():
    for n in (64, 65):
        keys, workgroups = cut([5000] * n, [4] * n, 4, 1, 128, _lib.TV_F32)
        assert (keys > 0) == (n == 64) and workgroups >= n


def test_invalid_lengths_are_refused():
    for prefixes, nodes in (([-1], [4]), ([4], [-1]), ([2 ** 31 - 1], [4])):
        with pytest.raises(Exception, match="invalid lengths"):
            cut(prefixes, nodes, 4, 1, 128, _lib.TV_F32)


def test_the_workspace_holds_one_partial_block_per_workgroup():
    """Sized by the workgroups the chip runs at a time, whatever the head count or chunks."""
    size = _lib.library().tv_tree_attention_fp32_workspace_bytes
    for queries, requests, q_heads, kv_heads, dim in ((64, 1, 32, 8, 128), (200, 8, 24, 8, 96), (1, 1, 1, 1, 512),
                                                      (400, 64, 32, 8, 192), (3000, 2, 4, 1, 80)):
        blocks = (queries * (q_heads // kv_heads) // BLOCK + requests + 1) * kv_heads
        slots = 512 if dim <= 128 else 256
        assert size(queries, requests, q_heads, kv_heads, dim) == -(-blocks // slots) * slots * BLOCK * (4 * dim + 8)
    assert size(64, 65, 32, 8, 128) == 0 and size(40000, 2, 32, 8, 128) == 0
