"""What a user of this framework has it do, as cases that can be timed and compared.

The framework is the tree-verification hot path of a speculative serving loop on one MI355X.
Per decoder layer a round appends the tree's K/V and runs the packed tree attention; once per
round it accepts tokens, builds the commit maps and moves the accepted K/V rows.  Each case is
one of those calls through the package's public entry points:

  attention   ``packed_tree_attention`` (one layer's verify launch, decode trees and prefill chunks)
  round       ``PackedVerifyGraph.verify`` (RoPE + scatter + attention of every layer, graph replay)
  accept      ``accept_batch_device`` -> ``truncate_accepted`` -> ``commit_slots``
  commit      ``copy_accepted_kv`` over every layer
  append      ``store_kvcache``

The layout of a batch (prefix lengths, tree shapes, accepted paths) follows from the case alone,
so its work does; the seed gives the page order, the values and the tokens.  K, V and Q are
N(0, 1) as in the benchmark, Q times ``gain`` (a gain of 1 gives the flat softmax of unnormalised
random heads, 2-3 the peaked one of trained heads).
"""
import os
import random
import sys
from types import SimpleNamespace

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "nano-vllm-jetspec_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_DEVICE = "cuda"


# --------------------------------------------------------------------------- cases
def _attention(**kw):
    case = {"kind": "attention", "dtype": "bf16", "kv_heads": 8, "groups": 4, "head_dim": 128, "page": 256,
            "backend": "auto", "out32": False, "requests": 0, "prefix_lo": 0, "prefix_hi": 0, "tree_lo": 16,
            "tree_hi": 64, "chunks": 0, "chunk_rows": 0, "chunk_prefix_hi": 0, "fill": 1.0, "gain": 1.0, "layout": 0}
    case.update(kw)
    return case


def listed():
    return [
        # One interactive request: short context, small tree.  Latency and launches count.
        _attention(name="verify_c1", requests=1, prefix_lo=512, prefix_hi=512, tree_lo=16, tree_hi=16, layout=1),
        # A small serving batch with ragged contexts and trees of 16 to 64 nodes.
        _attention(name="verify_c8", requests=8, prefix_lo=256, prefix_hi=4096, layout=2),
        # A full serving batch at long contexts in a nearly full pool: the largest case.
        _attention(name="verify_c64_long", requests=64, prefix_lo=8192, prefix_hi=32768, tree_lo=64, tree_hi=64,
                   fill=0.9, layout=4),
        # Prefill chunks (chain trees) scheduled beside decode trees in one launch.
        _attention(name="chunks_and_trees", requests=32, prefix_lo=2048, prefix_hi=8192, tree_lo=32, tree_hi=32,
                   chunks=16, chunk_rows=512, chunk_prefix_hi=16384, layout=5),
        # One tensor-parallel shard: a single KV head with 8 query heads, medium contexts.
        _attention(name="verify_shard_g8", requests=32, kv_heads=1, groups=8, prefix_lo=1024, prefix_hi=8192, gain=2.0,
                   layout=6),
        # The FP32-probability entry of a qualification run: f16, head size 64, FP32 output.
        _attention(name="verify_exact_d64", requests=8, dtype="f16", head_dim=64, backend="prefix", out32=True,
                   prefix_lo=256, prefix_hi=4096, gain=2.0, layout=7),
        # A float32 model, as the numerical oracle runs use.
        _attention(name="verify_f32", requests=8, dtype="f32", prefix_lo=256, prefix_hi=4096, layout=8),
        # A model outside the common head sizes, on 16-token pages.
        _attention(name="verify_d96_p16", requests=4, head_dim=96, groups=3, page=16, prefix_lo=256, prefix_hi=2048,
                   gain=2.0, layout=9),
        # A whole round of a 36-layer model through the graph cache.
        {"name": "round_c8", "kind": "round", "layers": 36, "requests": 8, "kv_heads": 8, "groups": 4, "head_dim": 128,
         "page": 256, "prefix_lo": 256, "prefix_hi": 2048, "tree_lo": 32, "tree_hi": 32, "gain": 1.0, "layout": 10},
        # Greedy acceptance of 64 requests x 64 nodes over a 151936-word vocabulary, to the commit maps.
        {"name": "accept_c64", "kind": "accept", "dtype": "bf16", "requests": 64, "tree_lo": 64, "tree_hi": 64,
         "vocab": 151936, "max_depth": 15, "prefix_lo": 8192, "prefix_hi": 32768, "page": 256, "layout": 11},
        # The accepted-only commit of 64 requests over 36 layers.
        {"name": "commit_c64", "kind": "commit", "dtype": "bf16", "layers": 36, "requests": 64, "kv_heads": 8,
         "head_dim": 128, "page": 256, "prefix_lo": 128, "prefix_hi": 1024, "tree_lo": 32, "tree_hi": 32, "layout": 3},
        # The K/V append of a prefill batch, one layer, with padding rows (slot -1).
        {"name": "append_prefill", "kind": "append", "dtype": "bf16", "rows": 8192, "kv_heads": 8, "head_dim": 128,
         "page": 256, "skip": 0.02, "slots64": False, "layout": 12},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    layout = rng.randrange(1, 1 << 30)
    kind = rng.choice(["short", "short", "long", "chunks", "shard", "exact", "f32", "general", "round", "accept",
                       "commit", "append"])
    top = _log(rng, 200, 4096)
    low = _log(rng, 33, top)
    tree_hi = _log(rng, 8, 64)
    tree_lo = rng.randint(max(1, tree_hi // 4), tree_hi)
    trees = {"tree_lo": tree_lo, "tree_hi": tree_hi, "prefix_lo": low, "prefix_hi": top}
    gain = rng.choice([1.0, 2.0, 3.0])
    if kind == "short":
        return _attention(requests=_log(rng, 1, 16), groups=rng.choice([1, 2, 4, 5, 8]), gain=gain,
                          dtype=rng.choice(["bf16", "bf16", "f16"]), out32=rng.random() < 0.2, layout=layout, **trees)
    if kind == "long":
        top = _log(rng, 4096, 32768)
        return _attention(requests=_log(rng, 4, 60), prefix_lo=top // 4, prefix_hi=top, tree_lo=max(1, tree_hi // 2),
                          tree_hi=tree_hi, fill=0.9, gain=gain, layout=layout)
    if kind == "chunks":
        return _attention(requests=rng.randint(0, 32), prefix_lo=1024, prefix_hi=8192, tree_lo=min(tree_lo, 16),
                          tree_hi=min(tree_hi, 32), chunks=rng.randint(1, 12), chunk_rows=_log(rng, 100, 512),
                          chunk_prefix_hi=_log(rng, 256, 16384), gain=gain, layout=layout)
    if kind == "shard":
        return _attention(requests=_log(rng, 8, 48), kv_heads=rng.choice([1, 2]), groups=rng.choice([4, 8, 16]),
                          prefix_lo=low, prefix_hi=2 * top, tree_lo=tree_lo, tree_hi=tree_hi, gain=gain, layout=layout)
    if kind == "exact":
        return _attention(requests=_log(rng, 1, 8), dtype=rng.choice(["bf16", "f16"]),
                          head_dim=rng.choice([64, 128, 256]), backend=rng.choice(["reference", "prefix"]),
                          out32=True, gain=gain, layout=layout, **trees)
    if kind == "f32":
        return _attention(requests=_log(rng, 1, 8), dtype="f32", groups=rng.choice([1, 2, 4, 8]),
                          head_dim=rng.choice([64, 128]), gain=gain, layout=layout, **trees)
    if kind == "general":
        return _attention(requests=_log(rng, 1, 4), head_dim=rng.choice([80, 96, 112, 128, 192]),
                          groups=rng.choice([3, 4, 7, 12]), page=rng.choice([16, 48]), gain=gain, layout=layout,
                          tree_lo=tree_lo, tree_hi=tree_hi, prefix_lo=min(low, 2048), prefix_hi=min(top, 2048),
                          kv_heads=rng.choice([2, 4, 8]), dtype=rng.choice(["bf16", "f16"]))
    if kind == "round":
        return {"kind": "round", "layers": rng.choice([12, 24, 36]), "requests": _log(rng, 1, 8), "kv_heads": 8,
                "groups": 4, "head_dim": 128, "page": 256, "prefix_lo": min(low, 2048), "prefix_hi": min(top, 2048),
                "tree_lo": tree_lo, "tree_hi": tree_hi, "gain": gain, "layout": layout}
    if kind == "accept":
        return {"kind": "accept", "dtype": rng.choice(["bf16", "bf16", "f32"]), "requests": _log(rng, 1, 32),
                "tree_lo": tree_lo, "tree_hi": tree_hi, "vocab": rng.choice([32000, 128256, 151936, 50257]),
                "max_depth": 15, "prefix_lo": low, "prefix_hi": top, "page": 256, "layout": layout}
    if kind == "commit":
        return {"kind": "commit", "dtype": rng.choice(["bf16", "f32"]), "layers": rng.choice([12, 24, 36]),
                "requests": _log(rng, 1, 32), "kv_heads": rng.choice([1, 2, 8]), "head_dim": rng.choice([64, 128]),
                "page": 256, "prefix_lo": min(low, 1024), "prefix_hi": min(top, 1024), "tree_lo": tree_lo,
                "tree_hi": tree_hi, "layout": layout}
    return {"kind": "append", "dtype": rng.choice(["bf16", "f32"]), "rows": _log(rng, 16, 8192),
            "kv_heads": rng.choice([1, 2, 8]), "head_dim": rng.choice([64, 128]), "page": 256, "skip": 0.02,
            "slots64": rng.random() < 0.5, "layout": layout}


# --------------------------------------------------------------------------- layouts (from the case alone)
def _random_tree(nodes, max_depth, rng):
    parents, depth = [-1], [0]
    for node in range(1, nodes):
        while True:
            parent = rng.randrange(node)
            if depth[parent] < max_depth:
                break
        parents.append(parent)
        depth.append(depth[parent] + 1)
    return parents, depth


def _layout(case):
    """Prefix lengths and (parents, depths) of every request."""
    rng = random.Random(case["layout"])
    prefixes, trees = [], []
    for _ in range(case.get("chunks", 0)):
        rows = case["chunk_rows"]
        prefixes.append(rng.randint(0, case["chunk_prefix_hi"]))
        trees.append((list(range(-1, rows - 1)), list(range(rows))))
    for _ in range(case["requests"]):
        prefixes.append(rng.randint(case["prefix_lo"], case["prefix_hi"]))
        trees.append(_random_tree(rng.randint(case["tree_lo"], case["tree_hi"]), 8, rng))
    return prefixes, trees


def _paths(case, trees):
    """One accepted root path per request, 1 to depth + 1 nodes."""
    rng = random.Random(case["layout"] + 1)
    paths = []
    for parents, depths in trees:
        length = rng.randint(1, max(depths) + 1)
        node = rng.choice([n for n in range(len(parents)) if depths[n] == length - 1])
        path = [node]
        while parents[path[-1]] >= 0:
            path.append(parents[path[-1]])
        paths.append(path[::-1])
    return paths


def _mask(parents):
    n = len(parents)
    mask = np.zeros((n, n), dtype=bool)
    for node, parent in enumerate(parents):
        if parent >= 0:
            mask[node] = mask[parent]
        mask[node, node] = True
    return mask


def _pages(case, prefixes, trees, seed, spare=0):
    """A shuffled pool: page tables of the prefixes (and `spare` further pages), tree scratch pages."""
    page = case["page"]
    order = np.random.default_rng([case["layout"], seed])
    need = [-(-(p + spare) // page) for p in prefixes]
    scratch = -(-sum(len(parents) for parents, _ in trees) // page)
    live = sum(need) + scratch
    total = max(live + 1, int(live / case.get("fill", 1.0)))
    shuffled = [int(x) for x in order.permutation(total)]
    tables, at = [], 0
    for n in need:
        tables.append(shuffled[at:at + n])
        at += n
    return tables, shuffled[at:at + scratch], total


def _normal(shape, dtype, generator, gain=1.0):
    x = torch.empty(shape, dtype=dtype, device=_DEVICE).normal_(generator=generator)
    return x if gain == 1.0 else x.mul_(gain)


def _generator(seed):
    return torch.Generator(device=_DEVICE).manual_seed(seed)


def _tree_slots(scratch, trees, page):
    total = sum(len(parents) for parents, _ in trees)
    node = np.arange(total)
    return np.asarray(scratch, dtype=np.int64)[node // page] * page + node % page


def _metadata(case, prefixes, trees, tables, scratch):
    from jetspec_amd import PackedTreeMetadata

    hosts = [SimpleNamespace(num_nodes=len(parents), host_ancestor=torch.from_numpy(_mask(parents)),
                             host_parents=parents, host_depths=depths) for parents, depths in trees]
    return PackedTreeMetadata.from_host_trees(prefixes, tables, hosts, scratch, case["page"], device=_DEVICE,
                                              request_ids=list(range(len(prefixes))))


# --------------------------------------------------------------------------- attention
def _attention_inputs(case, seed):
    prefixes, trees = _layout(case)
    tables, scratch, pages = _pages(case, prefixes, trees, seed)
    gen, dtype = _generator(seed), _DTYPES[case["dtype"]]
    shape = (pages, case["page"], case["kv_heads"], case["head_dim"])
    rows = sum(len(parents) for parents, _ in trees)
    k, v = _normal(shape, dtype, gen), _normal(shape, dtype, gen)
    q = _normal((rows, case["kv_heads"] * case["groups"], case["head_dim"]), dtype, gen, case["gain"])
    return prefixes, trees, tables, scratch, q, k, v


def _attention_prepare(case, seed):
    prefixes, trees, tables, scratch, q, k, v = _attention_inputs(case, seed)
    return {"case": case, "q": q, "k": k, "v": v, "metadata": _metadata(case, prefixes, trees, tables, scratch)}


def _attention_run(state):
    from jetspec_amd import packed_tree_attention

    case = state["case"]
    return packed_tree_attention(state["q"], state["k"], state["v"], state["metadata"], case["head_dim"] ** -0.5,
                                 case["groups"], backend=case["backend"],
                                 output_dtype=torch.float32 if case["out32"] else None)


def _attend(case, prefixes, trees, tables, slots, q, k, v):
    """Tree attention in 64 bits: [rows, heads, dim] over the pools k, v [pages, page, kv_heads, dim]."""
    hkv, groups, dim, page = case["kv_heads"], case["groups"], case["head_dim"], case["page"]
    out = torch.empty((q.shape[0], hkv * groups, dim), dtype=torch.float64, device=_DEVICE)
    flat_k, flat_v = k.reshape(-1, hkv, dim), v.reshape(-1, hkv, dim)
    start = 0
    for prefix, (parents, _), table in zip(prefixes, trees, tables):
        n = len(parents)
        pos = np.arange(prefix)
        index = np.concatenate([np.asarray(table, dtype=np.int64)[pos // page] * page + pos % page
                                if prefix else pos.astype(np.int64), slots[start:start + n]])
        index = torch.as_tensor(index, device=_DEVICE)
        hidden = torch.as_tensor(~_mask(parents), device=_DEVICE)
        rows = q[start:start + n].double().reshape(n, hkv, groups, dim)
        for h in range(hkv):
            keys = flat_k[index, h].double()
            values = flat_v[index, h].double()
            score = (rows[:, h].reshape(n * groups, dim) @ keys.T.contiguous()) * dim ** -0.5
            score.view(n, groups, -1)[:, :, prefix:].masked_fill_(hidden[:, None, :], float("-inf"))
            out[start:start + n, h * groups:(h + 1) * groups] = (torch.softmax(score, -1) @ values).view(n, groups, dim)
        start += n
    return out


def _attention_exact(case, seed):
    prefixes, trees, tables, scratch, q, k, v = _attention_inputs(case, seed)
    return _attend(case, prefixes, trees, tables, _tree_slots(scratch, trees, case["page"]), q, k, v)


def _attention_work(case, elem=None):
    prefixes, trees = _layout(case)
    elem = elem or _DTYPES[case["dtype"]].itemsize
    heads, dim = case["kv_heads"] * case["groups"], case["head_dim"]
    rows = sum(len(parents) for parents, _ in trees)
    keys = sum(p + len(parents) for p, (parents, _) in zip(prefixes, trees))
    pairs = sum(len(parents) * (p + 1) + sum(depths) for p, (parents, depths) in zip(prefixes, trees))
    out = 4 if case.get("out32") else elem
    return {"bytes": 2 * keys * case["kv_heads"] * dim * elem + rows * heads * dim * (elem + out),
            "flops": 4 * heads * dim * pairs}


# --------------------------------------------------------------------------- round
def _rope_cache(positions, dim):
    angles = torch.arange(positions, dtype=torch.float64)[:, None] * 1e6 ** (
        -torch.arange(0, dim, 2, dtype=torch.float64) / dim)
    return torch.cat((angles.cos(), angles.sin()), -1)


def _round_inputs(case, seed):
    prefixes, trees = _layout(case)
    tables, scratch, pages = _pages(case, prefixes, trees, seed)
    gen, layers = _generator(seed), case["layers"]
    rows = sum(len(parents) for parents, _ in trees)
    pool = _normal((2, layers, pages, case["page"], case["kv_heads"], case["head_dim"]), torch.bfloat16, gen)
    q = _normal((layers, rows, case["kv_heads"] * case["groups"], case["head_dim"]), torch.bfloat16, gen, case["gain"])
    k = _normal((layers, rows, case["kv_heads"], case["head_dim"]), torch.bfloat16, gen)
    v = _normal((layers, rows, case["kv_heads"], case["head_dim"]), torch.bfloat16, gen)
    positions = torch.tensor([p + d for p, (_, depths) in zip(prefixes, trees) for d in depths], dtype=torch.int64,
                             device=_DEVICE)
    cache = _rope_cache(4096, case["head_dim"]).to(_DEVICE).float()
    return prefixes, trees, tables, scratch, pool, q, k, v, positions, cache


def _round_prepare(case, seed):
    from jetspec_amd.target_graph import PackedVerifyGraph

    prefixes, trees, tables, scratch, pool, q, k, v, positions, cache = _round_inputs(case, seed)
    graph = PackedVerifyGraph(pool, cache, case["head_dim"] ** -0.5, 4096)
    return {"case": case, "graph": graph, "pool": pool, "q": q, "k": k, "v": v, "positions": positions,
            "metadata": _metadata(case, prefixes, trees, tables, scratch)}


def _round_run(state):
    out = state["graph"].verify(state["q"], state["k"], state["v"], state["positions"], state["metadata"])
    return {"attention": out, "pool": state["pool"]}


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    a, b = x[..., :half].double(), x[..., half:].double()
    return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)


def _round_exact(case, seed):
    prefixes, trees, tables, scratch, pool, q, k, v, positions, cache = _round_inputs(case, seed)
    slots = _tree_slots(scratch, trees, case["page"])
    at = torch.as_tensor(slots, device=_DEVICE)
    half = case["head_dim"] // 2
    cos, sin = cache[positions, None, :half].double(), cache[positions, None, half:].double()
    pool = pool.double()
    out = torch.empty(q.shape, dtype=torch.float64, device=_DEVICE)
    for layer in range(case["layers"]):
        k_pool, v_pool = pool[0, layer], pool[1, layer]
        k_pool.view(-1, *k_pool.shape[2:])[at] = _rotate(k[layer], cos, sin)
        v_pool.view(-1, *v_pool.shape[2:])[at] = v[layer].double()
        out[layer] = _attend(case, prefixes, trees, tables, slots, _rotate(q[layer], cos, sin), k_pool, v_pool)
    return {"attention": out, "pool": pool}


def _round_work(case):
    one = _attention_work(case, elem=2)
    rows = sum(len(parents) for parents, _ in _layout(case)[1])
    kv = 2 * 2 * rows * case["kv_heads"] * case["head_dim"]   # the tree K/V, written to its slots
    return {"bytes": case["layers"] * (one["bytes"] + kv), "flops": case["layers"] * one["flops"]}


# --------------------------------------------------------------------------- accept
def _accept_inputs(case, seed):
    prefixes, trees = _layout(case)
    paths = _paths(case, trees)
    tables, scratch, pages = _pages(case, prefixes, trees, seed, spare=case["max_depth"] + 1)
    rows, vocab = sum(len(parents) for parents, _ in trees), case["vocab"]
    logits = _normal((rows, vocab), _DTYPES[case["dtype"]], _generator(seed))
    greedy = logits.argmax(-1).cpu().numpy()
    rng = np.random.default_rng([case["layout"], seed, 1])
    tokens = rng.integers(0, vocab, size=rows)
    start = 0
    for (parents, _), path in zip(trees, paths):
        # The accepted path's nodes carry their parent's prediction, other children of the path do not.
        for node in range(1, len(parents)):
            want = greedy[start + parents[node]]
            if node in path:
                tokens[start + node] = want
            elif parents[node] in path and tokens[start + node] == want:
                tokens[start + node] = (want + 1) % vocab
        start += len(parents)
    width = max(len(t) for t in tables)
    padded = np.full((len(tables), width), -1, dtype=np.int32)
    for row, table in zip(padded, tables):
        row[:len(table)] = table
    offsets = np.cumsum([0] + [len(parents) for parents, _ in trees])
    # Budgets and the row that holds the EOS token go with the layout, as the committed row count does.
    fixed = np.random.default_rng([case["layout"], 2])
    budgets = [fixed.integers(1, 64) for _ in prefixes]
    eos = int(tokens[fixed.integers(rows)])
    return {"case": case, "logits": logits, "greedy": greedy, "tokens": tokens, "trees": trees, "paths": paths,
            "prefixes": prefixes, "tables": padded, "pages": pages, "offsets": offsets, "budgets": budgets, "eos": eos,
            "slots": _tree_slots(scratch, trees, case["page"])}


def _accept_prepare(case, seed):
    host = _accept_inputs(case, seed)

    def dev(x, dtype):
        return torch.as_tensor(np.asarray(x), dtype=dtype, device=_DEVICE)

    requests = len(host["prefixes"])
    return {"case": case, "logits": host["logits"], "tokens": dev(host["tokens"], torch.int64),
            "parents": dev([p for parents, _ in host["trees"] for p in parents], torch.int64),
            "depths": dev([d for _, depths in host["trees"] for d in depths], torch.int64),
            "cu": dev(host["offsets"], torch.int32), "budgets": dev(host["budgets"], torch.int32),
            "ignore_eos": torch.zeros(requests, dtype=torch.uint8, device=_DEVICE), "eos": [host["eos"]],
            "slots": dev(host["slots"], torch.int64), "tables": dev(host["tables"], torch.int32),
            "lens": dev(host["prefixes"], torch.int32), "pages": host["pages"]}


def _accept_run(state):
    from jetspec_amd import accept_batch_device, commit_slots, truncate_accepted

    case = state["case"]
    greedy, paths, lengths, corrections = accept_batch_device(
        state["logits"], state["tokens"], state["parents"], state["depths"], state["cu"], case["max_depth"])
    limits, emitted, commit_paths, commit_offsets = truncate_accepted(
        paths, lengths, corrections, state["tokens"], state["cu"], state["budgets"], state["ignore_eos"], state["eos"])
    source, destination = commit_slots(state["slots"], state["cu"], commit_paths, commit_offsets, state["tables"],
                                       state["lens"], case["page"], state["pages"])
    rows = int(commit_offsets[-1])   # the round's one host read: the commit's row count
    return {"greedy": greedy, "paths": paths, "lengths": lengths, "corrections": corrections, "limits": limits,
            "emitted": emitted, "offsets": commit_offsets, "source": source[:rows], "destination": destination[:rows]}


def _accept_exact(case, seed):
    host = _accept_inputs(case, seed)
    width, page = case["max_depth"] + 1, case["page"]
    requests = len(host["prefixes"])
    paths = np.full((requests, width), -1)
    emitted = np.full((requests, width), -1)
    lengths, corrections, limits, offsets, source, destination = [], [], [], [0], [], []
    for r, path in enumerate(host["paths"]):
        base, prefix = host["offsets"][r], host["prefixes"][r]
        paths[r, :len(path)] = path
        lengths.append(len(path) - 1)
        corrections.append(int(host["greedy"][base + path[-1]]))
        values = [int(host["tokens"][base + n]) for n in path[1:]] + [corrections[-1]]
        limit = min(len(values), int(host["budgets"][r]))
        if host["eos"] in values[:limit]:
            limit = values.index(host["eos"]) + 1
        limits.append(limit)
        emitted[r, :limit] = values[:limit]
        offsets.append(offsets[-1] + limit)
        for i, node in enumerate(path[:limit]):
            source.append(int(host["slots"][base + node]))
            pos = prefix + i
            destination.append(int(host["tables"][r, pos // page]) * page + pos % page)
    return {"greedy": torch.as_tensor(host["greedy"]), "paths": paths, "lengths": np.array(lengths),
            "corrections": np.array(corrections), "limits": np.array(limits), "emitted": emitted,
            "offsets": np.array(offsets), "source": np.array(source), "destination": np.array(destination)}


def _accept_work(case):
    rows = sum(len(parents) for parents, _ in _layout(case)[1])
    return {"bytes": rows * case["vocab"] * _DTYPES[case["dtype"]].itemsize, "flops": 0}


# --------------------------------------------------------------------------- commit
def _commit_inputs(case, seed):
    prefixes, trees = _layout(case)
    paths = _paths(case, trees)
    tables, scratch, pages = _pages(case, prefixes, trees, seed, spare=16)
    slots, page = _tree_slots(scratch, trees, case["page"]), case["page"]
    source, destination, start = [], [], 0
    for prefix, (parents, _), path, table in zip(prefixes, trees, paths, tables):
        source += [int(slots[start + n]) for n in path]
        destination += [table[pos // page] * page + pos % page for pos in range(prefix, prefix + len(path))]
        start += len(parents)
    pool = _normal((2, case["layers"], pages, page, case["kv_heads"], case["head_dim"]), _DTYPES[case["dtype"]],
                   _generator(seed))
    return pool, torch.tensor(source, device=_DEVICE), torch.tensor(destination, device=_DEVICE)


def _commit_prepare(case, seed):
    pool, source, destination = _commit_inputs(case, seed)
    return {"case": case, "pool": pool, "source": source, "destination": destination}


def _commit_run(state):
    from jetspec_amd import copy_accepted_kv

    payload = copy_accepted_kv(state["pool"], state["source"], state["destination"], state["case"]["page"])
    return {"payload": payload, "pool": state["pool"]}


def _commit_exact(case, seed):
    pool, source, destination = _commit_inputs(case, seed)
    rows = pool.view(2, case["layers"], -1, case["kv_heads"], case["head_dim"])
    rows[:, :, destination] = rows[:, :, source]
    return {"payload": 2 * case["layers"] * source.numel() * case["kv_heads"] * case["head_dim"] * pool.element_size(),
            "pool": pool}


def _commit_work(case):
    moved = sum(len(path) for path in _paths(case, _layout(case)[1]))
    row = case["kv_heads"] * case["head_dim"] * _DTYPES[case["dtype"]].itemsize
    return {"bytes": 2 * 2 * case["layers"] * moved * row, "flops": 0}


# --------------------------------------------------------------------------- append
def _append_inputs(case, seed):
    rng = np.random.default_rng([case["layout"], seed])
    gen, rows, page = _generator(seed), case["rows"], case["page"]
    pages = -(-rows // page) + 2
    shape = (pages, page, case["kv_heads"], case["head_dim"])
    dtype = _DTYPES[case["dtype"]]
    key, value = (_normal((rows, *shape[2:]), dtype, gen) for _ in range(2))
    k_cache, v_cache = _normal(shape, dtype, gen), _normal(shape, dtype, gen)
    node = np.arange(rows)
    slots = rng.permutation(pages)[node // page] * page + node % page
    skipped = np.random.default_rng(case["layout"]).random(rows) < case["skip"]
    slots[skipped] = -1
    return key, value, k_cache, v_cache, slots


def _append_prepare(case, seed):
    key, value, k_cache, v_cache, slots = _append_inputs(case, seed)
    mapping = torch.as_tensor(slots, dtype=torch.int64 if case["slots64"] else torch.int32, device=_DEVICE)
    return {"key": key, "value": value, "k_cache": k_cache, "v_cache": v_cache, "mapping": mapping}


def _append_run(state):
    from jetspec_amd import store_kvcache

    store_kvcache(state["key"], state["value"], state["k_cache"], state["v_cache"], state["mapping"])
    return {"k_cache": state["k_cache"], "v_cache": state["v_cache"]}


def _append_exact(case, seed):
    key, value, k_cache, v_cache, slots = _append_inputs(case, seed)
    kept = torch.as_tensor(np.flatnonzero(slots >= 0), device=_DEVICE)
    at = torch.as_tensor(slots[slots >= 0], device=_DEVICE)
    for rows, cache in ((key, k_cache), (value, v_cache)):
        cache.view(-1, *cache.shape[2:])[at] = rows[kept]
    return {"k_cache": k_cache, "v_cache": v_cache}


def _append_work(case):
    kept = int((np.random.default_rng(case["layout"]).random(case["rows"]) >= case["skip"]).sum())
    return {"bytes": 2 * 2 * kept * case["kv_heads"] * case["head_dim"] * _DTYPES[case["dtype"]].itemsize, "flops": 0}


# --------------------------------------------------------------------------- entry points
_PREPARE = {"attention": _attention_prepare, "round": _round_prepare, "accept": _accept_prepare,
            "commit": _commit_prepare, "append": _append_prepare}
_RUN = {"attention": _attention_run, "round": _round_run, "accept": _accept_run, "commit": _commit_run,
        "append": _append_run}
_EXACT = {"attention": _attention_exact, "round": _round_exact, "accept": _accept_exact, "commit": _commit_exact,
          "append": _append_exact}
_WORK = {"attention": _attention_work, "round": _round_work, "accept": _accept_work, "commit": _commit_work,
         "append": _append_work}


def prepare(case, seed):
    return {"kind": case["kind"], "state": _PREPARE[case["kind"]](case, seed)}


def run(state):
    return _RUN[state["kind"]](state["state"])


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def work(case):
    return _WORK[case["kind"]](case)


def tolerance(case):
    if case["kind"] in ("accept", "commit", "append"):
        return "exact"   # tokens, indices and moved bytes
    # About four times the difference from the 64-bit result over the declared ranges.
    if case["kind"] == "round":
        # bf16 products of the rotation, bf16 probabilities and output (5.4e-3 seen).
        return {"rel": 2e-2, "max": 0.4}
    if case["dtype"] == "f32":
        # fp32 sums of head_dim products and of every key (1.4e-6).
        return {"rel": 5e-6, "max": 8e-5}
    if case["out32"] and case["backend"] != "auto":
        # 16-bit operands and fp32 sums, probabilities to 2^-17 (bf16: 2.2e-6) or 2^-23 (f16: 8.4e-7).
        return {"rel": 8e-6, "max": 1e-4} if case["dtype"] == "bf16" else {"rel": 3.4e-6, "max": 4e-5}
    # The output, and the grouped path's probabilities, rounded once to 8 bits (2.4e-3) or 11 (3e-4).
    return {"rel": 1e-2, "max": 0.13} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 1.6e-2}
