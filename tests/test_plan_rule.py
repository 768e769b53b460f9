"""The planner's choice of the chunk target against an independent search over every target
(csrc/tv_plan_rule.h).  The device planner's items equal the host's in the GPU tests."""
from __future__ import annotations

import math
import random

import numpy as np
import pytest

from jetspec_amd.paged_backend import make_plan

CU, PAGE = 256, 256
MAX_CHUNK = 511 * PAGE // 32 * 32


def requests_of(prefixes, nodes, kv_heads, groups):
    """(prefix, nodes, cost weight, uncut items) of every request."""
    out = []
    for p, n in zip(prefixes, nodes):
        heads = 2 if n <= 4 * (32 // groups) and kv_heads >= 2 else 1
        out.append((p, n, 5 if heads == 2 else 4, -(-kv_heads // heads) * -(-n // ((8 // heads) * (32 // groups)))))
    return out


def limit(tau, weight):
    keys = np.maximum(64, tau // weight)
    return np.minimum(-(-keys // 32) * 32, MAX_CHUNK)


def counts(requests, taus):
    total = np.zeros(len(taus), dtype=np.int64)
    for p, _, weight, units in requests:
        total += units * (-(-p // limit(taus, weight)) if p else np.ones(len(taus), dtype=np.int64))
    return total


def span(requests, tau, score_rows):
    """The one-round estimate of a plan, from its items."""
    longest, partial, parts = 0, 0, 0
    for p, n, weight, _ in requests:
        chunks = int(-(-p // limit(np.int64(tau), weight))) if p else 1
        chunk = max(32, -(-(-(-p // chunks)) // 32) * 32)
        if chunks > 1:
            even, keep = -(-(-(-(p + 2 * n) // chunks)) // 32) * 32, (p - 1) // (chunks - 1) // 32 * 32
            chunk = max(chunk, min(even, keep, MAX_CHUNK))
            partial += chunks * n * score_rows
        ends = [min(p, chunk * i) for i in range(chunks)] + [p]
        costs = [weight * (b - a) for a, b in zip(ends, ends[1:])]
        costs[-1] += weight * n
        longest, parts = max(longest, *costs), max(parts, chunks)
    return 1500 + longest + 8 * partial // 256 + 60 * parts


def choice(requests, score_rows):
    """(items of the even share, rounds of the chosen plan or whether the balance was taken, its
    target), every target tried."""
    cost = sum(units * weight * (p + n) for p, n, weight, units in requests)
    target = max(64, cost // CU)
    now = int(counts(requests, np.array([target]))[0])
    if now > 4 * CU:
        return now, "even", target
    steps = 128 * np.arange(1, cost // 128 + 2)
    items = counts(requests, steps)
    if now <= CU:
        n = max(math.isqrt(cost // 5), sum(units for *_, units in requests))
        if n < now and (items <= n).any():
            tau = int(steps[np.argmax(items <= n)])
            if span(requests, tau, score_rows) * 104 < span(requests, target, score_rows) * 100:
                return now, "balance", tau
        return now, "even", target
    rounds = -(-now // CU)
    tau = target
    if now < rounds * CU:
        every = np.arange(1, target + 1)
        tau = int(every[np.argmax(counts(requests, every) <= rounds * CU)])
    best = (rounds * (tau + 1000) + 2 * rounds * CU, rounds, tau)
    for k in range(rounds - 1, 0, -1):
        if (items <= k * CU).any():
            t = int(steps[np.argmax(items <= k * CU)])
            estimate = k * (t + 1000) + 2 * k * CU
            if estimate < best[0]:
                best = (estimate, k, t)
    return now, best[1], best[2]


def check(prefixes, nodes, kv_heads, groups):
    requests = requests_of(prefixes, nodes, kv_heads, groups)
    now, rounds, tau = choice(requests, kv_heads * groups)
    plan = make_plan(prefixes, nodes, kv_heads, PAGE, CU, queries_per_kv=groups)
    assert plan["num_items"] == int(counts(requests, np.array([tau]))[0]) == len(plan["items"])
    if isinstance(rounds, int):
        assert plan["num_items"] <= rounds * CU
    per_request = np.bincount(plan["items"][:, 0], minlength=len(prefixes))
    for (p, _, weight, units), have in zip(requests, per_request):
        chunks = int(-(-p // limit(np.int64(tau), weight))) if p else 1
        assert have == units * chunks
    return now, rounds


def test_named_batches():
    rng = random.Random(1)
    # Two part-filled rounds at the even share, one round in the plan.
    now, rounds = check([rng.randint(1354, 4060) for _ in range(8)], [rng.randint(18, 54) for _ in range(8)], 8, 4)
    assert now > CU and rounds == 1
    # One round already: fewer items where their partial rows cost more than they spread, the even
    # share where the two are about level.
    now, rounds = check([1873, 2151], [7, 8], 8, 4)
    assert now == CU and rounds == "balance"
    now, rounds = check([500] * 3, [10] * 3, 8, 4)
    assert now <= CU and rounds == "even"
    # More uncut items than one round holds: two rounds are the fewest.
    now, rounds = check([rng.randint(2000, 9000) for _ in range(36)], [64] * 36, 8, 4)
    assert now > CU and rounds == 2
    # 136 uncut items: cut into one round they would be far longer than in two.
    now, rounds = check([16384] * 17, [64] * 17, 8, 4)
    assert CU < now and rounds == 2
    # Beyond four rounds the even share stands.
    now, rounds = check([300] * 200, [64] * 200, 8, 4)
    assert now > 4 * CU and rounds == "even"


def test_random_batches():
    rng, chosen = random.Random(7), {}
    for _ in range(250):
        n = rng.choice([1, 2, 5, 8, 20, 48, 64])
        top = rng.choice([200, 3000, 20000])
        _, rounds = check([rng.randint(0, top) for _ in range(n)], [rng.randint(1, rng.choice([8, 64, 300])) for _ in range(n)],
                          rng.choice([1, 2, 8]), rng.choice([1, 4, 5, 8, 16]))
        chosen[rounds] = chosen.get(rounds, 0) + 1
    assert all(chosen.get(k, 0) >= 3 for k in ("even", "balance", 1, 2, 3)), chosen


def test_counts_without_a_plan_are_the_plan_s():
    """The sizing call builds nothing; make_plan checks its counts against the second call's arrays."""
    plan = make_plan([5000, 70, 0], [64, 10, 33], 8, PAGE, CU, queries_per_kv=4)
    groups = plan["groups"]
    assert len(groups) == plan["num_groups"] and plan["num_partial_slots"] == int(groups[:, 5].sum())
    assert sorted(plan["items"][:, 6][plan["items"][:, 6] >= 0]) == list(range(plan["num_partial_slots"]))
