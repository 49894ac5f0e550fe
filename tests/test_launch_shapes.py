"""CPU models of the host's and the device's divisions of work (decode.hip, extend.hip): every unit
or row is taken exactly once, within the limits that the workspaces and the LDS assume.  No GPU."""

from __future__ import annotations

import random

import pytest

CUS = 256


def ceil_div(a, b):
    return -(-a // b)


def unit_shape(bs, kv, top_k):
    """unit_shape: waves per block and blocks per (request, KV head)."""
    units, pairs = top_k // 64, bs * kv
    cap8, cap4 = max(1, min(8, ceil_div(units, 8))), max(1, min(8, ceil_div(units, 4)))
    if units <= 4 * cap4 and pairs * cap4 <= CUS:
        return 4, cap4
    if pairs <= CUS:
        p8, p4 = max(1, min(cap8, CUS // pairs)), max(1, min(cap4, 2 * CUS // pairs))
        return (4, p4) if ceil_div(units, 4 * p4) < ceil_div(units, 8 * p8) else (8, p8)
    return 4, min(cap4, 3 if 3 * pairs <= 4 * CUS else 2 if 5 * pairs <= 8 * CUS else 1)


@pytest.mark.parametrize("kv", [1, 2, 4, 8])
@pytest.mark.parametrize("top_k", [64, 192, 256, 1024, 2048, 4096])
def test_every_unit_belongs_to_one_wave(kv, top_k):
    units = top_k // 64
    for bs in list(range(1, 70)) + [96, 128, 255, 512, 1000]:
        W, parts = unit_shape(bs, kv, top_k)
        assert W in (4, 8) and 1 <= parts <= min(8, units)  # the partials fit one chunk per 64 slots
        taken = []
        for part in range(parts):
            for wave in range(W):
                taken += range(wave * parts + part, units, parts * W)
        assert sorted(taken) == list(range(units))
        if bs * kv <= CUS:  # one round of resident blocks
            assert bs * kv * parts <= (2 * CUS if W == 4 else CUS)


def dense_plan(rows, blocks):
    """dense_store_plan_kernel: (request, KV head, first unit, end unit, part, parts) per block."""
    units = [max(ceil_div(n, 64), 1) for n in rows]
    bs, fit = len(rows), blocks // 4
    parts_of = lambda u, n: 1 if u <= 8 else ceil_div(u, n)  # noqa: E731
    if fit <= bs:
        return [(e // 4, e % 4, 0, units[e // 4], 0, 1) for e in range(4 * bs)]
    lo = max(ceil_div(sum(units), fit), 2)
    hi = max(lo, min(max(units), ceil_div(sum(units), fit - bs)))
    cands = [lo + ((hi - lo) * lane) // 63 for lane in range(64)]
    ok = [c for c in cands if sum(parts_of(u, c) for u in units) <= fit]
    assert ok, "the longest candidate fits"
    out = []
    for b, u in enumerate(units):
        p = parts_of(u, ok[0])
        out += [(b, h, u * i // p, u * (i + 1) // p, i, p) for h in range(4) for i in range(p)]
    return out


def test_dense_division_covers_every_unit_once():
    rng = random.Random(3)
    for _ in range(400):
        bs = rng.choice([1, 2, 3, 16, 60, 64, 65, 100, 300])
        width = rng.choice([1, 63, 200, 5000, 131072])
        rows = [rng.choice([0, 1, width, rng.randint(0, width)]) for _ in range(bs)]
        pairs = 4 * bs
        blocks = max(pairs, min(CUS, pairs * ceil_div(width, 64)))
        plan = dense_plan(rows, blocks)
        assert len(plan) <= blocks
        seen = {}
        for e, (b, h, u0, u1, part, parts) in enumerate(plan):
            assert u0 < u1 and part < parts <= CUS // 4  # the merge's LDS table
            seen.setdefault((b, h), []).append((e, u0, u1, part, parts))
        for b, n in enumerate(rows):
            for h in range(4):
                got = seen[b, h]
                assert [g[3] for g in got] == list(range(got[0][4]))  # consecutive blocks, in order
                assert [g[0] for g in got] == list(range(got[0][0], got[0][0] + len(got)))
                assert [g[1] for g in got] == [0] + [g[2] for g in got[:-1]]
                assert got[-1][2] == max(ceil_div(n, 64), 1)


def test_prefill_tiles_and_splits():
    """extend_tiles bounds the requests' 128-row tiles, and split_chunk covers a tile's K/V once."""
    rng = random.Random(4)
    for _ in range(500):
        G = rng.choice([1, 4, 5, 7, 8, 48])
        new = [rng.choice([0, 1, rng.randint(0, 700)]) for _ in range(rng.randint(1, 90))]
        assert sum(ceil_div(n * G, 128) for n in new) <= sum(new) * G // 128 + len(new)
        nt, splits = rng.randint(0, 300), rng.randint(1, 32)
        parts = max(min(splits, ceil_div(nt, 4)), 1)
        chunk = max(ceil_div(nt, parts), 1)
        got = [j for s in range(splits) for j in range(s * chunk, min(nt, s * chunk + chunk))]
        assert got == list(range(nt)) and ceil_div(nt, chunk) <= min(splits, 32)
