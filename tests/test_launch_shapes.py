"""The rules by which the launches divide their work (csrc/qq_rules.h, compiled here by the host's
C++ compiler): every unit or row is taken exactly once, within the limits that the workspaces and
the LDS assume.  No GPU."""

from __future__ import annotations

import ctypes
import heapq
import math
import os
import random
import shutil
import subprocess

import pytest

CUS, ROUND = 256, 64
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwenquest_amd", "csrc")

SHIM = """
#include "qq_rules.h"
using namespace qq::rules;
typedef int64_t L;
extern "C" {
L unit_shape_(L cus, L bs, L kv, L top_k) { auto u = unit_shape(cus, bs, kv, top_k); return u.W * 100 + u.parts; }
L unit_first_(L wave, L part, L parts) { return unit_first(wave, part, parts); }
L dense_units_(L rows) { return dense_units(rows); }
L dense_parts_(L units, L len) { return dense_parts(units, len); }
L dense_part_begin_(L units, L part, L parts) { return dense_part_begin(units, part, parts); }
L dense_fit_(L cus, L bs, L max_rows) { return dense_fit(cus, bs, max_rows); }
L dense_candidate_(L total, L longest, L bs, L fit, L round, L lane) {
  return dense_candidate(dense_range(total, longest, bs, fit, round), lane);
}
L dense_cost_(L total, L count, L len, L fit, L round) {  // ordered as the float is
  const float c = dense_cost(total, count, len, fit, round);
  int32_t bits;
  __builtin_memcpy(&bits, &c, 4);
  return bits;
}
L dense_all_whole_(L total, L longest, L bs, L round) { return dense_all_whole(total, longest, bs, round); }
L dense_one_round_(L bs, L round) { return dense_one_round(bs, round); }
L dense_first_(L units, L parts, L len) { return dense_first(units, parts, len); }
L extend_tiles_(L n, L bs, L G) { return extend_tiles(n, bs, G); }
L extend_request_tiles_(L n, L G) { return extend_request_tiles(n, G); }
L extend_splits_(L tiles, L kv, L max_rows) { return extend_splits(tiles, kv, max_rows); }
L split_chunk_(L nt, L splits) { return split_chunk(nt, splits); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    out = str(d / "librules.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-fPIC", "-shared", "-Wall", "-Werror", f"-I{CSRC}", "-o", out,
                    str(d / "shim.cpp")], check=True)
    lib = ctypes.CDLL(out)

    class Rules:
        def __getattr__(self, name):
            fn = getattr(lib, name + "_")
            fn.restype = ctypes.c_int64

            def call(*args):
                return fn(*(ctypes.c_int64(a) for a in args))

            return call

    return Rules()


def ceil_div(a, b):
    return -(-a // b)


@pytest.mark.parametrize("kv", [1, 2, 4, 8])
@pytest.mark.parametrize("top_k", [64, 192, 256, 1024, 2048, 4096])
def test_every_unit_belongs_to_one_wave(rules, kv, top_k):
    units = top_k // 64
    for bs in list(range(1, 70)) + [96, 128, 255, 512, 1000]:
        W, parts = divmod(rules.unit_shape(CUS, bs, kv, top_k), 100)
        assert W in (4, 8) and 1 <= parts <= min(8, units)  # the partials fit one chunk per 64 slots
        taken = []
        for part in range(parts):
            for wave in range(W):
                taken += range(rules.unit_first(wave, part, parts), units, parts * W)
        assert sorted(taken) == list(range(units))
        if bs * kv > CUS:  # a part fewer gives a wave more units
            assert parts == 1 or ceil_div(units, W * (parts - 1)) > ceil_div(units, W * parts)
        if bs * kv <= CUS:  # one round of resident blocks
            assert bs * kv * parts <= (2 * CUS if W == 4 else CUS)


def dense_plan(rules, rows, width):
    """dense_store_plan_kernel: (request, KV head, first unit, end unit, part, parts) per block."""
    units = [rules.dense_units(n) for n in rows]
    bs, fit = len(rows), rules.dense_fit(CUS, len(rows), width)
    total, best = min(sum(units), 1 << 24), None
    one_round = rules.dense_one_round(bs, ROUND)
    if fit <= bs or (not one_round and rules.dense_all_whole(total, max(units), bs, ROUND)):
        return [(e // 4, e % 4, 0, units[e // 4], 0, 1) for e in range(4 * bs)]
    for lane in range(64):
        n = rules.dense_candidate(total, max(units), bs, fit, ROUND, lane)
        count = sum(rules.dense_parts(u, n) for u in units)
        # plan_one_round takes the shortest that fits
        cost = int(count > fit) if one_round else rules.dense_cost(total, count, n, fit, ROUND)
        if best is None or cost < best[0]:
            best = cost, n, count
    cost, n, count = best
    if count > fit:  # a total past 2^24: no pair is split
        n, count = 1 << 30, bs
    out = []
    for first in (True, False) if count > ROUND else (None,):
        for b, u in enumerate(units):
            p = rules.dense_parts(u, n)
            if first is None or bool(rules.dense_first(u, p, n)) == first:
                out += [(b, h, rules.dense_part_begin(u, i, p), rules.dense_part_begin(u, i + 1, p), i, p)
                        for h in range(4) for i in range(p)]
    return out


def longest_run(plan):
    """Units on the busiest CU, blocks going to the first free one in their order."""
    cus = [0] * CUS
    heapq.heapify(cus)
    for _, _, u0, u1, _, _ in plan:
        heapq.heapreplace(cus, cus[0] + u1 - u0)
    return max(cus)


def test_dense_division_covers_every_unit_once(rules):
    rng = random.Random(3)
    for _ in range(150):
        bs = rng.choice([1, 2, 3, 16, 24, 25, 60, 64, 65, 100, 300])
        width = rng.choice([1, 63, 200, 513, 5000, 131072, 1 << 28, 1 << 30])
        rows = [rng.choice([0, 1, width, rng.randint(0, width)]) for _ in range(bs)]
        blocks = 4 * rules.dense_fit(CUS, bs, width)
        plan = dense_plan(rules, rows, width)
        assert len(plan) <= blocks and blocks <= 4 * bs + 512
        seen = {}
        for e, (b, h, u0, u1, part, parts) in enumerate(plan):
            assert u0 < u1 and part < parts <= 64  # the merge's LDS table
            seen.setdefault((b, h), []).append((e, u0, u1, part, parts))
        for b, n in enumerate(rows):
            for h in range(4):
                got = seen[b, h]
                assert [g[3] for g in got] == list(range(got[0][4]))  # consecutive blocks, in order
                assert [g[0] for g in got] == list(range(got[0][0], got[0][0] + len(got)))
                assert [g[1] for g in got] == [0] + [g[2] for g in got[:-1]]
                assert got[-1][2] == max(ceil_div(n, 64), 1)


def test_dense_blocks_grow_with_the_batch(rules):
    """A workspace for the request pool's size does for every smaller batch."""
    for width in (1, 64, 513, 700, 5000, 131072):
        fits = [rules.dense_fit(CUS, bs, width) for bs in range(1, 400)]
        assert fits == sorted(fits) and all(f >= bs for bs, f in enumerate(fits, 1))


@pytest.mark.parametrize("rows", [
    [100_000] + [2000] * 63,
    [131_072] + [500] * 62,
    [30_000] * 8 + [500] * 48,
    [100_000] * 2 + [300] * 126,
    [131_072] + [1] * 30,
    [10_000] * 70,
    [65_000, 2000] * 20,
    [131_072] + [8000] * 1500,  # more requests than the plan keeps in LDS
    [100] * 90 + [60_000] * 3 + [4000] * 30,
])
def test_dense_division_leaves_no_cu_with_a_long_run(rules, rows):
    """A CU's run stays near what the chip takes at its full rate: 8/5 of the mean is free (a CU
    alone reads that much faster), and half a mean's part may come last."""
    plan = dense_plan(rules, rows, 131_072)
    units = sum(u1 - u0 for _, _, u0, u1, _, _ in plan)
    assert longest_run(plan) <= 1.75 * units / CUS + 16


def test_dense_division_leaves_no_cu_with_a_long_run_in_random_batches(rules):
    rng = random.Random(9)
    for _ in range(200):
        bs = round(math.exp(rng.uniform(0, math.log(300))))
        lens = [round(math.exp(rng.uniform(math.log(50), math.log(131_072)))) for _ in range(rng.choice([1, 2, 3, bs]))]
        rows = [rng.choice(lens) for _ in range(bs)]
        plan = dense_plan(rules, rows, 131_072)
        units = sum(u1 - u0 for _, _, u0, u1, _, _ in plan)
        assert longest_run(plan) <= 1.75 * units / CUS + 16, rows


def test_prefill_tiles_and_splits(rules):
    """extend_tiles bounds the requests' 128-row tiles, and split_chunk covers a tile's K/V once."""
    rng = random.Random(4)
    for _ in range(500):
        G = rng.choice([1, 4, 5, 7, 8, 48])
        new = [rng.choice([0, 1, rng.randint(0, 700)]) for _ in range(rng.randint(1, 90))]
        tiles = rules.extend_tiles(sum(new), len(new), G)
        assert sum(rules.extend_request_tiles(n, G) for n in new) <= tiles
        assert all(rules.extend_request_tiles(n, G) == ceil_div(n * G, 128) for n in new)
        kv, width = rng.choice([1, 2, 4, 8]), rng.choice([1, 70, 1000, 131072])
        splits = rules.extend_splits(tiles, kv, width)
        assert 1 <= splits <= 32 and (splits == 1 or tiles * kv * splits <= CUS)
        nt, splits = rng.randint(0, 300), rng.randint(1, 32)
        chunk = rules.split_chunk(nt, splits)
        got = [j for s in range(splits) for j in range(s * chunk, min(nt, s * chunk + chunk))]
        assert got == list(range(nt)) and ceil_div(nt, chunk) <= min(splits, 32)
        assert nt <= chunk or ceil_div(nt, chunk) <= ceil_div(nt, 4)
