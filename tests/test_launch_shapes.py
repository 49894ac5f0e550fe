"""The rules by which the launches divide their work (csrc/qq_rules.h, compiled here by the host's
C++ compiler): every unit or row is taken exactly once, within the limits that the workspaces and
the LDS assume.  No GPU."""

from __future__ import annotations

import ctypes
import os
import random
import shutil
import subprocess

import pytest

CUS = 256
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
L dense_blocks_(L cus, L bs, L max_rows) { return dense_blocks(cus, bs, max_rows); }
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
        if bs * kv <= CUS:  # one round of resident blocks
            assert bs * kv * parts <= (2 * CUS if W == 4 else CUS)


def dense_plan(rules, rows, blocks):
    """dense_store_plan_kernel: (request, KV head, first unit, end unit, part, parts) per block."""
    units = [rules.dense_units(n) for n in rows]
    bs, fit = len(rows), blocks // 4
    if fit <= bs:
        return [(e // 4, e % 4, 0, units[e // 4], 0, 1) for e in range(4 * bs)]
    lo = max(ceil_div(sum(units), fit), 2)
    hi = max(lo, min(max(units), ceil_div(sum(units), fit - bs)))
    cands = [lo + ((hi - lo) * lane) // 63 for lane in range(64)]
    ok = [c for c in cands if sum(rules.dense_parts(u, c) for u in units) <= fit]
    assert ok, "the longest candidate fits"
    out = []
    for b, u in enumerate(units):
        p = rules.dense_parts(u, ok[0])
        out += [(b, h, rules.dense_part_begin(u, i, p), rules.dense_part_begin(u, i + 1, p), i, p)
                for h in range(4) for i in range(p)]
    return out


def test_dense_division_covers_every_unit_once(rules):
    rng = random.Random(3)
    for _ in range(150):
        bs = rng.choice([1, 2, 3, 16, 60, 64, 65, 100, 300])
        width = rng.choice([1, 63, 200, 5000, 131072])
        rows = [rng.choice([0, 1, width, rng.randint(0, width)]) for _ in range(bs)]
        blocks = rules.dense_blocks(CUS, bs, width)
        plan = dense_plan(rules, rows, blocks)
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
