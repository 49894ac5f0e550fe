"""Dense decode's division of a batch into parts (reference
``src/qwenquest/attention/dense.py:26-42``): (request, KV head) pairs whole and in up to 64 equal
parts, one part per block and blocks that take several, merges over one and several thread groups,
against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
KV, D = 4, 128


class Layer:
    layer_id, scaling = 0, D**-0.5


@pytest.mark.parametrize("heads,ctx,width", [
    (32, [8000], 8064),  # one request: 63 parts per KV head
    (16, [4097, 63], 4200),  # groups of 4: two thread groups merge
    (20, [2500, 1, 64, 65], 2600),  # groups of 5: threads past the merge's items
    (28, [700] * 3 + [3001], 3100),
    (4, [5000, 256], 5100),  # no grouping: eight thread groups merge
    (64, [3000, 17], 3100),  # groups of 16: two items per thread
    (8, [130, 0, 64], 200),  # a request without rows: zeros
    (32, [1 + 37 * i for i in range(70)], 2700),  # more requests than a round has parts
    (32, [20000, 300, 9000], 131072),  # several units per wave; a table far wider than the contexts
    (32, [9000] + [300] * 66, 9100),  # one long request among many: its parts go to blocks that are done
    (20, [4000, 100] * 15, 4100),  # fewer requests than a round has parts, two rounds
    (28, [1500] * 24 + [1600], 1700),  # 24 and 25 requests: the last batch of one round and the next
    (28, [1500] * 24, 1700),
    (8, [700, 0] * 40, 800),  # requests without rows among split ones
    (4, [9000, 1, 5000, 0] + [5] * 1100, 9100),  # more requests than the plan keeps in LDS
])
def test_dense_decode_matches_float64(heads, ctx, width):
    from qwenquest_amd.attention.dense import DenseBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    bs, G = len(ctx), heads // KV
    rtp = ReqToTokenPool(bs, width, DEV)
    kvp = MHATokenToKVPool(sum(ctx) + 1, 1, KV, D, torch.bfloat16, DEV)
    gen = torch.Generator(device=DEV).manual_seed(2)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    perm = (torch.randperm(sum(ctx), generator=torch.Generator().manual_seed(3)) + 1).to(torch.int32).to(DEV)
    at = 0
    for i, n in enumerate(ctx):
        rtp.req_to_token[i, :n] = perm[at : at + n]
        at += n
    be = DenseBackend(rtp, kvp)
    rpi, seq = torch.arange(bs, device=DEV), torch.tensor(ctx, device=DEV)
    loc = rtp.req_to_token[rpi, (seq - 1).clamp(min=0)].long()
    loc = torch.where(seq > 0, loc, sum(ctx) + 1)
    mk = lambda h: torch.empty((bs, h, D), device=DEV).normal_(generator=gen).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(heads), mk(KV), mk(KV)
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, loc, rtp, kvp, be)
    out = be.forward_decode(q, k, v, Layer(), batch)
    assert torch.equal(be.forward_decode(q, k, v, Layer(), batch), out)
    assert not be._sync.any()
    for i, n in enumerate(ctx):
        if n == 0:
            assert not out[i].any()
            continue
        rows = rtp.req_to_token[i, :n].long()
        kk, vv = kvp.k_all[0][rows].double(), kvp.v_all[0][rows].double()
        got = out[i].view(heads, D).double()
        for h in range(heads):
            p = torch.softmax((kk[:, h // G] @ q[i, h].double()) * D**-0.5, 0)
            ref = p @ vv[:, h // G]
            # half a bf16 ulp of the output, and of every weight (2^-9 each, at random signs
            # over the weights: their root sum of squares bounds it well)
            bound = 2.0**-8 * ref.abs() + 2.0**-8 * 3 * float((p * p).sum().sqrt()) + 1e-5
            assert bool(((got[h] - ref).abs() <= bound).all()), (i, h)


def test_columns_of_a_wider_table():
    """req_to_token as a slice of a wider table, at widths that give another number of blocks."""
    from qwenquest_amd.attention.dense import DenseBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    ctx, width = [300, 77], 320
    rtp = ReqToTokenPool(2, width, DEV)
    kvp = MHATokenToKVPool(2 * width, 1, KV, D, torch.bfloat16, DEV)
    gen = torch.Generator(device=DEV).manual_seed(8)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    rtp.req_to_token.copy_(torch.arange(1, 2 * width + 1, dtype=torch.int32).view(2, width))
    rpi, seq = torch.arange(2, device=DEV), torch.tensor(ctx, device=DEV)
    loc = rtp.req_to_token[rpi, seq - 1].long()
    mk = lambda h: torch.empty((2, h, D), device=DEV).normal_(generator=gen).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(32), mk(KV), mk(KV)
    out = []
    for wide in (0, 2000):
        if wide:
            table = torch.zeros((2, wide), dtype=torch.int32, device=DEV)
            table[:, 5 : 5 + width] = rtp.req_to_token
            rtp.req_to_token = table[:, 5 : 5 + width]
        be = DenseBackend(rtp, kvp)
        batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, loc, rtp, kvp, be)
        out.append(be.forward_decode(q, k, v, Layer(), batch))
    assert torch.equal(*out)


def batch_of(ctx, width, size, seed):
    from qwenquest_amd.attention.dense import DenseBackend
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    rtp = ReqToTokenPool(size, width, DEV)
    kvp = MHATokenToKVPool(sum(ctx), 1, KV, D, torch.bfloat16, DEV)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    at = 1
    for i, n in enumerate(ctx):
        rtp.req_to_token[i, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
    return rtp, kvp, DenseBackend(rtp, kvp), gen


def decode_call(rtp, kvp, be, gen, rpi, ctx):
    from qwenquest_amd.batch import ForwardBatch, ForwardMode

    rpi, seq = torch.tensor(rpi, device=DEV), torch.tensor(ctx, device=DEV)
    loc = rtp.req_to_token[rpi, seq - 1].long()
    q = torch.empty((len(ctx), 32, D), device=DEV).normal_(generator=gen).to(torch.bfloat16)
    k, v = kvp.k_all[0][loc].clone(), kvp.v_all[0][loc].clone()
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, loc, rtp, kvp, be)
    return lambda: be.forward_decode(q, k, v, Layer(), batch)


@pytest.mark.parametrize("first,rest", [([3000, 500], [4000] * 3), ([2500] + [300] * 30, [700] * 9)])
def test_a_captured_call_keeps_its_workspace(first, rest):
    """A graph captured with a small batch replays after a call with a larger one, and after other
    tensors took the memory that is free by then."""
    ctx = first + rest
    rtp, kvp, be, gen = batch_of(ctx, 4096, len(ctx), 5)
    small = decode_call(rtp, kvp, be, gen, list(range(len(first))), first)
    large = decode_call(rtp, kvp, be, gen, list(range(len(ctx))), ctx)
    want, all_want = small(), large()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = small()
    for i in range(3):
        assert torch.equal(large(), all_want)
        junk = [torch.full((1 << n,), -7, dtype=torch.int32, device=DEV) for n in range(4, 22)]
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        assert all(bool((x == -7).all()) for x in junk)
    assert not be._sync.any()


def test_calls_on_two_streams_share_nothing():
    """Batches of one backend on two streams at once: each call's division, counters and partial
    sums are its own."""
    a, b = [4000, 900, 64], [100] * 40 + [3000]
    rtp, kvp, be, gen = batch_of(a + b, 4096, len(a + b), 6)
    calls = [decode_call(rtp, kvp, be, gen, list(range(len(a))), a),
             decode_call(rtp, kvp, be, gen, list(range(len(a), len(a + b))), b)]
    want = [c() for c in calls]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[], []]
    for _ in range(20):
        for i in (0, 1):
            with torch.cuda.stream(streams[i]):
                got[i].append(calls[i]())
    torch.cuda.synchronize()
    for i in (0, 1):
        assert all(torch.equal(x, want[i]) for x in got[i])
