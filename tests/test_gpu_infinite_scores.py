"""Scores of -inf in the 64-row attention unit (reference ``src/qwenquest/attention/ops.py:48-66``):
rows whose scores are -inf weigh nothing, also where they fill a wave's first unit, in the dense
decode (dense.py:26-42) and the Quest layer step (quest_only.py:132-159); against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
D = 128
LOWEST = torch.finfo(torch.bfloat16).min


class Layer:
    layer_id, scaling = 0, D**-0.5


@pytest.mark.parametrize("backend,KV", [("dense", 4), ("quest", 1), ("quest", 2), ("quest", 4), ("quest", 8)])
@pytest.mark.parametrize("kind", ["infinite", "overflowing"])
def test_rows_of_infinite_scores_weigh_nothing(backend, KV, kind):
    from qwenquest_amd.attention import DenseBackend, QuestOnlyBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    H, ctx = 4 * KV, [100, 64 * 9, 2000, 300]
    dead = [64, 64 * 8, 1950, 300]  # leading rows of -inf: a unit, one per wave, nearly all, all
    rtp = ReqToTokenPool(len(ctx), 2048, DEV)
    kvp = MHATokenToKVPool(sum(ctx), 1, KV, D, torch.bfloat16, DEV)
    gen = torch.Generator(device=DEV).manual_seed(4)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    base = 1
    for i, n in enumerate(ctx):
        rows = torch.arange(base, base + n, dtype=torch.int32, device=DEV)
        rtp.req_to_token[i, :n] = rows
        if kind == "infinite":
            kvp.k_all[0, base : base + dead[i], :, 0] = -float("inf")
        else:  # the two products of a row overflow in their sum
            kvp.k_all[0, base : base + dead[i], :, :2] = LOWEST
        base += n
    if backend == "dense":
        be = DenseBackend(rtp, kvp)
    else:
        be = QuestOnlyBackend(rtp, kvp, {"algorithm": "quest", "top_k": 2048, "quest_page_size": 64})
        be._skip_first_decode_update.fill_(True)
    bs = len(ctx)
    rpi, seq = torch.arange(bs, device=DEV), torch.tensor(ctx, device=DEV)
    loc = rtp.req_to_token[rpi, seq - 1].long()
    q = torch.empty((bs, H, D), device=DEV).normal_(generator=gen).to(torch.bfloat16)
    q[:, :, :2] = 4.0
    k, v = kvp.k_all[0][loc].clone(), kvp.v_all[0][loc].clone()
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, loc, rtp, kvp, be)
    be.init_forward_metadata(batch)
    out = be.forward_decode(q, k, v, Layer(), batch)
    for i, n in enumerate(ctx):
        if dead[i] == n:  # nothing weighs anything: zeros
            assert not out[i].any()
            continue
        rows = rtp.req_to_token[i, dead[i] : n].long()
        kk, vv = kvp.k_all[0][rows].double(), kvp.v_all[0][rows].double()
        got = out[i].view(H, D).double()
        for h in range(H):
            p = torch.softmax((kk[:, h // 4] @ q[i, h].double()) * D**-0.5, 0)
            ref = p @ vv[:, h // 4]
            # half a bf16 ulp of the output, and of every weight (at random signs)
            bound = 2.0**-8 * ref.abs() + 2.0**-8 * 3 * float((p * p).sum().sqrt()) + 1e-5
            assert bool(((got[h] - ref).abs() <= bound).all()), (i, h)
