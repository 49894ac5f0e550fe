"""The fused layer step at 1, 2 and 8 KV heads (a model's heads split over ranks, or a model with
more of them): the flows and comparisons of the 4-head shapes, on those shapes."""

from __future__ import annotations

import pytest
import torch

from qwenquest_amd import _lib
from tests import test_gpu_hisparse as th
from tests import test_gpu_quest as tq

pytestmark = pytest.mark.gpu


# (layers, q heads, kv heads, head_dim, page, top_k, ctx, prompts, steps): long, short,
# exactly-top_k and one-past requests; groups of 1, 5, 7, 8 and 16; the recent window alone
@pytest.mark.parametrize("flow", [
    (1, 8, 1, 128, 64, 2048, 9000, {0: 8800, 1: 2046, 2: 2047, 3: 1000}, 3),
    (2, 10, 2, 128, 64, 256, 3000, {0: 2900, 1: 255, 2: 700}, 4),
    (1, 16, 1, 128, 64, 64, 700, {0: 650, 1: 63}, 3),
    (1, 8, 8, 128, 64, 512, 3000, {0: 2900, 1: 511, 2: 512}, 3),
    (1, 56, 8, 128, 64, 4096, 9000, {0: 8900, 1: 4000, 2: 4095}, 3),
    (1, 32, 2, 128, 64, 2048, 6000, {0: 5900, 1: 2100, 2: 300}, 3),
])
def test_engine_flow_against_the_oracle(flow, monkeypatch):
    monkeypatch.setattr(tq, "ENGINE_FLOWS", [flow])
    tq.test_forward_decode_fused_path_engine_flow(0)


@pytest.mark.parametrize("kv,heads", [(1, 7), (2, 16), (8, 32)])
@pytest.mark.parametrize("avoid", [False, True])
def test_quest_hisparse_is_bit_identical_to_quest(kv, heads, avoid, monkeypatch):
    shape = (heads, kv, 128, 256, 64, 384, 1200, {0: 700, 1: 1003}, 12)
    monkeypatch.setattr(th, "BIT_IDENTITY", [shape, None])  # not the 4-head shape, the list's last
    assert _lib.load().qq_quest_layer_step_fused(0, 0, 0, heads, kv, 128, 64, 256, 19) == 1
    th.test_quest_hisparse_is_bit_identical_to_quest(avoid, 0)


@pytest.mark.parametrize("kv,heads,bs", [(1, 8, 3), (2, 10, 40), (8, 32, 33), (8, 8, 70), (1, 8, 300)])
def test_fused_and_four_launch_steps_agree(kv, heads, bs):
    """Every launch shape (4-wave blocks with a unit per wave, one 8-wave block per CU, two
    4-wave blocks): the positions of the four launches, and their outputs to the bf16 rounding of
    weights and outputs."""
    from qwenquest_amd.attention.quest_only import QuestOnlyBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    D, CTX, TOP_K = 128, 1500, 1024
    rtp = ReqToTokenPool(bs, CTX, tq.DEV)
    kvp = MHATokenToKVPool(bs * CTX, 1, kv, D, torch.bfloat16, tq.DEV)
    gen = torch.Generator(device=tq.DEV).manual_seed(5)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    rtp.req_to_token.copy_((torch.randperm(bs * CTX, generator=torch.Generator().manual_seed(6)) + 1).view(bs, CTX))
    be = QuestOnlyBackend(rtp, kvp, {"algorithm": "quest", "top_k": TOP_K, "quest_page_size": 64})
    seq = torch.tensor([1499 - 13 * (i % 60) for i in range(bs)], device=tq.DEV)
    for r in range(bs):
        be.quest.update_prefill_representations_fused(r, kvp.k_all, rtp.req_to_token[r, : int(seq[r]) - 1])
        be._skip_first_decode_update[r] = True
    rpi = torch.arange(bs, device=tq.DEV)
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, rtp.req_to_token[rpi, seq - 1].long(), rtp, kvp, be)
    be.init_forward_metadata(batch)
    mk = lambda h: torch.randn((bs, h, D), generator=gen, device=tq.DEV).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(heads), mk(kv), mk(kv)

    class Layer:
        layer_id, scaling = 0, D**-0.5

    out = be.forward_decode(q, k, v, Layer(), batch)
    pos, sync = be._positions[:bs].clone(), be._step_sync
    assert not sync.any()
    be._step_sync = None
    four = be.forward_decode(q, k, v, Layer(), batch)
    assert torch.equal(be._positions[:bs], pos)
    err, scale = (out.double() - four.double()).abs(), four.double().abs().amax()
    assert float(err.max()) <= 2.0**-7 * float(scale) + 1e-4


@pytest.mark.parametrize("kv,group", [(1, 8), (1, 1), (2, 5), (2, 16), (8, 8), (8, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_scores_bit_exact_at_other_pages_per_wave(kv, group, dtype):
    tq.test_retrieve_scores_bit_exact_in_canonical_order(kv, 128, group, dtype)
