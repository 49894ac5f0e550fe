"""The work this framework is run for, as cases that can be timed and checked.

Five kinds of pass, each through the attention backends' (or the Quest algorithm's) public
entry points, on bf16 tensors as a serving engine holds them:

``quest``    one decode step of the quest backend: the step's bookkeeping, then every layer's
             new-token store, page scoring, selection and attention.  Decode steps are captured
             in a HIP graph and replayed, as bench.py and a serving loop do.
``dense``    one decode step of the dense backend (every row of every context).
``hisparse`` successive decode steps of one quest_hisparse layer: selection, swap-in of the
             missed rows from pinned host memory, attention over the hot buffer.
``extend``   one layer of prefill: the new K/V into the pool, then causal attention per request.
``bounds``   the page bounds of one prompt over every layer, as they are built after a prefill.

Contexts are never a multiple of the page size in the decode kinds: a pass is repeated on one
state, and the page that completes at such a length would be finalized by the repetition.
"""

from __future__ import annotations

import math
import random

import torch

PAGE = 64  # the reference's default quest page size
DEV = torch.device("cuda", 0)


def listed() -> list[dict]:
    return [
        # one interactive request at a short context: 48 layers of a 32/4-head model
        {"name": "quest_b1_8k", "kind": "quest", "bs": 1, "ctx_lo": 8192, "ctx_hi": 8192, "layers": 48,
         "heads": 32, "kv": 4, "top_k": 2048, "avoid": False},
        # the headline serving shape, long contexts (4 of its 48 layers: past the Infinity Cache)
        {"name": "quest_b16_128k", "kind": "quest", "bs": 16, "ctx_lo": 131072, "ctx_hi": 131072, "layers": 4,
         "heads": 32, "kv": 4, "top_k": 2048, "avoid": False},
        # a busy server: many requests of mixed lengths, the overlap option on
        {"name": "quest_b48_ragged", "kind": "quest", "bs": 48, "ctx_lo": 3000, "ctx_hi": 65536, "layers": 4,
         "heads": 32, "kv": 4, "top_k": 2048, "avoid": True},
        # a model with 8 KV heads
        {"name": "quest_kv8_b8_32k", "kind": "quest", "bs": 8, "ctx_lo": 32768, "ctx_hi": 32768, "layers": 8,
         "heads": 32, "kv": 8, "top_k": 2048, "avoid": False},
        # the 32/4-head model split over two ranks: 16 query heads, 2 KV heads each
        {"name": "quest_kv2_b16_64k", "kind": "quest", "bs": 16, "ctx_lo": 65536, "ctx_hi": 65536, "layers": 4,
         "heads": 16, "kv": 2, "top_k": 2048, "avoid": False},
        # dense decode of one short request: 24 layers
        {"name": "dense_b1_8k", "kind": "dense", "bs": 1, "ctx_lo": 8000, "ctx_hi": 8000, "layers": 24,
         "heads": 32, "kv": 4, "width": 32768},
        # dense decode of a mixed batch
        {"name": "dense_b16_ragged", "kind": "dense", "bs": 16, "ctx_lo": 2000, "ctx_hi": 65000, "layers": 2,
         "heads": 32, "kv": 4, "width": 131072},
        # the hierarchical cache: 8 decode steps of one layer, correlated queries
        {"name": "hisparse_b4_48k", "kind": "hisparse", "bs": 4, "ctx_lo": 49152, "ctx_hi": 49152, "steps": 8,
         "heads": 32, "kv": 4, "top_k": 2048, "avoid": False},
        # one short prompt
        {"name": "extend_1x600", "kind": "extend", "bs": 1, "new_lo": 600, "new_hi": 600, "prefix_lo": 0,
         "prefix_hi": 0, "heads": 32, "kv": 4},
        # several prompts at once, with cached prefixes
        {"name": "extend_6_ragged", "kind": "extend", "bs": 6, "new_lo": 200, "new_hi": 3000, "prefix_lo": 0,
         "prefix_hi": 4000, "heads": 32, "kv": 4},
        # one chunk of a long prompt
        {"name": "extend_8k_chunk", "kind": "extend", "bs": 1, "new_lo": 8192, "new_hi": 8192, "prefix_lo": 8192,
         "prefix_hi": 8192, "heads": 32, "kv": 4},
        # bounds of one 16K prompt over 48 layers
        {"name": "bounds_16k", "kind": "bounds", "tokens": 16384, "layers": 48, "kv": 4},
    ]


def _log(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["quest", "quest", "quest", "dense", "extend", "extend", "hisparse", "bounds"])
    kv = rng.choice([1, 2, 4, 4, 4, 8])
    heads = kv * rng.choice([4, 5, 7, 8])
    if kind == "quest":
        bs = _log(rng, 1, 64)
        hi = _log(rng, 4096, min(131072, 2_000_000 / bs))
        lo = rng.choice([hi, max(1500, hi // rng.randint(2, 16))])
        return {"kind": kind, "bs": bs, "ctx_lo": lo, "ctx_hi": hi, "layers": min(48, max(2, 2_000_000 // (bs * hi))),
                "heads": heads, "kv": kv, "top_k": rng.choice([1024, 2048, 2048, 4096]), "avoid": rng.random() < 0.5}
    if kind == "dense":
        bs = _log(rng, 1, 32)
        hi = _log(rng, 500, min(100_000, 1_000_000 / bs))
        lo = rng.choice([hi, max(100, hi // rng.randint(2, 16))])
        return {"kind": kind, "bs": bs, "ctx_lo": lo, "ctx_hi": hi, "layers": min(24, max(1, 1_500_000 // (bs * hi))),
                "heads": 4 * rng.choice([4, 5, 7, 8]), "kv": 4, "width": rng.choice([hi + 64, 131072])}
    if kind == "hisparse":
        ctx = _log(rng, 8192, 65536)
        return {"kind": kind, "bs": rng.randint(1, 6), "ctx_lo": ctx // rng.choice([1, 2]), "ctx_hi": ctx, "steps": 8,
                "heads": 4 * rng.choice([4, 8]), "kv": 4, "top_k": 2048, "avoid": rng.random() < 0.5}
    if kind == "bounds":
        return {"kind": kind, "tokens": _log(rng, 300, 32768), "layers": rng.choice([24, 36, 48]),
                "kv": rng.choice([2, 4, 8])}
    bs = rng.randint(1, 8)
    hi = _log(rng, 64, 8192 / bs)
    prefix = rng.choice([0, 0, _log(rng, 64, 8192)])
    return {"kind": "extend", "bs": bs, "new_lo": max(1, hi // rng.randint(1, 8)), "new_hi": hi,
            "prefix_lo": prefix // rng.randint(1, 4), "prefix_hi": prefix, "heads": heads, "kv": kv}


# ---------------------------------------------------------------- shapes of a case


def _head_dim(case: dict) -> int:
    return 128


def _spread(lo: int, hi: int, n: int, salt: int) -> list[int]:
    """n lengths in [lo, hi], fixed by the case alone: both ends, the rest log-uniform."""
    r = random.Random(f"{lo} {hi} {n} {salt}")
    if lo == hi or n == 1:
        return [hi] * n
    rest = [int(round(math.exp(r.uniform(math.log(max(lo, 1)), math.log(max(hi, 1)))))) for _ in range(n - 2)]
    out = [hi, lo, *rest]
    r.shuffle(out)
    return out


def _contexts(case: dict) -> list[int]:
    """Context lengths, the token being decoded included; none a multiple of the page size."""
    ctx = _spread(case["ctx_lo"], case["ctx_hi"], case["bs"], 1)
    return [s + 1 if s % PAGE == 0 else s for s in ctx]


def _extend_lens(case: dict) -> tuple[list[int], list[int]]:
    return (_spread(case["new_lo"], case["new_hi"], case["bs"], 2),
            _spread(case["prefix_lo"], case["prefix_hi"], case["bs"], 3))


def work(case: dict) -> dict:
    kind, kv, D = case["kind"], case["kv"], _head_dim(case)
    row = kv * D * 2  # bytes of one K or V row
    if kind == "bounds":
        n, layers = case["tokens"], case["layers"]
        return {"bytes": layers * (n * row + (n // PAGE) * 2 * row) + 4 * n, "flops": 2 * layers * n * kv * D}
    H = case["heads"]
    if kind == "extend":
        new, prefix = _extend_lens(case)
        pairs = sum(n * p + n * (n + 1) // 2 for n, p in zip(new, prefix))
        q = sum(new) * H * D * 2
        return {"bytes": 2 * q + 4 * row * sum(new) + 2 * row * sum(prefix), "flops": 4 * pairs * H * D}
    ctx = _contexts(case)
    token = 2 * H * D * 2 + 4 * row  # q, out, the new K/V read and written
    if kind == "dense":
        n = case["layers"]
        return {"bytes": n * sum(2 * row * s + token for s in ctx), "flops": n * sum(4 * s * H * D for s in ctx)}
    n = case["layers"] if kind == "quest" else case["steps"]
    top_k = case["top_k"]
    nbytes = flops = 0
    for s in ctx:
        rows = min(s, top_k)
        pages = s // PAGE if s > top_k else 0
        nbytes += pages * 2 * row + rows * 2 * row + token
        flops += 2 * pages * kv * D + 4 * rows * H * D
    return {"bytes": n * nbytes, "flops": n * flops}


def tolerance(case: dict):
    # bf16 outputs, about four times the error against 64 bits: decode rounds the softmax
    # weights to bf16 as well as the output (0.0021 to 0.0023), prefill only the output (0.0017)
    if case["kind"] == "bounds":
        return "exact"
    return {"rel": 7e-3} if case["kind"] == "extend" else {"rel": 9e-3}


# ---------------------------------------------------------------- inputs


class _Layer:
    def __init__(self, layer_id: int, head_dim: int):
        self.layer_id = layer_id
        self.scaling = head_dim**-0.5


def _randn(shape: tuple, gen: torch.Generator) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(generator=gen)


def _tables(rows_of: list[int], width: int, layers: int, kv: int, dim: int, gen: torch.Generator):
    """Pools holding each request's rows as one run, and the request table (row 0 is padding)."""
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    rtp = ReqToTokenPool(len(rows_of), width, DEV)
    kvp = MHATokenToKVPool(sum(rows_of), layers, kv, dim, torch.bfloat16, DEV)
    for layer in range(layers):
        kvp.k_all[layer].normal_(generator=gen)
        kvp.v_all[layer].normal_(generator=gen)
    base = 1
    for i, n in enumerate(rows_of):
        rtp.req_to_token[i, :n] = torch.arange(base, base + n, dtype=torch.int32, device=DEV)
        base += n
    return rtp, kvp


def prepare(case: dict, seed: int):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return {"quest": _prepare_decode, "dense": _prepare_decode, "hisparse": _prepare_hisparse,
            "extend": _prepare_extend, "bounds": _prepare_bounds}[case["kind"]](case, gen)


def _decode_inputs(case: dict, n: int, gen: torch.Generator):
    bs, H, KV, D = case["bs"], case["heads"], case["kv"], _head_dim(case)
    return _randn((n, bs, H, D), gen), _randn((n, bs, KV, D), gen), _randn((n, bs, KV, D), gen)


def _prepare_decode(case: dict, gen: torch.Generator) -> dict:
    from qwenquest_amd.attention import DenseBackend, QuestOnlyBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode

    ctx, layers, D = _contexts(case), case["layers"], _head_dim(case)
    width = max(case.get("width", 0), max(ctx) + PAGE)
    rtp, kvp = _tables(ctx, width, layers, case["kv"], D, gen)
    if case["kind"] == "dense":
        be = DenseBackend(rtp, kvp)
    else:
        be = QuestOnlyBackend(rtp, kvp, {"algorithm": "quest", "top_k": case["top_k"], "quest_page_size": PAGE,
                                         "avoid_recent_overlap": case["avoid"]})
        for i, s in enumerate(ctx):  # the prompt's bounds, as the prefill leaves them
            be.quest.update_prefill_representations_fused(i, kvp.k_all, rtp.req_to_token[i, : s - 1])
    q, k, v = _decode_inputs(case, layers, gen)
    seq = torch.tensor(ctx, dtype=torch.int64, device=DEV)
    rpi = torch.arange(case["bs"], dtype=torch.int64, device=DEV)
    loc = rtp.req_to_token[rpi, seq - 1].to(torch.int64)
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, loc, rtp, kvp, be)
    mods = [_Layer(i, D) for i in range(layers)]

    def step():
        be.init_forward_metadata(batch)
        return [be.forward_decode(q[i], k[i], v[i], mods[i], batch) for i in range(layers)]

    return _captured({"be": be, "q": q, "k": k, "v": v, "batch": batch, "ctx": ctx}, step)


def _captured(state: dict, step) -> dict:
    step()  # workspaces, and the kernels' code on the device
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["out"] = step()
    state["graph"] = graph
    return state


def _prepare_hisparse(case: dict, gen: torch.Generator) -> dict:
    from qwenquest_amd.attention import QuestHiSparseBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode

    ctx, steps, D, bs, rho = _contexts(case), case["steps"], _head_dim(case), case["bs"], 0.9
    rtp, kvp = _tables(ctx, max(ctx) + PAGE, 1, case["kv"], D, gen)
    be = QuestHiSparseBackend(rtp, kvp, {"algorithm": "quest", "top_k": case["top_k"], "quest_page_size": PAGE,
                                         "device_buffer_size": 2 * case["top_k"],
                                         "avoid_recent_overlap": case["avoid"]}, host_pool_size=sum(ctx) + 64)
    be.on_extend_finished(ForwardBatch(ForwardMode.EXTEND, None, None, torch.arange(bs), torch.tensor(ctx) - 1, None,
                                       rtp, kvp, be))
    q, k, v = _decode_inputs(case, steps, gen)
    x = q[0].float()
    for i in range(1, steps):  # consecutive tokens' queries are correlated
        x = rho * x + (1 - rho**2) ** 0.5 * q[i].float()
        q[i] = x.to(torch.bfloat16)
    seq = torch.tensor(ctx, dtype=torch.int64, device=DEV)
    rpi = torch.arange(bs, dtype=torch.int64, device=DEV)
    batch = ForwardBatch(ForwardMode.DECODE, None, None, rpi, seq, None, rtp, kvp, be)
    layer = _Layer(0, D)
    # a whole step would take a host row per request for good, which a repeated pass cannot
    be.quest.prepare_step(seq)

    def step():
        return [be.forward_decode(q[i], k[i], v[i], layer, batch) for i in range(steps)]

    return _captured({"be": be, "q": q, "k": k, "v": v, "batch": batch, "ctx": ctx}, step)


def _prepare_extend(case: dict, gen: torch.Generator) -> dict:
    from qwenquest_amd.attention import DenseBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode

    new, prefix = _extend_lens(case)
    total = [n + p for n, p in zip(new, prefix)]
    H, KV, D = case["heads"], case["kv"], _head_dim(case)
    rtp, kvp = _tables(total, max(total) + PAGE, 1, KV, D, gen)
    be = DenseBackend(rtp, kvp)
    loc = torch.cat([rtp.req_to_token[i, p : p + n] for i, (n, p) in enumerate(zip(new, prefix))]).to(torch.int64)

    def i64(x):
        return torch.tensor(x, dtype=torch.int64, device=DEV)

    batch = ForwardBatch(ForwardMode.EXTEND, None, None, i64(list(range(len(new)))), i64(total), loc, rtp, kvp, be,
                         extend_prefix_lens=i64(prefix), extend_seq_lens=i64(new))
    n = sum(new)
    return {"be": be, "q": _randn((n, H, D), gen), "k": _randn((n, KV, D), gen), "v": _randn((n, KV, D), gen),
            "batch": batch, "layer": _Layer(0, D), "new": new, "prefix": prefix}


def _prepare_bounds(case: dict, gen: torch.Generator) -> dict:
    from qwenquest_amd.quest import QuestAlgorithm

    n, layers, KV, D = case["tokens"], case["layers"], case["kv"], _head_dim(case)
    k_all = _randn((layers, n + 1, KV, D), gen)
    qa = QuestAlgorithm(2048, PAGE, DEV)
    qa.init_storage(0, layers, 1, n + PAGE, KV, D)
    idx = torch.arange(1, n + 1, dtype=torch.int32, device=DEV)
    return {"qa": qa, "k_all": k_all, "idx": idx}


# ---------------------------------------------------------------- one pass


def run(state: dict):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "qa" in state:
        qa = state["qa"]
        qa.update_prefill_representations_fused(0, state["k_all"], state["idx"])
        return [qa.page_k_bounds, qa.running_k_min, qa.running_k_max, qa.running_token_count, qa.running_page_idx]
    return state["be"].forward_extend(state["q"], state["k"], state["v"], state["layer"], state["batch"])


# ---------------------------------------------------------------- the same in 64 bits


def _attend64(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float, mask=None) -> torch.Tensor:
    """q [n, H, D], k/v [m, KV, D] -> [n, H*D] in float64; mask [n, m] True where attended."""
    n, H, D = q.shape
    KV = k.shape[1]
    out = torch.empty((n, H, D), dtype=torch.float64, device=q.device)
    for h in range(KV):
        kh, vh = k[:, h].double(), v[:, h].double()
        for g in range(H // KV):
            s = (q[:, h * (H // KV) + g].double() @ kh.T) * scale
            if mask is not None:
                s.masked_fill_(~mask, -math.inf)
            out[:, h * (H // KV) + g] = torch.softmax(s, dim=-1) @ vh
    return out.view(n, H * D)


def exact(case: dict, seed: int):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "bounds":
        n, k_all = case["tokens"], state["k_all"]
        layers, _, KV, D = k_all.shape
        full, inf = n // PAGE, torch.finfo(torch.bfloat16).max
        pages = k_all[:, 1 : 1 + full * PAGE].view(layers, full, PAGE, KV, D)
        bounds = torch.empty((layers, 1, (n + 2 * PAGE - 1) // PAGE, KV, D, 2), dtype=torch.float64, device=DEV)
        bounds[..., 0], bounds[..., 1] = inf, -inf
        bounds[:, 0, :full, :, :, 0] = pages.amin(2).double()
        bounds[:, 0, :full, :, :, 1] = pages.amax(2).double()
        tail = k_all[:, 1 + full * PAGE :]
        lo, hi = torch.full((2, layers, 1, KV, D), inf, dtype=torch.float64, device=DEV).unbind(0)
        lo, hi = lo.clone(), -hi
        if tail.shape[1]:
            lo[:, 0], hi[:, 0] = tail.amin(1).double(), tail.amax(1).double()
        count = torch.tensor([n % PAGE], dtype=torch.int32, device=DEV)
        return [bounds, lo, hi, count, torch.tensor([full], dtype=torch.int32, device=DEV)]
    batch, scale = state["batch"], _head_dim(case) ** -0.5
    kvp, r2t = batch.token_to_kv_pool, batch.req_to_token_pool.req_to_token
    if kind == "extend":
        kvp.k_all[0][batch.out_cache_loc] = state["k"]
        kvp.v_all[0][batch.out_cache_loc] = state["v"]
        outs, at = [], 0
        for i, (n, p) in enumerate(zip(state["new"], state["prefix"])):
            rows = r2t[i, : n + p].long()
            k, v = kvp.k_all[0][rows], kvp.v_all[0][rows]
            kpos = torch.arange(n + p, device=DEV)
            for a in range(0, n, 2048):
                b = min(n, a + 2048)
                mask = kpos[None] <= (p + torch.arange(a, b, device=DEV))[:, None]
                outs.append(_attend64(state["q"][at + a : at + b], k, v, scale, mask))
            at += n
        return torch.cat(outs)
    n = case["layers"] if kind != "hisparse" else case["steps"]
    return [_exact_decode(case, state, i, kvp, r2t, scale) for i in range(n)]


def _exact_decode(case: dict, state: dict, i: int, kvp, r2t: torch.Tensor, scale: float) -> torch.Tensor:
    layer = i if case["kind"] != "hisparse" else 0
    H, KV, D = case["heads"], case["kv"], _head_dim(case)
    out = torch.empty((case["bs"], H * D), dtype=torch.float64, device=DEV)
    for b, s in enumerate(state["ctx"]):
        rows = r2t[b, :s].long()
        k, v = kvp.k_all[layer][rows], kvp.v_all[layer][rows]
        k[s - 1], v[s - 1] = state["k"][i, b], state["v"][i, b]
        if case["kind"] != "dense" and s > case["top_k"]:
            pages = s // PAGE
            lim = max(pages - 1, 0) if case["avoid"] else pages
            kp = k[: pages * PAGE].view(pages, PAGE, KV, D)
            acc = torch.zeros((KV, D), dtype=torch.float32, device=DEV)
            for g in range(H // KV):  # the mean query is part of the method: bf16, summed in head order
                acc = acc + state["q"][i, b].view(KV, H // KV, D)[:, g].float()
            qbar = (acc / (H // KV)).to(torch.bfloat16).double()
            sc = torch.where(qbar >= 0, qbar * kp.amax(1).double(), qbar * kp.amin(1).double()).sum((1, 2))[:lim]
            top = torch.sort(sc, descending=True, stable=True).indices[: case["top_k"] // PAGE - 1]
            pos = torch.cat([(top[:, None] * PAGE + torch.arange(PAGE, device=DEV)).flatten(),
                             torch.arange(s - PAGE, s, device=DEV)])
            k, v = k[pos], v[pos]
        out[b] = _attend64(state["q"][i, b][None], k, v, scale)[0]
    return out
