"""Batched prefill attention (reference ``src/qwenquest/attention/base.py:65-93``, ops.py:18-45):
the HIP kernel against float64 and against the request-by-request path."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)


class Layer:
    def __init__(self, d):
        self.layer_id, self.scaling = 0, d**-0.5


def make(new, prefix, H, KV, seed, width=None, qscale=1.0):
    from qwenquest_amd.attention.dense import DenseBackend
    from qwenquest_amd.batch import ForwardBatch, ForwardMode
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

    total = [n + p for n, p in zip(new, prefix)]
    bs, D = len(new), 128
    rtp = ReqToTokenPool(bs + 1, width or max(total) + 5, DEV)
    kvp = MHATokenToKVPool(sum(total), 1, KV, D, torch.bfloat16, DEV)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    kvp.k_all.normal_(generator=gen)
    kvp.v_all.normal_(generator=gen)
    perm = torch.from_numpy(np.random.default_rng(seed).permutation(sum(total)).astype(np.int32) + 1).to(DEV)
    slots = list(range(1, bs + 1))[::-1]  # request i in table row bs - i
    at = 0
    for i, n in enumerate(total):
        rtp.req_to_token[slots[i], :n] = perm[at : at + n]
        at += n
    be = DenseBackend(rtp, kvp)
    loc = torch.cat([rtp.req_to_token[slots[i], p : p + n] for i, (n, p) in enumerate(zip(new, prefix))]).long()
    n = sum(new)
    mk = lambda h: torch.empty((n, h, D), device=DEV).normal_(generator=gen).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(H) * qscale, mk(KV), mk(KV)
    t = lambda x: torch.tensor(x, dtype=torch.int64, device=DEV)  # noqa: E731
    batch = ForwardBatch(ForwardMode.EXTEND, None, None, t(slots), t(total), loc, rtp, kvp, be,
                         extend_prefix_lens=t(prefix), extend_seq_lens=t(new))
    return be, q, k, v, batch, Layer(D), slots


def launch(be, q, batch, layer):
    """The launch alone, as a captured call runs it: nothing is read on the host."""
    from qwenquest_amd.attention.ops import extend_attention_batch

    k_buf, v_buf = batch.token_to_kv_pool.get_kv_buffer(0)
    return extend_attention_batch(q, k_buf, v_buf, be.req_to_token, batch.req_pool_indices, batch.seq_lens,
                                  batch.extend_prefix_lens, batch.extend_seq_lens, layer.scaling)


def exact(batch, slots, q, new, prefix, KV):
    """float64 causal attention over the pool's rows."""
    kvp, r2t = batch.token_to_kv_pool, batch.req_to_token_pool.req_to_token
    H, D = q.shape[1:]
    outs, at = [], 0
    for i, (n, p) in enumerate(zip(new, prefix)):
        rows = r2t[slots[i], : n + p].long()
        k, v = kvp.k_all[0][rows].double(), kvp.v_all[0][rows].double()
        mask = torch.arange(n + p, device=DEV)[None] <= (p + torch.arange(n, device=DEV))[:, None]
        o = torch.empty((n, H, D), dtype=torch.float64, device=DEV)
        for h in range(H):
            s = (q[at : at + n, h].double() @ k[:, h // (H // KV)].T.contiguous()) * D**-0.5
            o[:, h] = torch.softmax(s.masked_fill(~mask, -float("inf")), -1) @ v[:, h // (H // KV)].contiguous()
        outs.append(o.view(n, H * D))
        at += n
    return torch.cat(outs)


def close(got, ref):
    """Half a bf16 ulp of the result (2^-8 of it) and the fp32 sums' own error."""
    err = (got.double() - ref).abs()
    assert bool((err <= 2.0**-8 * ref.abs() + 1e-5).all()), float((err - 2.0**-8 * ref.abs()).max())


@pytest.mark.parametrize("H,KV,new,prefix", [
    (32, 4, [1], [0]),
    (32, 4, [16], [0]),  # one block's rows
    (32, 4, [17, 15, 1, 64], [0, 63, 64, 65]),  # edges of the query and of the K/V tile
    (32, 4, [600], [0]),
    (20, 4, [77, 130], [5, 0]),  # groups of 5: a tile ends inside a token
    (28, 4, [33, 200], [0, 129]),
    (4, 4, [129, 1], [0, 300]),  # no grouping
    (5, 1, [300], [40]),
    (14, 2, [190, 31], [0, 12]),
    (64, 8, [100, 9], [64, 1]),
    (96, 2, [21], [7]),  # 48 heads per KV head
    (32, 4, [5], [6000]),  # few rows, long prefix: K/V splits and the merge
    (8, 2, [3, 40], [2047, 513]),  # splits for one request, none for the other
    (32, 4, [2, 0, 3] + [1] * 66, [1, 4, 0] + [9] * 66),  # an empty request; more than 64 requests
])
def test_extend_batch_matches_float64_and_the_general_path(H, KV, new, prefix, monkeypatch):
    be, q, k, v, batch, layer, slots = make(new, prefix, H, KV, 3, width=8192 if max(prefix) > 2000 else None)
    got = be.forward_extend(q, k, v, layer, batch)
    assert got.shape == (sum(new), H * 128) and got.dtype == torch.bfloat16
    close(got, exact(batch, slots, q, new, prefix, KV))
    again = be.forward_extend(q, k, v, layer, batch)
    assert torch.equal(got, again)
    monkeypatch.setattr(be, "_extend_fast", lambda *a: False)
    ref = be.forward_extend(q, k, v, layer, batch).double()
    err = (got.double() - ref).abs()  # one rounding each, of sums 1e-5 apart
    assert bool((err <= 2.0**-7 * ref.abs() + 2e-5).all())


def test_extend_batch_sharp_scores_and_other_forms():
    """Scores up to hundreds (one weight near 1, the rest tiny); lengths as CPU and int32 tensors,
    q as a view with gaps; a captured call replays."""
    new, prefix = [70, 130], [0, 100]
    be, q, k, v, batch, layer, slots = make(new, prefix, 32, 4, 9, qscale=40.0)
    got = be.forward_extend(q, k, v, layer, batch)
    ref = exact(batch, slots, q, new, prefix, 4)
    # an fp32 score of 400 is off by up to 2e-5, and its weight by that share
    assert bool(((got.double() - ref).abs() <= 2.0**-8 * ref.abs() + 4e-4).all())
    wide = torch.zeros((q.shape[0], 40, 128), dtype=q.dtype, device=DEV)
    wide[:, :32] = q
    batch.seq_lens, batch.req_pool_indices = batch.seq_lens.cpu(), batch.req_pool_indices.to(torch.int32)
    batch.extend_prefix_lens = batch.extend_prefix_lens.cpu()
    assert torch.equal(be.forward_extend(wide[:, :32], k, v, layer, batch), got)
    batch.seq_lens, batch.extend_prefix_lens = batch.seq_lens.to(DEV), batch.extend_prefix_lens.to(DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = be.forward_extend(q, k, v, layer, batch)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, got)


def test_extend_batch_rows_outside_their_tables():
    """A request index past the table raises, a row past the pool gives NaN, the others get their
    answer, and negative ones count from the end; a context longer than the table is cut to it, as a slice is."""
    new, prefix = [40, 50, 60], [0, 30, 0]
    be, q, k, v, batch, layer, slots = make(new, prefix, 32, 4, 5)
    want = be.forward_extend(q, k, v, layer, batch)
    batch.req_pool_indices[2] = 99
    with pytest.raises(IndexError):  # as the request-by-request path
        be.forward_extend(q, k, v, layer, batch)
    got = launch(be, q, batch, layer)
    assert torch.equal(got[:90], want[:90]) and bool(got[90:].isnan().all())
    batch.req_pool_indices[2] = slots[2] - batch.req_to_token_pool.size  # counts from the table's end
    assert torch.equal(be.forward_extend(q, k, v, layer, batch), want)
    assert torch.equal(launch(be, q, batch, layer), want)
    batch.req_pool_indices[2] = slots[2]
    r2t = batch.req_to_token_pool.req_to_token
    keep = int(r2t[slots[1], 10])
    r2t[slots[1], 10] = keep - batch.token_to_kv_pool.rows  # a negative row counts from the pool's end
    assert torch.equal(be.forward_extend(q, k, v, layer, batch), want)
    r2t[slots[1], 10] = 1 << 20
    got = be.forward_extend(q, k, v, layer, batch)
    assert torch.equal(got[:40], want[:40]) and torch.equal(got[90:], want[90:])
    assert bool(got[40:90].isnan().all())
    r2t[slots[1], 10] = keep
    batch.seq_lens[1] = 10_000
    batch.extend_prefix_lens[1] = r2t.shape[1] - 50
    r2t[slots[1], 80:] = 1
    got = be.forward_extend(q, k, v, layer, batch)
    batch.seq_lens[1] = r2t.shape[1]
    assert torch.equal(be.forward_extend(q, k, v, layer, batch), got)


@pytest.mark.parametrize("H,KV,n,ext", [
    (32, 4, 6, [5]),  # the request's partial tile is the last one that the rows can fill
    (32, 4, 31, [30]),
    (4, 4, 255, [254]),
    (8, 2, 63, [50, 12]),
    (32, 4, 700, [33, 1, 17]),  # many tiles past the requests'
    (20, 4, 40, [0, 0]),  # no tokens at all
])
def test_rows_past_the_requests_tokens_are_nan(H, KV, n, ext):
    """q with more rows than the requests have tokens: the rows past them are written."""
    from qwenquest_amd.attention.ops import extend_attention_batch

    be, q, k, v, batch, layer, slots = make([max(e, 1) for e in ext], [3] * len(ext), H, KV, 7)
    lens = torch.tensor(ext, device=DEV)
    total = sum(ext)
    k_buf, v_buf = batch.token_to_kv_pool.get_kv_buffer(0)
    qp = torch.ones((n, H, 128), dtype=torch.bfloat16, device=DEV)
    qp[:total] = q[:total]

    def call(x):
        stale = [torch.ones((n, H * 128), dtype=torch.bfloat16, device=DEV) for _ in range(4)]
        del stale  # the output's memory holds numbers before the call
        return extend_attention_batch(x, k_buf, v_buf, be.req_to_token, batch.req_pool_indices, lens + 3,
                                      batch.extend_prefix_lens, lens, layer.scaling)

    got = call(qp)
    assert got.shape == (n, H * 128) and bool(got[total:].isnan().all())
    if total:
        assert torch.equal(got[:total], call(qp[:total].contiguous()))


@pytest.mark.parametrize("where", ["cuda", "cpu"])
def test_calls_that_the_request_by_request_path_takes_or_refuses(where, monkeypatch):
    """The batched path against the loop over the forms of a call: the same rows, values to one
    rounding of each, and the same refusals."""
    new, prefix = [40, 0, 30], [0, 5, 70]
    be, q, k, v, batch, layer, slots = make(new, prefix, 8, 2, 11)
    names = ("req_pool_indices", "seq_lens", "extend_prefix_lens", "extend_seq_lens")
    for name in names:
        setattr(batch, name, getattr(batch, name).to(where))
    fields = {name: getattr(batch, name) for name in names}
    fast = be._extend_fast

    def both(q=q, **changed):
        got = []
        for loop in (False, True):
            for name in names:
                setattr(batch, name, changed.get(name, fields[name]))
            monkeypatch.setattr(be, "_extend_fast", (lambda *a: False) if loop else fast)
            try:
                got.append(be.forward_extend(q, k, v, layer, batch))
            except (IndexError, RuntimeError) as e:
                got.append(type(e))
        a, b = got
        if isinstance(b, type):
            assert a is b
            return a
        assert a.shape == b.shape
        err = (a.double() - b.double()).abs()
        assert bool((err <= 2.0**-7 * b.double().abs() + 2e-5).all())
        return a

    def t(*x):
        return torch.tensor(x, device=where)

    full = both()
    padded = torch.cat([q, torch.ones_like(q[:9])])
    assert torch.equal(both(q=padded), full)  # the requests' rows and no others
    assert torch.equal(both(q=q[:60].contiguous()), full[:60])  # fewer: the last request has what is left
    assert torch.equal(both(req_pool_indices=t(*(s - batch.req_to_token_pool.size for s in slots))), full)
    assert both(req_pool_indices=t(slots[0], slots[1], batch.req_to_token_pool.size)) is IndexError
    assert both(req_pool_indices=t(-batch.req_to_token_pool.size - 1, *slots[1:])) is IndexError
    for name in names[1:]:  # fewer lengths than requests
        assert both(**{name: fields[name][:2]}) is IndexError
    for name in names[1:]:  # and more of them
        assert torch.equal(both(**{name: torch.cat([fields[name], t(7)])}), full)
    both(extend_seq_lens=t(0, 0, 0), q=q[:0])
    both(seq_lens=t(40, 5, 10_000))  # longer than the table: cut to its width


@pytest.mark.parametrize("new,prefix", [([5], [600]), ([70, 3], [0, 200])])
def test_columns_of_a_wider_table(new, prefix):
    """req_to_token as a slice of a table whose width asks for other K/V splits; a context longer
    than the slice is cut to the slice, not to the table."""
    be, q, k, v, batch, layer, slots = make(new, prefix, 8, 1, 13)
    want = be.forward_extend(q, k, v, layer, batch)
    narrow = be.req_to_token
    wide = torch.full((narrow.shape[0], 9000), 1 << 20, dtype=torch.int32, device=DEV)  # rows past the pool
    wide[:, 11 : 11 + narrow.shape[1]] = narrow
    batch.req_to_token_pool.req_to_token = wide[:, 11 : 11 + narrow.shape[1]]
    exact_err(be.forward_extend(q, k, v, layer, batch), want)
    batch.seq_lens[0] = 9000
    batch.extend_prefix_lens[0] = narrow.shape[1] - new[0]
    got = be.forward_extend(q, k, v, layer, batch)
    batch.req_to_token_pool.req_to_token = narrow
    exact_err(got, be.forward_extend(q, k, v, layer, batch))


def exact_err(got, want):
    """Other splits of the same sums: one rounding of each."""
    assert not bool(got.isnan().any())
    err = (got.double() - want.double()).abs()
    assert bool((err <= 2.0**-7 * want.double().abs() + 2e-5).all())


def test_derivatives_and_subclasses_go_through_torch():
    """A gradient, a tangent or a subclass keeps what torch does with it."""
    from torch.autograd import forward_ad as fwad
    from torch.nn.attention import SDPBackend, sdpa_kernel

    be, q, k, v, batch, layer, slots = make([20, 13], [0, 30], 4, 2, 17)
    dq = torch.randn_like(q)
    run = lambda x: be.forward_extend(x, k, v, layer, batch)  # noqa: E731
    want = run(q)
    x = q.clone().requires_grad_()
    run(x).sum().backward()
    assert bool(x.grad.abs().sum() > 0)
    with sdpa_kernel(SDPBackend.MATH):  # the one form with forward derivatives
        with fwad.dual_level():
            out = fwad.unpack_dual(run(fwad.make_dual(q, dq)))
        assert out.tangent is not None and bool(out.tangent.abs().sum() > 0)
        exact_err(out.primal, want)

    class Seen(torch.Tensor):
        pass

    assert type(run(q.as_subclass(Seen))) is Seen


@pytest.mark.parametrize("new,prefix,width", [([200, 40], [0, 30], None), ([6], [3000], 8192)])
def test_infinite_values(new, prefix, width):
    """An infinite value of an attended row makes the output infinite (also through K/V splits and
    their merge), a NaN makes it NaN, and other channels stay as they are."""
    be, q, k, v, batch, layer, slots = make(new, prefix, 4, 2, 19, width=width)
    want = be.forward_extend(q, k, v, layer, batch).view(-1, 4, 128)
    inf = float("inf")
    pool, r2t = batch.token_to_kv_pool, batch.req_to_token_pool.req_to_token
    at, ones = 0, torch.ones(4, device=DEV)
    for i, (n, p) in enumerate(zip(new, prefix)):
        rows = r2t[slots[i]].long()
        old = sorted({0, p + n // 2})
        for pos, c, val in ((0, 5, inf), (old[-1], 9, -inf), (old[-1], 11, float("nan"))):
            if pos >= p:
                v[at + pos - p, :, c] = val
            else:
                pool.v_all[0, rows[pos], :, c] = val
        at += n
    got = be.forward_extend(q, k, v, layer, batch).view(-1, 4, 128)
    at = 0
    for i, (n, p) in enumerate(zip(new, prefix)):
        mid = n // 2  # the first of the request's tokens that attends the second position
        assert torch.equal(got[at : at + n, :, 5].float(), inf * ones.expand(n, 4))
        assert torch.equal(got[at + mid : at + n, :, 9].float(), -inf * ones.expand(n - mid, 4))
        assert bool(got[at + mid : at + n, :, 11].isnan().all())
        at += n
    rest = [c for c in range(128) if c not in (5, 9, 11)]
    assert torch.equal(got[..., rest], want[..., rest])


def test_a_row_outside_the_pool_in_the_new_tokens():
    """Every token that attends the row gets NaN, and tokens before it keep their answer up to the
    tile of 128 query rows that holds it."""
    H, KV, n, at = 32, 4, 600, 300
    be, q, k, v, batch, layer, slots = make([n, 20], [0, 9], H, KV, 23)
    want = be.forward_extend(q, k, v, layer, batch)
    batch.req_to_token_pool.req_to_token[slots[0], at] = 1 << 20
    got = launch(be, q, batch, layer)
    tile = 128 // (H // KV)  # tokens of a tile
    first = at // tile * tile
    assert torch.equal(got[:first], want[:first]) and torch.equal(got[n:], want[n:])
    assert bool(got[at:n].isnan().all())


def test_threads_on_their_own_streams():
    """Calls of several threads, some of them refused, each with its own verdict."""
    import threading

    cases = [make([50 + 30 * i], [10 * i], 8, 2, 30 + i) for i in range(3)]
    want = [be.forward_extend(q, k, v, layer, batch) for be, q, k, v, batch, layer, _ in cases]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        be, q, k, v, batch, layer, slots = cases[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                if not torch.equal(be.forward_extend(q, k, v, layer, batch), want[i]):
                    wrong.append(i)
                good, batch.req_pool_indices = batch.req_pool_indices, torch.full((1,), 9, device=DEV)
                try:
                    be.forward_extend(q, k, v, layer, batch)
                    wrong.append(i)
                except IndexError:
                    pass
                batch.req_pool_indices = good
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
