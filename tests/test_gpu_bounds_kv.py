"""Prefill page bounds at KV*D = 128, 256, 512 and 1024 (1, 2, 4 and 8 KV heads x 128): the wave-per-page
folds against the per-element fold of the same keys as fp32 (reference quest.py:231-280)."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_quest import DEV, new_quest, rand_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [1, 2, 4, 8])
@pytest.mark.parametrize("page,n", [(64, 0), (64, 1), (64, 63), (64, 777), (16, 100), (32, 65), (128, 333), (200, 777)])
@pytest.mark.parametrize("kind", ["plain", "special", "bad_rows", "zeros"])
def test_prefill_bounds_match_the_per_element_fold(kv, page, n, kind):
    pool = rand_bf16((1100, kv, 128), seed=n + page)
    gen = torch.Generator().manual_seed(kv)
    if kind == "special":  # NaN, both zeros and both infinities, several to a page
        bits = pool.view(torch.int16).view(-1)
        for val in (0x7FC0, 0x0000, -0x8000, 0x7F80, 0xFF80 - 65536):
            bits[torch.randint(0, bits.numel(), (60 * kv,), generator=gen)] = val
    if kind == "zeros":  # by channel: all of one zero, clamped at one, with a few of the other, NaNs
        x = pool.view(1100, kv * 128)
        zero, neg = torch.zeros((), dtype=x.dtype), -torch.zeros((), dtype=x.dtype)
        for c in range(kv * 128):
            z, other = (zero, neg) if c % 2 else (neg, zero)
            how = (c // 2) % 8
            if how == 1:
                x[:, c] = z
            elif how in (2, 3, 4):
                x[:, c] = torch.where((x[:, c] < 0) if how == 2 else (x[:, c] > 0), z, x[:, c])
            if how in (1, 3) and c % 5 == 0:
                x[torch.randint(0, 1100, (9,), generator=gen), c] = other
            if how == 4 and c % 31 == 0:
                x[torch.randint(0, 1100, (2,), generator=gen), c] = float("nan")
    idx = torch.randperm(1100, generator=gen)[:n].to(torch.int32 if page != 128 else torch.int64)
    if kind == "bad_rows" and n > 3:
        idx[[0, n // 2, n - 1]] = torch.tensor([-1, 5000, 1100], dtype=idx.dtype)
    qb, _ = new_quest(page * 4, page, 2, 4, 1024, kv, 128)
    qf, _ = new_quest(page * 4, page, 2, 4, 1024, kv, 128)
    for layer in range(2):
        qb.update_prefill_representations(layer, 2, pool.to(DEV), idx.to(DEV))
        qf.update_prefill_representations(layer, 2, pool.float().to(DEV), idx.to(DEV))
    for name in ("page_k_bounds", "running_k_min", "running_k_max"):
        assert torch.equal(getattr(qb, name).view(torch.int16), getattr(qf, name).view(torch.int16)), name
    for name in ("running_token_count", "running_page_idx"):
        assert torch.equal(getattr(qb, name), getattr(qf, name)), name


@pytest.mark.parametrize("kv", [1, 2, 4, 8])
def test_row_counts_past_32_bits_take_the_general_fold(kv):
    """A pool said to hold more than 2^31 rows (the indices are small): the same bounds."""
    pool = rand_bf16((500, kv, 128), seed=kv).to(DEV)
    idx = torch.randperm(500, generator=torch.Generator().manual_seed(kv))[:333].to(DEV)
    got = []
    for rows in (500, 1 << 32):
        q, _ = new_quest(256, 64, 1, 1, 1024, kv, 128)
        q._prefill(pool, 0, rows, 0, idx, 0, 1, True)
        got.append([t.clone() for t in (q.page_k_bounds, q.running_k_min, q.running_k_max, q.running_page_idx)])
    for a, b in zip(*got, strict=True):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
