"""Attention-backend interface (reference ``src/qwenquest/attention/base.py:20-112``).

The drop-in boundary: per forward the engine calls ``init_forward_metadata``
once, then the model calls ``forward`` once per layer.  ``layer`` is any object
with ``layer_id`` and ``scaling`` (the reference's ``RadixAttention``).
"""

from __future__ import annotations

from abc import ABC, abstractmethod
from typing import TYPE_CHECKING, Any

import torch
from torch.autograd import forward_ad

from qwenquest_amd.attention.ops import extend_attention, extend_attention_batch, extend_attention_batch_checked

if TYPE_CHECKING:
    from qwenquest_amd.batch import ForwardBatch
    from qwenquest_amd.memory import MHATokenToKVPool, ReqToTokenPool

__all__ = ["AttentionBackend"]


def _plain(t: torch.Tensor) -> bool:
    """Whether torch would only compute with ``t``: no gradient to record, no tangent to carry and
    no subclass that sees the operations."""
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and not (t.requires_grad and torch.is_grad_enabled())
            and forward_ad.unpack_dual(t).tangent is None)


class AttentionBackend(ABC):
    #: SGLang backend this class stands in for.
    name: str = ""
    #: Whether a decode token's K/V goes to the shared device token pool.
    uses_token_pool_for_decode: bool = True
    #: Whether the engine may free the prefill's token-pool slots after on_extend_finished.
    frees_prefill_kv_after_admission: bool = False

    def __init__(self, req_to_token_pool: ReqToTokenPool, token_to_kv_pool: MHATokenToKVPool):
        self.req_to_token_pool = req_to_token_pool
        self.token_to_kv_pool = token_to_kv_pool

    @property
    def req_to_token(self) -> torch.Tensor:
        return self.req_to_token_pool.req_to_token

    def init_forward_metadata(self, batch: ForwardBatch) -> None:  # noqa: B027 - optional hook
        """Per-forward preparation (once, before layer 0)."""

    def forward(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer: Any, batch: ForwardBatch) -> torch.Tensor:
        if batch.forward_mode.is_decode():
            return self.forward_decode(q, k, v, layer, batch)
        return self.forward_extend(q, k, v, layer, batch)

    def forward_extend(self, q, k, v, layer, batch: ForwardBatch) -> torch.Tensor:
        """Dense causal prefill: save the new K/V, then attend per request (base.py:65-93).

        bf16 with head_dim 128 runs the whole batch in one launch, which reads the lengths
        on the device; a batch that the launch does not answer as the loop below does goes
        through the loop (which raises IndexError for a request index outside the table).
        Other shapes go request by request through ``extend_attention``.  Inside a graph
        capture, which the loop refuses, a request index outside the table gives NaN, as do
        rows of ``q`` past the requests' tokens.
        """
        assert batch.out_cache_loc is not None and batch.extend_prefix_lens is not None
        pool = self.token_to_kv_pool
        pool.set_kv_buffer(layer.layer_id, batch.out_cache_loc, k, v)
        k_buf, v_buf = pool.get_kv_buffer(layer.layer_id)
        if self._extend_fast(q, k_buf, v_buf, layer.scaling, batch):
            attend = (extend_attention_batch if torch.cuda.is_current_stream_capturing()
                      else extend_attention_batch_checked)
            out = attend(q, k_buf, v_buf, self.req_to_token, batch.req_pool_indices, batch.seq_lens,
                         batch.extend_prefix_lens, batch.extend_seq_lens, float(layer.scaling))
            if out is not None:
                return out
        offsets = batch.extend_token_offsets()
        outputs = []
        for i in range(batch.batch_size):
            req = int(batch.req_pool_indices[i])
            seq_len = int(batch.seq_lens[i])
            locs = self.req_to_token[req, :seq_len].long()
            outputs.append(
                extend_attention(q[offsets[i] : offsets[i + 1]], k_buf[locs], v_buf[locs],
                                 prefix_len=int(batch.extend_prefix_lens[i]), scaling=layer.scaling)
            )
        return torch.cat(outputs, dim=0)

    def _extend_fast(self, q: torch.Tensor, k_buf: torch.Tensor, v_buf: torch.Tensor, scaling: float,
                     batch: ForwardBatch) -> bool:
        """Whether the batched prefill kernel takes this call: its tile is 128 channels wide, a
        row's maximum is taken before the scale, which therefore has to be positive, it reads the
        pool in 16-byte pieces, and it records and carries no derivative."""
        pool, r2t, ext, bs = self.token_to_kv_pool, self.req_to_token, batch.extend_seq_lens, batch.batch_size
        dev = q.device
        if (q.dim() != 3 or q.dtype != torch.bfloat16 or pool.dtype != torch.bfloat16 or pool.head_dim != 128
                or bs == 0 or ext is None or not float(scaling) > 0.0 or not q.is_cuda or not _plain(q)
                or torch._C._get_tracing_state() is not None):
            return False
        n, heads, dim = q.shape
        if n == 0 or heads == 0 or dim != 128 or heads % pool.kv_heads:
            return False
        for b in (k_buf, v_buf):
            if b.device != dev or b.data_ptr() % 16 or not b.is_contiguous() or b.requires_grad:
                return False
        for t in (batch.req_pool_indices, batch.seq_lens, batch.extend_prefix_lens, ext):
            if t.dim() != 1 or t.shape[0] < bs:
                return False
        row, col = r2t.stride()
        return r2t.dtype == torch.int32 and col == 1 and row >= r2t.shape[1] and r2t.device == dev

    @abstractmethod
    def forward_decode(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, layer: Any, batch: ForwardBatch) -> torch.Tensor:
        """``q [bs, H, D]``, ``k/v [bs, KV, D]`` of the new tokens -> ``[bs, H*D]``."""

    def on_extend_finished(self, batch: ForwardBatch) -> None:  # noqa: B027 - optional hook
        """Called by the engine after a whole prefill forward (all layers)."""

    def on_request_finished(self, req_pool_idx: int) -> None:  # noqa: B027 - optional hook
        """Called by the engine before a request slot is reused."""

    def poll_errors(self) -> None:  # noqa: B027 - optional hook
        """Raise an error the device detected in a decode step whose kernels have finished,
        without a synchronisation.  A caller that replays a captured decode step calls it after
        each replay, since no Python check runs inside a replay.  Backends without
        device-detected errors have nothing to raise."""
