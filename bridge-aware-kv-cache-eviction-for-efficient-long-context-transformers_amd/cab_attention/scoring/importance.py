"""Cumulative-attention (H2O) importance tracking (reference:
``cab_attention/scoring/importance.py`` :17-133). The running totals are
summed by ``cab_key_sums`` on the GPU; the top-k runs in ``cab_evict_select``."""

from __future__ import annotations

from typing import Optional

import torch

from .. import _native as nat
from ..eviction._select import BRIDGE_NONE, select_positions

_DTYPES = (torch.float32, torch.float16, torch.bfloat16)

def _kernel_sums(rows: int, n_k: int, key_stride: int = 1) -> bool:
    """Whether ``cab_key_sums`` takes a sum over ``rows`` (batch x heads x queries)
    of ``n_k`` keys; torch's sum the rest. The kernel's workgroups are one per 64
    keys, each over all rows: one launch instead of several, but too few of them
    where many rows meet few keys, and slower than torch's wide loads once they
    run in several rounds. bf16 (fp32), us an update, torch -> kernel:
    32 rows of 4500 keys 13.3 -> 6.5 (9.2 -> 6.3), 512 of 300 15.8 -> 13.3
    (12.1 -> 11.7), 512 of 24000 29.6 -> 25.5 (28.4 -> 22.1), 512 of 32768 24.1 ->
    25.8; 256 of 32768 14.5 -> 13.2 (13.3 -> 12.5), 256 of 50000 20.1 -> 25.1; 8 of
    131072 13.0 -> 6.8, 64 of 131072 14.2 -> 14.8 (9.8 -> 14.1); 1024 of 8192 16.7 ->
    25.2 (14.0 -> 22.3), 1024 of 12000 52.2 -> 31.0 (50.0 -> 23.7), 4096 of 24000
    196 -> 189 (290 -> 155), 16000 of 500 23 -> 424. The fp32 sums' rms error is not
    above torch's anywhere in it. Keys apart in memory (a transposed tensor) cost a
    cache line each: 32 rows of 4500 keys 13.8 -> 6.5 (10.2 -> 6.8), 512 of 300 14.2 ->
    15.8 (10.2 -> 15.8)."""
    if key_stride != 1 and rows > 32:
        return False
    if n_k <= 24000:
        return rows <= 512 or (n_k >= 12000 and rows <= 4096)
    return rows * n_k <= (1 << 23 if n_k <= 32768 else 1 << 20)


class ImportanceTracker:
    """Running sum of the attention each cached position receives."""

    def __init__(self, device: str = "cuda"):
        self.device = device
        self.cumulative_scores = None
        self.total_queries = 0

    def reset(self):
        self.cumulative_scores = None
        self.total_queries = 0

    def update(self, attention_weights: torch.Tensor):
        """Adds ``attention_weights [B, H, N_q, N_kv]`` summed over batch,
        heads and queries; a longer N_kv extends the totals with zeros."""
        if self._update_on_device(attention_weights):
            return
        position_scores = attention_weights.sum(dim=(0, 1, 2)).float()
        if self.cumulative_scores is None:
            self.cumulative_scores = position_scores
        else:
            cur, cached = position_scores.numel(), self.cumulative_scores.numel()
            if cur > cached:
                self.cumulative_scores = torch.cat([
                    self.cumulative_scores,
                    torch.zeros(cur - cached, device=self.cumulative_scores.device,
                                dtype=self.cumulative_scores.dtype)])
            self.cumulative_scores[:cur] += position_scores
        self.total_queries += attention_weights.shape[2]

    def _update_on_device(self, w: torch.Tensor) -> bool:
        """:meth:`update` in one launch (``cab_key_sums``), the extension
        included. False, and nothing done, for what it does not take."""
        old = self.cumulative_scores
        if (w.device.type != "cuda" or w.dim() != 4 or w.dtype not in _DTYPES or w.numel() == 0
                or (w.requires_grad and torch.is_grad_enabled()) or not nat.addressable(w)):
            return False
        if w.dtype != torch.float32 and torch.is_autocast_enabled("cuda"):
            return False  # autocast sums in fp32 and does not round
        B, H, n_q, n_k = w.shape
        if not _kernel_sums(B * H * n_q, n_k, w.stride(3)):
            return False
        if old is None:
            n_old = 0
        elif (old.device != w.device or old.dtype != torch.float32 or old.dim() != 1
              or not old.is_contiguous() or old.requires_grad):
            return False
        else:
            n_old = old.numel()
            if n_old >= n_k and nat.closed(old):
                return False
        # Totals that reach far enough are added to in place, shorter ones extended.
        sums = old if n_old >= n_k else torch.empty(n_k, dtype=torch.float32, device=w.device)
        with nat.on_device(w.device):
            st = nat.load().cab_key_sums(w.data_ptr(), nat.dtype_code(w), B, H, n_q, n_k,
                                         nat.strides4(w), nat.ptr(old), n_old, sums.data_ptr(),
                                         nat.stream_ptr(w.device))
        nat.check("cab_key_sums", st)
        if sums is old:
            nat.wrote(sums)
        self.cumulative_scores = sums
        self.total_queries += n_q
        return True

    def add_scores(self, position_scores: torch.Tensor, n_queries: int = 1):
        """Adds per-position totals already summed over queries (for example
        the key totals of ``flash_attention_with_cumulative_scores``, summed
        over batch and heads)."""
        self.update(position_scores.reshape(1, 1, 1, -1))
        self.total_queries += n_queries - 1

    def get_top_k_indices(self, k: int, exclude_indices: Optional[torch.Tensor] = None) -> torch.Tensor:
        """The k highest-scoring positions, highest first (equal scores in
        position order), or an empty tensor before any update."""
        if self.cumulative_scores is None:
            return torch.arange(0, 0, device=self.device)
        scores = self.cumulative_scores
        if exclude_indices is not None and len(exclude_indices) > 0:
            scores = scores.clone()
            scores[exclude_indices] = -float("inf")
        n = scores.numel()
        k = min(k, n)
        keep, _, _, _ = select_positions(n, scores, 0, k, 0, False, BRIDGE_NONE, scores.device)
        vals = scores[keep]
        nan = torch.isnan(vals)
        order = torch.sort(torch.where(nan, torch.full_like(vals, float("inf")), vals), stable=True,
                           descending=True).indices
        order = order[torch.sort(nan[order].to(torch.uint8), stable=True, descending=True).indices]
        return keep[order]

    def get_scores(self) -> Optional[torch.Tensor]:
        return self.cumulative_scores

    def prune(self, keep_indices: torch.Tensor):
        """Keeps the totals of the kept positions (in order)."""
        if self.cumulative_scores is not None:
            valid = keep_indices[keep_indices < self.cumulative_scores.numel()]
            self.cumulative_scores = self.cumulative_scores[valid] if valid.numel() > 0 else None

    def __len__(self) -> int:
        return 0 if self.cumulative_scores is None else self.cumulative_scores.numel()
