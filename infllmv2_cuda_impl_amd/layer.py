"""Caller-side glue: an attention layer that strings the operators together the way a MiniCPM4-style model does.

The reference ships only the operators; its callers (the model code, README.md:36-60, 118-140) build the
compressed keys, call ``infllmv2_attn_stage1``, pool, take the top-k and call ``infllmv2_attn_varlen_func`` (prefill)
or ``infllmv2_attn_with_kvcache`` (decode).  This module is that sequence, so that the kernels can be exercised and
validated inside one layer: a prefill over packed sequences, a single-sequence decode loop and a batched decode step
(``BatchCache`` / ``decode_batch``) that keep the K/V caches and the two compressed-key caches up to date (a new
compressed key every ``stride`` tokens).

Conventions (the ones the operators assume):
* block size 64, compressed keys kernel 32 / stride 16, log-sum-exp over kernel 128 / stride 64;
* ``topk`` counts the forced blocks (``init_blocks`` first ones, the query's own block and ``local_blocks`` before it);
* sequences of at most ``dense_len`` tokens skip the selection and attend densely (every block selected);
* in decode the single query scores every complete compressed key of the cache (non-causal Stage 1: all of them
  lie in its past), its block index is ``cache_len // 64`` (``max_pooling_1d`` with ``cache_len``), and the top-k
  indices go to the decode kernel as ``(1, nheads_k, 1, topk)``.  A decode step then selects and attends exactly as
  the prefill does for the last token of the same sequence, except at lengths L with L % 16 == 15 or
  L % 64 == 63, where the causal Stage-1 rule of the prefill (truncating division, mask.h:273-281) hides the newest
  compressed key from the last token.
"""
from __future__ import annotations

from dataclasses import dataclass

import torch

from . import _lib
from .attention import HEAD_DIM, attend_varlen, infllmv2_attn_with_kvcache, pad_head_dim
from .selection import compress_keys, compress_keys_cache


@dataclass
class SequenceCache:
    """K/V cache of one sequence plus its compressed keys.  ``length`` tokens are valid."""
    k: torch.Tensor                  # (1, capacity, nheads_k, d)
    v: torch.Tensor
    k_fine: torch.Tensor             # (capacity // stride, nheads_k, d): stride-16 compressed keys
    k_coarse: torch.Tensor           # (capacity // (4 * stride), nheads_k, d)
    length: int = 0

    @staticmethod
    def empty(capacity: int, nheads_k: int, head_dim: int, device, stride: int = 16, dtype=torch.bfloat16):
        z = lambda n: torch.zeros((n, nheads_k, head_dim), dtype=dtype, device=device)
        return SequenceCache(z(capacity).unsqueeze(0), z(capacity).unsqueeze(0), z(capacity // stride + 1),
                             z(capacity // (4 * stride) + 1), 0)


@dataclass
class BatchCache:
    """K/V caches of a batch of sequences plus their compressed keys, for batched decoding.  All lengths live on the
    device (no host read per step); ``max_length`` is the host's upper bound of ``lengths``."""
    k: torch.Tensor                  # (batch, capacity, nheads_k, d)
    v: torch.Tensor
    k_fine: torch.Tensor             # (batch, capacity // stride + 1, nheads_k, d)
    k_coarse: torch.Tensor           # (batch, capacity // (4 * stride) + 1, nheads_k, d)
    lengths: torch.Tensor            # int32 (batch,): tokens held per sequence
    fine_lens: torch.Tensor          # int32 (batch,): rows of k_fine that are valid
    coarse_lens: torch.Tensor
    max_length: int = 0

    @staticmethod
    def empty(batch: int, capacity: int, nheads_k: int, head_dim: int, device, stride: int = 16, dtype=torch.bfloat16):
        z = lambda n: torch.zeros((batch, n, nheads_k, head_dim), dtype=dtype, device=device)
        i = lambda: torch.zeros(batch, dtype=torch.int32, device=device)
        return BatchCache(z(capacity), z(capacity), z(capacity // stride + 1), z(capacity // (4 * stride) + 1),
                          i(), i(), i(), 0)


def _dense(x):
    return x if x.stride(-1) == 1 else x.contiguous()


class InfLLMv2Attention(torch.nn.Module):
    """Sparse attention over 64-token key blocks chosen per query token and KV head (no parameters).

    ``selection`` picks the branch a model layer runs: ``"sparse"`` (default) scores the compressed keys and takes the
    top-k blocks; ``"window"`` attends only the forced blocks (the first ``init_blocks`` and the query's own block with
    the ``local_blocks`` before it: a sliding window in 64-token blocks plus attention sinks, no scoring at all);
    ``"dense"`` attends everything.  Sequences of at most ``dense_len`` tokens are dense whatever the branch."""

    def __init__(self, topk: int = 64, local_blocks: int = 31, init_blocks: int = 1, dense_len: int = 0,
                 kernel_size: int = 32, stride: int = 16, block_size: int = 64, softmax_scale: float | None = None,
                 selection: str = "sparse"):
        super().__init__()
        if selection not in ("sparse", "window", "dense"):
            raise ValueError("selection must be 'sparse', 'window' or 'dense'")
        self.selection = selection
        self.topk, self.local_blocks, self.init_blocks = topk, local_blocks, init_blocks
        self.dense_len = dense_len
        self.kernel_size, self.stride, self.block_size = kernel_size, stride, block_size
        self.softmax_scale = softmax_scale

    def _window_blocks(self, nheads_k: int, rows: int, cu_seqlens_q, positions, max_seqlen_q: int, max_position: int):
        """The forced blocks alone as a selection: what the pooling operator marks +inf, with every other block
        dropped.  ``rows``: packed query tokens; ``positions`` int32 (batch) or None: tokens before each sequence's
        first query.  Returns ``(topk_idx, block_mask)`` with ``init_blocks + local_blocks + 1`` index slots."""
        return _lib.host.window_blocks(nheads_k, rows, cu_seqlens_q, positions, max_seqlen_q, max_position, self.local_blocks,
                                       self.init_blocks, self.block_size)

    # ---- prefill / training ----
    def forward(self, q, k, v, cu_seqlens, max_seqlen: int, cache: SequenceCache | None = None):
        """q ``(total, nheads, d)``, k/v ``(total, nheads_k, d)`` packed; returns ``(total, nheads, d)``.
        With ``cache`` (one sequence only) the keys, values and compressed keys are also stored for decoding."""
        topk_idx = mask = images = None
        if self.selection == "window" and max_seqlen > self.dense_len:
            topk_idx, mask = self._window_blocks(k.shape[1], q.shape[0], cu_seqlens, None, max_seqlen, 0)
        elif self.selection == "sparse" and max_seqlen > self.dense_len:
            if self.topk < 1:
                raise RuntimeError("topk: the sparse selection takes at least one block per row")
            # the selection writes the packed mask Stage 2 walks, no list, and the block images of k and v
            scale = q.shape[-1] ** (-0.5) if self.softmax_scale is None else self.softmax_scale
            qs, ks = (q, k) if q.shape[-1] == HEAD_DIM else pad_head_dim(q, k)
            topk_idx, mask, images = _lib.host.select_mask(qs.detach(), ks.detach(), v.detach(), cu_seqlens, max_seqlen, self.topk, self.local_blocks,
                                                           self.init_blocks, scale, self.kernel_size, self.stride, self.block_size)
        out = attend_varlen(q, k, v, cu_seqlens, cu_seqlens, max_seqlen, max_seqlen, softmax_scale=self.softmax_scale, causal=True, topk_idx=topk_idx,
                            block_mask=mask, alike=self.selection == "window", images=images)
        if cache is not None:
            if cu_seqlens.numel() != 2:
                raise RuntimeError("a SequenceCache holds one sequence")
            n = k.shape[0]
            cache.k[0, :n], cache.v[0, :n] = k.detach(), v.detach()
            cache.length = n
            self._extend_compressed(cache, 0)
        return out

    def _extend_compressed(self, cache: SequenceCache, old_length: int):
        """Brings the compressed keys up to ``cache.length`` tokens; only windows completed since ``old_length`` are
        computed."""
        n = cache.length
        cu = torch.tensor([0, n], dtype=torch.int32, device=cache.k.device)
        rows = lambda length, ks, st: (length - ks) // st + 1 if length >= ks else 0
        for buf, ks, st in ((cache.k_fine, self.kernel_size, self.stride),
                            (cache.k_coarse, 4 * self.kernel_size, 4 * self.stride)):
            if rows(n, ks, st) > rows(old_length, ks, st):
                compress_keys(cache.k[0, :n], cu, n, ks, st, out=buf, first_row=rows(old_length, ks, st))

    # ---- decode ----
    def _step(self, q, k_new, v_new, k, v, k_fine, k_coarse, lens, host_len, fine_lens, coarse_lens, max_len, window_mask):
        """One decode step: append, compressed keys, selection, attention.  ``window_mask()`` gives the block mask
        ``(batch, nheads_k, 1, words)`` of the window branch.  Returns the output and the lengths after the step (device)."""
        scale = q.shape[-1] ** (-0.5) if self.softmax_scale is None else self.softmax_scale
        step = (q, k_new, v_new, k, v, k_fine, k_coarse, lens, host_len, fine_lens, coarse_lens, max_len, self.kernel_size, self.stride,
                self.block_size)
        if self.selection == "sparse" and max_len > self.dense_len:
            return _lib.host.decode_sparse(*step, self.topk, self.local_blocks, self.init_blocks, scale)
        new, _ = _lib.host.decode_step(*step, 0, self.local_blocks, self.init_blocks, scale)
        mask = window_mask() if self.selection == "window" and max_len > self.dense_len else None
        return infllmv2_attn_with_kvcache(q, k, v, cache_seqlens=new, softmax_scale=self.softmax_scale, block_mask=mask), new

    def decode(self, q, k_new, v_new, cache: SequenceCache):
        """One token of one sequence: q ``(1, 1, nheads, d)``, k_new/v_new ``(1, 1, nheads_k, d)``.  Appends the token
        to the cache (K/V, and the compressed keys when a window completes), selects blocks and attends.  Returns
        ``(1, 1, nheads, d)``."""
        pos = cache.length                                     # position of the new token
        if pos >= cache.k.shape[1]:
            raise IndexError(f"index {pos} is out of bounds: the K/V cache holds {cache.k.shape[1]} tokens")
        n = pos + 1
        q, k_new, v_new = _dense(q), _dense(k_new), _dense(v_new)

        def window_mask():
            dev = q.device
            _, mask = self._window_blocks(cache.k.shape[2], 1, torch.tensor([0, 1], dtype=torch.int32, device=dev),
                                          torch.tensor([pos], dtype=torch.int32, device=dev), 1, pos)
            return mask.transpose(0, 1).unsqueeze(2).contiguous()

        out, _ = self._step(q, k_new, v_new, cache.k, cache.v, cache.k_fine.unsqueeze(0), cache.k_coarse.unsqueeze(0), None, pos, None, None,
                            n, window_mask)
        cache.length = n
        return out

    # ---- batched decode ----
    def fill_cache(self, cache: BatchCache, k, v, seqlens):
        """Stores packed keys/values ``(total, nheads_k, d)`` of ``len(seqlens)`` sequences (host list of lengths) in
        ``cache`` and builds their compressed keys, as after a prefill."""
        if len(seqlens) != cache.k.shape[0]:
            raise RuntimeError("one length per cached sequence")
        start = 0
        for b, n in enumerate(seqlens):
            cache.k[b, :n], cache.v[b, :n] = k[start:start + n].detach(), v[start:start + n].detach()
            start += n
        cache.lengths.copy_(torch.tensor(list(seqlens), dtype=torch.int32))
        cache.max_length = max(seqlens)
        for buf, lens, ks, st in ((cache.k_fine, cache.fine_lens, self.kernel_size, self.stride),
                                  (cache.k_coarse, cache.coarse_lens, 4 * self.kernel_size, 4 * self.stride)):
            compress_keys_cache(cache.k, cache.lengths, ks, st, out=buf, out_lens=lens)

    def decode_batch(self, q, k_new, v_new, cache: BatchCache):
        """One token for every sequence of the batch: q ``(batch, 1, nheads, d)``, k_new/v_new
        ``(batch, 1, nheads_k, d)``.  Per sequence exactly what :meth:`decode` does, in a fixed number of launches
        for the whole batch and without reading anything back to the host: append, extend the compressed keys where a
        window completes, Stage 1 over each sequence's compressed-key cache, pooling at the sequence's own position,
        top-k, split decode attention.  Returns ``(batch, 1, nheads, d)``."""
        batch = q.shape[0]
        if cache.max_length + 1 > cache.k.shape[1]:
            raise RuntimeError("the K/V cache is full")
        q, k_new, v_new = _dense(q), _dense(k_new), _dense(v_new)

        def window_mask():
            cu_one = torch.arange(batch + 1, dtype=torch.int32, device=q.device)
            _, mask = self._window_blocks(cache.k.shape[2], batch, cu_one, cache.lengths, 1, cache.max_length)
            return mask.transpose(0, 1).unsqueeze(2).contiguous()                    # (Hk, batch, words) -> (batch, Hk, 1, words)

        out, new = self._step(q, k_new, v_new, cache.k, cache.v, cache.k_fine, cache.k_coarse, cache.lengths, 0, cache.fine_lens,
                              cache.coarse_lens, cache.max_length + 1, window_mask)
        cache.lengths = new
        cache.max_length += 1
        return out
