"""Chooses the attention kernels for a step.

float32 storage: the 32-bit matrix-core kernel for the head sizes it is built for, the plain kernel for all others; a
row's keys are visited in an order fixed by their positions in both.
bfloat16 storage: MFMA kernels where the geometry fits them (head size from the
instantiated list, page size a multiple of 8): split-K decode for the requests that
bring one row, flash for the others; the plain kernel otherwise.
"""
from __future__ import annotations

import torch

from . import ops

TARGET_WAVES = 1024   # split-K aims at about this many waves (measured: more, shorter waves cost more than they hide)
MAX_SPLITS = 128      # the kernels take up to 256
MIN_KEYS_PER_SPLIT = 512   # of the longest request the engine admits, beyond 32 parts
SHORTEST_PART = 64         # keys of the longest request in one part, at least


class Workspace:
    """Geometry checks and the split-K scratch of one attention shape, sized once."""

    def __init__(self, ctx, heads: int, kv_heads: int, head_dim: int):
        self.max_reqs = ctx.max_reqs
        # measured on MI355X (head 128, 8 kv heads): one request of 2k-4k keys is fastest with 32 parts,
        # of 32k with 64, of 128k with 128; the count may not depend on the lengths of a step (a captured
        # graph must stay valid), so it is bounded by the longest request the engine admits
        longest = ctx.max_seq_len or 4096
        self.max_splits = min(MAX_SPLITS, max(32, longest // MIN_KEYS_PER_SPLIT))
        # an engine for short requests: no part shorter than 64 keys of the longest, so up to 256 keys there are at
        # most four parts, which meet inside the workgroup and need no merge kernel (28 layers of 1,024 wide, 256
        # keys: 1.17 -> 1.0x ms a step at one request)
        self.max_splits = max(1, min(self.max_splits, -(-longest // SHORTEST_PART)))
        self.mfma = (ctx.dtype == torch.bfloat16 and ops.attn_mfma_supports(head_dim, ctx.page_size, heads, kv_heads))
        self.f32 = ctx.dtype == torch.float32 and ops.attn_f32_supports(head_dim, ctx.page_size, heads, kv_heads)
        self.split_k = self.mfma and heads // kv_heads <= 16
        self.part = None
        self.kv_heads = kv_heads
        # a step of single rows: the split-K kernel can take the per-head norms, the rotation and the cache write along
        self.decode_takes_post = self.split_k and ops.attn_decode_post_supports(head_dim)
        if self.split_k:
            max_units = max(max(self.splits(n), self.splits_beside(n)) * n for n in range(1, ctx.max_reqs + 1)) * kv_heads
            elems = max_units * (heads // kv_heads) * (head_dim + 4)
            self.part = ctx.workspace.buffer("attn_partials", elems, dtype=torch.float32, rows=1)

    def splits(self, num_reqs: int) -> int:
        """Parts per request: a function of the batch size only, so a captured graph stays valid."""
        return max(1, min(self.max_splits, TARGET_WAVES // (num_reqs * self.kv_heads)))

    def splits_beside(self, num_reqs: int) -> int:
        """The same where at least one of the requests brings a longer run of rows: the others are cut as a step of their own where
        their parts then come to the waves aimed at exactly. 8 kv heads, us cut with the others and without: 8 rows of 900 keys
        15.7 and 13.3, 16 of 2,458 33.7 and 32.8, 32 of 900 27.7 and 25.4, 64 of 2,458 124 and 112; parts that come to
        fewer waves go either way (5 rows of 2,458 20.0 and 18.7, 7 21.2 and 22.6, 10 of 900 15.1 and 15.7)."""
        singles = max(num_reqs - 1, 1)
        return self.splits(singles if TARGET_WAVES % (singles * self.kv_heads) == 0 else num_reqs)


def decode_with_post(qkv, out, k_cache, v_cache, batch, group: int, ws: Workspace, *, write: bool, **kw):
    """A step in which every request brings one row (ws.decode_takes_post): norms, rotation, cache write and attention
    in one kernel (and the merge of its parts). kw: geometry, norm and rotation as ops.attn_decode_post takes them."""
    B = batch.num_reqs
    return ops.attn_decode_post(qkv, out, ws.part, k_cache, v_cache, batch.block_table[group], batch.seq_lens, B,
                                ws.splits(B), slot_mapping=batch.slot_mapping[group] if write else None, **kw)


def paged_attention(qkv: torch.Tensor, out: torch.Tensor, k_cache, v_cache, batch, group: int, ws: Workspace, *,
                    scale: float, window: int, heads: int, kv_heads: int, head_dim: int, page_size: int):
    """q is read from the first heads*head_dim columns of qkv; out [T, heads*head_dim]."""
    geo = dict(scale=scale, window=window, heads=heads, kv_heads=kv_heads, head_dim=head_dim, page_size=page_size)
    bt = batch.block_table[group]
    B, T = batch.num_reqs, batch.num_tokens
    # (requests are the y of that kernel's grid)
    if ws.f32 and B <= 65535 and all(t.stride(0) % 4 == 0 and t.data_ptr() % 16 == 0 for t in (qkv, out)):
        return ops.attn_f32(qkv, out, k_cache, v_cache, bt, batch.cu_seqlens, batch.seq_lens, B, T, batch.max_q_len, **geo)
    if not ws.mfma:
        return ops.attn_paged_ref(qkv, out, k_cache, v_cache, bt, batch.cu_seqlens, batch.seq_lens, B, T, **geo)
    singles = batch.num_singles if ws.split_k else 0
    # a few single rows beside long portions are not worth two more launches
    use_decode = singles == B or singles >= 4
    if use_decode:
        ops.attn_decode(qkv, out, ws.part, k_cache, v_cache, bt, None if singles == B else batch.cu_seqlens,
                        batch.seq_lens, B, ws.splits(B) if singles == B else ws.splits_beside(B), **geo)
        if singles == B:
            return out
    return ops.attn_flash(qkv, out, k_cache, v_cache, bt, batch.cu_seqlens, batch.seq_lens, B, T, batch.max_q_len,
                          skip_single=use_decode, **geo)
