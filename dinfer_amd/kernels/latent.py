"""Chooses the latent-attention kernels for a step.

float32 storage: always the plain kernel (fixed key order, any sizes). bfloat16 storage: the MFMA kernel where the
sizes fit it (latent a multiple of 16 up to 512, rotated part a multiple of 8 up to 128, pages of a multiple of 8), with the keys of single rows cut into parts on the
device; the plain kernel otherwise.

Steps with many rows a request make the heads' keys and values again (Expanded) where the lengths of the requests are known and
that is the lesser work.
"""
from __future__ import annotations

import numpy as np
import torch

from . import ops

TARGET_WORKGROUPS = 256   # measured at 16 heads of 512 + 64, 2,048 keys: 64 requests are fastest with 4 parts, 8 with 16 to 32
MAX_SPLITS = 64
SHORTEST_PART = 128    # keys of the longest request in one part (its four waves take a quarter each), at least


class Workspace:
    """Geometry checks and the split-K scratch of one latent shape, sized once."""

    def __init__(self, ctx, heads: int, rank: int, rot_dim: int):
        self.heads, self.rank, self.rot_dim = heads, rank, rot_dim
        self.mfma = ctx.dtype == torch.bfloat16 and ops.latent_mfma_supports(rank, rot_dim, ctx.page_size)
        longest = ctx.max_seq_len or 4096
        self.max_splits = max(1, min(MAX_SPLITS, -(-longest // SHORTEST_PART)))
        self.part = None
        if self.mfma:
            units = max(self.splits(n) * n for n in range(1, ctx.max_reqs + 1)) * heads
            self.part = ctx.workspace.buffer("latent_partials", units * (rank + 4), dtype=torch.float32, rows=1)

    def splits(self, num_reqs: int) -> int:
        """Parts per request in a step of single rows: a function of the batch size only, so a captured graph stays valid."""
        tiles = -(-self.heads // 16)
        return max(1, min(self.max_splits, TARGET_WORKGROUPS // max(1, num_reqs * tiles)))


def paged_attention(qa: torch.Tensor, out: torch.Tensor, cache: torch.Tensor, cache_t, batch, group: int, ws: Workspace, *,
                    scale: float, window: int, heads: int, rank: int, rot_dim: int, page_size: int):
    """qa [T, heads * (rank + rot_dim)] -> out [T, heads * rank] (the attention's output in latent space)."""
    geo = dict(scale=scale, window=window, heads=heads, rank=rank, rot_dim=rot_dim, page_size=page_size)
    bt = batch.block_table[group]
    B, T = batch.num_reqs, batch.num_tokens
    if not ws.mfma:
        return ops.latent_attn_ref(qa, out, cache, bt, batch.cu_seqlens, batch.seq_lens, B, T, **geo)
    splits = ws.splits(B) if batch.all_decode else 1
    return ops.latent_attn_mfma(qa, out, cache, cache_t, bt, batch.cu_seqlens, batch.seq_lens, B, T, splits, ws.part, **geo)


EXPANDED_BYTES = 512 << 20     # scratch for expanded keys and values, at most: 32 or 64 thousand keys of 32 or 16 heads
EXPANDED_SHARE = 32            # and of the device's free memory: what is left is the cache's


class Expanded:
    """Attention over keys and values made again from the latents (csrc/latent_expand.hip): scratch, sized once and shared by the
    layers of one geometry, and the choice for a step."""

    ROWS = 128      # a request, from which on a step may gain
    cus = 256       # of the device

    def __init__(self, ctx, heads: int, rank: int):
        self.heads, self.rank = heads, rank
        per_chunk = 2 * heads * 4096 + 2048
        longest, room = ctx.max_seq_len or 4096, EXPANDED_BYTES
        if ctx.device.type == "cuda":
            room = min(room, torch.cuda.mem_get_info(ctx.device)[0] // EXPANDED_SHARE)
            self.cus = torch.cuda.get_device_properties(ctx.device).multi_processor_count
        # (no more requests than can bring ROWS rows each; a chunk at least, whose step then finds no room)
        self.chunks = max(1, min(min(ctx.max_reqs, ctx.max_tokens // self.ROWS) * (-(-longest // 16) + 1), room // per_chunk))
        buf = ctx.workspace.buffer
        self.keys, self.values = (buf(f"latent_expanded_{n}", heads * 2048, rows=self.chunks) for n in ("keys", "values"))
        self.rot = buf("latent_expanded_rot", 1024, rows=self.chunks)

    @staticmethod
    def supports(ctx, dim: int, rot_dim: int, vdim: int, rank: int) -> bool:
        return (ctx.dtype == torch.bfloat16 and ctx.max_tokens >= Expanded.ROWS
                and ops.latent_expanded_supports(dim, rot_dim, vdim, rank, ctx.page_size))

    def plan(self, starts, counts):
        """[(first request, requests, their keys, longest portion)] of the launches for requests of `counts` rows behind `starts`
        keys, or None where the queries' side is the better one (see weigh)."""
        planned = self.weigh(starts, counts)
        return planned and planned[0]

    def weigh(self, starts, counts):
        """(launches as plan() has them, us of the queries' side), or None.

        Both sides' times in us as measured with 16 heads of 128 + 64 over latents of 512. Queries' side: 77 ns a key of a round of
        256 workgroups of 64 (row, head) pairs and 15.5 ns a row for the products around them; keys' side: 5.5 ns a key
        and 2.3 us for 64 keys of 256 workgroups of 256 rows of a head, 1.7 where few run. 16 x 256 rows behind 1,000: 437
        and 164; 16 x 130 87 and 45, behind 500 179 and 96; 16 x 128 behind 2,000 321 and 268; 16 x 64 behind 6,000 457 and 735;
        2,048 rows from nothing 200 and 84; 512 behind 4,000 317 and 150."""
        starts, counts = np.asarray(starts, dtype=np.float64), np.asarray(counts, dtype=np.float64)
        scale = self.heads * self.rank / (16 * 512)
        ends, middle = starts + counts, starts + counts / 2
        groups = counts * self.heads / 64
        queries = 0.077 * self.rank / 512 * max((groups * middle).sum() / self.cus, ends.max()) + 0.0155 * scale * counts.sum()
        tiles = np.ceil(counts / 256) * self.heads
        keys = 0.0055 * scale * ends.sum() + max((tiles * middle).sum() / self.cus * 2.3, ends.max() * 1.7) / 64
        if keys > 0.9 * queries:
            return None
        lengths, rows = ends.astype(np.int64), counts.astype(np.int64)
        launches, first, total = [], 0, 0
        for i, n in enumerate(lengths.tolist()):
            if n // 16 + 1 > self.chunks:
                return None
            if i > first and (total + n) // 16 + i - first + 1 > self.chunks:
                launches.append((first, i - first, total, int(rows[first:i].max())))
                first, total = i, 0
            total += n
        launches.append((first, len(lengths) - first, total, int(rows[first:].max())))
        return launches, float(queries)

    def _weighed(self, batch):
        """weigh() of the step in `batch`, worked out once a step; None for a step whose lengths are not known."""
        if not batch.lengths_known or batch.num_tokens < self.ROWS * batch.num_reqs:
            return None
        key = ("latent", self.heads, self.rank, self.chunks)
        if key not in batch.notes:
            B = batch.num_reqs
            counts = np.diff(batch.h["cu_seqlens"][:B + 1])
            batch.notes[key] = self.weigh(batch.h["seq_lens"][:B] - counts, counts)
        return batch.notes[key]

    def launches(self, batch):
        """plan() of the step in `batch`."""
        weighed = self._weighed(batch)
        return weighed and weighed[0]

    def usual_way(self, batch):
        """us of the queries' side where the keys' side is better, else None (see Part.choices)."""
        weighed = self._weighed(batch)
        return weighed and weighed[1]

    def attention(self, launches, q, q_off: int, qa, uk, uv, out, cache, batch, group: int, *, scale: float, page_size: int, gate,
                  gate_off: int, gate_entries: bool):
        """out [T, heads * 128]: the gated outputs of the heads."""
        for first, reqs, total, longest in launches:
            ops.latent_attn_expanded(q, qa, uk, uv, out, cache, batch.block_table[group], batch.cu_seqlens, batch.seq_lens, reqs, total,
                                     longest, self.keys, self.values, self.rot, scale=scale, q_off=q_off, rank=self.rank,
                                     page_size=page_size, gate=gate, gate_off=gate_off, gate_entries=gate_entries, first=first)
        return out
