"""Latent attention with the heads' keys and values made again (csrc/latent_expand.hip), and which steps take it."""
import random
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from dinfer_amd.kernels import latent, ops
from dinfer_amd.parts import DecoderModel
from dinfer_amd.parts.latent_attention import LatentAttention
from dinfer_amd.parts.spec import part

DEV = "cuda"


def made(heads, rank, chunks):
    ex = latent.Expanded.__new__(latent.Expanded)
    ex.heads, ex.rank, ex.chunks = heads, rank, chunks
    return ex


def test_many_rows_a_request_take_the_keys_side_and_few_do_not():
    ex = made(16, 512, 65536 // 16)
    for starts, counts in (([1000] * 16, [256] * 16), ([0] * 16, [130] * 16), ([0], [2048]), ([4000], [512]), ([12000], [130])):
        assert ex.plan(starts, counts) == [(0, len(counts), sum(starts) + sum(counts), max(counts))]
    for starts, counts in (([6000] * 16, [64] * 16), ([2000] * 64, [1] * 64), ([3000] * 31 + [1024], [1] * 31 + [512]), ([500] * 16, [18] * 16)):
        assert ex.plan(starts, counts) is None


def test_requests_are_dealt_to_launches_that_fit_the_scratch():
    ex, rng = made(16, 512, 300), random.Random(3)
    for _ in range(200):
        n = rng.randint(1, 9)
        starts, counts = [rng.randint(0, 900) for _ in range(n)], [rng.randint(128, 600) for _ in range(n)]
        launches = ex.plan(starts, counts)
        if launches is None:
            continue
        assert [f for f, *_ in launches] == [sum(r for _, r, *_ in launches[:i]) for i in range(len(launches))]
        assert sum(r for _, r, *_ in launches) == n
        for first, reqs, total, longest in launches:
            part = range(first, first + reqs)
            assert total == sum(starts[i] + counts[i] for i in part) and longest == max(counts[i] for i in part)
            assert sum(-(-(starts[i] + counts[i]) // 16) for i in part) <= total // 16 + reqs <= ex.chunks
    assert ex.plan([100], [300 * 16]) is None and ex.plan([0], [299 * 16]) is not None     # one that never fits


def test_lengths_that_are_not_known_are_not_used():
    ex = made(16, 512, 4096)
    step = SimpleNamespace(lengths_known=False, num_tokens=4096, num_reqs=16, notes={})
    assert ex.launches(step) is None and not step.notes


def test_scratch_holds_what_a_step_can_bring_and_no_more():
    sizes = {}
    def ctx(**kw):
        buffer = lambda name, cols, rows: sizes.__setitem__(name, (rows, cols))
        return SimpleNamespace(**{**dict(device=torch.device("cpu"), dtype=torch.bfloat16, max_tokens=2048, max_reqs=257, max_seq_len=1000,
                                         page_size=16, workspace=SimpleNamespace(buffer=buffer)), **kw})
    assert latent.Expanded(ctx(), 2, 512).chunks == 16 * 64          # of 257 requests 16 can bring 128 rows
    assert latent.Expanded(ctx(max_reqs=3), 2, 512).chunks == 3 * 64
    ex = latent.Expanded(ctx(max_seq_len=40960), 16, 512)
    assert 500 << 20 < sum(r * c * 2 for r, c in sizes.values()) <= 512 << 20 and sizes["latent_expanded_rot"] == (ex.chunks, 1024)
    assert latent.Expanded.supports(ctx(), 128, 64, 128, 512)
    for other in (dict(max_tokens=127), dict(dtype=torch.float32), dict(page_size=24)):
        assert not latent.Expanded.supports(ctx(**other), 128, 64, 128, 512)


@pytest.mark.parametrize("q_rank,gated,window,taken", [(96, "entries", None, True), (98, "entries", None, False), (98, True, None, True),
                                                       (None, "entries", None, True), (96, "entries", 64, False)])
def test_an_entry_gate_that_begins_anywhere_keeps_its_way(q_rank, gated, window, taken):
    position = part("rotary", theta=10000.0, max_positions=64, rotary_dim=64)
    mixer = LatentAttention(256, 4, 128, 64, 128, 128, 0.1, position, part("rmsnorm", eps=1e-6, weight_name=""), gated=gated, q_rank=q_rank,
                            window=window)
    assert mixer.may_expand == taken


@pytest.mark.gpu
@pytest.mark.parametrize("H,R,page,hist,new,gate", [
    (16, 512, 16, [1000, 0, 17, 255, 256, 5], [256, 300, 5, 257, 1, 250], "heads"),   # edges of tiles of 256 keys and rows, of pieces of 16
    (3, 128, 32, [33, 0], [200, 64], None), (4, 384, 8, [0, 700, 9], [15, 513, 7], "entries"), (5, 160, 64, [100], [300], "heads"),
    (2, 256, 16, [4000], [140], None),
    (4, 128, 1, [i % 3 for i in range(4000)], [1 + i % 2 for i in range(4000)], "heads"),   # more tiles a workgroup than it looks up at once
    (33, 128, 16, [700, 0, 31], [40, 1500, 2], None)])                                      # several tiles a workgroup, of keys and of values
def test_expanded_attention(H, R, page, hist, new, gate):
    g = torch.Generator().manual_seed(H + R)
    rn = lambda *s: torch.randn(*s, generator=g)
    total, T, B = [h + n for h, n in zip(hist, new)], sum(new), len(new)
    need = [-(-t // page) for t in total]
    order = list(range(sum(need) + 3))
    random.Random(R).shuffle(order)
    cache = rn(len(order), page, R + 64)
    cache[..., :R] /= cache[..., :R].pow(2).mean(-1, keepdim=True).sqrt()
    cache = cache.bfloat16()
    bt = torch.full((B, max(need) + 1), -1, dtype=torch.int32)
    for b, n in enumerate(need):
        bt[b, :n] = torch.tensor([order.pop() for _ in range(n)])
    for b in range(B):      # what a page holds past its request's keys is no number
        cache[bt[b, need[b] - 1], (total[b] - 1) % page + 1:] = float("nan")
    g_size = {None: 0, "heads": H, "entries": H * 128}[gate]
    width = -(-(24 + H * 192 + g_size) // 8) * 8
    proj = (rn(T, width) * 2).bfloat16()
    uk, uv = ((rn(H, 128, R) * R ** -0.5).bfloat16() for _ in range(2))
    qa = torch.full((T, H * (R + 64)), float("nan")).bfloat16()
    q = proj[:, 24:24 + H * 192].reshape(T, H, 192)
    qa.view(T, H, R + 64)[:, :, R:] = q[:, :, 128:]
    cu = torch.tensor([0] + torch.tensor(new).cumsum(0).tolist(), dtype=torch.int32)
    want, at = torch.empty(T, H, 128, dtype=torch.double), 0
    for b in range(B):
        rows = cache[bt[b, :need[b]].long()].reshape(-1, R + 64)[:total[b]].double()
        hidden = torch.arange(total[b])[None] > torch.arange(hist[b], total[b])[:, None]
        for h in range(H):
            k = torch.cat([rows[:, :R] @ uk[h].double().T, rows[:, R:]], 1)
            w = (q[at:at + new[b], h].double() @ k.T * 192 ** -0.5).masked_fill(hidden, float("-inf")).softmax(-1)
            want[at:at + new[b], h] = w @ (rows[:, :R] @ uv[h].double().T)
        at += new[b]
    if gate:
        z = torch.sigmoid(proj[:, 24 + H * 192:24 + H * 192 + g_size].double())
        want = want * (z[:, :, None] if gate == "heads" else z.view(T, H, 128))
    chunks = sum(total) // 16 + B
    room = lambda n: torch.full((chunks, n), float("nan"), device=DEV, dtype=torch.bfloat16)
    out = torch.full((T + 1, H * 128), 7.0, device=DEV, dtype=torch.bfloat16)
    keys, values, rot = room(H * 2048), room(H * 2048), room(1024)
    d = {n: t.to(DEV) for n, t in dict(proj=proj, qa=qa, uk=uk, uv=uv, cache=cache, bt=bt, cu=cu, sl=torch.tensor(total, dtype=torch.int32)).items()}
    assert ops.latent_expanded_supports(128, 64, 128, R, page)
    cut = B // 2     # in two launches: the second's scratch begins anew
    for first, n in ((0, B),) if cut == 0 else ((0, cut), (cut, B - cut)):
        mine = range(first, first + n)
        ops.latent_attn_expanded(d["proj"], d["qa"], d["uk"], d["uv"], out, d["cache"], d["bt"], d["cu"], d["sl"], n, sum(total[i] for i in mine),
                                 max(new[i] for i in mine), keys, values, rot, scale=192 ** -0.5, q_off=24, rank=R, page_size=page,
                                 gate=d["proj"] if gate else None, gate_off=24 + H * 192, gate_entries=gate == "entries", first=first)
    # rounded to 8 bits on the way: keys (a score of size 4 is off by 0.01 or so), weights, values, the result
    torch.testing.assert_close(out[:-1].double().cpu().view(T, H, 128), want, rtol=2e-2, atol=2e-2)
    assert (out[-1] == 7.0).all()


def step_of(starts, counts, known=True):
    cu, lens = np.concatenate([[0], np.cumsum(counts)]), np.add(starts, counts)
    return SimpleNamespace(lengths_known=known, num_tokens=sum(counts), num_reqs=len(counts), notes={}, h=dict(cu_seqlens=cu, seq_lens=lens))


def test_a_step_leaves_the_graphs_only_where_that_pays():
    """Eight heads over 512: a layer of 10 million weights is launched slower than it runs, unless the attention is long; one of 316 million
    never; and where the queries' side is the better one nothing is gained by launching."""
    ex = made(8, 512, 65536 // 16)
    wants = lambda step, weights: DecoderModel.wants_lengths(SimpleNamespace(_choices=[(ex, 8)], run=[None] * 8, _weights=weights), step)
    for starts, counts in (([0], [128]), ([0], [384]), ([0] * 8, [130] * 8), ([0, 0], [256, 256])):
        assert ex.plan(starts, counts) and not wants(step_of(starts, counts), 10e6) and wants(step_of(starts, counts), 316e6)
        assert not wants(step_of(starts, counts, known=False), 316e6)
    for starts, counts in (([0], [512]), ([1000], [128]), ([300] * 3, [200] * 3)):
        assert wants(step_of(starts, counts), 10e6)
    ex = made(16, 512, 65536 // 16)
    for starts, counts in (([3000] * 31 + [1024], [1] * 31 + [512]), ([100] * 4, [20] * 4), ([70000], [512])):   # few rows a request; no room
        assert ex.launches(step_of(starts, counts)) is None and not wants(step_of(starts, counts), 316e6)
    assert not DecoderModel.wants_lengths(SimpleNamespace(_choices=[], run=[None], _weights=10**9), step_of([0], [2048]))
