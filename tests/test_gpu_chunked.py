"""Recurrences over prompt portions in chunks of 64 tokens (chunked.hip) against the recurrence token by token in 64 bits, and
beside the token-by-token kernels of the same sums in 32 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def plain(q, k, v, decay, gain, delta, S):
    """One request in 64 bits: q, k [n, H, D], v [n, H, V], decay and gain [n, H], S [H, D, V]."""
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = decay[t, :, None, None] * S
        u = v[t] - (k[t, :, None] @ S)[:, 0] if delta else v[t]
        S = S + k[t, :, :, None] * (gain[t, :, None] * u)[:, None]
        out[t] = (q[t, :, None] @ S)[:, 0]
    return out, S


# delta, groups, heads, dim, vdim, rows a request, rows before (0: from nothing), chunks of scratch, one decay a head
CASES = [
    (True, 2, 2, 128, 128, [128], [0], 64, False),              # the fewest rows, whole chunks
    (True, 1, 2, 64, 48, [129, 1, 191, 64], [5, 3, 0, 0], 64, False),    # ragged ends, rows that go token by token between
    (True, 2, 4, 128, 16, [500, 300], [0, 7], 3, False),        # a scratch that the step goes through in turns
    (True, 1, 1, 64, 64, [256] + [1] * 70, [0] * 71, 64, False),   # more requests than a wave has lanes
    (False, 2, 2, 128, 128, [128], [0], 64, True),
    (False, 1, 3, 64, 48, [129, 1, 191, 64], [5, 3, 0, 0], 64, False),
    (False, 2, 8, 128, 64, [500, 300], [0, 7], 3, False),
    (False, 1, 16, 64, 16, [4500], [9], 64, False),             # more chunks than a buffer; heads that share k . q
]


@pytest.mark.parametrize("case", CASES)
def test_against_token_by_token(case):
    from dinfer_amd.kernels import ops
    delta, G, H, D, V, new, before, chunks, fixed = case
    g = torch.Generator().manual_seed(sum(new) + D)
    T, B = sum(new), len(new)
    cu = [0]
    for n in new:
        cu.append(cu[-1] + n)
    unit = torch.nn.functional.normalize
    # neighbouring keys alike, so that the triangular system is far from the identity; a decay of zero, and some of one
    k = torch.randn(T, G, D, generator=g)
    k[1::2] = k[0::2][:k[1::2].shape[0]] + 0.5 * k[1::2]
    k, q = unit(k, dim=-1), unit(torch.randn(T, G, D, generator=g), dim=-1)
    v = torch.randn(T, H, V, generator=g)
    gain = torch.rand(T, H, generator=g)
    decay = 1 - 0.2 * torch.rand(T, H, generator=g) ** 2
    if fixed:
        decay = torch.tensor([1.0, 0.97]).expand(T, H).contiguous()
        gain = torch.ones(T, H)
    else:
        decay[T // 2, 0] = 0.0
        decay[T // 3:T // 3 + 20] = 1.0
    slots = torch.randperm(B + 2, generator=g)[:B]
    state0 = torch.randn(B + 2, H, V, D, generator=g)
    cols = ops.delta_work_columns(G, H, D, V)
    work = torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1), gain, decay], dim=1)
    work = torch.nn.functional.pad(work, (0, -(-cols // 4) * 4 - cols)).cuda()
    size = ops.chunk_scratch(delta, G, H, D, V, T, B)
    i32 = dict(dtype=torch.int32, device="cuda")
    common = dict(state_slots=slots.to(**i32), cu_seqlens=torch.tensor(cu, **i32),
                  seq_lens=torch.tensor([a + b for a, b in zip(new, before)], **i32), num_reqs=B, heads=H, dim=D, vdim=V)
    got = {}
    for chunked in (False, True):
        state = state0.cuda()
        out = torch.full((T + 1, H * V), 7.0, device="cuda")
        more = dict(tokens=T, scratch=torch.full((min(size[0], chunks), size[1]), float("nan"), device="cuda")) if chunked else {}
        if delta:
            ops.delta_recurrence(work, state, out, qk_heads=G, **common, **more)
        else:
            qk, ve = G * D, 2 * G * D + H * V
            ops.decay_recurrence(work[:, :qk], work[:, qk:2 * qk], work[:, 2 * qk:ve],
                                 decay[0].cuda() if fixed else work[:, ve + H:ve + 2 * H],
                                 None if fixed else work[:, ve:ve + H], state, out, groups=G, **common, **more)
        torch.cuda.synchronize()
        assert (out[T] == 7.0).all()
        got[chunked] = out[:T].double().cpu(), state.double().cpu()
    rep = H // G
    q, k = q.double().repeat_interleave(rep, 1), k.double().repeat_interleave(rep, 1)
    v, gain, decay = v.double(), gain.double(), decay.double()
    want, want_state = torch.empty(T, H * V, dtype=torch.float64), state0.double()
    for b in range(B):
        s = slice(cu[b], cu[b + 1])
        S = state0[slots[b]].double().transpose(1, 2) if before[b] else torch.zeros(H, D, V, dtype=torch.float64)
        o, S = plain(q[s], k[s], v[s], decay[s], gain[s], delta, S)
        want[s] = o.reshape(-1, H * V)
        want_state[slots[b]] = S.transpose(1, 2)
    for i, w in ((0, want), (1, want_state)):
        # both forms round each product and each partial sum to 2^-24 of itself: some 2 log2(D) roundings of a sum over D in
        # trees, as many of a sum over a chunk; and the chunked form is to be no further off than the other
        top = w.abs().max().item()
        worst, rms = {}, {}
        for c in got:
            e = (got[c][i] - w) / top
            worst[c], rms[c] = e.abs().max().item(), e.pow(2).mean().sqrt().item()
        assert worst[True] < 4 * (7 + 6) * 2.0 ** -24, (worst, rms)
        assert rms[True] <= 1.02 * rms[False], (worst, rms)


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("G,H,D,V,B", [(1, 2, 128, 128, 3), (2, 4, 68, 40, 1), (1, 3, 100, 9, 70), (2, 2, 128, 33, 5), (1, 1, 64, 32, 2)])
def test_single_rows_have_the_same_bits(delta, G, H, D, V, B):
    """A step of single rows, told so, against the kernel for any rows: the same arithmetic, so the same bits; columns that fill
    no workgroup, heads that fill no half wave, a request that starts from nothing."""
    from dinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(D + V)
    cols = ops.delta_work_columns(G, H, D, V) + 3
    work = torch.rand(B, cols, generator=g).cuda()
    state0 = torch.randn(B + 2, H, V, D, generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    common = dict(state_slots=torch.randperm(B + 2, generator=g)[:B].to(**i32), cu_seqlens=torch.arange(B + 1, **i32),
                  seq_lens=torch.tensor([1 + b % 3 for b in range(B)], **i32), num_reqs=B, heads=H, dim=D, vdim=V)
    got = []
    for told in (dict(), dict(tokens=B)):
        state, out = state0.cuda(), torch.full((B + 1, H * V), 7.0, device="cuda")
        if delta:
            ops.delta_recurrence(work, state, out, qk_heads=G, **common, **told)
        else:
            qk, ve = G * D, 2 * G * D + H * V
            ops.decay_recurrence(work[:, :qk], work[:, qk:2 * qk], work[:, 2 * qk:ve], work[:, ve + H:ve + 2 * H], work[:, ve:ve + H],
                                 state, out, groups=G, **common, **told)
        got.append((out, state))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("rows,tokens", [
    ([100], 200),            # a lone request of fewer rows than the step is long: it is not left out
    ([1], 128), ([128], 128), ([70], 4300),
    ([2, 0, 1], 3),          # as many rows as requests, but not one each
    ([0, 0, 3, 1, 1], 5),
])
def test_steps_longer_than_their_rows(delta, rows, tokens):
    """`tokens` says how long a step may be; what a request gets follows its own rows."""
    from dinfer_amd.kernels import ops
    G, H, D, V, B = 1, 2, 128, 32, len(rows)
    g = torch.Generator().manual_seed(sum(rows) + tokens)
    work = torch.rand(tokens, ops.delta_work_columns(G, H, D, V) + 2, generator=g) / 8
    state0 = torch.randn(B + 1, H, V, D, generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    cu = torch.tensor([0] + rows).cumsum(0)
    common = dict(state_slots=torch.arange(B, **i32), cu_seqlens=cu.to(**i32), seq_lens=torch.tensor([9 + n for n in rows], **i32),
                  num_reqs=B, heads=H, dim=D, vdim=V)
    size = ops.chunk_scratch(delta, G, H, D, V, 4300, B)
    got = []
    for more in (dict(), dict(tokens=tokens, scratch=torch.zeros(size, device="cuda"), one_row_each=False)):
        w, state, out = work.cuda(), state0.cuda(), torch.full((tokens, H * V), 7.0, device="cuda")
        w = torch.nn.functional.pad(w, (0, -w.shape[1] % 4))
        if delta:
            ops.delta_recurrence(w, state, out, qk_heads=G, **common, **more)
        else:
            qk, ve = G * D, 2 * G * D + H * V
            ops.decay_recurrence(w[:, :qk], w[:, qk:2 * qk], w[:, 2 * qk:ve], w[:, ve + H:ve + 2 * H], w[:, ve:ve + H], state, out, groups=G,
                                 **common, **more)
        got.append((out, state))
    # (both in 32 bits, sums of 128 products in two orders)
    for a, b in zip(*got):
        torch.testing.assert_close(b, a, rtol=1e-5, atol=1e-5 * a.abs().max().item())
    assert (got[1][0][sum(rows):] == 7.0).all()


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [64 + 21, 64 + 15, 0, 130])
@pytest.mark.parametrize("what", ["q", "k", "v", "gain", "decay", "state"])
@pytest.mark.parametrize("delta,D,V", [(True, 128, 32), (False, 128, 16), (True, 64, 16), (False, 64, 16)])
def test_a_bad_number_stays_with_what_follows_it(delta, D, V, what, at, bad):
    """An infinity or NaN of one token: what the token-by-token kernel leaves finite is finite and the same in chunks, and what it
    does not is not; the tokens before it, in its own block of 16 and chunk of 64 too, keep their numbers."""
    from dinfer_amd.kernels import ops
    G, H, T = 2, 2, 150
    g = torch.Generator().manual_seed(at + D)
    unit = torch.nn.functional.normalize
    q, k = (unit(torch.randn(T, G, D, generator=g), dim=-1) for _ in range(2))
    v, gain, decay = torch.randn(T, H, V, generator=g), 0.2 + 0.8 * torch.rand(T, H, generator=g), 1 - 0.1 * torch.rand(T, H, generator=g)
    state0 = torch.randn(1, H, V, D, generator=g)
    {"q": q[at, 1], "k": k[at, 1], "v": v[at, 1], "gain": gain[at], "decay": decay[at], "state": state0[0, 1, 3]}[what][1] = bad
    cols = ops.delta_work_columns(G, H, D, V)
    work = torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1), gain, decay], dim=1)
    work = torch.nn.functional.pad(work, (0, -(-cols // 4) * 4 - cols)).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    common = dict(state_slots=torch.zeros(1, **i32), cu_seqlens=torch.tensor([0, T], **i32), seq_lens=torch.tensor([T + 5], **i32), num_reqs=1,
                  heads=H, dim=D, vdim=V)
    got = []
    for more in (dict(), dict(tokens=T, scratch=torch.zeros(ops.chunk_scratch(delta, G, H, D, V, T, 1), device="cuda"))):
        state, out = state0.cuda(), torch.full((T, H * V), 7.0, device="cuda")
        if delta:
            ops.delta_recurrence(work, state, out, qk_heads=G, **common, **more)
        else:
            qk, ve = G * D, 2 * G * D + H * V
            ops.decay_recurrence(work[:, :qk], work[:, qk:2 * qk], work[:, 2 * qk:ve], work[:, ve + H:ve + 2 * H], work[:, ve:ve + H], state, out,
                                 groups=G, **common, **more)
        got.append((out, state))
    for want, have in zip(*got):
        fine = torch.isfinite(want)
        assert torch.equal(fine, torch.isfinite(have))
        torch.testing.assert_close(have[fine], want[fine], rtol=1e-5, atol=1e-5)     # (32 bits, two orders)
    if what != "state":
        assert torch.isfinite(got[1][0][:at]).all() and not torch.isfinite(got[1][0]).all()


@pytest.mark.parametrize("delta", [True, False])
@pytest.mark.parametrize("rows,max_rows,calls_made", [([18] * 16, 18, 1), ([127, 3], 127, 1), ([127, 3], None, 2), ([128, 3], 128, 2)])
def test_steps_of_short_portions_launch_nothing_for_long_ones(monkeypatch, delta, rows, max_rows, calls_made):
    """Where the longest portion is known to be short, nothing of the chunked form is launched; the results are the same bits."""
    from dinfer_amd.kernels import lib, ops
    G, H, D, V, B, T = 1, 2, 64, 32, len(rows), sum(rows)
    g = torch.Generator().manual_seed(T)
    cols = -(-ops.delta_work_columns(G, H, D, V) // 4) * 4
    work = (torch.rand(T, cols, generator=g) / 8).cuda()
    state0 = torch.randn(B + 1, H, V, D, generator=g)
    i32 = dict(dtype=torch.int32, device="cuda")
    common = dict(state_slots=torch.arange(B, **i32), cu_seqlens=torch.tensor([0] + rows).cumsum(0).to(**i32),
                  seq_lens=torch.tensor([5 + n for n in rows], **i32), num_reqs=B, heads=H, dim=D, vdim=V, one_row_each=False, tokens=T,
                  scratch=torch.zeros(ops.chunk_scratch(delta, G, H, D, V, T, B), device="cuda"))
    calls, call, got = [], lib.call, []
    monkeypatch.setattr(lib, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    for more in (dict(), dict(max_rows=max_rows)):
        state, out = state0.cuda(), torch.zeros(T, H * V, device="cuda")
        calls.clear()
        if delta:
            ops.delta_recurrence(work, state, out, qk_heads=G, **common, **more)
        else:
            qk, ve = G * D, 2 * G * D + H * V
            ops.decay_recurrence(work[:, :qk], work[:, qk:2 * qk], work[:, 2 * qk:ve], work[:, ve + H:ve + 2 * H], work[:, ve:ve + H],
                                 state, out, groups=G, **common, **more)
        got.append((out, state))
    assert len(calls) == calls_made
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
