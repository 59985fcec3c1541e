"""The experts' and heads' products of many rows (csrc/grouped.hip) at the edges of their tiles, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def act(z, name):
    return {None: lambda x: x, "silu": lambda x: x * torch.sigmoid(x), "relu2": lambda x: torch.relu(x) ** 2,
            "gelu": lambda x: torch.nn.functional.gelu(x)}[name](z)


def close(out, want):
    """bfloat16 results of float sums: half a unit of 2^-8 of the value, and sums of K products of size one that carry at
    most K 2^-24 each, far below."""
    err = (out.double() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 2e-3).all(), f"off by {err.max().item()}"


# rows an expert gets: none, one, the edges of blocks of 32 and of tiles of 128
COUNTS = [0, 1, 31, 32, 33, 64, 65, 96, 127, 0, 128, 129, 160, 300]


def sorted_entries(counts, top, tokens, seed):
    """A list of choices in which expert e is chosen counts[e] times, in a random order; entry i belongs to token i // top."""
    flat = torch.tensor([e for e, c in enumerate(counts) for _ in range(c)], dtype=torch.int32)
    g = torch.Generator().manual_seed(seed)
    return flat[torch.randperm(flat.numel(), generator=g)]


# columns: fewer than a wave's, two waves beside two, a last wave in part, no whole 16-byte pieces, several workgroups
# K: one piece, a step and a piece, whole steps, a part of a step
@pytest.mark.parametrize("N,K,kind", [(40, 8, None), (128, 72, "silu"), (130, 64, "gelu"), (256, 136, "relu2"), (300, 128, None),
                                      (1408, 256, "gelu"), (24, 64, "gated"), (64, 200, "gated"), (72, 64, "gated"), (132, 328, "gated")])
def test_experts_of_many_rows(N, K, kind):
    from dinfer_amd.kernels import ops
    E, n = len(COUNTS), sum(COUNTS)
    top = 3
    idx = sorted_entries(COUNTS, top, n, N)
    tokens = -(-n // top)
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(tokens, K, generator=g, device=DEV).to(torch.bfloat16)
    gated = kind == "gated"
    w = (torch.randn(E, 2 * N if gated else N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device=DEV)
    perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.zeros((ops.moe_max_tiles(n, E, 16), 2), **i32)
    rows = ops.moe_tile_rows(torch.bfloat16, n, E, K, K)
    assert rows == 128
    ops.moe_scatter(idx.to(DEV), n, E, offsets, perm, tiles, rows)
    scale = torch.rand(n, generator=g, device=DEV) + 0.5
    for row_scale in (None, scale):
        for to_perm in (True, False):
            out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
            ops.experts_nt(x, w, out, n, tiles, offsets, perm, gated=gated, a_div=top, c_to_perm=to_perm, tile_rows=rows,
                           act=None if gated else kind, row_scale=row_scale)
            e = idx.to(DEV).long()
            y = torch.empty(n, w.shape[1], dtype=torch.float64, device=DEV)
            for k in range(E):
                at = (e == k).nonzero().flatten()
                y[at] = x[at // top].double() @ w[k].double().T
            if row_scale is not None:
                y = y * row_scale.double()[:, None]
            want = act(y[:, :N], "silu") * y[:, N:] if gated else act(y, kind)
            close(out, want if to_perm else want[perm.long()])
    # the second product's form: the rows of A are the sorted places themselves
    if not gated:
        out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
        a = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
        ops.experts_nt(a, w, out, n, tiles, offsets, perm, gated=False, a_div=0, c_to_perm=True, tile_rows=rows)
        for k in range(E):
            places = slice(int(offsets[k]), int(offsets[k + 1]))
            close(out[perm[places].long()], a[places].double() @ w[k].double().T)


@pytest.mark.parametrize("gate", [None, "head", "entry"])
@pytest.mark.parametrize("M,N,K,extra", [(17, 128, 64, 0), (128, 512, 128, 0), (129, 96, 40, 8), (300, 260, 72, 0), (64, 33, 8, 5)])
def test_heads_of_many_rows(M, N, K, extra, gate):
    from dinfer_amd.kernels import ops
    H = 3
    g = torch.Generator(device=DEV).manual_seed(M)
    a = torch.randn(M, H * K + 8, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(H, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    out = torch.full((M, H * (N + extra)), 7.0, dtype=torch.bfloat16, device=DEV)
    gates = torch.randn(M, H * N, generator=g, device=DEV).to(torch.bfloat16)
    ops.heads_nt(a, 8, K, w, out, 0, N + extra, M, **({} if gate is None else dict(gate=gates, gate_entries=gate == "entry")))
    for h in range(H):
        want = a[:, 8 + h * K:8 + (h + 1) * K].double() @ w[h].double().T
        if gate == "head":
            want = want * torch.sigmoid(gates[:, h:h + 1].double())
        elif gate == "entry":
            want = want * torch.sigmoid(gates[:, h * N:(h + 1) * N].double())
        close(out[:, h * (N + extra):h * (N + extra) + N], want)
        assert (out[:, h * (N + extra) + N:(h + 1) * (N + extra)] == 7.0).all()


# few rows: up to 16 an expert (full tiles, one row, none), columns in part of a workgroup's 32, k in part of a step and in
# more steps than are in flight
@pytest.mark.parametrize("N,K,kind", [(32, 8, None), (33, 64, "silu"), (40, 72, "gelu"), (96, 520, "relu2"), (1408, 2048, None),
                                      (24, 64, "gated"), (70, 200, "gated"), (64, 1408, "gated")])
def test_experts_of_few_rows(N, K, kind):
    from dinfer_amd.kernels import ops
    counts = [0, 1, 16, 15, 2, 0, 9, 17, 3, 1]
    E, n, top = len(counts), sum(counts), 3
    idx = sorted_entries(counts, top, n, N)
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(-(-n // top), K, generator=g, device=DEV).to(torch.bfloat16)
    gated = kind == "gated"
    w = (torch.randn(E, 2 * N if gated else N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device=DEV)
    perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.zeros((ops.moe_max_tiles(n, E, 16), 2), **i32)
    rows = ops.moe_tile_rows(torch.bfloat16, n, E, K, K)
    assert rows == 16
    ops.moe_scatter(idx.to(DEV), n, E, offsets, perm, tiles, rows)
    out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.experts_nt(x, w, out, n, tiles, offsets, perm, gated=gated, a_div=top, c_to_perm=True, tile_rows=rows, act=None if gated else kind)
    e = idx.to(DEV).long()
    y = torch.stack([w[int(e[i])].double() @ x[i // top].double() for i in range(n)])
    close(out, act(y[:, :N], "silu") * y[:, N:] if gated else act(y, kind))


@pytest.mark.parametrize("M", [1, 5, 16])
def test_heads_of_few_rows(M):
    from dinfer_amd.kernels import ops
    H, N, K = 3, 72, 136
    g = torch.Generator(device=DEV).manual_seed(M)
    a = torch.randn(M, H * K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(H, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    out = torch.full((M, H * N), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.heads_nt(a, 0, K, w, out, 0, N, M)
    close(out, torch.cat([a[:, h * K:(h + 1) * K].double() @ w[h].double().T for h in range(H)], dim=1))


@pytest.mark.parametrize("entries,experts,real,tile_rows", [(1, 1, 1, 128), (63, 64, 64, 16), (1024, 65, 60, 128), (8193, 130, 130, 128), (20000, 200, 190, 32)])
def test_entries_are_sorted_by_expert(entries, experts, real, tile_rows):
    from dinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(entries)
    idx = (torch.rand(entries, generator=g) ** 2 * experts).to(torch.int32)
    most = -(-entries // tile_rows) + experts
    offsets, perm, tiles = (torch.full((n,), -7, dtype=torch.int32, device=DEV) for n in (experts + 1, entries + 1, 2 * most))
    ops.lib.call("dinfer_moe_scatter", idx.to(DEV).data_ptr(), entries, experts, tile_rows, offsets.data_ptr(), perm.data_ptr(),
                 tiles.data_ptr(), most, real, ops._stream())
    counts = torch.bincount(idx.long(), minlength=experts)
    off = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)])
    assert torch.equal(offsets.cpu().long(), off) and perm[entries].item() == -7
    p = perm[:entries].cpu().long()
    assert torch.equal(p.sort().values, torch.arange(entries))
    assert torch.equal(idx[p].long(), torch.arange(experts).repeat_interleave(counts))
    want = sorted((e, int(off[e]) + r) for e in range(real) for r in range(0, int(counts[e]), tile_rows))
    got = [tuple(t) for t in tiles.cpu().view(-1, 2).tolist()]
    assert sorted(t for t in got if t[0] >= 0) == want and len(got) == most


@pytest.mark.parametrize("places", [65504, 65505, 65535])
def test_work_lists_of_the_longest_length(places):
    """As many places as a grid has in y, and the last counts before: the tiles named by the last places are worked off."""
    from dinfer_amd.kernels import ops
    E, N, K, n = 3, 24, 16, 300
    g = torch.Generator(device=DEV).manual_seed(places)
    a = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.randn(E, N, K, generator=g, device=DEV).to(torch.bfloat16)
    out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
    offsets = torch.tensor([0, 100, 150, n], dtype=torch.int32, device=DEV)
    perm = torch.arange(n, dtype=torch.int32, device=DEV)
    tiles = torch.full((places, 2), -1, dtype=torch.int32)
    for at, tile in ((0, (0, 0)), (places // 2, (1, 100)), (places - 2, (2, 150)), (places - 1, (2, 278))):
        tiles[at] = torch.tensor(tile, dtype=torch.int32)
    tiles = tiles.to(DEV)
    ops.lib.call("dinfer_experts_nt", ops.dtype_code(a.dtype), 0, a.data_ptr(), K, w.data_ptr(), K, N * K, out.data_ptr(), N, N, K,
                 tiles.data_ptr(), places, 128, offsets.data_ptr(), perm.data_ptr(), 0, 1, 0, 0.0, 0.0, n, ops._stream())
    for e, (lo, hi) in enumerate(((0, 100), (100, 150), (150, n))):
        close(out[lo:hi], a[lo:hi].double() @ w[e].double().T)


@pytest.mark.parametrize("gated", [False, True])
def test_an_expert_of_more_than_2_gb(gated):
    from dinfer_amd.kernels import ops
    E, N, K, n = 2, 280008, 4096, 70
    g = torch.Generator(device=DEV).manual_seed(3)
    a = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
    w = torch.empty(E, N, K, dtype=torch.bfloat16, device=DEV)
    for e in range(E):
        for lo in range(0, N, 20000):
            w[e, lo:lo + 20000] = torch.randn(min(20000, N - lo), K, generator=g, device=DEV) / K ** 0.5
    i32 = dict(dtype=torch.int32, device=DEV)
    idx = (torch.arange(n, **i32) * 7 % 3 > 0).to(torch.int32)
    perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.zeros((ops.moe_max_tiles(n, E, 128), 2), **i32)
    rows = ops.moe_tile_rows(torch.bfloat16, n, E, K, K)
    assert rows == 128
    ops.moe_scatter(idx, n, E, offsets, perm, tiles, rows)
    cols = N // 2 if gated else N
    out = torch.full((n, cols), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.experts_nt(a, w, out, n, tiles, offsets, perm, gated=gated, a_div=1, c_to_perm=True, tile_rows=rows)
    pick = torch.cat([torch.arange(300), torch.arange(0, cols, 997), torch.arange(cols - 300, cols)]).to(DEV)
    for e in range(E):
        at = (idx == e).nonzero().flatten()
        y = a[at].double() @ w[e, pick].double().T
        if gated:
            y = act(y, "silu") * (a[at].double() @ w[e, pick + cols].double().T)
        close(out[at][:, pick], y)


def test_rows_too_wide_for_32_bit_offsets_take_tiles_of_16():
    from dinfer_amd.kernels import ops
    wide = 2 ** 26
    assert ops.moe_tile_rows(torch.bfloat16, 1000, 2, wide - 8, 64) == 128
    assert ops.moe_tile_rows(torch.bfloat16, 1000, 2, wide, 64) == 16 and ops.moe_tile_rows(torch.bfloat16, 1000, 2, 64, wide) == 16


# the last k of the form for products that are soon over, and the first of the other; columns in part of a workgroup's, odd widths
@pytest.mark.parametrize("N,K,kind", [(33, 512, "silu"), (33, 520, None), (257, 584, "gelu"), (70, 256, "gated"), (70, 264, "gated"), (33, 328, "gated")])
def test_experts_of_few_rows_in_both_forms(N, K, kind):
    test_experts_of_few_rows(N, K, kind)


@pytest.mark.parametrize("M,N,K", [(16, 33, 512), (1, 33, 520), (9, 72, 1032), (16, 130, 584)])
def test_heads_of_few_rows_in_both_forms(M, N, K):
    from dinfer_amd.kernels import ops
    H = 3
    g = torch.Generator(device=DEV).manual_seed(M)
    a = torch.randn(M, H * K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(H, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    gates = torch.randn(M, H * N, generator=g, device=DEV).to(torch.bfloat16)
    for gate in (None, gates):
        out = torch.full((M, H * N + 1), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.heads_nt(a, 0, K, w, out, 0, N, M, **({} if gate is None else dict(gate=gate, gate_entries=True)))
        want = torch.cat([a[:, h * K:(h + 1) * K].double() @ w[h].double().T for h in range(H)], dim=1)
        close(out[:, :H * N], want if gate is None else want * torch.sigmoid(gate.double()))
        assert (out[:, H * N] == 7.0).all()


# rows of the result that do not begin at 16 bytes: odd widths, halves of a wave's columns, blocks of rows in part
@pytest.mark.parametrize("N,K,kind", [(257, 64, None), (65, 72, "silu"), (1001, 128, "relu2"), (33, 64, "gated"), (129, 72, "gated"), (508, 64, "gated")])
def test_experts_of_many_rows_and_odd_widths(N, K, kind):
    test_experts_of_many_rows(N, K, kind)


@pytest.mark.parametrize("gate", [None, "head", "entry"])
@pytest.mark.parametrize("M,N,K,extra", [(130, 257, 64, 0), (300, 127, 72, 0), (17, 511, 64, 3), (200, 130, 40, 0)])
def test_heads_of_many_rows_and_odd_widths(M, N, K, extra, gate):
    test_heads_of_many_rows(M, N, K, extra, gate)


# many tiles (the bound of the entries says so, not the rows that are there): workgroups walk them; columns in part of a workgroup's
# 256 and of a wave's, k in the fewest steps and in odd and even numbers
@pytest.mark.parametrize("N,K,kind,top,to_perm,factor", [
    (200, 192, None, 0, True, False), (256, 256, "gelu", 3, False, False), (33, 448, "silu", 3, True, True),
    (300, 192, "relu2", 0, False, False), (130, 320, "gated", 3, True, False), (72, 192, "clamped", 3, False, True), (600, 1408, None, 0, True, False)])
def test_experts_that_walk_their_tiles(N, K, kind, top, to_perm, factor):
    from dinfer_amd.kernels import ops
    E, n, gated = len(COUNTS), sum(COUNTS), kind in ("gated", "clamped")
    idx = sorted_entries(COUNTS, top, n, N).to(DEV)
    g = torch.Generator(device=DEV).manual_seed(N + K)
    a = torch.randn(-(-n // top) if top else n, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, 2 * N if gated else N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    scale = torch.rand(n, generator=g, device=DEV) if factor else None
    limit, slope = (0.7, 1.3) if kind == "clamped" else (0.0, 0.0)
    i32 = dict(dtype=torch.int32, device=DEV)
    perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.full((ops.moe_max_tiles(n, E, 16), 2), -1, **i32)
    ops.moe_scatter(idx, n, E, offsets, perm, tiles, 128)
    out = torch.full((n + 1, N), 7.0, dtype=torch.bfloat16, device=DEV)
    form = 1 if gated else {None: 0, "silu": 2, "gelu": 3, "relu2": 4}[kind]
    ops.lib.call("dinfer_experts_nt", ops.dtype_code(a.dtype), form, a.data_ptr(), K, w.data_ptr(), K, w.shape[1] * K, out.data_ptr(), N, N, K,
                 tiles.data_ptr(), tiles.shape[0], 128, offsets.data_ptr(), perm.data_ptr(), top, int(to_perm),
                 0 if scale is None else scale.data_ptr(), limit, slope, 704 * 128, ops._stream())
    assert (out[n] == 7.0).all()
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        entry = perm[lo:hi].long()
        rows = (a[entry // top] if top else a[lo:hi]).double()
        z = rows @ w[e].double().T
        if scale is not None:
            z = z * scale[entry].double()[:, None]
        if kind == "clamped":
            gate, up = z[:, :N].clamp(max=limit), z[:, N:].clamp(-limit, limit)
            want = gate * torch.sigmoid(slope * gate) * (up + 1)
        else:
            want = act(z[:, :N], "silu") * z[:, N:] if gated else act(z, kind)
        close(out[entry] if to_perm else out[lo:hi], want)


def test_a_walk_past_what_is_looked_up_at_once():
    """A work list with places left empty, and more tiles a workgroup than it keeps in mind (tiles named twice write the same)."""
    from dinfer_amd.kernels import ops
    E, N, K, n, places = 3, 40, 192, 700, 9000
    g = torch.Generator(device=DEV).manual_seed(9)
    a = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
    ends = [0, 400, 400, n]
    perm = torch.randperm(n, generator=torch.Generator().manual_seed(1)).to(torch.int32).to(DEV)
    offsets = torch.tensor(ends, dtype=torch.int32, device=DEV)
    there = [(e, at) for e in range(E) for at in range(ends[e], ends[e + 1], 128)]
    tiles = torch.full((places, 2), -1, dtype=torch.int32)
    for at in range(places):
        if at % 5 and at not in (places - 1, places - 2):
            tiles[at] = torch.tensor(there[at % (len(there) - 1)], dtype=torch.int32)
    tiles[places - 1] = torch.tensor(there[-1], dtype=torch.int32)
    tiles = tiles.to(DEV)
    ops.lib.call("dinfer_experts_nt", ops.dtype_code(a.dtype), 0, a.data_ptr(), K, w.data_ptr(), K, N * K, out.data_ptr(), N, N, K,
                 tiles.data_ptr(), places, 128, offsets.data_ptr(), perm.data_ptr(), 0, 1, 0, 0.0, 0.0, 704 * 128, ops._stream())
    want = torch.empty(n, N, dtype=torch.double, device=DEV)
    for e in range(E):
        want[perm[ends[e]:ends[e + 1]].long()] = a[ends[e]:ends[e + 1]].double() @ w[e].double().T
    close(out, want)


# rows an expert gets: none, one, the edges of blocks of 16 a half and of tiles of 224, two to four tiles of equal heights
TALL_COUNTS = [0, 1, 16, 17, 32, 33, 63, 64, 65, 192, 193, 223, 224, 225, 0, 256, 300, 448, 449, 672, 700]


def cut_evenly(count):
    """The first rows of an expert's tiles: as few tiles as 224 rows allow, of one height in whole blocks of 32."""
    n = -(-count // 224)
    height = -(-(-(-count // n)) // 32) * 32 if n else 224
    return list(range(0, count, height))


# columns: fewer than a wave's, two waves beside two, a last wave in part, odd widths, more tiles than a workgroup looks up at once;
# k: the fewest steps that are kept ahead, one more, many
@pytest.mark.parametrize("N,K,kind", [(40, 192, None), (130, 256, "gelu"), (255, 320, "relu2"), (1408, 1024, "silu"), (300, 2048, None),
                                      (26000, 192, "relu2"), (24, 192, "gated"), (132, 448, "gated"), (1000, 256, "gated"), (13100, 192, "gated")])
def test_experts_in_tall_tiles(N, K, kind):
    from dinfer_amd.kernels import ops
    E, n, top = len(TALL_COUNTS), sum(TALL_COUNTS), 3
    idx = sorted_entries(TALL_COUNTS, top, n, N)
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(-(-n // top), K, generator=g, device=DEV).to(torch.bfloat16)
    gated = kind == "gated"
    w = (torch.randn(E, 2 * N if gated else N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device=DEV)
    perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.zeros((ops.moe_max_tiles(n, E, 224), 2), **i32)
    ops.moe_scatter(idx.to(DEV), n, E, offsets, perm, tiles, 224)
    off = [0] + torch.tensor(TALL_COUNTS).cumsum(0).tolist()
    want = sorted((e, off[e] + r) for e in range(E) for r in cut_evenly(TALL_COUNTS[e]))
    assert sorted(tuple(t) for t in tiles.tolist() if t[0] >= 0) == want
    pick = torch.arange(N, device=DEV) if N <= 2048 else torch.cat([torch.arange(300), torch.arange(0, N, 97), torch.arange(N - 300, N)]).to(DEV)
    e = idx.to(DEV).long()

    def products(rows_of):
        y = torch.empty(n, pick.numel(), dtype=torch.float64, device=DEV)
        u = torch.empty_like(y) if gated else None
        for k in range(E):
            at, rows = rows_of(k)
            y[at] = rows.double() @ w[k, pick].double().T
            if gated:
                u[at] = rows.double() @ w[k, pick + N].double().T
        return y, u

    def by_entry(k):
        at = (e == k).nonzero().flatten()
        return at, x[at // top]

    scale = torch.rand(n, generator=g, device=DEV) + 0.5
    for row_scale in (None, scale):
        for to_perm in (True, False):
            out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
            ops.experts_nt(x, w, out, n, tiles, offsets, perm, gated=gated, a_div=top, c_to_perm=to_perm, tile_rows=224,
                           act=None if gated else kind, row_scale=row_scale)
            y, u = products(by_entry)
            if row_scale is not None:
                y = y * row_scale.double()[:, None]
                u = u * row_scale.double()[:, None] if gated else None
            z = act(y, "silu") * u if gated else act(y, kind)
            close(out[:, pick], z if to_perm else z[perm.long()])
    if gated:
        out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.experts_nt(x, w, out, n, tiles, offsets, perm, gated=True, a_div=top, c_to_perm=True, tile_rows=224, clamp=(1.0, 1.7))
        y, u = products(by_entry)
        y, u = y.clamp(max=1.0), u.clamp(-1.0, 1.0)
        close(out[:, pick], y * torch.sigmoid(1.7 * y) * (u + 1.0))
    else:
        out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
        a = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
        ops.experts_nt(a, w, out, n, tiles, offsets, perm, gated=False, a_div=0, c_to_perm=True, tile_rows=224)
        y, _ = products(lambda k: (perm[off[k]:off[k + 1]].long(), a[off[k]:off[k + 1]]))
        close(out[:, pick], y)


def test_which_tiles_a_routed_layer_takes():
    """Tall ones from 112 rows an expert on, where their k and their number allow it; what they do not take falls to 128 or 64 as before."""
    from dinfer_amd.kernels import lib, ops
    BF = torch.bfloat16
    rows = lambda avg, e, k_in, k_mid: ops.moe_tile_rows(BF, avg * e, e, k_in, k_mid)
    assert rows(111, 64, 2048, 1408) == 128 and rows(112, 64, 2048, 1408) == 224 and rows(384, 64, 2048, 1408) == 224
    assert all(rows(avg, 64, 2048, 1408) == 224 for avg in (176, 190, 223, 224)) and rows(190, 8, 4096, 14336) == 224
    assert rows(384, 64, 2048, 1400) == 128 and rows(384, 64, 2048, 128) == 128 and rows(384, 64, 1024, 512) == 128
    assert rows(384, 2, 65536, 32768) == 128 and rows(16, 64, 2048, 1408) == 16 and ops.moe_tile_rows(torch.float32, 9999, 8, 2048, 1408) == 64
    x, w = torch.zeros(8, 200, device=DEV, dtype=BF), torch.zeros(1, 64, 200, device=DEV, dtype=BF)
    i32 = dict(dtype=torch.int32, device=DEV)
    with pytest.raises(lib.KernelError):      # depth
        ops.experts_nt(x, w, torch.zeros(8, 64, device=DEV, dtype=BF), 8, torch.zeros(2, 2, **i32), torch.zeros(2, **i32), torch.zeros(8, **i32),
                       gated=False, a_div=1, c_to_perm=True, tile_rows=224)


# few tiles on an XCD: every workgroup of the walk has places that hold some
@pytest.mark.parametrize("counts", [[700], [130, 0, 0, 129], [256] * 8, [128] * 9 + [1]])
def test_walked_tiles_of_few_experts(counts):
    from dinfer_amd.kernels import ops
    N, K, E, n = 14336, 256, len(counts), sum(counts)
    idx = sorted_entries(counts, 1, n, 3)
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(n, K, generator=g, device=DEV).to(torch.bfloat16)
    w = (torch.randn(E, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    i32 = dict(dtype=torch.int32, device=DEV)
    for rows in (128, 224):
        perm, offsets, tiles = torch.zeros(n, **i32), torch.zeros(E + 1, **i32), torch.zeros((ops.moe_max_tiles(n, E, rows), 2), **i32)
        ops.moe_scatter(idx.to(DEV), n, E, offsets, perm, tiles, rows)
        out = torch.full((n, N), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.experts_nt(x, w, out, n, tiles, offsets, perm, gated=False, a_div=1, c_to_perm=True, tile_rows=rows)
        for k in range(E):
            at = (idx.to(DEV) == k).nonzero().flatten()
            close(out[at], x[at].double() @ w[k].double().T)


@pytest.mark.parametrize("all_scores", [0, 1, 2])
def test_a_row_that_is_no_number_still_names_experts(all_scores):
    """Logits that are NaN choose no expert by comparison; the indices lie among the experts all the same, each row's result is its own, and
    what such a row weighs by is no number or nothing."""
    from dinfer_amd.kernels import ops
    T, E, top, width = 9, 40, 6, 64
    g = torch.Generator().manual_seed(3)
    x = torch.randn(T, width, generator=g).to(torch.bfloat16)
    x[4] = float("nan")
    router = torch.randn(E, width, generator=g)
    some = router.clone()
    some[3:] = float("nan")          # three logits of every row compare
    for w in (router, some):
        idx = torch.full((T, top), -7, dtype=torch.int32, device="cuda")
        share = torch.full((T, top), 7.0, device="cuda")
        ops.moe_route(x.cuda(), w.cuda(), None, idx, share, None, T, top, torch.empty(T * (E + 1), device="cuda"), all_scores=all_scores)
        assert bool(((idx >= 0) & (idx < E)).all())
        bad = share[4].cpu()
        assert bool((bad.isnan() | (bad == 0)).all())
        if w is router:
            z = x.double() @ w.double().T
            good = [t for t in range(T) if t != 4]
            assert torch.equal(idx.cpu()[good].long().sort(1).values, z[good].topk(top, 1).indices.sort(1).values)


@pytest.mark.parametrize("all_scores", [0, 1, 2])
@pytest.mark.parametrize("E", [1, 40, 63, 64, 65, 200, 1024])
def test_the_lowest_of_equal_experts_is_chosen(E, all_scores):
    """Logits of which many are equal (whole numbers, exact in every order of summation): the choices in descending order, the lowest index
    among equals, wherever the lanes' own share of the experts ends."""
    from dinfer_amd.kernels import ops
    T, top, width = 70, min(6, E), 32
    g = torch.Generator().manual_seed(E)
    x = torch.randint(-2, 3, (T, width), generator=g).to(torch.bfloat16)
    router = torch.randint(-1, 2, (5, width), generator=g).float()[torch.randint(0, 5, (E,), generator=g)].contiguous()
    idx = torch.full((T, top), -7, dtype=torch.int32, device="cuda")
    share = torch.zeros(T, top, device="cuda")
    ops.moe_route(x.cuda(), router.cuda(), None, idx, share, None, T, top, torch.empty(T * (E + 1), device="cuda"), all_scores=all_scores)
    z = x.double() @ router.double().T
    want = torch.sort(z, dim=1, descending=True, stable=True).indices[:, :top]
    if all_scores == 1:      # by the softmax in float, where logits far below the largest are equal to nothing
        p = torch.softmax(z, 1)
        got = torch.gather(p, 1, idx.cpu().long())
        assert bool((got - torch.gather(p, 1, want)).abs().max() < 1e-6)
        assert all(len(set(r)) == top for r in idx.cpu().tolist())
    else:
        assert torch.equal(idx.cpu().long(), want)
