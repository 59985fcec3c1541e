"""Kernels for steps of many rows against the ones for few or for any rows, and against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def ops():
    from dinfer_amd.kernels import ops as o
    return o


def _slots(portions, page, blocks):
    """Slots of portions (first position, tokens), each on pages of its own in shuffled order."""
    order, out, g = torch.randperm(blocks, generator=torch.Generator().manual_seed(page)).tolist(), [], 0
    for first, n in portions:
        pages = [order[g + i] for i in range((first + n - 1) // page + 1)]
        g += len(pages)
        out += [pages[p // page] * page + p % page for p in range(first, first + n)]
    return out


@pytest.mark.parametrize("H,Hkv,D,style,extras", [(6, 3, 64, 0, True), (16, 8, 128, 0, False), (9, 1, 128, 1, True), (5, 5, 256, 0, True), (4, 2, 256, 1, False)])
@pytest.mark.parametrize("portions", [[(0, 64)], [(5, 1), (0, 3), (3, 61), (8, 7), (16, 8), (1, 40)], [(i, 37 + i) for i in range(12)],
                                      [(0, 512)], [(i, 43 + i) for i in range(12)]])     # from 512 tokens on four heads a workgroup
def test_qkv_post_of_portions(H, Hkv, D, style, extras, portions):
    """The kernel for prompt portions leaves the bits of the kernel that takes single tokens, wherever portions begin."""
    page, blocks = 16, sum((a + n - 1) // 16 + 1 for a, n in portions)
    g = torch.Generator().manual_seed(D + style)
    T, cols = sum(n for _, n in portions), (H + 2 * Hkv) * D
    x = torch.randn(T, cols, generator=g).to(BF).cuda()
    slots = _slots(portions, page, blocks)
    slots[T // 2] = -1
    slots = torch.tensor(slots).cuda()
    ang = torch.rand(300, D // 2, generator=g) * 6
    table = torch.cat([ang.cos(), ang.sin()], 1).cuda()
    pos = torch.randint(0, 300, (T,), generator=g, dtype=torch.int32).cuda()
    gains = [(1 + 0.2 * torch.randn(D, generator=g)).to(torch.float32 if extras else BF).cuda() for _ in range(2)]
    more = dict(bias=torch.randn(cols, generator=g).cuda(), q_temp=(0.1, 16), q_head_scale=torch.rand(H, generator=g).cuda(),
                v_first=torch.randn(T, Hkv * D, generator=g).to(BF).cuda(), v_share=0.3) if extras else {}
    got = []
    for runs in (False, True):
        buf = x.clone()
        kc = torch.full((blocks, Hkv, D // 8, page, 8), 9.0, dtype=BF, device="cuda")
        vc = torch.full((blocks, Hkv, D, page), 9.0, dtype=BF, device="cuda")
        ops().qkv_post(buf, T, heads=H, kv_heads=Hkv, head_dim=D, q_off=0, k_off=H * D, v_off=(H + Hkv) * D, q_gain=gains[0],
                       k_gain=gains[1], eps=1e-6, gain_offset=0.5, positions=pos, cos_sin=table, rotary_dim=D, rope_style=style,
                       k_cache=kc, v_cache=vc, slot_mapping=slots, page_size=page, token_runs=runs, **more)
        got.append((buf, kc, vc))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("H,Hkv,D", [(16, 8, 128), (3, 2, 64), (2, 1, 256), (2, 2, 320)])
@pytest.mark.parametrize("portions", [[(0, 127)], [(0, 128)], [(5, 100), (16, 20), (3, 9)], [(7, 255)], [(i, 37 + i) for i in range(12)]])
def test_qkv_post_of_portions_in_32_bits(H, Hkv, D, portions):
    """From 128 tokens on neighbours share an XCD: the same bits, whatever the number of tokens leaves of the last 128."""
    page, blocks = 16, sum((a + n - 1) // 16 + 1 for a, n in portions)
    g = torch.Generator().manual_seed(D)
    T, cols = sum(n for _, n in portions), (H + 2 * Hkv) * D
    x = torch.randn(T, cols, generator=g).cuda()
    slots = _slots(portions, page, blocks)
    slots[T // 2] = -1
    slots = torch.tensor(slots).cuda()
    ang = torch.rand(300, D // 2, generator=g) * 6
    table = torch.cat([ang.cos(), ang.sin()], 1).cuda()
    pos = torch.randint(0, 300, (T,), generator=g, dtype=torch.int32).cuda()
    gains = [(1 + 0.2 * torch.randn(D, generator=g)).cuda() for _ in range(2)]
    got = []
    for runs in (False, True):
        buf = torch.cat([x, torch.full((3, cols), 9.0, device="cuda")])
        kc = torch.full((blocks, Hkv, D // 8, page, 8), 9.0, device="cuda")
        vc = torch.full((blocks, Hkv, D, page), 9.0, device="cuda")
        ops().qkv_post(buf, T, heads=H, kv_heads=Hkv, head_dim=D, q_off=0, k_off=H * D, v_off=(H + Hkv) * D, q_gain=gains[0],
                       k_gain=gains[1], eps=1e-6, gain_offset=0.0, positions=pos, cos_sin=table, rotary_dim=D, rope_style=0,
                       k_cache=kc, v_cache=vc, slot_mapping=slots, page_size=page, token_runs=runs)
        got.append((buf, kc, vc))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    assert bool((got[1][0][T:] == 9).all())


@pytest.mark.parametrize("rows,width", [(1023, 2048), (1024, 8), (1025, 520), (1030, 2048), (1024, 2056), (1027, 4096), (1024, 4104)])
@pytest.mark.parametrize("x_dtype,out_dtype,branch", [(BF, BF, True), (torch.float32, BF, False), (torch.float32, torch.float32, True)])
def test_layernorm_of_many_rows(rows, width, x_dtype, out_dtype, branch):
    g = torch.Generator().manual_seed(rows + width)
    x = (torch.randn(rows, width, generator=g) + 0.5).to(x_dtype).cuda()
    stream = torch.randn(rows, width, generator=g).cuda() if branch else None
    w, b = torch.randn(width, generator=g).cuda(), torch.randn(width, generator=g).cuda()
    out = torch.empty(rows, width, dtype=out_dtype, device="cuda")
    y = x.double() + (stream.double() if branch else 0)
    total = x.float() + stream if branch else None
    ops().layernorm(x, w, b, out, 1e-5, rows, residual=stream)
    want = torch.nn.functional.layer_norm(y, (width,), w.double(), b.double(), 1e-5)
    if branch:
        assert torch.equal(stream, total)
    # sums of up to 4,104 floats, then one rounding: 2^-9 in bfloat16, some 2^-18 in float
    tol = 2.0 ** -8 if out_dtype == BF else 2.0 ** -16
    assert ((out.double() - want).abs() <= tol * (want.abs() + 1)).all()


@pytest.mark.parametrize("rows,n", [(131073, 8), (14564, 72), (400, 2816), (600, 2056), (9, 16392 * 8)])
def test_activations_in_16_byte_pieces(rows, n):
    """Rows that begin at a 16-byte piece against the same rows two entries further on, which are taken one by one: rows of one
    piece, more than a launch takes, and rows of more pieces than its workgroups of a row."""
    assert rows * n >= 1 << 20      # fewer numbers are taken one by one wherever they begin
    g = torch.Generator().manual_seed(n)
    x, gates = torch.randn(rows, n, generator=g).to(BF) * 3, torch.randn(rows, n, generator=g).to(BF)
    for kind in ("silu", "relu2", "gelu", "gelu_tanh", "sigmoid"):
        got = []
        for at in (0, 2):
            a, b, o = (torch.zeros(rows, n + 8, dtype=BF, device="cuda") for _ in range(3))
            a[:, at:at + n] = x.cuda()
            b[:, at:at + n] = gates.cuda()
            ops().act(a[:, at:at + n], o[:, at:at + n], rows, kind)
            ys = [o[:, at:at + n]]
            for group in (1, 8):
                z = torch.zeros(rows, n + 8, dtype=BF, device="cuda")
                z[:, at:at + n] = x.cuda()
                ops().gate(z[:, at:at + n], b[:, at:at + n // group], rows, kind, group=group)
                ys.append(z[:, at:at + n])
                assert not z[:, :at].any() and not z[:, at + n:].any()
            got.append(ys)
        for a, b in zip(*got):
            assert torch.equal(a, b)


@pytest.mark.parametrize("tokens,experts,width,gate", [(1024, 1, 32, False), (1030, 64, 2048, True), (1025, 47, 544, False), (1100, 130, 96, True), (1024, 64, 40, True)])
def test_router_logits_of_many_tokens(tokens, experts, width, gate):
    """The logits against 64 bits: as near as the kernel for few tokens (which a step of 1,000 of them gets), and the choice
    made from them; an infinity of one token stays with that token."""
    g = torch.Generator().manual_seed(tokens + experts)
    x = torch.randn(tokens, width, generator=g).to(BF).cuda()
    x[7, 3] = float("inf")
    w, sg = torch.randn(experts, width, generator=g).cuda(), torch.randn(width, generator=g).cuda() if gate else None
    top = min(2, experts)
    want = x.double() @ torch.cat([w] + ([sg[None]] if gate else [])).double().t()
    err = []
    for n in (tokens, 1000):
        idx, share = torch.zeros(n * top, dtype=torch.int32, device="cuda"), torch.zeros(n * top, device="cuda")
        z = torch.zeros(n * (experts + 1), device="cuda")
        ops().moe_route(x, w, sg, idx, share, torch.zeros(n, device="cuda"), n, top, z, all_scores=0, correction=None)
        z = z.view(n, experts + 1)[:, :want.shape[1]]
        keep = torch.arange(n, device="cuda") != 7
        assert not torch.isfinite(z[7]).any()
        err.append(((z.double() - want[:n])[keep].norm() / want[:n][keep].norm()).item())
        assert torch.equal(idx.view(n, top)[keep, 0].long(), z[keep][:, :experts].argmax(1))
    assert err[0] <= 1.1 * err[1] and err[0] < 2e-7


@pytest.mark.parametrize("width", [4, 1020, 1024, 1025, 1028, 4100, 5120, 5121])
def test_float_rows(width):
    """The norm of float rows at the edges of the widths that registers hold; norms and gated
    activations wherever the rows begin, the latter bit for bit."""
    g = torch.Generator().manual_seed(width)
    T, eps = 5, 1e-6
    x, res, w = torch.randn(T, width, generator=g).cuda(), torch.randn(T, width, generator=g).cuda(), torch.randn(width, generator=g).cuda()
    x[3, width - 1] = float("inf")
    gu = torch.randn(T, 2 * width, generator=g).cuda()
    norms, acts = [], []
    for at in (0, 1):
        a, r, z = (torch.zeros(T, n + 4, device="cuda") for n in (width, width, 2 * width))
        a[:, at:at + width], r[:, at:at + width], z[:, at:at + 2 * width] = x, res, gu
        o, y = torch.full((T + 1, width), 7.0, device="cuda"), torch.full((T + 1, width), 7.0, device="cuda")
        ops().rmsnorm(a[:, at:at + width], w, o, eps, T, residual=r[:, at:at + width], weight_offset=1.0)
        ops().gated_act(z[:, at:at + 2 * width], y, T, "silu")
        assert torch.equal(r[:, at:at + width], x + res) and not r[:, at + width:].any() and (o[T] == 7.0).all() and (y[T] == 7.0).all()
        norms.append(o[:T]), acts.append(y[:T])
    assert torch.equal(*acts)
    keep = [0, 1, 2, 4]
    s = (x + res).double()[keep]
    want = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + eps) * (w.double() + 1)
    for o in norms:   # a sum of squares of up to 20 terms a thread, 8 levels of tree, a root, three products: 2^-24 each
        assert ((o[keep].double() - want).abs() <= 32 * 2.0 ** -24 * want.abs()).all()
        assert not torch.isfinite(o[3, -1])
