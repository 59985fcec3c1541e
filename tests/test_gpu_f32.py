"""The 32-bit path's matrix-core kernels (csrc/f32.hip) against float64, at the edges of their tiles, and the promise
that a row's result does not depend on how many rows ran with it."""
import pytest
import torch

from test_gpu_kernels import DEV, expected_attention, ops, paged_case

pytestmark = pytest.mark.gpu


def product(M, N, K, seed=0, lda=None, spread=1.0):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, lda or K, generator=g)[:, :K] * spread
    w = torch.randn(N, K, generator=g)
    if lda is not None:
        a = torch.randn(M, lda, generator=g).to(DEV)[:, :K]
    return a.to(DEV), w.to(DEV)


# rows: the few-row kernel's last (16), the tiles' edges; K: shorter than a piece of 16, a segment and one more, no whole
# step, many segments (more than the few-row kernel has waves)
@pytest.mark.parametrize("K", [4, 20, 256, 260, 1024, 2300, 6144])
@pytest.mark.parametrize("M,N", [(1, 16), (1, 331), (16, 40), (17, 96), (33, 65), (64, 64), (100, 130), (500, 1024)])
def test_gemm_f32(M, N, K):
    a, w = product(M, N, K, seed=M + N + K)
    out = torch.full((M + 1, N), 7.0, device=DEV)
    ops().gemm_f32(a, w, out, M)
    want = a.double() @ w.double().T
    # every product and sum rounds by 2^-24 of a partial sum: segments of 256 terms and K / 256 additions. The standard
    # deviation of a sum of K unit products is sqrt(K); 16 roundings' worth at that size is far beyond what is seen
    # (the largest of half a million entries: 6) and far below one term lost
    bound = 16 * 2.0 ** -24 * K ** 0.5 * max(1.0, (min(K, 256) / 4 + K / 256) ** 0.5)
    assert (out[:M].double() - want).abs().max().item() <= bound
    assert (out[M] == 7.0).all()
    # fewer rows, the last of them: the same bits
    for m in (1, 16, 17, 40):
        if m <= M:
            part = torch.empty(m, N, device=DEV)
            ops().gemm_f32(a[M - m:].contiguous(), w, part, m)
            assert torch.equal(part, out[M - m:M]), f"{m} rows differ"


# sizes that lead to each of the six tiles, none whole; K: less than a step, a segment and a piece, an odd number of segments
@pytest.mark.parametrize("K", [20, 260, 1284])
@pytest.mark.parametrize("M,N", [(250, 6150), (193, 9000), (130, 4090), (300, 4090), (1001, 331), (33, 1027)])
def test_gemm_f32_tiles(M, N, K):
    a, w = product(M, N, K, seed=M + N + K, lda=K + 8)
    out = torch.full((M + 1, N + 2), 7.0, device=DEV)
    ops().gemm_f32(a, w, out[:, :N], M)
    bound = 16 * 2.0 ** -24 * K ** 0.5 * max(1.0, (min(K, 256) / 4 + K / 256) ** 0.5)   # as above
    assert (out[:M, :N].double() - a.double() @ w.double().T).abs().max().item() <= bound
    assert (out[M] == 7.0).all() and (out[:, N:] == 7.0).all()
    part = torch.empty(16, N, device=DEV)
    ops().gemm_f32(a[M - 16:].contiguous(), w, part, 16)
    assert torch.equal(part, out[M - 16:M, :N])


def test_gemm_f32_strides_and_what_it_leaves_to_the_plain_kernel():
    a, w = product(40, 48, 64, seed=5, lda=100)
    assert ops().gemm_f32_supports(a, w)
    out = torch.zeros(40, 60, device=DEV)[:, :48]
    ops().gemm_f32(a, w, out, 40)
    torch.testing.assert_close(out.double(), a.double() @ w.double().T, rtol=1e-5, atol=1e-4)
    assert not ops().gemm_f32_supports(a[:, 1:61], w[:, :60])           # rows that do not begin at 16 bytes
    assert not ops().gemm_f32_supports(torch.zeros(4, 37, device=DEV), torch.zeros(4, 37, device=DEV))
    from dinfer_amd.kernels import gemm
    b, v = product(9, 33, 37, seed=6)
    out = torch.empty(9, 33, device=DEV)
    torch.testing.assert_close(gemm.matmul_nt(b, v, out, 9).double(), b.double() @ v.double().T, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("M", [32 * 65535 + 1, 64 * 65535])
def test_gemm_f32_takes_as_many_rows_as_the_plain_kernel(M):
    a, w = product(M, 5, 8, seed=9)
    out = torch.empty(M, 5, device=DEV)
    ops().gemm_f32(a, w, out, M)
    torch.testing.assert_close(out.double(), a.double() @ w.double().T, rtol=1e-5, atol=1e-5)


def test_gemm_f32_keeps_infinities_to_their_row():
    a, w = product(50, 70, 300, seed=8)
    clean = torch.empty(50, 70, device=DEV)
    ops().gemm_f32(a, w, clean, 50)
    a[13, 299], a[20, 5] = float("inf"), float("nan")
    out = torch.empty(50, 70, device=DEV)
    ops().gemm_f32(a, w, out, 50)
    rows = [r for r in range(50) if r not in (13, 20)]
    assert torch.equal(out[rows], clean[rows])
    assert out[13].isinf().all() and out[20].isnan().all()


def attend(q, kc, vc, m, B, T, max_q, **geo):
    out = torch.full((T, geo["heads"] * geo["head_dim"]), 9.0, device=DEV)
    ops().attn_f32(q, out, kc, vc, m["bt"], m["cu"], m["sl"], B, T, max_q, scale=geo["head_dim"] ** -0.5, **geo)
    return out


@pytest.mark.parametrize("window", [0, 40, 64])
@pytest.mark.parametrize("H,Hkv,D,page", [(16, 8, 128, 16), (4, 2, 16, 4), (6, 2, 48, 8), (5, 1, 64, 64), (3, 3, 80, 12),
                                         (8, 4, 96, 16), (2, 1, 112, 8), (4, 4, 192, 16), (3, 1, 256, 32), (32, 1, 32, 16)])
def test_attn_f32(H, Hkv, D, page, window):
    # tails of tiles and key blocks, histories that end inside a page, single rows, blocks enough for every wave
    hist, new = [0, 0, 11, 0, 70, 300, 6], [1, 17, 3, 64, 1, 90, 1]
    q, kc, vc, m, outs = paged_case(torch.float32, H, Hkv, D, page, hist, new, seed=D + page)
    if window:      # what lies behind every row's window has been given back
        for b, h in enumerate(hist):
            m["bt"][b, :max(0, h - window + 1) // page] = -1
    geo = dict(window=window, heads=H, kv_heads=Hkv, head_dim=D, page_size=page)
    out = attend(q, kc, vc, m, len(hist), sum(new), max(new), **geo)
    want = expected_attention(outs, hist, D ** -0.5, window)
    # scores of size 1 to 5 carry D roundings each, a mean of at most 400 values another few: below 1e-5
    torch.testing.assert_close(out.double().cpu().view(-1, H, D), want, rtol=1e-5, atol=1e-5)


def test_attn_f32_rows_do_not_depend_on_the_cut():
    H, Hkv, D, page, n, window = 8, 2, 64, 16, 203, 0
    q, kc, vc, m, _ = paged_case(torch.float32, H, Hkv, D, page, [0], [n], seed=4)
    geo = dict(window=window, heads=H, kv_heads=Hkv, head_dim=D, page_size=page)
    whole = attend(q, kc, vc, m, 1, n, n, **geo)
    for start, rows in ((0, 1), (1, 2), (63, 1), (64, 4), (65, 70), (130, 73), (202, 1)):
        part = dict(m, cu=torch.tensor([0, rows], dtype=torch.int32, device=DEV), sl=torch.tensor([start + rows], dtype=torch.int32, device=DEV))
        got = attend(q[start:start + rows].contiguous(), kc, vc, part, 1, rows, rows, **geo)
        assert torch.equal(got, whole[start:start + rows]), f"rows {start} to {start + rows}"


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attn_f32_keeps_a_bad_value_to_the_rows_that_see_it(bad):
    H, Hkv, D, page, n, at = 4, 2, 64, 16, 100, 70
    q, kc, vc, m, _ = paged_case(torch.float32, H, Hkv, D, page, [0], [n], seed=5)
    geo = dict(window=0, heads=H, kv_heads=Hkv, head_dim=D, page_size=page)
    clean = attend(q, kc, vc, m, 1, n, n, **geo)
    vc[m["bt"][0, at // page].long(), :, 3, at % page] = bad
    out = attend(q, kc, vc, m, 1, n, n, **geo)
    assert torch.isfinite(out[:at]).all()
    torch.testing.assert_close(out[:at], clean[:at], rtol=1e-5, atol=1e-6)      # (key by key there: another order)
    assert not torch.isfinite(out[at:].view(-1, H, D)[:, :, 3]).any()
    assert torch.isfinite(out[at:].view(-1, H, D)[:, :, 4]).all()
