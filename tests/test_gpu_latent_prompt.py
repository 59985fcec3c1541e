"""Latent attention over prompt portions at the sizes of the kernel that shares a block of keys among 64 rows, against
float64: edges of its row groups and key blocks, histories, windows, short pages."""
import math

import pytest
import torch

from test_gpu_kudurax import latent_case, latent_plain

pytestmark = pytest.mark.gpu

CASES = [
    # seqs, q_lens, H, R, dr, page, window, far (request, token, head, key it looks at)
    ([300], [300], 4, 128, 32, 8, 0, (0, 299, 2, 3)),                   # pages shorter than a block; tails of both
    ([33, 64, 31, 1], [33, 64, 31, 1], 16, 128, 0, 16, 0, (1, 63, 7, 0)),  # no rotated part; a prompt of one token among others
    ([500, 64, 33], [37, 1, 33], 16, 256, 64, 32, 0, (0, 36, 9, 0)),    # histories; a single row
    ([200, 90], [64, 2], 3, 128, 96, 64, 50, (0, 10, 1, 200 - 64 + 10 - 49)),   # a window: the oldest key a row still sees
    ([200, 90], [64, 2], 3, 128, 96, 64, 50, (0, 10, 1, 200 - 64 + 10 - 50)),   # ... and the first it does not; rows of 28 pieces
    ([150, 70], [150, 3], 5, 512, 64, 16, 0, (0, 149, 1, 5)),           # the widest rows
    ([700], [130], 16, 512, 64, 16, 0, (0, 129, 15, 31)),               # several groups behind a history
    ([70] * 66, [2] * 66, 16, 128, 32, 16, 0, (65, 1, 3, 64)),          # more requests than a wave counts at once
    ([200, 120, 75, 10], [150, 120, 40, 10], 16, 512, 64, 8, 0, (2, 39, 1, 70)),   # more row groups than two rounds over the XCDs take
]


@pytest.mark.parametrize("case_no", range(len(CASES)))
def test_latent_prompt_portions(case_no):
    from dinfer_amd.kernels import ops
    seqs, q_lens, H, R, dr, page, window, far = CASES[case_no]
    case = latent_case(seqs, q_lens, H, R, dr, page, 500 + case_no, torch.bfloat16, far)
    scale = 0.7 / math.sqrt(R + dr)
    want = latent_plain(case, q_lens, seqs, H, R, dr, scale, window)
    dev = {k: v.cuda() for k, v in case.items() if k != "keys"}
    if window:      # what lies behind every row's window has been given back
        for b, (s, n) in enumerate(zip(seqs, q_lens)):
            dev["bt"][b, :max(0, s - n - window + 1) // page] = -1
    T, B = sum(q_lens), len(seqs)
    out = torch.zeros(T, H * R, dtype=torch.bfloat16, device="cuda")
    cache_t = dev["cache"][:, :, :R].transpose(1, 2).contiguous()
    part = torch.zeros(T * H * (R + 4), dtype=torch.float32, device="cuda")
    ops.latent_attn_mfma(dev["qa"], out, dev["cache"], cache_t, dev["bt"], dev["cu"], dev["seq"], B, T, 1, part, scale=scale,
                         window=window, heads=H, rank=R, rot_dim=dr, page_size=page)
    got = out.double().cpu()
    # weights and results rounded to 2^-9 each, values of size one: a few times that of the largest
    assert (got - want).abs().max().item() < 0.015 * max(1.0, want.abs().max().item())
    b, i, h, j = far
    t, p = sum(q_lens[:b]) + i, seqs[b] - q_lens[b] + i
    seen = j <= p and (not window or j > p - window)
    close = (got[t, h * R:(h + 1) * R] - case["keys"][b][j][:R].double()).abs().max().item()
    assert (close < 0.1) == seen


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("n,hist,H,R,dr,page,at", [(100, 0, 1, 128, 32, 16, 40), (40, 9, 2, 512, 64, 64, 33), (300, 70, 4, 256, 64, 8, 300)])
def test_a_bad_key_stays_away_from_rows_before_it(n, hist, H, R, dr, page, at, bad):
    """An infinity or NaN that a later token left in the cache does not reach a tile of 16 rows that ends before its block of 32 keys."""
    from dinfer_amd.kernels import ops
    case = latent_case([hist + n], [n], H, R, dr, page, at, torch.bfloat16)
    args = lambda c: (c["cache"], c["cache"][:, :, :R].transpose(1, 2).contiguous(), dev["bt"], dev["cu"], dev["seq"], 1, n, 1,
                      torch.zeros(n * H * (R + 4), device="cuda"))
    dev = {k: v.cuda() for k, v in case.items() if k != "keys"}
    got = []
    for value in (None, bad):
        c = dict(cache=dev["cache"].clone())
        if value is not None:
            c["cache"][int(case["bt"][0, at // page]), at % page, :] = value
        out = torch.zeros(n, H * R, dtype=torch.bfloat16, device="cuda")
        ops.latent_attn_mfma(dev["qa"], out, *args(c), scale=0.1, window=0, heads=H, rank=R, rot_dim=dr, page_size=page)
        got.append(out)
    safe, sees = (at // 32 * 32 - hist) * H // 16 * 16 // H, at - hist      # tokens of the tiles before the block; the first that sees it
    assert safe > 0 and torch.equal(got[1][:safe], got[0][:safe])
    assert torch.isfinite(got[0]).all() and not torch.isfinite(got[1][sees:]).any()


def test_pages_whose_offsets_pass_32_bits():
    """A page of 2^22 tokens (4.3 GB, and as much again transposed): the kernel that keeps 32-bit offsets leaves it alone."""
    from dinfer_amd.kernels import ops
    n, H, R, page = 40, 2, 512, 1 << 22
    g = torch.Generator().manual_seed(1)
    keys, qa = torch.randn(n, R, generator=g).to(torch.bfloat16), (0.3 * torch.randn(n, H * R, generator=g)).to(torch.bfloat16)
    cache, cache_t = torch.zeros(1, page, R, dtype=torch.bfloat16, device="cuda"), torch.zeros(1, R, page, dtype=torch.bfloat16, device="cuda")
    cache[0, :n], cache_t[0, :, :n] = keys.cuda(), keys.T.cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    out = torch.zeros(n, H * R, dtype=torch.bfloat16, device="cuda")
    ops.latent_attn_mfma(qa.cuda(), out, cache, cache_t, torch.zeros(1, 1, **i32), torch.tensor([0, n], **i32), torch.tensor([n], **i32), 1, n, 1,
                         torch.zeros(n * H * (R + 4), device="cuda"), scale=0.1, window=0, heads=H, rank=R, rot_dim=0, page_size=page)
    want = latent_plain(dict(qa=qa, cache=keys[None], bt=torch.zeros(1, 1, dtype=torch.int32)), [n], [n], H, R, 0, 0.1)
    assert (out.double().cpu() - want).abs().max().item() < 0.015 * max(1.0, want.abs().max().item())
