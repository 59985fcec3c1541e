"""Attention with options over steps of single rows: the heads of a group share the tile (attention_tile.cuh, HEADS), against
the plain kernel on the same pages, and beside the tile of rows, which serves the same rows when told of longer portions."""
import random

import pytest
import torch

pytestmark = pytest.mark.gpu

# heads, kv heads, key size, value size, page, options, keys a request
CASES = [
    (16, 4, 128, 128, 64, {}, [1, 31, 32, 33, 257, 4100]),                       # runs of no block, one block, many
    (3, 3, 32, 64, 16, dict(slope_exp=8.0), [1, 300, 1025]),                     # groups of one head
    (16, 1, 64, 64, 32, dict(window=100, keep_first=5, sinks=True), [3, 100, 101, 107, 900]),    # a full tile of heads
    (18, 2, 48, 48, 24, dict(sinks=True, softcap=3.0), [7, 500]),                # pages of no power of two
    (32, 2, 128, 96, 128, dict(chunk=192), [192, 193, 385, 1000]),
    (6, 2, 96, 128, 64, dict(window=64, keep_first=40), [20, 64, 65, 90, 129, 2000]),
    (4, 2, 256, 256, 16, dict(out_scale=0.5), [1, 1500]),
    (12, 4, 64, 128, 32, dict(sigmoid=True, slope_exp=4.0), [1, 40, 700]),
    (17, 1, 64, 64, 32, {}, [1, 600]),                                           # more heads than a tile: rows as before
]


@pytest.mark.parametrize("case", CASES)
def test_heads_of_a_group_share_the_tile(case):
    from dinfer_amd.kernels import ops
    H, G, D, V, page, options, lens = case
    opts = dict(options)
    g = torch.Generator().manual_seed(D + H)
    if opts.pop("sinks", False):
        opts["sinks"] = torch.randn(H, generator=g).cuda()
    if opts.pop("sigmoid", False):
        opts["sigmoid_bias"] = (torch.randn(H, generator=g) - 3).cuda()
    B, blocks = len(lens), sum(-(-n // page) for n in lens)
    ids = list(range(blocks + 1))
    random.Random(H).shuffle(ids)
    kp = torch.full((blocks + 1, G, page, D), float("nan"), dtype=torch.bfloat16)     # what no request holds must not count
    vp = torch.full((blocks + 1, G, page, V), float("nan"), dtype=torch.bfloat16)
    table = torch.full((B, max(-(-n // page) for n in lens)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        for i in range(-(-n // page)):
            m = min(page, n - i * page)
            table[b, i] = ids[at]
            kp[ids[at], :, :m] = torch.randn(G, m, D, generator=g).to(torch.bfloat16)
            vp[ids[at], :, :m] = torch.randn(G, m, V, generator=g).to(torch.bfloat16)
            at += 1
    q = (2 * torch.randn(B, H * D, generator=g)).to(torch.bfloat16).cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    args = (ops.k_cache_pack(kp).cuda(), vp.permute(0, 1, 3, 2).contiguous().cuda(), table.cuda(),
            torch.arange(B + 1, **i32), torch.tensor(lens, **i32), B)
    opts = dict(scale=D ** -0.5, heads=H, kv_heads=G, head_dim=D, v_dim=V, page_size=page, **{"window": 0, **opts})
    new, rows, want = (torch.full((B, H * V), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(3))
    ops.attn_flash_ext(q, new, *args, 1, **opts)
    ops.attn_flash_ext(q, rows, *args, 2, **opts)
    ops.attn_paged_ext(q, want, *args, B, **opts)
    # weights and results are rounded to bfloat16 (2^-9 each) in sums that no value exceeds (sigmoid weights: sums of many)
    top = max(want.float().abs().max().item(), vp.nan_to_num().float().abs().max().item())
    for name, got in (("heads", new), ("rows", rows)):
        err = (got.double() - want.double()).abs().max().item()
        assert err < 2.0 ** -7 * top, f"{name}: off by {err} of {top}"


@pytest.mark.parametrize("case", [
    (8, 4, 64, 64, 32, {}, [32 * n - n % 3 for n in range(1, 28)]),     # every count of key blocks up to three a wave and beyond
    (8, 4, 48, 32, 16, dict(window=250, keep_first=33, sinks=True), list(range(20, 1100, 90))),
    (16, 4, 256, 256, 16, {}, [40 * n + 1 for n in range(16)]),         # heads of 256: 256 rows in groups of four,
    (4, 2, 256, 256, 32, dict(slope_exp=8.0), [7 + n % 130 for n in range(256)]),   # 1,024 in groups of two
    (16, 4, 256, 256, 16, dict(softcap=5.0), [1, 900]),                 # ... and fewer: rows
    (16, 16, 32, 32, 16, {}, [5, 77, 130, 200, 64, 1, 300, 31]),        # groups of one: 128 rows,
    (16, 16, 32, 32, 16, {}, [5, 77, 130, 200, 64, 1, 300, 31, 9]),     # and more
    (16, 4, 128, 128, 16, dict(window=1024, keep_first=4, sinks=True), [300, 1500]),   # 32 rows and a window: rows; one wider: heads
    (16, 4, 128, 128, 16, dict(window=1025, keep_first=4), [300, 1500]),
])
def test_runs_of_keys_and_the_choice_of_the_tile(case):
    test_heads_of_a_group_share_the_tile(case)
