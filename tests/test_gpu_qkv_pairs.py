"""Norm, rotation of pairs (2i, 2i + 1) and cache write of whole heads in bfloat16: the kernel of 16-byte accesses against the
general kernel, which the same rows get where they start at a column that is no multiple of 8."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,Hkv,D,tokens,page,rotated,extras", [
    (3, 1, 64, 1, 16, True, False), (16, 4, 128, 70, 32, True, True), (8, 2, 128, 520, 64, True, False), (5, 5, 256, 65, 8, True, True),
    (4, 2, 128, 9, 24, False, False)])
def test_neighbouring_pairs(H, Hkv, D, tokens, page, rotated, extras):
    from dinfer_amd.kernels import ops
    g = torch.Generator().manual_seed(D + tokens)
    cols = (H + 2 * Hkv) * D
    x = torch.randn(tokens, cols, generator=g).to(torch.bfloat16)
    ang = torch.rand(300, D // 2, generator=g) * 6
    table = torch.cat([ang.cos(), ang.sin()], 1).cuda() if rotated else None
    pos = torch.randint(0, 300, (tokens,), generator=g, dtype=torch.int32).cuda()
    gains = [(1 + 0.2 * torch.randn(D, generator=g)).to(torch.bfloat16).cuda() for _ in range(2)]
    blocks = -(-tokens // page) + 1
    slots = torch.arange(3, tokens + 3)
    slots[tokens // 2] = -1                                   # a row that is not cached
    more = dict(bias=torch.randn(cols, generator=g).cuda(), q_temp=(0.1, 16), q_head_scale=torch.rand(H, generator=g).cuda()) if extras else {}
    got = []
    for shift in (0, 4):
        buf = torch.zeros(tokens, cols + 8, dtype=torch.bfloat16)
        buf[:, shift:shift + cols] = x
        buf = buf.cuda()
        kc = torch.full((blocks, Hkv, D // 8, page, 8), 9.0, dtype=torch.bfloat16, device="cuda")
        vc = torch.full((blocks, Hkv, D, page), 9.0, dtype=torch.bfloat16, device="cuda")
        ops.qkv_post(buf, tokens, heads=H, kv_heads=Hkv, head_dim=D, q_off=shift, k_off=shift + H * D, v_off=shift + (H + Hkv) * D,
                     q_gain=gains[0], k_gain=gains[1], eps=1e-6, gain_offset=0.0, positions=pos, cos_sin=table, rotary_dim=D,
                     rope_style=1, k_cache=kc, v_cache=vc, slot_mapping=slots.cuda(), page_size=page, **more)
        got.append((buf[:, shift:shift + H * D].float(), kc.float(), vc.float()))
    for a, b in zip(*got):
        # the sum of squares is added up in another order: a float rounding, which may move a result by one step of bfloat16
        assert ((a - b).abs() <= 2.0 ** -7 * b.abs() + 1e-6).all()
        assert (a != b).float().mean().item() < 1e-2
    assert torch.equal(got[0][2], got[1][2])
