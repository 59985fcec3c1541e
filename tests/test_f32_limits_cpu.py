"""What the 32-bit matrix-core kernels (csrc/f32.hip) leave to the plain ones, as the host decides it."""
from types import SimpleNamespace

import pytest
import torch

from dinfer_amd.kernels import attention, lib, ops


@pytest.mark.parametrize("K,taken", [(0, False), (4, True), (1022, False), (2 ** 31 - 4, False), (2 ** 31 - 68, False), (2 ** 31 - 512, False),
                                     (2 ** 31 - 516, True)])
def test_products_whose_offsets_fit(K, taken):
    """Steps of 64 k are fetched two ahead, in 32-bit numbers: k must end two segments before those do."""
    fn = lib.get("dinfer_gemm_f32_supports")
    assert bool(fn(4096, max(K, 4), 8192, max(K, 4), K)) == taken


@pytest.mark.parametrize("reqs,cols,shift,plain", [(1, 128, 0, False), (65535, 128, 0, False), (65536, 128, 0, True), (3, 130, 0, True),
                                                   (3, 128, 1, True)])
def test_attention_the_grid_takes(monkeypatch, reqs, cols, shift, plain):
    """More requests than a grid's y has places, and rows that do not begin at 16 bytes, go to the plain kernel."""
    monkeypatch.setattr(ops, "attn_f32", lambda *a, **k: False)
    monkeypatch.setattr(ops, "attn_paged_ref", lambda *a, **k: True)
    ws = SimpleNamespace(f32=True, mfma=False)
    batch = SimpleNamespace(block_table=[None], num_reqs=reqs, num_tokens=reqs, max_q_len=1, cu_seqlens=None, seq_lens=None)
    rows = torch.empty(4 * cols + 4)
    qkv, out = rows[shift:shift + 4 * cols].view(4, cols), torch.empty(4, 128)
    assert attention.paged_attention(qkv, out, None, None, batch, 0, ws, scale=1.0, window=0, heads=4, kv_heads=2, head_dim=16,
                                     page_size=16) is plain
