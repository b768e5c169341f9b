"""gsvk_decode_attention split by heads (csrc/gsvk_attention.hip attn_heads): every piece width, the
edges of its key rounds and the line to the key chunks, against the oracle with the tolerance of
test_gpu_attention.py; an infinite value in the last cached row."""
import numpy as np
import pytest
import torch

import gsvk
from gpu_util import BF16, F16, F32
from test_gpu_attention import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 33, 65, 130])  # 8, 16, 32 and 64 lanes per key
@pytest.mark.parametrize("kv_dt,out_dt", [(F16, F16), (F32, F32), (BF16, F16)])
def test_piece_widths(B, kv_dt, out_dt):
    max_len = 150
    pos = np.arange(B) * 37 % max_len
    pos[-1] = max_len - 1
    case(B, 16, 32, max_len, pos, kv_dt, out_dt, seed=300 + B, poison=True)


@pytest.mark.parametrize("H,HD", [(2, 32), (8, 64), (4, 128), (1, 512), (8, 8), (6, 32), (3, 64)])
def test_head_shapes(H, HD):
    """(6 x 32 and 3 x 64: 24 lanes, pieces of 8.)"""
    case(5, H, HD, 140, [0, 1, 63, 64, 139], F16, F32, seed=320 + HD + H, poison=True)


@pytest.mark.parametrize("pos", [[0], [255, 256, 257], [511, 8, 512]])
def test_key_rounds(pos):
    case(len(pos), 16, 32, 600, pos, F16, F16, seed=340 + pos[0])


@pytest.mark.parametrize("B,max_len,kv_dt", [(23, 1000, F16), (23, 1001, F16), (24, 1001, F16),
                                              (47, 500, F32), (47, 501, F32), (48, 501, F32)])
def test_either_side_of_the_line(B, max_len, kv_dt):
    pos = np.random.default_rng(B).integers(0, max_len, B)
    case(B, 4, 32, max_len, pos, kv_dt, F32, seed=350 + B)


def test_infinite_value_in_the_last_cached_row():
    """It reaches its own output as the reference's sum takes it, not as NaN through a reread."""
    B, H, HD, max_len = 2, 16, 32, 64
    g = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    qkv, k, v = r(B, 1536), r(B, max_len, 512).half(), r(B, max_len, 512).half()
    pos = torch.tensor([40, 63], device="cuda")
    v[0, 39, 100] = float("inf")
    out = torch.empty(B, 512, device="cuda")
    gsvk.decode_attention(qkv, k, v, pos, out, H)
    torch.cuda.synchronize()
    assert torch.isinf(out[0, 100]) and torch.isfinite(out).sum() == out.numel() - 1
