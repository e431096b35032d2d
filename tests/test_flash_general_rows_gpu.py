"""Key masks that are no prefix, through both ways they are served: inside the attention
kernel, and by the kernel beside the prefix-only ones, whose few blocks walk a larger grid.
Batches mix prefix rows, left padding, holes and a row without a valid key; against float64."""
from __future__ import annotations

import pytest
import torch

from techjam2026_amd import _lib as L
from techjam2026_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")

# 2-norm error of softmax(q k) v at each operand precision: one rounding of q, k, v and p to
# 11 bits; 22-bit operands with fp32 accumulation
TOL = {L.MMA_F16: 1.5e-3, L.MMA_F16X3: 3e-6, L.MMA_BF16X3: 6e-5}


def _masks(B, S, g):
    pos = torch.arange(S, device=DEV)[None]
    keep = pos < torch.randint(1, S + 1, (B, 1), device=DEV, generator=g)       # prefix rows
    keep[1::4] = pos >= torch.randint(0, S, (len(keep[1::4]), 1), device=DEV, generator=g)
    keep[2::4] = torch.rand(len(keep[2::4]), S, device=DEV, generator=g) < 0.5
    if B > 6:
        keep[6] = False
    return keep


@pytest.mark.parametrize("mode", [L.MMA_F16, L.MMA_F16X3, L.MMA_BF16X3])
@pytest.mark.parametrize("hd", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("B,H,S", [(3, 1, 1), (5, 2, 31), (4, 3, 65), (2, 2, 333), (44, 16, 130)])
@pytest.mark.parametrize("causal", [True, False])
def test_mixed_masks_match_float64(mode, hd, B, H, S, causal):
    g = torch.Generator(device=DEV).manual_seed(hd + S)
    dt = torch.float16 if mode == L.MMA_F16 else torch.float32
    q, k, v = (torch.randn(B, H, S, hd, device=DEV, generator=g).to(dt) for _ in range(3))
    keep = _masks(B, S, g)
    kd = (hd + B) % 3                           # the mask as bool, fp32 or fp16
    got = K.flash_attention(q, k, v, keep=(keep, keep.float(), keep.half())[kd], causal=causal, mode=mode)
    s = torch.matmul(q.double(), k.double().transpose(-2, -1).contiguous()) * hd ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1), -float("inf"))
    s = s.masked_fill(~keep[:, None, None], -float("inf"))
    want = torch.matmul(torch.softmax(s, -1).nan_to_num(0.0), v.double())
    err = float((got.double() - want).norm() / want.norm().clamp(min=1e-30))
    assert err < TOL[mode], f"off by {err:.2e}"
    dead = ~(s > -float("inf")).any(-1)
    assert torch.count_nonzero(got[dead]) == 0


@pytest.mark.parametrize("mode", [L.MMA_F16, L.MMA_F16X3, L.MMA_BF16X3])
@pytest.mark.parametrize("hd", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("B,H,S", [(1, 1, 1), (2, 3, 65), (2, 2, 333), (40, 8, 130)])
@pytest.mark.parametrize("causal", [True, False])
def test_no_mask_equals_a_mask_of_ones(mode, hd, B, H, S, causal):
    """Calls without a mask run instantiations without the mask code: the same bits."""
    g = torch.Generator(device=DEV).manual_seed(hd + S)
    dt = torch.float16 if mode == L.MMA_F16 else torch.float32
    q, k, v = (torch.randn(B, H, S, hd, device=DEV, generator=g).to(dt) for _ in range(3))
    ones = torch.ones(B, S, dtype=torch.bool, device=DEV)
    want = K.flash_attention(q, k, v, keep=ones, causal=causal, mode=mode)
    got = K.flash_attention(q, k, v, causal=causal, mode=mode)
    assert torch.equal(got, want)
    p16 = [K.flash_attention(q, k, v, keep=m, causal=causal, mode=mode, p16=True) for m in (None, ones)]
    assert torch.equal(*p16)


@pytest.mark.parametrize("mode", [L.MMA_F16, L.MMA_F16X3, L.MMA_BF16X3])
@pytest.mark.parametrize("hd", [8, 64, 128])
@pytest.mark.parametrize("B,H,S", [(300, 5, 4), (270, 4, 33), (1030, 1, 64), (140, 8, 65)])
def test_short_sequences_beyond_the_grid_match_float64(mode, hd, B, H, S):
    """More (row, head) pairs than the general kernel has blocks, at and around the length up to
    which it takes 64-row blocks."""
    test_mixed_masks_match_float64(mode, hd, B, H, S, True)
