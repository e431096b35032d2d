"""The erf-GELU of the kernels' epilogues against float64, from the smallest fp16 inputs to the
largest, through an identity product (fp16 values pass it exactly)."""
from __future__ import annotations

import pytest
import torch

from techjam2026_amd import _lib as L
from techjam2026_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("scale", [6e-8, 1e-3, 0.3, 1.0, 3.0, 8.0, 200.0, 65504.0])
def test_gelu_matches_float64(scale):
    n = 64
    w = K.PreparedLinear(torch.eye(n, device=DEV), None, L.MMA_F16)
    x = (torch.linspace(-1, 1, 4096 * n, device=DEV) * scale).half().view(-1, n)
    got = K.linear(x, w, act=L.ACT_GELU_ERF, out_dtype=torch.float32).double()
    xd = x.double()
    want = 0.5 * xd * torch.special.erfc(-xd * 0.5 ** 0.5)
    # Phi is off by at most a few fp32 roundings of values up to 1 (4 * 2^-24), and the last
    # product adds one of its own
    assert bool(((got - want).abs() <= 2.5e-7 * xd.abs() + 1e-45).all())
    assert bool((got[xd <= -14] == 0).all()), "the lower tail underflows to zero"
