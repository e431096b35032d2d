"""The graph path launches its first and last kernels around the captured ones, on the
caller's input and into a new output: equal to the eager forward bit for bit over replays with
new inputs, whatever their strides and the mask's type, with eager work in between, in and
outside inference mode, one layer deep (nothing but attention is captured) and deeper."""
from __future__ import annotations

import pytest
import torch

from techjam2026_amd.model import TransformerConfig
from techjam2026_amd.optimized import LADDER, build_shared
from tests.test_stack_gpu import make_model

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


@pytest.mark.parametrize("d,H,F,layers", [(128, 4, 192, 1), (64, 8, 64, 3), (512, 8, 512, 2)])
@pytest.mark.parametrize("mask", ["bool", "float", None])
def test_replays_equal_the_eager_forward(d, H, F, layers, mask):
    B, S = 3, 45
    base = make_model(TransformerConfig(B, S, d, H, F, layers, True), device=DEV)
    eager = build_shared(base.config, LADDER["f16x3"], base)
    graphed = build_shared(base.config, LADDER["graph"], base)
    g = torch.Generator(device=DEV).manual_seed(1)
    held = []
    for i in range(4):
        x = torch.randn(B, S, 2 * d, device=DEV, generator=g)
        x = (x[..., :d].contiguous(), x[..., :d], x[..., ::2], x.reshape(-1)[1:B * S * d + 1].view(B, S, d))[i]
        m = None
        if mask:
            m = torch.arange(S, device=DEV)[None] < torch.randint(1, S + 1, (B, 1), device=DEV, generator=g)
            m = m.float() if mask == "float" else m
        with torch.inference_mode(i % 2 == 0), torch.no_grad():
            want = eager(x, m)
            got = graphed(x, m)
            held.append((got, want))
            torch.cuda.synchronize()
    assert len(graphed._graphs) == 1
    for i, (got, want) in enumerate(held):
        assert torch.equal(got, want), f"call {i}"
