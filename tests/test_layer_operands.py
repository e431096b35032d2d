"""kf_layer_block's wrapper refuses operands that the kernel would read past their ends: each wrong
operand is named before anything is launched (on the CPU: operands that fit get as far as the
demand for device tensors)."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from techjam2026_amd import _lib as L
from techjam2026_amd import kernels as K
from techjam2026_amd.model import TransformerConfig
from techjam2026_amd.optimized import LADDER, FusedTransformer

M, D, F, B, S, H = 12, 64, 96, 2, 6, 4


def _linear(n, k, mode=L.MMA_F16X3, bias=True):
    return SimpleNamespace(N=n, K=k, mode=mode, hi=torch.zeros(n, k, dtype=torch.float16), lo=None,
                           bias=torch.zeros(n) if bias else None)


def _norm(d=D, dtype=torch.float32):
    return torch.ones(d, dtype=dtype), torch.zeros(d, dtype=dtype), 1e-5


def _planes(m=M, d=D, dtype=torch.float16):
    return K.Planes(torch.zeros(m, d, dtype=dtype), torch.zeros(m, d, dtype=dtype))


def _operands(**change):
    o = dict(keep=torch.ones(M, dtype=torch.uint8), norm=_norm(), ctx=_planes(), out=_linear(D, D),
             norm2=_norm(), f1=_linear(F, D), f2=_linear(D, F), w=_linear(3 * D, D), B=B, S=S, H=H,
             Dh=D // H, single=False)
    o.update(change)
    return (o["keep"], o["norm"]), dict(tail=(o["ctx"], o["out"], o["norm2"], o["f1"], o["f2"]),
                                        qkv=(o["w"], o["B"], o["S"], o["H"], o["Dh"], o["single"]))


def test_operands_that_fit_reach_the_device_check():
    for change in ({}, {"keep": None}, {"ctx": torch.zeros(M, D, dtype=torch.float16),
                                        "out": _linear(D, D, L.MMA_F16X2)}):
        args, options = _operands(**change)
        with pytest.raises(RuntimeError, match="device tensors"):
            K.LayerBlock(M, D, "cpu", *args, **options)


@pytest.mark.parametrize("change", [
    {"keep": torch.ones(M - 1, dtype=torch.uint8)}, {"keep": torch.ones(M)},
    {"keep": torch.ones(2 * M, dtype=torch.uint8)[::2]},
    {"norm": _norm(D - 4)}, {"norm": _norm(dtype=torch.float16)}, {"norm2": _norm(D // 2)},
    {"ctx": _planes(M - 1)}, {"ctx": _planes(M, D // 2)}, {"ctx": _planes(dtype=torch.bfloat16)},
    {"ctx": torch.zeros(M, D, dtype=torch.float16)},                   # one plane for f16x3
    {"ctx": K.Planes(*(torch.zeros(M, 2 * D, dtype=torch.float16)[:, :D] for _ in "ab"))},
    {"out": _linear(D, D - 32)}, {"out": _linear(D, D, L.MMA_BF16X3)}, {"out": _linear(D, D, bias=False)},
    {"f1": _linear(F, D // 2)}, {"f1": _linear(F + 32, D)}, {"f2": _linear(D, F - 32)},
    {"f2": _linear(D - 32, F)}, {"w": _linear(2 * D, D)}, {"w": _linear(3 * D, D, L.MMA_F32)},
    {"S": S + 1}, {"B": 1}, {"H": 2}, {"w": _linear(3 * D, D, L.MMA_F16), "single": True},
])
def test_operands_that_do_not_fit_are_refused(change):
    args, options = _operands(**change)
    with pytest.raises(AssertionError):
        K.LayerBlock(M, D, "cpu", *args, **options)


def test_a_model_whose_weights_do_not_fit_keeps_the_separate_kernels():
    """The stack checks its weights once: layers changed after construction (a pruned
    feed-forward, a bias taken away) run the row kernel where it serves them."""
    def fused(modes=(L.MMA_F16X3,) * 4, **change):
        model = FusedTransformer(TransformerConfig(B, S, D, H, F, 2, True), LADDER["graph"])
        good = dict(qkv=_linear(3 * D, D), out=_linear(D, D), ffn_in=_linear(F, D), ffn_out=_linear(D, F))
        model._layers_w = [good, dict(good, **change)]
        return model._rows_fused(torch.float32, modes)

    assert fused()
    assert fused(ffn_in=_linear(F - 32, D), ffn_out=_linear(D, F - 32))
    assert not fused(ffn_in=_linear(F - 8, D), ffn_out=_linear(D, F - 8))
    assert not fused(ffn_out=_linear(D, F - 32))
    assert not fused(out=_linear(D, D, bias=False))
    assert not fused(modes=(L.MMA_BF16X3,) * 4)


@pytest.mark.parametrize("d,ffn,planes,row_kernel", [
    (256, 1024, 2, True), (256, 3072, 2, True), (256, 4096, 2, False), (256, 8192, 1, False),
    (256, 6144, 1, True), (128, 4096, 2, True), (32, 4096, 2, True)])
def test_layers_of_many_weights_keep_the_separate_kernels(d, ffn, planes, row_kernel):
    mode = L.MMA_F16X3 if planes == 2 else L.MMA_F16

    def lin(n, k):
        w = _linear(n, k, mode)
        w.lo = w.hi if planes == 2 else None
        return w

    model = FusedTransformer(TransformerConfig(1, 64, d, 1, 32, 1, True), LADDER["graph"])
    model._layers_w = [dict(qkv=lin(3 * d, d), out=lin(d, d), ffn_in=lin(ffn, d), ffn_out=lin(d, ffn))]
    assert model._rows_fused(torch.float32, (mode,) * 4) == row_kernel
