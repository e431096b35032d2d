"""The graph path's host side on the CPU: which inputs reach the entry kernels as they are, that
threads which share a runner keep their own data, and which calls capture the whole stack."""
from __future__ import annotations

import threading
import time
from types import SimpleNamespace

import pytest
import torch

from techjam2026_amd.model import TransformerConfig
from techjam2026_amd.optimized import LADDER, FusedTransformer, GraphRunner, _entry_rows

D, S = 32, 12


@pytest.mark.parametrize("make,as_is", [
    (lambda t: t[: S * D].view(S, D), True),
    (lambda t: t[: 2 * S * D].view(S, 2 * D)[:, :D], True),         # rows of a wider tensor
    (lambda t: t[4: 4 + S * D].view(S, D), True),
    (lambda t: t[1: 1 + S * D].view(S, D), False),                  # 4-byte aligned
    (lambda t: t[: S * (D + 2)].view(S, D + 2)[:, :D], False),      # every other row aligned
    (lambda t: t[: 2 * S * D].view(S, 2 * D)[:, ::2], False),
    (lambda t: t[: S * D].view(D, S).t(), False),
    (lambda t: t[:D].expand(S, D), False),                          # one row repeated
    (lambda t: t.unfold(0, D, 16)[:S], False),                      # overlapping frames
    (lambda t: t.unfold(0, D, 4)[:S], False),
    (lambda t: t[:D].expand(5, D)[:1], False),                      # one row of stride 0
])
def test_entry_rows_are_dense_and_aligned(make, as_is):
    storage = torch.randn(4 * S * D)
    assert storage.data_ptr() % 16 == 0
    rows = make(storage)
    got = _entry_rows(rows)
    assert torch.equal(got, rows)
    assert (got.data_ptr() == rows.data_ptr()) == as_is
    assert got.stride(1) == 1 and got.stride(0) >= D
    assert got.stride(0) % 4 == 0 and got.data_ptr() % 16 == 0


class _OneLayerModel:
    """The two ends of a one-layer narrow model as `GraphRunner` calls them: the last kernel
    takes the rows that the first one returned, and the buffer between them is shared."""

    def _enter(self, p, x, into_graph=False):
        p["buffer"] = float(x[0])
        return x

    def _leave(self, p, first):
        return float(first[0]), p["buffer"]


class _SlowGraph:
    def replay(self):
        time.sleep(0.002)


def test_threads_that_share_a_runner_keep_their_own_rows():
    runner = GraphRunner.__new__(GraphRunner)            # no device: the captured part is a stand-in
    runner.lock, runner.x, runner.mask = threading.Lock(), None, None
    runner.state, runner.graph = {}, _SlowGraph()
    wrong, model = [], _OneLayerModel()

    def calls(value):
        for i in range(20):
            x = torch.full((4,), float(value * 100 + i))
            got = runner(model, x, None)
            if got != (float(x[0]), float(x[0])):
                wrong.append((value, i, got))

    threads = [threading.Thread(target=calls, args=(v,)) for v in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(30)
    assert not wrong and not any(t.is_alive() for t in threads)


@pytest.mark.parametrize("narrow,d,F,layers,B,S,whole", [
    (True, 32, 32, 1, 1, 16, True), (False, 32, 32, 1, 1, 16, True),
    (False, 128, 256, 1, 32, 128, True), (False, 512, 1024, 1, 2, 128, True),
    (True, 128, 256, 1, 128, 128, False), (True, 128, 128, 4, 1, 128, False),
    (False, 512, 1024, 1, 16, 128, False), (False, 512, 2048, 6, 16, 512, False),
    (True, 64, 64, 1, 1, 4096, False),                   # attention over one long sequence
])
def test_calls_that_wait_for_the_host_capture_the_whole_stack(narrow, d, F, layers, B, S, whole):
    model = FusedTransformer(TransformerConfig(B, S, d, max(1, d // 64), F, layers, True), LADDER["graph"])
    plane = {"qkv": 3 * d * d, "out": d * d, "ffn_in": d * F, "ffn_out": d * F}
    model._layers_w = [{k: SimpleNamespace(hi=torch.empty(n, dtype=torch.float16),
                                           lo=torch.empty(n, dtype=torch.float16))
                        for k, n in plane.items()} for _ in range(layers)]
    assert model._copies_pay(SimpleNamespace(B=B, S=S, narrow=narrow)) == whole
