"""The fused transformer stack on gfx950, expressed as a plan.

Mirrors `kernelforge/optimized.py` (`Plan` :54-121, `LADDER` :126-145,
`FusedTransformer` :166-585, `GraphRunner` :588-625, `build_shared` :632-651). Every
device op of the forward is a libkf950 kernel:

    mask_prep                               once per forward (kv_len / prefix per sequence)
    add_mask_ln(x, -, keep, norm1[0])       entry LayerNorm
    per layer:
      gemm(h, Wqkv)                         fused QKV projection      -> qkv [M, 3d]
      flash(q, k, v views of qkv)           causal + key padding      -> ctx [B, S, H, Dh]
      gemm(ctx, Wo)                         out_proj
      add_mask_ln(res, attn, keep, norm2)   residual + mask + LN
      gemm(h, W1) + erf-GELU epilogue       ffn_in
      gemm(f, W2)                           ffn_out
      add_mask_ln(res, ffn, keep, next)     next layer's norm1, or final_norm + mask

Precision is chosen per stage ("attn" = QKV GEMM + attention, "out_proj", "ffn1",
"ffn2"): "f16x3" / "bf16x3" (split fp32 on the fp16/bf16 MFMA, fp32-level accuracy),
"f16x3p" (f16x3 with the attention probabilities as one fp16 plane in P.V),
"f16x2" (activation one fp16 plane, weight hi/lo planes: two MFMAs; for "attn" the QKV
GEMM, the attention staying f16x3), "f16x2p" (f16x2 with the probabilities as one plane),
"f16x3s" (attention only: an f16x3 QKV GEMM feeding the single-pass fp16 attention),
"float16" / "bfloat16" (single pass), "float32" (fp32 MFMA). The residual stream is
fp32; each activation is stored in the operand format of the stage that consumes it (X2
planes for a split stage, 16-bit for a single-pass one); the QKV GEMM writes q, k split
and v transposed (the attention layout). Mask placement follows docs/EQUIVALENCE.md of
the reference: rows are zeroed at each block boundary inside the fused LayerNorm, and
after the final norm.
"""
from __future__ import annotations

import dataclasses
from typing import Dict, List, Optional, Tuple

import torch
import torch.nn as nn

from . import _lib as L
from . import kernels as K
from .model import BaselineTransformer, TransformerConfig, reference_forward

DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16}
STAGES = ("attn", "out_proj", "ffn1", "ffn2")
PRECISIONS = ("auto", "float32", "float16", "bfloat16", "f16x3", "bf16x3", "f16x3p", "f16x2",
              "f16x2p", "f16x3s")


@dataclasses.dataclass(frozen=True)
class Plan:
    """A point in the optimization space (field names of `optimized.py:54-82`).

    `compute_dtype` and `overrides` name a stage precision from PRECISIONS ("auto" is the
    I/O dtype). `fuse_qkv` and `fused_norm` are always on in the native path and kept for
    the table schema; `torch_compile` is accepted in tables but never used (no tracing
    compiler on this path); `flash_block` is (BLOCK_M, BLOCK_N, wavefronts, LDS stages);
    `smem_kb` is the LDS budget (160 KB per CU on gfx950). `match_score_rounding` rounds
    the attention scores as the reference's narrow forward does (16-bit I/O whose attention
    stage runs the single-pass MFMA of that type; KF_FLASH_ROUND_SCORES).
    """

    name: str = "default"
    compute_dtype: str = "f16x3"
    residual_dtype: str = "float32"
    fuse_qkv: bool = True
    attention: str = "flash"          # flash | baseline
    fused_norm: bool = True
    cuda_graph: bool = False          # hipGraph capture of the whole stack
    torch_compile: Optional[str] = None
    flash_block: Optional[Tuple[int, int, int, int]] = None
    smem_kb: float = K.LDS_KB
    overrides: Tuple[Tuple[str, str], ...] = ()
    match_score_rounding: bool = False

    def stage_precision(self, stage: str, io_dtype: torch.dtype) -> str:
        name = dict(self.overrides).get(stage, self.compute_dtype)
        if name == "auto":
            name = {torch.float32: "float32", torch.float16: "float16",
                    torch.bfloat16: "bfloat16"}[io_dtype]
        if name not in K.MODES:
            raise ValueError(f"unknown stage precision {name!r}")
        return name

    def stage_mode(self, stage: str, io_dtype: torch.dtype) -> int:
        return K.MODES[self.stage_precision(stage, io_dtype)]

    def residual_torch_dtype(self, io_dtype: torch.dtype) -> torch.dtype:
        return io_dtype if self.residual_dtype == "auto" else DTYPES[self.residual_dtype]

    def with_override(self, stage: str, precision: str) -> "Plan":
        kept = tuple((s, d) for s, d in self.overrides if s != stage)
        return dataclasses.replace(self, overrides=kept + ((stage, precision),),
                                   name=f"{self.name}+{stage}:{precision}")

    def describe(self) -> str:
        bits = [f"compute={self.compute_dtype}", f"residual={self.residual_dtype}",
                f"attn={self.attention}"]
        if self.cuda_graph:
            bits.append("hip-graph")
        if self.match_score_rounding:
            bits.append("score-rounding")
        if self.overrides:
            bits.append("[" + ",".join(f"{s}={d}" for s, d in self.overrides) + "]")
        if self.flash_block:
            bits.append(f"block={self.flash_block}")
        return " ".join(bits)


LADDER: Dict[str, Plan] = {
    "baseline": Plan("baseline", compute_dtype="auto", residual_dtype="auto",
                     fuse_qkv=False, attention="baseline", fused_norm=False),
    "fp32": Plan("fp32", compute_dtype="float32"),
    "bf16x3": Plan("bf16x3", compute_dtype="bf16x3"),
    "f16x3": Plan("f16x3", compute_dtype="f16x3"),
    "graph": Plan("graph", compute_dtype="f16x3", cuda_graph=True),
    "half": Plan("half", compute_dtype="float16"),
    "half_graph": Plan("half_graph", compute_dtype="float16", cuda_graph=True),
    "f16x3p": Plan("f16x3p", compute_dtype="f16x3", overrides=(("attn", "f16x3p"),)),
    "f16x2": Plan("f16x2", compute_dtype="f16x2", overrides=(("attn", "f16x2p"),)),
    "f16x3s": Plan("f16x3s", compute_dtype="f16x3", overrides=(("attn", "f16x3s"),)),
}


@dataclasses.dataclass(frozen=True)
class MemoryModel:
    """How many sequences one pass of the native forward may hold.

    The reference sizes its batch slices from a calibrated peak working set
    (`kernelforge/optimized.py:288-364`): LIVE_TENSORS activation tensors of the layer's
    widest row (max(d_model, ffn_dim) elements) per sequence, and a pass may take
    `headroom` of what is left once the whole output is allocated. Those two constants are
    the reference's calibration and are kept as data. Sizing needs only shapes and a byte
    count, so it is testable without a device; the device is queried only when a whole
    batch's working set passes `probe_above`.
    """
    widest: int
    d_model: int
    live_tensors: int = 32
    headroom: float = 0.55
    probe_above: int = 8 * 2**30

    @staticmethod
    def of(config: TransformerConfig) -> "MemoryModel":
        return MemoryModel(max(config.d_model, config.ffn_dim), config.d_model)

    def working_set(self, sequences: int, seq_len: int, itemsize: int) -> int:
        """Modelled peak bytes of one pass over `sequences` sequences."""
        return sequences * seq_len * self.widest * self.live_tensors * itemsize

    def sequences_per_pass(self, batch: int, seq_len: int, itemsize: int, free: int) -> int:
        """Largest pass (1 .. batch sequences) whose working set fits `free` bytes."""
        if batch <= 1:
            return batch
        output = batch * seq_len * self.d_model * itemsize
        usable = int((free - output) * self.headroom)
        per_sequence = max(1, self.working_set(1, seq_len, itemsize))
        return min(batch, max(1, usable // per_sequence))


class FusedTransformer(BaselineTransformer):
    """Drop-in for `BaselineTransformer` (same parameters) running the native stack.

    Weight planes for the chosen stage precisions are derived lazily on the first
    forward (inside the caller's warm-up) and dropped whenever parameters are reloaded
    or moved.
    """

    memory_budget_bytes = None   # a cap on a pass's working set; None: what the device has free

    def __init__(self, config: TransformerConfig, plan: Optional[Plan] = None):
        super().__init__(config)
        self.plan = plan or LADDER["graph"]
        self._prepared_key: Optional[tuple] = None
        self._layers_w: List[dict] = []
        self._graphs: Dict[tuple, "GraphRunner"] = {}

    # --- weight preparation --------------------------------------------------
    def _invalidate(self) -> None:
        self._prepared_key = None
        self._layers_w = []
        self._graphs = {}

    def _load_from_state_dict(self, *args, **kwargs):
        self._invalidate()
        return super()._load_from_state_dict(*args, **kwargs)

    def _apply(self, fn, *args, **kwargs):
        self._invalidate()
        return super()._apply(fn, *args, **kwargs)

    def _prepare(self, io_dtype: torch.dtype, device: torch.device) -> None:
        modes = tuple(self.plan.stage_mode(s, io_dtype) for s in STAGES)
        key = (modes, device)
        if self._prepared_key == key:
            return
        m_attn, m_out, m_f1, m_f2 = modes
        prepared = []
        with torch.no_grad():
            for layer in self.layers:
                a = layer.attention
                wqkv = torch.cat([a.q_proj.weight, a.k_proj.weight, a.v_proj.weight], 0)
                bqkv = torch.cat([a.q_proj.bias, a.k_proj.bias, a.v_proj.bias], 0)
                prepared.append({
                    "qkv": K.PreparedLinear(wqkv, bqkv, m_attn),
                    "out": K.PreparedLinear(a.out_proj.weight, a.out_proj.bias, m_out),
                    "ffn_in": K.PreparedLinear(layer.ffn_in.weight, layer.ffn_in.bias, m_f1),
                    "ffn_out": K.PreparedLinear(layer.ffn_out.weight, layer.ffn_out.bias, m_f2),
                })
        self._layers_w = prepared
        self._prepared_key = key

    # --- forward ---------------------------------------------------------------
    def forward(self, x: torch.Tensor,
                valid_token_mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        if self.plan.attention == "baseline":
            # the reference forward itself (restated op for op, `model.reference_forward`,
            # so that no bf16 batched product takes a transposed right operand); with
            # cuda_graph it is replayed from a hipGraph (same kernels, same arithmetic:
            # bit-exact, minus the per-op launches)
            if self.plan.cuda_graph and x.is_cuda and not torch.cuda.is_current_stream_capturing():
                return self._graph_forward(x, valid_token_mask)
            return reference_forward(self, x, valid_token_mask)
        if not x.is_cuda:
            raise RuntimeError("FusedTransformer runs on the GPU; the input is on "
                               f"{x.device}")
        chunk = self._batch_chunk(x)
        if chunk < x.shape[0]:
            return self._chunked_forward(x, valid_token_mask, chunk)
        if self.plan.cuda_graph and not torch.cuda.is_current_stream_capturing():
            return self._graph_forward(x, valid_token_mask)
        try:
            return self._eager_forward(x, valid_token_mask)
        except torch.cuda.OutOfMemoryError:
            if x.shape[0] <= 1:
                raise
            torch.cuda.empty_cache()
            return self._chunked_forward(x, valid_token_mask, 1)

    def set_memory_budget(self, budget_bytes):
        """Cap the bytes one pass may use (`optimized.py:301-311`), e.g. when another
        model shares the card; None sizes passes by what the device reports free.
        Smaller caps mean more, smaller passes and the same result."""
        if budget_bytes is not None and budget_bytes <= 0:
            raise ValueError("memory budget must be positive, or None")
        self.memory_budget_bytes = budget_bytes
        return self

    def _chunk_for_budget(self, B, S, dtype, free_bytes) -> int:
        """Sequences per pass for a [B, S] batch of `dtype` given `free_bytes`."""
        return MemoryModel.of(self.config).sequences_per_pass(B, S, dtype.itemsize, free_bytes)

    def _batch_chunk(self, x) -> int:
        """Sequences per pass for this input: the whole batch unless its modelled working
        set passes the probe threshold (or a budget is set), then what fits."""
        B, S, _ = x.shape
        if B <= 1 or not x.is_cuda:
            return B
        mm = MemoryModel.of(self.config)
        free = self.memory_budget_bytes
        if free is None:
            if mm.working_set(B, S, 4) < mm.probe_above:
                return B                       # no driver query for ordinary shapes
            try:
                free = torch.cuda.mem_get_info(x.device)[0]
            except RuntimeError:               # pragma: no cover
                return B
        return mm.sequences_per_pass(B, S, 4, free)

    def _chunked_forward(self, x, valid_token_mask, chunk):
        """The forward in passes of at most `chunk` sequences, written into one output.

        No op mixes sequences, so a pass over rows [lo, hi) is the forward of those rows.
        A pass that runs out of memory is split in two halves, each run (and split again)
        in turn; the largest pass that succeeded bounds the passes planned after it. Rows
        already written stay written; a single sequence that does not fit re-raises."""
        B = x.shape[0]
        out = torch.empty_like(x)

        def run(lo: int, hi: int) -> int:
            try:
                keep = None if valid_token_mask is None else valid_token_mask[lo:hi]
                out[lo:hi] = self._eager_forward(x[lo:hi], keep)
                return hi - lo
            except torch.cuda.OutOfMemoryError:
                if hi - lo == 1:
                    raise
            torch.cuda.empty_cache()
            mid = lo + (hi - lo) // 2
            return max(run(lo, mid), run(mid, hi))

        cap, lo = max(1, chunk), 0
        while lo < B:
            hi = min(B, lo + cap)
            cap = min(cap, run(lo, hi))
            lo = hi
        return out

    def _eager_forward(self, x: torch.Tensor,
                       valid_token_mask: Optional[torch.Tensor]) -> torch.Tensor:
        cfg = self.config
        B, S, d = x.shape
        M, H = B * S, cfg.num_heads
        Dh = d // H
        io_dtype = x.dtype
        if io_dtype not in (torch.float32, torch.float16, torch.bfloat16):
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     f"native path takes float32/16-bit I/O, got {io_dtype}")
        if io_dtype != torch.float32 and self.plan.residual_dtype != "float32":
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     "16-bit I/O runs the native stack with a float32 "
                                     "residual stream only")
        if not K.flash_supported(Dh):
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     f"head_dim {Dh} has no flash kernel")
        self._prepare(io_dtype, x.device)
        rdtype = self.plan.residual_torch_dtype(io_dtype)
        m_attn, m_out, m_f1, m_f2 = (self.plan.stage_mode(s, io_dtype) for s in STAGES)
        # Each producer writes its consumer's operand format: X2 planes for a split-mode
        # GEMM, the 16-bit type for a single-pass one, fp32 for the fp32 MFMA.
        h_attn = K.planes_format(m_attn)                  # LN output -> QKV GEMM
        h_ffn = K.planes_format(m_f1)                     # LN output -> ffn_in
        ctx_fmt = K.planes_format(m_out)                  # attention output -> out_proj
        hid_fmt = K.planes_format(m_f2)                   # GELU output -> ffn_out
        single_attn = self.plan.stage_precision("attn", io_dtype) in K.SINGLE_ATTN_PRECISIONS
        flash_mode = (L.MMA_F16 if single_attn else
                      m_attn if m_attn not in (L.MMA_F32, L.MMA_F16X2) else L.MMA_F16X3)
        K.check_block(self.plan.flash_block, S, Dh, self.plan.smem_kb, flash_mode)
        p16 = self.plan.stage_precision("attn", io_dtype) in K.P16_PRECISIONS
        # the reference's narrow score rounding (`optimized.py:523`): only where attention
        # runs the single-pass MFMA of the 16-bit I/O type
        rs = (self.plan.match_score_rounding
              and flash_mode == {torch.float16: L.MMA_F16, torch.bfloat16: L.MMA_BF16}.get(io_dtype))

        keep = kv_len = prefix = None
        if valid_token_mask is not None:
            keep2d = valid_token_mask
            if keep2d.dtype != torch.bool:
                keep2d = keep2d != 0
            keep2d = keep2d.contiguous().view(torch.uint8)
            keep = keep2d.reshape(M)
            kv_len, prefix = K.mask_prep(keep2d)
        else:
            keep2d = None

        res = x.reshape(M, d)
        if io_dtype != torch.float32:        # 16-bit input: widened once, fp32 inside
            res = res.float()
        if self._rows_fused(rdtype, (m_attn, m_out, m_f1, m_f2)):
            return self._narrow_stack(res, keep, keep2d, kv_len, prefix, B, S, io_dtype,
                                      ctx_fmt, single_attn, p16, rs).view(B, S, d)
        res, h = K.add_mask_layernorm(res, None, keep, self.layers[0].norm1.weight,
                                      self.layers[0].norm1.bias, self.layers[0].norm1.eps,
                                      out_dtype=h_attn, residual_dtype=rdtype)
        n = len(self.layers)
        for i, layer in enumerate(self.layers):
            w = self._layers_w[i]
            ctx = K._alloc((B, S, H, Dh), ctx_fmt, x.device)
            if m_attn != L.MMA_F32:
                # QKV GEMM writes q, split k and transposed v^T for the attention kernel
                ops = K.linear_qkv(h, w["qkv"], B, S, H, Dh, single=single_attn)
                K.flash_attention_ops(ops, keep=keep2d, causal=cfg.causal, sm_scale=Dh ** -0.5,
                                      out=ctx.permute(0, 2, 1, 3), kv_len=kv_len,
                                      prefix=prefix, skip_pad_rows=keep is not None,
                                      p16=p16, round_scores=rs)
            else:
                qkv = K.linear(h, w["qkv"], out_dtype=torch.float32)      # [M, 3d]
                q5 = qkv.view(B, S, 3, H, Dh)
                q, k, v = (q5[:, :, j].permute(0, 2, 1, 3) for j in range(3))
                K.flash_attention(q, k, v, keep=keep2d, causal=cfg.causal, sm_scale=Dh ** -0.5,
                                  out=ctx.permute(0, 2, 1, 3), mode=flash_mode,
                                  kv_len=kv_len, prefix=prefix, skip_pad_rows=keep is not None,
                                  p16=p16, round_scores_to=io_dtype if rs else None)
            attn = K.linear(ctx.view(M, d), w["out"], out_dtype=torch.float32)
            res, h = K.add_mask_layernorm(res, attn, keep, layer.norm2.weight,
                                          layer.norm2.bias, layer.norm2.eps,
                                          out_dtype=h_ffn, residual_dtype=rdtype)
            f = K.linear(h, w["ffn_in"], act=L.ACT_GELU_ERF, out_dtype=hid_fmt)
            f = K.linear(f, w["ffn_out"], out_dtype=torch.float32)
            last = i == n - 1
            nxt = self.final_norm if last else self.layers[i + 1].norm1
            res, h = K.add_mask_layernorm(res, f, keep, nxt.weight, nxt.bias, nxt.eps,
                                          mask_out=last,
                                          out_dtype=io_dtype if last else h_attn,
                                          residual_dtype=rdtype, want_residual=not last)
        return h.view(B, S, d)

    def _rows_fused(self, rdtype, modes) -> bool:
        """Whether the row-wise part of each layer runs as one kernel (kf_layer_block): a
        width it serves, fp16-family stages and fp32 norm parameters (16-bit models keep
        theirs in 16 bits) that it can read in 16-byte pieces."""
        cfg = self.config
        norms = [n for layer in self.layers for n in (layer.norm1, layer.norm2)] + [self.final_norm]
        return (rdtype == torch.float32
                and K.layer_block_supported(cfg.d_model, cfg.ffn_dim, modes)
                and all(t.dtype == torch.float32 and t.is_contiguous() and t.data_ptr() % 16 == 0
                        for n in norms for t in (n.weight, n.bias)))

    def _narrow_stack(self, res, keep, keep2d, kv_len, prefix, B, S, io_dtype, ctx_fmt,
                      single_attn, p16, rs):
        """The stack of a narrow model: per layer attention and one row kernel from the
        attention output to the next layer's q, k, v^T (the last one: to the output)."""
        cfg = self.config
        H, Dh = cfg.num_heads, cfg.d_model // cfg.num_heads
        M = B * S

        def norm(ln):
            return ln.weight, ln.bias, ln.eps

        def qkv(i):
            return self._layers_w[i]["qkv"], B, S, H, Dh, single_attn

        if res.stride(1) != 1 or res.stride(0) % 4 or res.data_ptr() % 16:
            res = res.clone(memory_format=torch.contiguous_format)
        # the first residual is x itself: the row kernel applies the mask where it reads it
        _, ops = K.layer_block(res, keep, norm(self.layers[0].norm1), qkv=qkv(0),
                               want_residual=False)
        for i, layer in enumerate(self.layers):
            w = self._layers_w[i]
            last = i + 1 == len(self.layers)
            ctx = K._alloc((B, S, H, Dh), ctx_fmt, res.device)
            K.flash_attention_ops(ops, keep=keep2d, causal=cfg.causal, sm_scale=Dh ** -0.5,
                                  out=ctx.permute(0, 2, 1, 3), kv_len=kv_len, prefix=prefix,
                                  skip_pad_rows=keep is not None, p16=p16, round_scores=rs)
            tail = (ctx.view(M, cfg.d_model), w["out"], norm(layer.norm2), w["ffn_in"], w["ffn_out"])
            if last:
                return K.layer_block(res, keep, norm(self.final_norm), tail=tail,
                                     want_residual=False, out_dtype=io_dtype)[1]
            res, ops = K.layer_block(res, keep, norm(self.layers[i + 1].norm1), tail=tail,
                                     qkv=qkv(i + 1))

    # --- graph path --------------------------------------------------------------
    def _body(self, x, valid_token_mask):
        """What a graph captures: the native stack, or the reference forward."""
        if self.plan.attention == "baseline":
            return reference_forward(self, x, valid_token_mask)
        return self._eager_forward(x, valid_token_mask)

    def _graph_forward(self, x, valid_token_mask):
        key = (tuple(x.shape), x.dtype, x.device,
               None if valid_token_mask is None else
               (tuple(valid_token_mask.shape), valid_token_mask.dtype))
        runner = self._graphs.get(key)
        if runner is None:
            runner = GraphRunner(self, x, valid_token_mask)
            self._graphs[key] = runner
        return runner(x, valid_token_mask)


class GraphRunner:
    """The whole stack captured once per (shape, dtype, mask shape) in a HIP graph
    (`optimized.py:588-625`): warm-up on a side stream, capture, then replay against
    static buffers; the output is cloned so a held result survives the next replay.

    The runner keeps no reference to its model (the model holds its runners): without the
    cycle a graph and its memory pool go when the model does, not at whatever later
    allocation the cyclic garbage collector runs on."""

    def __init__(self, model: FusedTransformer, x, mask):
        self.static_x = x.clone()
        self.static_mask = None if mask is None else mask.clone()
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for _ in range(2):
                model._body(self.static_x, self.static_mask)
        torch.cuda.current_stream().wait_stream(stream)
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.static_out = model._body(self.static_x, self.static_mask)

    def __call__(self, x, mask):
        self.static_x.copy_(x)
        if self.static_mask is not None and mask is not None:
            self.static_mask.copy_(mask)
        self.graph.replay()
        return self.static_out.clone()


def build(config: TransformerConfig, plan: Plan) -> FusedTransformer:
    return FusedTransformer(config, plan)


def build_shared(config: TransformerConfig, plan: Plan,
                 reference: nn.Module) -> FusedTransformer:
    """A candidate sharing `reference`'s parameter tensors (`optimized.py:632-651`)."""
    with torch.device("meta"):
        model = FusedTransformer(config, plan)
    model.load_state_dict(reference.state_dict(), assign=True)
    return model.eval()
