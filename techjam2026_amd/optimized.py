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

In narrow models (`FusedTransformer._rows_fused`) one kernel, kf_layer_block, does all of a
layer but the attention: from its output to the next layer's q, k, v^T.

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
import threading
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
        p = self._plan_pass(x, valid_token_mask)
        p.res = self._enter(p, x)
        self._layer_steps(p)
        return self._leave(p, p.res)

    # A forward in three parts: `_enter` launches the kernel that reads x, `_layer_steps`
    # everything between, `_leave` the kernel that writes the output. `GraphRunner` captures
    # the middle and launches the two ends around it.
    def _plan_pass(self, x: torch.Tensor, valid_token_mask: Optional[torch.Tensor]) -> "_Pass":
        """Checks, weight planes and operand formats of a forward; launches no layer kernel."""
        cfg = self.config
        B, S, d = x.shape
        io_dtype = x.dtype
        if io_dtype not in (torch.float32, torch.float16, torch.bfloat16):
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     f"native path takes float32/16-bit I/O, got {io_dtype}")
        if io_dtype != torch.float32 and self.plan.residual_dtype != "float32":
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     "16-bit I/O runs the native stack with a float32 "
                                     "residual stream only")
        Dh = d // cfg.num_heads
        if not K.flash_supported(Dh):
            raise L.UnsupportedError("FusedTransformer", L.EUNSUPPORTED,
                                     f"head_dim {Dh} has no flash kernel")
        self._prepare(io_dtype, x.device)
        modes = m_attn, m_out, m_f1, m_f2 = tuple(self.plan.stage_mode(s, io_dtype) for s in STAGES)
        rdtype = self.plan.residual_torch_dtype(io_dtype)
        attn_name = self.plan.stage_precision("attn", io_dtype)
        single_attn = attn_name in K.SINGLE_ATTN_PRECISIONS
        flash_mode = (L.MMA_F16 if single_attn else
                      m_attn if m_attn not in (L.MMA_F32, L.MMA_F16X2) else L.MMA_F16X3)
        K.check_block(self.plan.flash_block, S, Dh, self.plan.smem_kb, flash_mode)
        # the reference's narrow score rounding (`optimized.py:523`): only where attention
        # runs the single-pass MFMA of the 16-bit I/O type
        rs = (self.plan.match_score_rounding
              and flash_mode == {torch.float16: L.MMA_F16, torch.bfloat16: L.MMA_BF16}.get(io_dtype))
        keep2d = valid_token_mask
        if keep2d is not None:
            if keep2d.dtype != torch.bool:
                keep2d = keep2d != 0
            keep2d = keep2d.contiguous().view(torch.uint8)
        # Each producer writes its consumer's operand format: X2 planes for a split-mode
        # GEMM, the 16-bit type for a single-pass one, fp32 for the fp32 MFMA.
        return _Pass(B, S, cfg.num_heads, Dh, io_dtype, rdtype, m_attn, single_attn, flash_mode,
                     attn_name in K.P16_PRECISIONS, rs,
                     h_attn=K.planes_format(m_attn), ctx_fmt=K.planes_format(m_out),
                     h_ffn=K.planes_format(m_f1), hid_fmt=K.planes_format(m_f2),
                     narrow=self._rows_fused(rdtype, modes), keep2d=keep2d,
                     keep=None if keep2d is None else keep2d.reshape(B * S))

    def _enter(self, p: "_Pass", x: torch.Tensor, into_graph: bool = False) -> torch.Tensor:
        """The entry LayerNorm (narrow models: with the first q, k, v^T); returns the residual
        rows. `into_graph`: the outputs are the graph's inputs, buffers of their own, written
        again by each call; rows that no captured layer reads are the caller's own, and `p`
        does not keep them."""
        M, d = p.B * p.S, p.H * p.Dh
        res = x.reshape(M, d)
        if p.io_dtype != torch.float32:      # 16-bit input: widened once, fp32 inside
            res = res.float()
        res = _entry_rows(res)
        if p.narrow:
            if p.entry is None:
                # the first residual is x itself (the row kernel applies the mask where it
                # reads it), unless a captured layer reads it
                p.entry = K.LayerBlock(M, d, x.device, p.keep, _norm_of(self.layers[0].norm1),
                                       qkv=self._qkv_of(p, 0),
                                       want_residual=into_graph and len(self.layers) > 1,
                                       check=False)
            s, p.ops = p.entry(res)
            return res if s is None else s
        first = self.layers[0].norm1
        s, p.h = K.add_mask_layernorm(res, None, p.keep, first.weight, first.bias, first.eps,
                                      out_dtype=p.h_attn, residual_dtype=p.rdtype,
                                      s_out=p.res, h_out=p.h)
        return s

    def _layer_steps(self, p: "_Pass") -> None:
        """From the entry kernel's outputs to the last kernel's inputs."""
        if p.keep2d is not None:
            p.kv_len, p.prefix = K.mask_prep(p.keep2d)
        if p.narrow:
            self._narrow_steps(p)
        else:
            self._wide_steps(p)

    def _leave(self, p: "_Pass", first: torch.Tensor) -> torch.Tensor:
        """The last kernel of the stack, into a new tensor; `first`: what `_enter` returned."""
        norm = self.final_norm
        if p.narrow:
            if p.exit is None:
                p.exit = K.LayerBlock(p.B * p.S, p.H * p.Dh, p.ctx.hi.device if isinstance(
                                          p.ctx, K.Planes) else p.ctx.device, p.keep, _norm_of(norm),
                                      tail=self._tail_of(p, len(self.layers) - 1),
                                      want_residual=False, out_dtype=p.io_dtype, check=False)
            out = p.exit(first if len(self.layers) == 1 else p.last_res)[1]
        else:
            out = K.add_mask_layernorm(p.last_res, p.f, p.keep, norm.weight, norm.bias, norm.eps,
                                       mask_out=True, out_dtype=p.io_dtype,
                                       residual_dtype=p.rdtype, want_residual=False)[1]
        return out.view(p.B, p.S, p.H * p.Dh)

    def _attend(self, p: "_Pass", ops) -> "K.Act":
        """Attention on operands in its layout -> ctx [B, S, H, Dh] in out_proj's format."""
        ctx = K._alloc((p.B, p.S, p.H, p.Dh), p.ctx_fmt, ops.q.device)
        K.flash_attention_ops(ops, keep=p.keep2d, causal=self.config.causal,
                              sm_scale=p.Dh ** -0.5, out=ctx.permute(0, 2, 1, 3),
                              kv_len=p.kv_len, prefix=p.prefix,
                              skip_pad_rows=p.keep2d is not None, p16=p.p16, round_scores=p.rs)
        return ctx

    # --- wide models: one kernel per operation -----------------------------------
    def _wide_steps(self, p: "_Pass") -> None:
        B, S, H, Dh, M, d = p.B, p.S, p.H, p.Dh, p.B * p.S, p.H * p.Dh
        res, h, n = p.res, p.h, len(self.layers)
        for i, layer in enumerate(self.layers):
            w = self._layers_w[i]
            if p.m_attn != L.MMA_F32:
                # QKV GEMM writes q, split k and transposed v^T for the attention kernel
                ctx = self._attend(p, K.linear_qkv(h, w["qkv"], B, S, H, Dh, single=p.single_attn))
            else:
                ctx = K._alloc((B, S, H, Dh), p.ctx_fmt, res.device)
                qkv = K.linear(h, w["qkv"], out_dtype=torch.float32)      # [M, 3d]
                q5 = qkv.view(B, S, 3, H, Dh)
                q, k, v = (q5[:, :, j].permute(0, 2, 1, 3) for j in range(3))
                K.flash_attention(q, k, v, keep=p.keep2d, causal=self.config.causal,
                                  sm_scale=Dh ** -0.5, out=ctx.permute(0, 2, 1, 3),
                                  mode=p.flash_mode, kv_len=p.kv_len, prefix=p.prefix,
                                  skip_pad_rows=p.keep2d is not None, p16=p.p16,
                                  round_scores_to=p.io_dtype if p.rs else None)
            attn = K.linear(ctx.view(M, d), w["out"], out_dtype=torch.float32)
            res, h = K.add_mask_layernorm(res, attn, p.keep, layer.norm2.weight,
                                          layer.norm2.bias, layer.norm2.eps,
                                          out_dtype=p.h_ffn, residual_dtype=p.rdtype)
            f = K.linear(h, w["ffn_in"], act=L.ACT_GELU_ERF, out_dtype=p.hid_fmt)
            f = K.linear(f, w["ffn_out"], out_dtype=torch.float32)
            if i + 1 < n:
                nxt = self.layers[i + 1].norm1
                res, h = K.add_mask_layernorm(res, f, p.keep, nxt.weight, nxt.bias, nxt.eps,
                                              out_dtype=p.h_attn, residual_dtype=p.rdtype)
        p.last_res, p.f = res, f

    # --- narrow models: one kernel per layer beside attention ----------------------
    # The most weight bytes of a layer that the row kernel takes. Each of its blocks streams all
    # of them at about 100 GB/s, the chain of a launch however few the rows, where separate
    # kernels spread them over the chip. Six layers, f16x3, row kernel / today's separate
    # kernels / separate kernels with 128 x 128 GEMM tiles, us: d 128, F 512 (0.8 MB), 256 rows
    # 124 / 190 / 312; d 256, F 1024 (3.1 MB), 256 rows 272 / 212 / 430, 4096 rows 350 / 456 / 535,
    # 16384 rows 862 / 1045 / 1103; d 256, F 4096 (9.4 MB), 64 rows 664 / 264 / 682, 4096 rows
    # 737 / 776 / 993; F 8192 (17.8 MB), 64 rows 1177 / 355 / 1065. The line lies where the row
    # kernel would lose to what it replaced. With few rows the separate kernels win earlier
    # (from 2 MB at 256 rows), but a rule on rows would give a sequence other last bits in
    # another batch.
    ROW_KERNEL_BYTES = 8 << 20

    def _rows_fused(self, rdtype, modes) -> bool:
        """Whether the row-wise part of each layer runs as one kernel (kf_layer_block): a
        width it serves, fp16-family stages, weights of the shapes it reads, not too many of
        them for one block to stream, and fp32 norm parameters (16-bit models keep theirs in 16 bits) that it can read in 16-byte pieces."""
        d = self.config.d_model

        def fits(w):
            qkv, out, f1, f2 = w["qkv"], w["out"], w["ffn_in"], w["ffn_out"]
            return (K.layer_block_supported(d, f1.N, modes)
                    and (qkv.N, qkv.K, out.N, out.K, f1.K, f2.N, f2.K) == (3 * d, d, d, d, d, d, f1.N)
                    and all(lin.bias is not None and lin.bias.shape == (lin.N,)
                            for lin in (qkv, out, f1, f2)))

        norms = [n for layer in self.layers for n in (layer.norm1, layer.norm2)] + [self.final_norm]
        return (rdtype == torch.float32
                and all(fits(w) for w in self._layers_w)
                and max(self._layer_weight_bytes()) <= self.ROW_KERNEL_BYTES
                and all(t.dtype == torch.float32 and t.shape == (d,) and t.is_contiguous()
                        and t.data_ptr() % 16 == 0 for n in norms for t in (n.weight, n.bias)))

    def _qkv_of(self, p: "_Pass", i: int):
        return self._layers_w[i]["qkv"], p.B, p.S, p.H, p.Dh, p.single_attn

    def _tail_of(self, p: "_Pass", i: int):
        w = self._layers_w[i]
        return (p.ctx.view(p.B * p.S, p.H * p.Dh), w["out"], _norm_of(self.layers[i].norm2),
                w["ffn_in"], w["ffn_out"])

    def _narrow_steps(self, p: "_Pass") -> None:
        """Per layer attention, and one row kernel from its output to the next layer's q, k,
        v^T; the last row kernel is `_leave`."""
        res, ops = p.res, p.ops
        for i in range(len(self.layers)):
            p.ctx = self._attend(p, ops)
            if i + 1 < len(self.layers):
                res, ops = K.layer_block(res, p.keep, _norm_of(self.layers[i + 1].norm1),
                                         tail=self._tail_of(p, i), qkv=self._qkv_of(p, i + 1),
                                         check=False)
        p.last_res = res

    # --- graph path --------------------------------------------------------------
    def _layer_weight_bytes(self) -> List[int]:
        return [sum(t.numel() * t.element_size() for lin in w.values() for t in (lin.hi, lin.lo)
                    if t is not None) for w in self._layers_w]

    def _copies_pay(self, p: "_Pass") -> bool:
        """Whether a call of this shape waits for the host, so that two small copies around a
        graph of the whole stack cost less than launching its two ends beside the graph: those
        launches take the host 55 us a call in narrow models and 70 in wide ones, a copy in and
        a copy out 43 and 46, while on the device the copies add 6 to 10. The device's time is
        estimated from its launches, the weights (each block of the row kernel streams all of
        them) and the operations. Measured, ends / whole: one layer, d 32, 16 rows 53 / 41 us;
        d 128, 4096 rows 55 / 43, 16384 rows 54 / 60; in separate kernels d 32, 16 rows
        69 / 46, d 512, 256 rows 70 / 64, 1024 rows 73 / 79; four layers of d 128, 128 rows
        80 / 86 and, in separate kernels, 122 / 126."""
        cfg, layers = self.config, len(self.layers)
        weights = sum(self._layer_weight_bytes())
        d = cfg.d_model
        flops = p.B * p.S * layers * (8 * d * d + 4 * d * cfg.ffn_dim + 4 * p.S * d)
        if p.narrow:
            return 5.3 * (2 * layers + 2) + weights / 1e5 + flops / 1e8 < 42
        return 2.8 * (7 * layers + 2) + weights / 1.2e6 + flops / 1e8 < 45

    def _graph_forward(self, x, valid_token_mask):
        key = (tuple(x.shape), x.dtype, x.device,
               None if valid_token_mask is None else
               (tuple(valid_token_mask.shape), valid_token_mask.dtype))
        runner = self._graphs.get(key)
        if runner is None:
            kind = _BaselineGraph if self.plan.attention == "baseline" else GraphRunner
            runner = kind(self, x, valid_token_mask)
            self._graphs[key] = runner
        return runner(self, x, valid_token_mask)


def _entry_rows(rows: torch.Tensor) -> torch.Tensor:
    """Rows that the entry kernels read in 16-byte pieces: [M, d] itself, or a dense copy where
    rows overlap or repeat (x expanded over the batch or the sequence, frames of a signal: the
    kernels take row strides of at least d), are not of unit stride or are not 16-byte aligned
    (16384 unaligned rows of d 1024, one layer: 1110 us a forward copied, 1165 through the unaligned
    LayerNorm path)."""
    ld, unit = rows.stride()
    if unit == 1 and ld >= rows.shape[1] and ld % 4 == 0 and rows.data_ptr() % 16 == 0:
        return rows
    return rows.clone(memory_format=torch.contiguous_format)


def _norm_of(ln):
    return ln.weight, ln.bias, ln.eps


@dataclasses.dataclass
class _Pass:
    """One forward's settings and the tensors that pass between its parts."""
    B: int
    S: int
    H: int
    Dh: int
    io_dtype: torch.dtype
    rdtype: torch.dtype
    m_attn: int
    single_attn: bool
    flash_mode: int
    p16: bool
    rs: bool
    h_attn: object                          # LayerNorm output -> QKV GEMM
    ctx_fmt: object                         # attention output -> out_proj
    h_ffn: object                           # LayerNorm output -> ffn_in
    hid_fmt: object                         # GELU output -> ffn_out
    narrow: bool
    keep2d: Optional[torch.Tensor] = None   # [B, S] uint8
    keep: Optional[torch.Tensor] = None     # the same as [B * S]
    kv_len: Optional[torch.Tensor] = None
    prefix: Optional[torch.Tensor] = None
    res: Optional[torch.Tensor] = None      # residual rows after the entry kernel
    h: object = None                        # wide: its normalised rows
    ops: object = None                      # narrow: the first layer's q, k, v^T
    ctx: object = None                      # narrow: the last attention's output
    f: Optional[torch.Tensor] = None        # wide: the last ffn_out
    last_res: Optional[torch.Tensor] = None # residual rows before the last kernel
    entry: Optional[K.LayerBlock] = None    # narrow: the first and last row kernels
    exit: Optional[K.LayerBlock] = None


def _capture(warm, body):
    """A HIP graph of `body`, after two runs of `warm` on a side stream."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(2):
            warm()
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = body()
    return graph, out


class GraphRunner:
    """The stack captured once per (shape, dtype, mask shape) in a HIP graph
    (`optimized.py:588-625`): warm-up on a side stream, capture, then replay.

    Only the kernels between the first and the last are captured. The entry LayerNorm is
    launched on the caller's x and writes the graph's input buffers, the final one writes
    a new output tensor, so no call copies its input in or its output out (two passes over
    the activation: 490 of 2710 us for 10000 x 128 rows of d 128), and a held result survives
    the next replay. Calls so short that the host's launches are their time
    (`FusedTransformer._copies_pay`) capture the whole stack, between a copy of x and one of
    the output.

    The runner keeps no reference to its model (the model holds its runners): without the
    cycle a graph and its memory pool go when the model does, not at whatever later
    allocation the cyclic garbage collector runs on.

    The graph's buffers are the runner's: a call holds the lock from the first write of them to
    the launch of the last read, so threads that share a model and a stream each get the
    forward of their own x. Calls on different streams are the caller's to order."""

    def __init__(self, model: FusedTransformer, x, mask):
        self.lock = threading.Lock()
        with torch.inference_mode(False):
            # written by every call, from inference mode or not
            self.mask = None if mask is None else torch.empty(mask.shape, dtype=torch.bool,
                                                              device=mask.device)
        self._take_mask(mask)
        self.x = None
        p = self.state = model._plan_pass(x, self.mask)
        if model._copies_pay(p):
            with torch.inference_mode(False):
                self.x = torch.empty(x.shape, dtype=x.dtype, device=x.device)
            self.x.copy_(x.detach())

            def body():
                return model._eager_forward(self.x, self.mask)

            self.graph, self.out = _capture(body, body)
            return
        first = model._enter(p, x, into_graph=True)
        if len(model.layers) > 1 or not p.narrow:
            p.res = first                      # a buffer that the captured kernels read
        self.graph, _ = _capture(lambda: model._eager_forward(x, self.mask),
                                 lambda: model._layer_steps(p))

    def _take_mask(self, mask):
        if mask is not None:
            if mask.dtype == torch.bool:
                self.mask.copy_(mask)
            else:
                torch.ne(mask, 0, out=self.mask)

    def __call__(self, model, x, mask):
        with self.lock:
            self._take_mask(mask)
            if self.x is not None:
                self.x.copy_(x.detach() if x.requires_grad else x)
                self.graph.replay()
                return self.out.clone()
            first = model._enter(self.state, x, into_graph=True)
            self.graph.replay()
            return model._leave(self.state, first)


class _BaselineGraph:
    """The reference forward replayed from a HIP graph: the same kernels and arithmetic,
    bit for bit, minus the per-op launches. Static input and mask, cloned output."""

    def __init__(self, model: FusedTransformer, x, mask):
        self.static_x = x.clone()
        self.static_mask = None if mask is None else mask.clone()

        def body():
            return reference_forward(model, self.static_x, self.static_mask)

        self.graph, self.static_out = _capture(body, body)

    def __call__(self, model, x, mask):
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
