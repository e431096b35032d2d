"""What a user of the stack has it do, as cases that can be timed and compared.

`listed()` names the cases, `draw(rng)` gives more of the same ranges. Each case is a dict
of plain values; `kind` says which public entry points it goes through:

* "call":      `submission.UserOptimizedTransformer`, the drop-in, with the plan that the
               dispatch table gives for the shape
* "layer":     `optimized.build_shared` with a plan of the table's kind, one layer deep (entry
               norm, attention, feed-forward, final norm)
* "attention": `kernels.flash_attention` on q, k, v views of one packed projection
* "mlp":       `kernels.add_mask_layernorm` and the two `kernels.linear` of a feed-forward block
* "norm":      `kernels.add_mask_layernorm`

Masks: "ones" (every position valid, what the organizer's harness passes without padding),
"prefix" (valid lengths uniform in [lo * S, S], the rest padding), "left" (padding in front,
up to a third of the row), "none" (no mask passed).
"""
import math

import torch

from techjam2026_amd import _lib as L
from techjam2026_amd import kernels as K
from techjam2026_amd.model import BaselineTransformer, TransformerConfig
from techjam2026_amd.optimized import Plan, build_shared
from techjam2026_amd.submission import UserOptimizedTransformer

DEVICE = "cuda"


def _model_case(name, kind, B, S, d, H, F, layers, plan="table", mask="ones", lo=1.0, causal=True):
    case = {"kind": kind, "B": B, "S": S, "d": d, "H": H, "F": F, "L": layers, "plan": plan,
            "mask": mask, "lo": lo, "causal": causal}
    return dict(case, name=name) if name else case


def _attention_case(name, B, H, S, hd, dtype, mask="prefix", lo=0.5, causal=True):
    case = {"kind": "attention", "B": B, "H": H, "S": S, "hd": hd, "dtype": dtype, "mask": mask,
            "lo": lo, "causal": causal}
    return dict(case, name=name) if name else case


def _mlp_case(name, M, d, F, mode):
    case = {"kind": "mlp", "M": M, "d": d, "F": F, "mode": mode}
    return dict(case, name=name) if name else case


def _norm_case(name, M, d, out):
    case = {"kind": "norm", "M": M, "d": d, "out": out}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the drop-in on one short sequence: launch latency is all there is
        _model_case("call_b1_s128_d128", "call", 1, 128, 128, 4, 128, 4),
        # the drop-in on an ordinary encoder: six layers, width 512, ragged lengths
        _model_case("call_b16_s512_d512", "call", 16, 512, 512, 8, 2048, 6, mask="prefix", lo=0.125),
        # a small batch through one layer, the feed-forward and out_proj in single-pass fp16
        _model_case("layer_b2_s128_d256", "layer", 2, 128, 256, 4, 1024, 1, "f16x3+half_rest",
                    "prefix", 0.5),
        # bulk scoring of many short sequences with a narrow model: activations larger than caches
        _model_case("layer_b10000_s128_d128", "layer", 10000, 128, 128, 4, 128, 1, "f16x3p"),
        # tiny heads: head_dim 8, width 64
        _model_case("layer_b64_s1024_d64", "layer", 64, 1024, 64, 8, 256, 1, "f16x3+f16x2_out",
                    "prefix", 0.125),
        # wide heads and a wide feed-forward over a long context
        _model_case("layer_b8_s4096_d1024", "layer", 8, 4096, 1024, 4, 4096, 1, "f16x3s+half_ffn",
                    "prefix", 0.25),
        # a wide model on short sequences at the default precision
        _model_case("layer_b64_s128_d1024", "layer", 64, 128, 1024, 4, 1024, 1, "f16x3p"),
        # sizes that divide by nothing, padding in front, bidirectional
        _model_case("layer_b5_s333_d192", "layer", 5, 333, 192, 6, 768, 1, "f16x3", "left", 1.0,
                    causal=False),
        # attention alone over a long context, fp16 tensors
        _attention_case("attention_fp16_s16384_hd64", 2, 16, 16384, 64, "float16"),
        # attention alone on fp32 tensors of an odd length, bidirectional, no mask
        _attention_case("attention_fp32_s1001_hd128", 4, 8, 1001, 128, "float32", "none", 1.0,
                        causal=False),
        # a feed-forward block on a ragged number of tokens, bf16 operands
        _mlp_case("mlp_bf16_3001x768x3072", 3001, 768, 3072, "bfloat16"),
        # residual add, mask and norm of a large activation
        _norm_case("norm_32768x1024", 32768, 1024, "float32"),
    ]


# ------------------------------------------------------------------ plans
# (attention, out_proj, ffn_in, ffn_out) precision of the plans a "layer" case may name
PLANS = {
    "f16x3": ("f16x3", "f16x3", "f16x3", "f16x3"),
    "f16x3p": ("f16x3p", "f16x3", "f16x3", "f16x3"),
    "f16x3+half_rest": ("f16x3", "float16", "float16", "float16"),
    "f16x3+f16x2_out": ("f16x3", "f16x2", "f16x3", "f16x2"),
    "f16x3p+half_in": ("f16x3p", "f16x3", "float16", "f16x3"),
    "f16x3s+half_ffn": ("f16x3s", "f16x3", "float16", "float16"),
    "bf16x3": ("bf16x3", "bf16x3", "bf16x3", "bf16x3"),
    "half": ("float16", "float16", "float16", "float16"),
}


def _plan(name):
    p = PLANS[name]
    return Plan(name=name, compute_dtype="f16x3", cuda_graph=True,
                overrides=tuple(zip(("attn", "out_proj", "ffn1", "ffn2"), p)))


# ------------------------------------------------------------------ drawn cases
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_any(rng):
    kind = rng.choice(("call", "layer", "layer", "layer", "attention", "mlp", "norm"))
    if kind in ("call", "layer"):
        hd = rng.choice((8, 16, 32, 64, 128, 256))
        H = rng.randint(1, max(1, min(16, 1024 // hd)))
        d = hd * H
        if d % 32:
            d, H = 32 * (d // 32 + 1), 32 * (d // 32 + 1) // hd
        S = _log_int(rng, 24, 4096)
        B = _log_int(rng, 1, max(1, 300000 // S))
        F = d * rng.choice((1, 2, 3, 4))
        mask = rng.choice(("ones", "prefix", "prefix", "left", "none"))
        plan = "table" if kind == "call" else rng.choice(sorted(PLANS))
        return _model_case(None, kind, B, S, d, H, F, rng.choice((1, 2, 4)) if kind == "call" else 1,
                           plan, mask, rng.choice((0.125, 0.5)), rng.random() < 0.7)
    if kind == "attention":
        S = _log_int(rng, 32, 16384)
        BH = _log_int(rng, 4, max(4, min(2048, 400000 // S)))
        H = rng.choice((1, 2, 4, 6, 8, 16))
        return _attention_case(None, max(1, BH // H), H, S, rng.choice((8, 16, 32, 64, 128, 256)),
                               rng.choice(("float16", "bfloat16", "float32")),
                               rng.choice(("prefix", "none", "left")), 0.5, rng.random() < 0.7)
    if kind == "mlp":
        d = 32 * rng.randint(2, 32)
        return _mlp_case(None, _log_int(rng, 16, 40000), d, d * rng.choice((1, 2, 4)),
                         rng.choice(("float16", "bfloat16", "f16x3", "f16x2", "bf16x3")))
    d = 4 * _log_int(rng, 8, 1024)
    return _norm_case(None, _log_int(rng, 64, max(64, 50000000 // d)), d,
                      rng.choice(("float32", "float16", "bfloat16")))


def _cost(case):
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 3e14


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_any(rng)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _mask(case, g):
    B, S = case["B"], case["S"]
    pos = torch.arange(S, device=DEVICE)[None, :]
    if case["mask"] == "none":
        return None
    if case["mask"] == "ones":
        return torch.ones(B, S, dtype=torch.bool, device=DEVICE)
    if case["mask"] == "prefix":
        low = max(1, int(round(S * case["lo"])))
        lengths = torch.randint(low, S + 1, (B, 1), generator=g, device=DEVICE)
        return pos < lengths
    start = torch.randint(0, max(1, S // 3) + 1, (B, 1), generator=g, device=DEVICE)
    return pos >= torch.clamp(start, max=S - 1)


def _linear(g, n, k):
    """Xavier-uniform weight and nn.Linear's default bias."""
    w = (torch.rand(n, k, generator=g, device=DEVICE) * 2 - 1) * math.sqrt(6.0 / (n + k))
    b = (torch.rand(n, generator=g, device=DEVICE) * 2 - 1) / math.sqrt(k)
    return w, b


def _config(case):
    return TransformerConfig(case["B"], case["S"], case["d"], case["H"], case["F"], case["L"],
                             case["causal"])


def _weights(case, g):
    """A state dict of the stack: Xavier weights, norms near one."""
    d, F = case["d"], case["F"]
    state = {}

    def norm(name):
        state[name + ".weight"] = 1 + 0.1 * torch.randn(d, generator=g, device=DEVICE)
        state[name + ".bias"] = 0.1 * torch.randn(d, generator=g, device=DEVICE)

    def linear(name, n, k):
        state[name + ".weight"], state[name + ".bias"] = _linear(g, n, k)

    for i in range(case["L"]):
        p = f"layers.{i}."
        norm(p + "norm1")
        for t in ("q_proj", "k_proj", "v_proj", "out_proj"):
            linear(p + "attention." + t, d, d)
        norm(p + "norm2")
        linear(p + "ffn_in", F, d)
        linear(p + "ffn_out", d, F)
    norm("final_norm")
    return state


def _model_inputs(case, seed):
    g = _gen(seed)
    state = _weights(case, g)
    mask = _mask(case, g)
    x = torch.randn(case["B"], case["S"], case["d"], generator=g, device=DEVICE)
    if mask is not None:
        x.mul_(mask[..., None])
    return state, mask, x


def _attention_inputs(case, seed):
    g = _gen(seed)
    B, S, H, hd = case["B"], case["S"], case["H"], case["hd"]
    mask = _mask(case, g)
    qkv = torch.randn(B, S, 3, H, hd, generator=g, device=DEVICE).to(getattr(torch, case["dtype"]))
    q, k, v = (qkv[:, :, j].permute(0, 2, 1, 3) for j in range(3))
    return q, k, v, mask


def _norm_inputs(case, g):
    M, d = case["M"], case["d"]
    x = torch.randn(M, d, generator=g, device=DEVICE)
    y = torch.randn(M, d, generator=g, device=DEVICE)
    keep = torch.rand(M, generator=g, device=DEVICE) < 0.8
    w = 1 + 0.1 * torch.randn(d, generator=g, device=DEVICE)
    b = 0.1 * torch.randn(d, generator=g, device=DEVICE)
    return x, y, keep, w, b


def _mlp_inputs(case, seed):
    g = _gen(seed)
    norm = _norm_inputs(case, g)
    return norm, _linear(g, case["F"], case["d"]), _linear(g, case["d"], case["F"])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("call", "layer"):
        state, mask, x = _model_inputs(case, seed)
        if kind == "call":
            with torch.device("meta"):
                model = UserOptimizedTransformer(_config(case))
            model.load_state_dict(state, assign=True)
            model.eval()
        else:
            with torch.device("meta"):
                reference = BaselineTransformer(_config(case))
            reference.load_state_dict(state, assign=True)
            model = build_shared(_config(case), _plan(case["plan"]), reference)
        with torch.inference_mode():
            model(x, mask)              # a program warms its model up: plan, weight planes, graph
        return {"kind": kind, "model": model, "x": x, "mask": mask}
    if kind == "attention":
        q, k, v, mask = _attention_inputs(case, seed)
        return {"kind": kind, "q": q, "k": k, "v": v, "mask": mask, "causal": case["causal"]}
    if kind == "mlp":
        norm, w1, w2 = _mlp_inputs(case, seed)
        mode = K.MODES[case["mode"]]
        return {"kind": kind, "norm": norm, "w1": K.PreparedLinear(*w1, mode),
                "w2": K.PreparedLinear(*w2, mode), "format": K.planes_format(mode)}
    return {"kind": kind, "norm": _norm_inputs(case, _gen(seed)), "out": getattr(torch, case["out"])}


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    with torch.inference_mode():
        if kind in ("call", "layer"):
            return state["model"](state["x"], state["mask"])
        if kind == "attention":
            return K.flash_attention(state["q"], state["k"], state["v"], keep=state["mask"],
                                     causal=state["causal"])
        x, y, keep, w, b = state["norm"]
        if kind == "mlp":
            s, h = K.add_mask_layernorm(x, y, keep, w, b, out_dtype=state["format"])
            f = K.linear(h, state["w1"], act=L.ACT_GELU_ERF, out_dtype=state["format"])
            return s, K.linear(f, state["w2"])
        return K.add_mask_layernorm(x, y, keep, w, b, out_dtype=state["out"])


# ------------------------------------------------------------------ work
def _pairs(case):
    """Expected number of (query, key) pairs per head over the batch; padded queries of a
    "layer" or "call" need no attention (their rows are zeroed)."""
    B, S = case["B"], case["S"]
    stack = case["kind"] != "attention"

    def of(first, n):                         # valid keys [first, first + n)
        if not case["causal"]:
            return n * (n if stack else S)
        inside = n * (n + 1) / 2
        return inside + (0 if stack else (S - first - n) * n)

    if case["mask"] == "prefix":
        low = max(1, int(round(S * case["lo"])))
        lens = [low + (S - low) * i / 64 for i in range(65)]
        return B * sum(of(0, n) for n in lens) / len(lens)
    if case["mask"] == "left":
        starts = [max(1, S // 3) * i / 64 for i in range(65)]
        return B * sum(of(s, S - s) for s in starts) / len(starts)
    return B * of(0, S)


def work(case):
    kind = case["kind"]
    if kind in ("call", "layer"):
        M, d, F, layers = case["B"] * case["S"], case["d"], case["F"], case["L"]
        weights = layers * (4 * d * d + 2 * d * F)
        mask = 0 if case["mask"] == "none" else M
        return {"bytes": 8 * M * d + 4 * weights + mask,
                "flops": 2 * M * weights + layers * 4 * d * _pairs(case)}
    if kind == "attention":
        size = 4 if case["dtype"] == "float32" else 2
        n = case["B"] * case["H"] * case["S"] * case["hd"]
        mask = 0 if case["mask"] == "none" else case["B"] * case["S"]
        return {"bytes": 4 * n * size + mask, "flops": 4 * case["H"] * case["hd"] * _pairs(case)}
    M, d = case["M"], case["d"]
    if kind == "mlp":
        F = case["F"]
        size = 2 if case["mode"] in ("float16", "bfloat16") else 4
        return {"bytes": 16 * M * d + M + 2 * d * F * size, "flops": 4 * M * d * F}
    return {"bytes": M * d * (12 + (4 if case["out"] == "float32" else 2)) + M + 8 * d,
            "flops": 8 * M * d}


# ------------------------------------------------------------------ tolerances
# About four times what the outputs are off `exact` by at these precisions (one layer or six:
# f16x3 3.1e-7, f16x3p 3.7e-5 and 5.5e-5, the fp16 stages 1.0e-4 to 2.5e-4; bf16 3.5e-3).
_MODE_REL = {"float16": 1.6e-3, "bfloat16": 1.4e-2, "f16x3": 3e-6, "f16x2": 1e-3, "bf16x3": 4e-5}
_PLAN_REL = {"f16x3": 3e-6, "f16x3p": 2e-4, "f16x3+half_rest": 8e-4, "f16x3+f16x2_out": 5e-4,
             "f16x3p+half_in": 1e-3, "f16x3s+half_ffn": 8e-4, "bf16x3": 4e-5, "half": 1.5e-3,
             "table": 1e-3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("call", "layer"):
        return {"rel": _PLAN_REL[case["plan"]]}
    if kind == "attention":
        return {"rel": {"float16": 1.4e-3, "bfloat16": 1.1e-2, "float32": 3e-6}[case["dtype"]]}
    if kind == "mlp":
        return {"rel": _MODE_REL[case["mode"]]}
    return {"rel": {"float32": 4e-7, "float16": 1e-3, "bfloat16": 8e-3}[case["out"]]}


# ------------------------------------------------------------------ 64-bit results
def _attend(q, k, v, mask, causal, scale):
    """softmax(q k^T scale + masks) v in float64 for [B, H, S, hd], a (row, head) at a time
    where the scores are large; rows without a valid key give zeros."""
    B, H, S, hd = q.shape
    out = torch.empty((B, H, S, hd), dtype=torch.float64, device=q.device)
    rows = max(1, min(S, (1 << 27) // S))                   # query rows at a time
    nb = max(1, (1 << 27) // max(1, H * S * S)) if rows == S else 1
    heads = H if rows == S and H * S * S <= (1 << 27) else 1
    key = torch.arange(S, device=q.device)
    for b in range(0, B, nb):
        for h in range(0, H, heads):
            sl = (slice(b, b + nb), slice(h, h + heads))
            kt = k[sl].double().transpose(-2, -1).contiguous()
            vv = v[sl].double().contiguous()
            for r in range(0, S, rows):
                n = min(S, r + rows) if causal else S
                s = torch.matmul(q[sl][:, :, r:r + rows].double().contiguous(),
                                 kt[..., :n].contiguous()).mul_(scale)
                if causal:
                    qi = torch.arange(r, min(S, r + rows), device=q.device)
                    s.masked_fill_(key[None, :n] > qi[:, None], -math.inf)
                if mask is not None:
                    s.masked_fill_(~mask[sl[0], None, None, :n], -math.inf)
                p = torch.softmax(s, dim=-1).nan_to_num_(0.0)
                out[sl][:, :, r:r + rows] = torch.matmul(p, vv[:, :, :n].contiguous())
                del s, p
    return out


def _ln(x, w, b, eps=1e-5):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w.double(), b.double(), eps)


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x * math.sqrt(0.5)))


def _exact_model(case, state, mask, x):
    B, S, d, H = case["B"], case["S"], case["d"], case["H"]
    drop = None if mask is None else ~mask[..., None]
    step = max(1, 400000000 // (S * max(3 * d, case["F"]) * 8))   # sequences at a time

    def lin(t, name):
        return t @ state[name + ".weight"].double().t() + state[name + ".bias"].double()

    out = torch.empty((B, S, d), dtype=torch.float64, device=x.device)
    for lo in range(0, B, step):
        sl = slice(lo, min(B, lo + step))
        t = x[sl].double()
        m = None if mask is None else mask[sl]
        dr = None if drop is None else drop[sl]
        for i in range(case["L"]):
            p = f"layers.{i}."
            h = _ln(t, state[p + "norm1.weight"], state[p + "norm1.bias"])
            q, k, v = (lin(h, p + "attention." + n).view(-1, S, H, d // H).permute(0, 2, 1, 3)
                       for n in ("q_proj", "k_proj", "v_proj"))
            a = _attend(q, k, v, m, case["causal"], (d // H) ** -0.5)
            a = lin(a.permute(0, 2, 1, 3).reshape(-1, S, d), p + "attention.out_proj")
            t = t + (a if dr is None else a.masked_fill(dr, 0.0))
            h = _ln(t, state[p + "norm2.weight"], state[p + "norm2.bias"])
            t = t + lin(_gelu(lin(h, p + "ffn_in")), p + "ffn_out")
            if dr is not None:
                t = t.masked_fill(dr, 0.0)
        t = _ln(t, state["final_norm.weight"], state["final_norm.bias"])
        out[sl] = t if dr is None else t.masked_fill(dr, 0.0)
    return out


def exact(case, seed):
    kind = case["kind"]
    with torch.inference_mode():
        if kind in ("call", "layer"):
            return _exact_model(case, *_model_inputs(case, seed))
        if kind == "attention":
            q, k, v, mask = _attention_inputs(case, seed)
            return _attend(q, k, v, mask, case["causal"], case["hd"] ** -0.5)
        norm = _mlp_inputs(case, seed)[0] if kind == "mlp" else _norm_inputs(case, _gen(seed))
        x, y, keep, w, b = norm
        s = (x.double() + y.double()) * keep[:, None]
        h = _ln(s, w, b)
        if kind == "norm":
            return s, h
        _, w1, w2 = _mlp_inputs(case, seed)
        f = _gelu(h @ w1[0].double().t() + w1[1].double())
        return s, f @ w2[0].double().t() + w2[1].double()
