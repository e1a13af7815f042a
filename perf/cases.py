"""Performance cases of the mixed FP16/FP32 causal-Transformer forward on one GPU.

Each case is one call that a program using this package makes: a whole forward, one attention or
FFN sub-block of a wide layer, the fused tail of a narrow layer, or a single operator.  Sizes come
from the benchmark configurations, the 14-case suite and the tests, with ragged sizes beside them.
``draw`` gives further cases of the same ranges.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from tiktoktechjam2026_amd.config import TransformerConfig
from tiktoktechjam2026_amd.custom_kernel.hip_attention import attention
from tiktoktechjam2026_amd.harness import HipGraphModel
from tiktoktechjam2026_amd.mixed_precision import MixedPrecisionTransformer
from tiktoktechjam2026_amd.mixed_precision.hip_fused import fused_layer_tail
from tiktoktechjam2026_amd.mixed_precision.hip_linear import mixed_add_layer_norm, mixed_linear

DEVICE = "cuda"
HEAD_DIMS = (8, 16, 32, 64, 128, 256)
TAIL_SHAPES = ((32, 32), (32, 64), (32, 128), (64, 64), (64, 128), (64, 256), (128, 128))


# --------------------------------------------------------------------------- the cases


def _forward(batch, seq, d, heads, ffn, layers, causal=True, padding=0.0, graph=False):
    return {"path": "forward", "batch": batch, "seq": seq, "d": d, "heads": heads, "ffn": ffn, "layers": layers,
            "causal": causal, "padding": padding, "graph": graph}


def _attention_block(batch, seq, d, heads, causal=True, padding=0.0):
    return {"path": "attention_block", "batch": batch, "seq": seq, "d": d, "heads": heads, "causal": causal,
            "padding": padding}


def _ffn_block(rows, d, ffn):
    return {"path": "ffn_block", "rows": rows, "d": d, "ffn": ffn}


def _layer_tail(rows, d, ffn, last=False):
    return {"path": "layer_tail", "rows": rows, "d": d, "ffn": ffn, "last": last}


def _attention(batch, seq, heads, head_dim, causal=True, padding=0.0, fp32=False):
    return {"path": "attention", "batch": batch, "seq": seq, "heads": heads, "head_dim": head_dim, "causal": causal,
            "padding": padding, "fp32": fp32}


def _linear(rows, n, k, gelu=False, fp32_in=False, fp32_out=False):
    return {"path": "linear", "rows": rows, "n": n, "k": k, "gelu": gelu, "fp32_in": fp32_in, "fp32_out": fp32_out}


def _add_norm(rows, d, fp32_out=False):
    return {"path": "add_norm", "rows": rows, "d": d, "fp32_out": fp32_out}


def listed():
    return [
        # the smallest whole call: one short sequence through a narrow model, eager; launches and
        # host work count
        {"name": "forward_b1_s128_d128", **_forward(1, 128, 128, 4, 128, 4)},
        # the ordinary narrow model at full batch, replayed from a HIP graph as the command line does
        {"name": "forward_graph_b64_s1024_d128", **_forward(64, 1024, 128, 4, 128, 4, graph=True)},
        # the suite's wide model: short sequences, head dim 256, square projections of 8192 rows
        {"name": "forward_b64_s128_d1024", **_forward(64, 128, 1024, 4, 1024, 4)},
        # attention half of a d_model 512 layer: QKV projection, causal attention at head dim 64,
        # out-projection + residual + LayerNorm
        {"name": "attention_block_b16_s2048_d512", **_attention_block(16, 2048, 512, 8)},
        # the largest: the attention half of a d_model 256 layer over a 64-sequence microbatch
        {"name": "attention_block_b64_s4096_d256", **_attention_block(64, 4096, 256, 8)},
        # FFN half of a d_model 512 layer (projection + GELU, projection + residual, LayerNorm)
        {"name": "ffn_block_32768_d512", **_ffn_block(32768, 512, 2048)},
        # everything after attention in a narrow layer, at a ragged row count
        {"name": "layer_tail_4099_d64", **_layer_tail(4099, 64, 256)},
        # bidirectional attention over a padded batch (key mask), ragged length
        {"name": "attention_padded_b24_s1000_hd64", **_attention(24, 1000, 8, 64, causal=False, padding=0.5)},
        # causal attention at head dim 128, an odd length
        {"name": "attention_b8_s1531_hd128", **_attention(8, 1531, 8, 128)},
        # the FP32-input attention operator
        {"name": "attention_fp32_b16_s1024_hd32", **_attention(16, 1024, 4, 32, fp32=True)},
        # one projection + GELU over a handful of rows
        {"name": "linear_gelu_77x2048x512", **_linear(77, 2048, 512, gelu=True)},
        # residual add + LayerNorm between the GEMMs of a wide layer
        {"name": "add_norm_8192x1024", **_add_norm(8192, 1024)},
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))))


# Bounds of a drawn case: each keeps its time below that of the largest listed case.
_MAX_FLOPS = 1.2e11       # matrix operations at the rate of a small or ragged call
_MAX_BYTES = 6.0e8
_MAX_SCORES = 4.0e8       # attention scores, whatever the head dim
_MAX_ROWS = 70000


def _scores(case):
    return case["batch"] * case["heads"] * case["seq"] ** 2 * case.get("layers", 1)


def _cheap(case):
    w = work(case)
    if w["flops"] > _MAX_FLOPS or w["bytes"] > _MAX_BYTES:
        return False
    if "seq" in case and (_scores(case) > _MAX_SCORES or case["batch"] * case["seq"] > _MAX_ROWS):
        return False
    return True


def _draw_once(rng):
    path = rng.choice(["forward", "attention_block", "ffn_block", "layer_tail", "attention", "attention", "linear",
                       "add_norm"])
    padding = rng.choice([0.0, 0.0, 0.25, 0.5])
    causal = rng.random() < 0.75
    if path == "forward":
        d = rng.choice([32, 64, 128, 256, 512, 1024])
        heads = rng.choice([h for h in (1, 2, 4, 8, 16) if d // h in HEAD_DIMS])
        graph = padding == 0.0 and rng.random() < 0.5
        return _forward(_log_int(rng, 1, 128), _log_int(rng, 8, 2048), d, heads, d * rng.choice([1, 2, 4]),
                        rng.randint(1, 4), causal, padding, graph)
    if path == "attention_block":
        d = rng.choice([256, 512, 768, 1024])
        heads = rng.choice([h for h in (2, 4, 6, 8, 12, 16, 24) if d % h == 0 and d // h in HEAD_DIMS])
        return _attention_block(_log_int(rng, 1, 64), _log_int(rng, 16, 4096), d, heads, causal, padding)
    if path == "ffn_block":
        d = rng.choice([256, 512, 768, 1024])
        return _ffn_block(_log_int(rng, 16, 40000), d, d * rng.choice([1, 2, 4]))
    if path == "layer_tail":
        d, ffn = rng.choice(TAIL_SHAPES)
        return _layer_tail(_log_int(rng, 16, 65536), d, ffn, rng.random() < 0.3)
    if path == "attention":
        return _attention(_log_int(rng, 1, 64), _log_int(rng, 16, 4096), rng.choice([1, 2, 3, 4, 8, 16]),
                          rng.choice(HEAD_DIMS), causal, padding, rng.random() < 0.25)
    if path == "linear":
        widths = [32, 64, 128, 200, 256, 384, 512, 768, 1024, 1536, 2048, 3072]
        return _linear(_log_int(rng, 1, 65536), rng.choice(widths), rng.choice(widths[:-1]), rng.random() < 0.4,
                       rng.random() < 0.2, rng.random() < 0.2)
    return _add_norm(_log_int(rng, 1, 65536), rng.choice([32, 128, 256, 512, 768, 1024, 2048]), rng.random() < 0.3)


def draw(rng):
    while True:
        case = _draw_once(rng)
        if _cheap(case):
            return case


# --------------------------------------------------------------------------- inputs


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEVICE) * scale).to(dtype)


def _linear_params(g, n, k):
    """FP16 weight and bias in nn.Linear's default range."""
    bound = k ** -0.5
    w = (torch.rand(n, k, generator=g, device=DEVICE) * 2 - 1) * bound
    b = (torch.rand(n, generator=g, device=DEVICE) * 2 - 1) * bound
    return w.half(), b.half()


def _norm_params(g, d):
    return 1 + _randn(g, d, scale=0.1), _randn(g, d, scale=0.1)


def _valid_mask(g, batch, seq, padding):
    """Right-padded sequences: lengths uniform in [(1 - padding) seq, seq]."""
    if padding <= 0:
        return None
    low = max(1, int(round(seq * (1 - padding))))
    lengths = torch.randint(low, seq + 1, (batch,), generator=g, device=DEVICE)
    return torch.arange(seq, device=DEVICE)[None, :] < lengths[:, None]


def _layer_params(g, d, ffn):
    p = {}
    p["norm1.weight"], p["norm1.bias"] = _norm_params(g, d)
    p["norm2.weight"], p["norm2.bias"] = _norm_params(g, d)
    for name, n, k in (("attention.qkv_proj", 3 * d, d), ("attention.out_proj", d, d), ("ffn_in", ffn, d),
                       ("ffn_out", d, ffn)):
        p[name + ".weight"], p[name + ".bias"] = _linear_params(g, n, k)
    return p


def _model_params(g, case):
    layers = case.get("layers", 1)
    params = {}
    for i in range(layers):
        for key, value in _layer_params(g, case["d"], case.get("ffn", case["d"])).items():
            params[f"layers.{i}.{key}"] = value
    params["final_norm.weight"], params["final_norm.bias"] = _norm_params(g, case["d"])
    return params


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g = _generator(seed)
    path = case["path"]
    if path == "forward":
        b, s, d = case["batch"], case["seq"], case["d"]
        return {"x": _randn(g, b, s, d), "mask": _valid_mask(g, b, s, case["padding"]), "params": _model_params(g, case)}
    if path == "attention_block":
        b, s, d = case["batch"], case["seq"], case["d"]
        return {"x": _randn(g, b, s, d, dtype=torch.float16), "residual": _randn(g, b, s, d),
                "mask": _valid_mask(g, b, s, case["padding"]), "params": _model_params(g, case)}
    if path == "ffn_block":
        rows, d = case["rows"], case["d"]
        return {"x": _randn(g, 1, rows, d, dtype=torch.float16), "residual": _randn(g, 1, rows, d),
                "params": _model_params(g, case)}
    if path == "layer_tail":
        rows, d = case["rows"], case["d"]
        return {"x": _randn(g, rows, d, dtype=torch.float16, scale=0.5), "residual": _randn(g, rows, d),
                "params": _model_params(g, case), "next_norm": _norm_params(g, d), "next_qkv": _linear_params(g, 3 * d, d)}
    if path == "attention":
        b, s, h, hd = case["batch"], case["seq"], case["heads"], case["head_dim"]
        dtype = torch.float32 if case["fp32"] else torch.float16
        return {"qkv": _randn(g, b, s, 3, h, hd, dtype=dtype), "mask": _valid_mask(g, b, s, case["padding"])}
    if path == "linear":
        dtype = torch.float32 if case["fp32_in"] else torch.float16
        return {"x": _randn(g, case["rows"], case["k"], dtype=dtype), "linear": _linear_params(g, case["n"], case["k"])}
    rows, d = case["rows"], case["d"]
    return {"x": _randn(g, rows, d), "update": _randn(g, rows, d), "norm": _norm_params(g, d)}


def _linear_module(params):
    w, b = params
    module = torch.nn.Linear(w.shape[1], w.shape[0], device="meta", dtype=torch.float16)
    module.weight = torch.nn.Parameter(w, requires_grad=False)
    module.bias = torch.nn.Parameter(b, requires_grad=False)
    return module


def _norm_module(params):
    w, b = params
    module = torch.nn.LayerNorm(w.shape[0], device="meta")
    module.weight = torch.nn.Parameter(w, requires_grad=False)
    module.bias = torch.nn.Parameter(b, requires_grad=False)
    return module


def _model(case, params):
    config = TransformerConfig(case.get("batch", 1), case.get("seq", case.get("rows")), case["d"],
                               case.get("heads", max(1, case["d"] // 64)), case.get("ffn", case["d"]), case.get("layers", 1),
                               bool(case.get("causal", True)))
    with torch.device(DEVICE):
        model = MixedPrecisionTransformer(config)
    model.convert_projections_to_fp16()
    model.load_state_dict(params, strict=True)
    model.assume_all_tokens_valid = case.get("padding", 0.0) <= 0
    return model.eval().requires_grad_(False)


def prepare(case, seed):
    t = _inputs(case, seed)
    path = case["path"]
    state = {"path": path, "case": case}
    if path == "forward":
        model = _model(case, t["params"])
        state.update(model=HipGraphModel(model) if case["graph"] else model, x=t["x"], mask=t["mask"])
        if case["graph"]:
            with torch.inference_mode():
                state["model"](t["x"])  # a program captures the graph once, at start-up
    elif path in ("attention_block", "ffn_block"):
        model = _model(case, t["params"])
        state.update(layer=model.layers[0], final_norm=model.final_norm, x=t["x"], residual=t["residual"],
                     mask=t.get("mask"))
    elif path == "layer_tail":
        layer = _model(case, t["params"]).layers[0]
        state.update(layer=layer, x=t["x"], residual=t["residual"], next_norm=_norm_module(t["next_norm"]),
                     next_qkv=None if case["last"] else _linear_module(t["next_qkv"]))
    elif path == "attention":
        q, k, v = t["qkv"].permute(2, 0, 3, 1, 4).unbind(0)
        state.update(q=q, k=k, v=v, mask=t["mask"])
    elif path == "linear":
        state.update(x=t["x"], linear=_linear_module(t["linear"]))
    else:
        state.update(x=t["x"], update=t["update"], norm=_norm_module(t["norm"]))
    return state


def run(state):
    case, path = state["case"], state["path"]
    with torch.inference_mode():
        if path == "forward":
            return state["model"](state["x"], state["mask"])
        if path == "attention_block":
            layer = state["layer"]
            return layer.attention(state["x"], state["mask"], case["causal"], residual_fp32=state["residual"],
                                   next_norm=layer.norm2)
        if path == "ffn_block":
            return state["layer"].ffn(state["x"], state["residual"], state["final_norm"], torch.float16)
        if path == "layer_tail":
            layer = state["layer"]
            return fused_layer_tail(state["x"], state["residual"], layer.attention.out_proj, layer.norm2,
                                    layer.ffn_in, layer.ffn_out, state["next_norm"], state["next_qkv"])
        if path == "attention":
            return attention(state["q"], state["k"], state["v"], case["head_dim"] ** -0.5, causal=case["causal"],
                             key_valid=state["mask"])
        if path == "linear":
            return mixed_linear(state["x"], state["linear"],
                                output_dtype=torch.float32 if case["fp32_out"] else torch.float16,
                                fuse_gelu=case["gelu"])
        return mixed_add_layer_norm(state["x"], state["update"], state["norm"],
                                    normalized_dtype=torch.float32 if case["fp32_out"] else torch.float16)


# --------------------------------------------------------------------------- the work of one pass


def _pairs(case):
    """(query, visible key) pairs of one head and sequence; padded keys at their mean count."""
    s = case["seq"]
    keys = s * (1 - case["padding"] / 2)
    if not case["causal"]:
        return s * keys
    return s * (s + 1) / 2 - (s - keys) * (s - keys + 1) / 2


def _tail_work(rows, d, ffn, last):
    flops = 2.0 * rows * (d * d + 2 * d * ffn + (0 if last else 3 * d * d))
    weights = 2.0 * (d * d + 2 * d * ffn + (0 if last else 3 * d * d))
    return {"bytes": rows * d * (2 + 4 + 4 + (4 if last else 6)) + weights, "flops": flops}


def work(case):
    path = case["path"]
    if path == "forward":
        rows, d, ffn, layers = case["batch"] * case["seq"], case["d"], case["ffn"], case["layers"]
        flops = layers * (2.0 * rows * (4 * d * d + 2 * d * ffn) + 4.0 * case["batch"] * d * _pairs(case))
        return {"bytes": 8.0 * rows * d + layers * 2.0 * (4 * d * d + 2 * d * ffn), "flops": flops}
    if path == "attention_block":
        rows, d = case["batch"] * case["seq"], case["d"]
        flops = 2.0 * rows * 4 * d * d + 4.0 * case["batch"] * d * _pairs(case)
        return {"bytes": rows * d * (2.0 + 4 + 4 + 2) + 8.0 * d * d, "flops": flops}
    if path == "ffn_block":
        rows, d, ffn = case["rows"], case["d"], case["ffn"]
        return {"bytes": rows * d * (2.0 + 4 + 4 + 2) + 4.0 * d * ffn, "flops": 4.0 * rows * d * ffn}
    if path == "layer_tail":
        return _tail_work(case["rows"], case["d"], case["ffn"], case["last"])
    if path == "attention":
        size = case["batch"] * case["seq"] * case["heads"] * case["head_dim"]
        return {"bytes": size * 4.0 * (4 if case["fp32"] else 2),
                "flops": 4.0 * case["batch"] * case["heads"] * case["head_dim"] * _pairs(case)}
    if path == "linear":
        rows, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": rows * k * (4.0 if case["fp32_in"] else 2.0) + 2.0 * n * k
                + rows * n * (4.0 if case["fp32_out"] else 2.0), "flops": 2.0 * rows * n * k}
    return {"bytes": case["rows"] * case["d"] * (12.0 + (4 if case["fp32_out"] else 2)), "flops": 0.0}


# --------------------------------------------------------------------------- tolerance


# About four times the largest error against ``exact`` that was measured over the listed cases and 90
# drawn ones (rel: 2-norm; max: one element, over the result's root mean square).
def tolerance(case):
    path = case["path"]
    if path == "forward":  # FP32 output of a model with FP16 operands: 1.3e-4, 1.1e-3
        return {"rel": 6e-4, "max": 6e-3}
    if path == "attention":
        if case["fp32"]:  # operands rounded to an 11-bit significand: 4.4e-4, 2.2e-2
            return {"rel": 1.8e-3, "max": 8e-2}
        return {"rel": 1.2e-3, "max": 4e-2}  # FP16 weights and output: 2.9e-4, 1.0e-2
    if path == "layer_tail":  # FP16 normalized operand and QKV output: 3.0e-4, 2.4e-3
        return {"rel": 1.2e-3, "max": 1e-2}
    if path == "linear":
        if case["fp32_in"]:  # the input is rounded to FP16: 3.0e-4, 4.0e-3
            return {"rel": 1.2e-3, "max": 1.6e-2}
        if case["fp32_out"]:  # 32-bit sums of exact products: 1.4e-7 at K 128, growing with K; 1.8e-6
            return {"rel": 4e-6, "max": 4e-5}
        return {"rel": 1e-3, "max": 1.2e-2}  # FP16 output: 2.1e-4, 2.8e-3
    if path == "add_norm" and case["fp32_out"]:  # 32-bit sums: 6.3e-8, 6e-7
        return {"rel": 5e-7, "max": 4e-6}
    return {"rel": 1e-3, "max": 1e-2}  # FP16 normalized output: 2.1e-4, 2.0e-3


# --------------------------------------------------------------------------- 64-bit results


def _linear64(x, params):
    w, b = params
    return x @ w.double().t() + b.double()


def _norm64(x, params, eps=1e-5):
    mean = x.mean(-1, keepdim=True)
    c = x - mean
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + eps) * params[0].double() + params[1].double()


def _gelu64(x):
    return 0.5 * x * (1 + torch.erf(x * 0.5 ** 0.5))


def _attention64(q, k, v, scale, causal, mask):
    """[B, H, S, hd] FP64 -> [B, S, H, hd], one sequence at a time."""
    b, h, s, hd = q.shape
    out = torch.empty(b, s, h, hd, dtype=torch.float64, device=q.device)
    future = torch.ones(s, s, dtype=torch.bool, device=q.device).triu(1) if causal else None
    for i in range(b):
        scores = torch.matmul(q[i].contiguous() * scale, k[i].transpose(-1, -2).contiguous())
        if causal:
            scores.masked_fill_(future, -math.inf)
        if mask is not None:
            scores.masked_fill_(~mask[i][None, None, :], -math.inf)
        out[i] = torch.matmul(torch.softmax(scores, -1), v[i].contiguous()).transpose(0, 1)
    return out


def _pick(params, prefix):
    return params[prefix + ".weight"], params[prefix + ".bias"]


def _attention_half64(x, residual, mask, case, params, prefix):
    b, s, d = x.shape
    h = case["heads"]
    qkv = _linear64(x, _pick(params, prefix + "attention.qkv_proj")).view(b, s, 3, h, d // h).permute(2, 0, 3, 1, 4)
    ctx = _attention64(qkv[0], qkv[1], qkv[2], (d // h) ** -0.5, case["causal"], mask).reshape(b, s, d)
    x1 = _linear64(ctx, _pick(params, prefix + "attention.out_proj")) + residual
    return x1, _norm64(x1, _pick(params, prefix + "norm2"))


def _ffn_half64(normalized, residual, params, prefix, next_norm):
    hidden = _gelu64(_linear64(normalized, _pick(params, prefix + "ffn_in")))
    x2 = _linear64(hidden, _pick(params, prefix + "ffn_out")) + residual
    return x2, _norm64(x2, next_norm)


def exact(case, seed):
    t = _inputs(case, seed)
    path = case["path"]
    with torch.inference_mode():
        if path == "forward":
            params, mask = t["params"], t["mask"]
            x = t["x"].double()
            normalized = _norm64(x, _pick(params, "layers.0.norm1"))
            for i in range(case["layers"]):
                prefix = f"layers.{i}."
                last = i + 1 == case["layers"]
                x, normalized = _attention_half64(normalized, x, mask, case, params, prefix)
                next_norm = _pick(params, "final_norm" if last else f"layers.{i + 1}.norm1")
                x, normalized = _ffn_half64(normalized, x, params, prefix, next_norm)
            if mask is not None:
                normalized = normalized.masked_fill(~mask[..., None], 0)
            return normalized
        if path == "attention_block":
            return _attention_half64(t["x"].double(), t["residual"].double(), t["mask"], case, t["params"], "layers.0.")
        if path == "ffn_block":
            return _ffn_half64(t["x"].double(), t["residual"].double(), t["params"], "layers.0.",
                               _pick(t["params"], "final_norm"))
        if path == "layer_tail":
            params = t["params"]
            x1 = _linear64(t["x"].double(), _pick(params, "layers.0.attention.out_proj")) + t["residual"].double()
            x2, normalized = _ffn_half64(_norm64(x1, _pick(params, "layers.0.norm2")), x1, params, "layers.0.",
                                         t["next_norm"])
            return x2, (normalized if case["last"] else _linear64(normalized, t["next_qkv"]))
        if path == "attention":
            q, k, v = t["qkv"].double().permute(2, 0, 3, 1, 4).unbind(0)
            return _attention64(q, k, v, case["head_dim"] ** -0.5, case["causal"], t["mask"])
        if path == "linear":
            y = _linear64(t["x"].double(), t["linear"])
            return _gelu64(y) if case["gelu"] else y
        r = t["x"].double() + t["update"].double()
        return r, _norm64(r, t["norm"])
