"""The workloads this package's speed is judged by, each through its public entry points.

A case is a dict of plain values.  ``kind`` names the entry point:

* ``tensor``   ``WeightQuantizer.quantize_tensor`` on one weight (1x128 blocks)
* ``plan``     a ``QuantPlan`` over the linears of some decoder layers (the weight sync)
* ``experts``  ``quantize_fp8_blockwise`` on a stack of expert matrices (128x128 tiles)
* ``state``    ``WeightQuantizer.quantize_state_dict`` (the drop-in, outputs and plans made per call)
* ``unstate``  ``WeightQuantizer.dequantize_state_dict`` (back to bf16)
* ``act``      ``act_qdq``: the activation fake-quant of the FP8 rollout linear
* ``kv``       ``FP8KVCacheQuantizer.recalibrate_scales`` over a model's q/k/v projections
* ``loader``   ``DynamicWeightLoader.load_weights`` with FP8 on (unscaled e4m3 cast)
* ``linear``   a linear patched by ``FP8RolloutQuantizer.quantize_model``, one forward
* ``mlp``      a SwiGLU MLP whose three linears are patched the same way

The sizes are Qwen3-8B's, or generic ones of the same range; ``draw`` spreads
them over hidden sizes from 1024 to 8192, 1 to 8192 tokens, and the data types
and options a trainer or a rollout engine uses.
"""

from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "lumen-rl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from lumenrl_amd.engine.inference import DynamicWeightLoader  # noqa: E402
from lumenrl_amd.quantization import (  # noqa: E402
    FP8Config,
    FP8KVCacheQuantizer,
    FP8RolloutQuantizer,
    QuantPlan,
    WeightQuantizer,
    act_qdq,
    quantize_fp8_blockwise,
)

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_E4M3 = torch.float8_e4m3fn
_MAX = 448.0
#: no drawn case costs more than the largest listed linear
_MOST_MACS = 8192 * 4096 * 12288
_MOST_WEIGHTS = 4 * 192_937_984


def listed():
    return [
        # one k_proj of Qwen3-8B, quantized by itself: the smallest call, launch and host latency
        {"name": "tensor_k_proj", "kind": "tensor", "dtype": "bf16", "rows": 1024, "cols": 4096, "pow2": False},
        # the trainer -> rollout sync in vLLM's per-block layout: four Qwen3-8B layers per plan
        {"name": "sync_fp8_128x128", "kind": "plan", "fmt": "fp8_block", "block": 128, "dtype": "bf16",
         "hidden": 4096, "inter": 12288, "q": 4096, "kv": 1024, "layers": 4},
        # the same sync for an MXFP4 rollout engine, two layers
        {"name": "sync_mxfp4", "kind": "plan", "fmt": "mxfp4", "block": 32, "dtype": "bf16",
         "hidden": 4096, "inter": 12288, "q": 4096, "kv": 1024, "layers": 2},
        # the down projections of 128 experts cut four ways (768 -> 192 columns: ragged tiles)
        {"name": "experts_down_tp4", "kind": "experts", "dtype": "bf16", "experts": 128, "rows": 2048, "cols": 192},
        # the reference's own call per sync: a state dict in, codes and bf16 scales out
        {"name": "state_dict_2_layers", "kind": "state", "dtype": "bf16",
         "hidden": 4096, "inter": 12288, "q": 4096, "kv": 1024, "layers": 2},
        # the way back, as a checkpoint export or an evaluation in bf16 does it
        {"name": "dequantize_2_layers", "kind": "unstate", "hidden": 4096, "inter": 12288, "q": 4096, "kv": 1024,
         "layers": 2},
        # the input of a Qwen3-8B attention block at prefill
        {"name": "act_prefill_8192", "kind": "act", "dtype": "bf16", "tokens": 8192, "cols": 4096, "pow2": False},
        # the per-step KV scales of a 16-layer model
        {"name": "kv_scales_16_layers", "kind": "kv", "dtype": "bf16", "hidden": 4096, "q": 4096, "kv": 1024,
         "layers": 16},
        # one decoder layer with its norms and the embedding, loaded into an engine in e4m3
        {"name": "loader_embed_and_layer", "kind": "loader", "dtype": "bf16", "hidden": 4096, "inter": 12288,
         "q": 4096, "kv": 1024, "layers": 1, "vocab": 151936},
        # the rollout linear at its smallest: o_proj for the one token of a single decoding sequence
        {"name": "linear_decode_1", "kind": "linear", "dtype": "bf16", "tokens": 1, "cols": 4096, "out": 4096,
         "bias": False, "pow2": False},
        # a decoding step of 48 sequences through one layer's MLP
        {"name": "mlp_decode_48", "kind": "mlp", "dtype": "bf16", "tokens": 48, "hidden": 4096, "inter": 12288,
         "pow2": False},
        # gate_proj over the prompts of a rollout batch
        {"name": "linear_prefill_8192", "kind": "linear", "dtype": "bf16", "tokens": 8192, "cols": 4096, "out": 12288,
         "bias": False, "pow2": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _decoder(rng, layers):
    hidden = 128 * _log(rng, 8, 64)
    case = {"hidden": hidden, "inter": 128 * _log(rng, hidden // 64, hidden // 32), "q": 128 * _log(rng, 8, 64),
            "kv": 128 * _log(rng, 2, 8), "layers": layers}
    while case["layers"] > 1 and sum(r * c for _, r, c in _linears(case)) > _MOST_WEIGHTS:
        case["layers"] -= 1
    return case


def draw(rng):
    kind = rng.choice(["tensor", "plan", "plan", "experts", "state", "unstate", "act", "kv", "loader",
                       "linear", "linear", "linear", "linear", "mlp"])
    dt = rng.choice(["bf16", "bf16", "bf16", "f16"])
    pow2 = rng.random() < 0.25
    tokens = _log(rng, 1, 8192)
    if kind == "tensor":
        return {"kind": kind, "dtype": rng.choice(["bf16", "f16", "f32"]), "rows": _log(rng, 256, 32768),
                "cols": 128 * _log(rng, 8, 96), "pow2": pow2}
    if kind == "plan":
        fmt, block = rng.choice([("fp8_block", 128), ("fp8_block", 1), ("mxfp8", 32), ("mxfp4", 32)])
        return {"kind": kind, "fmt": fmt, "block": block, "dtype": rng.choice(["bf16", "bf16", "f32"]),
                **_decoder(rng, rng.randint(1, 4))}
    if kind == "experts":
        # whole experts, or cut by tensor parallelism to widths that 128 does not divide
        rows, cols = rng.choice([(1536, 2048), (2048, 768), (768, 2048), (2048, 384), (384, 2048), (2048, 192)])
        return {"kind": kind, "dtype": dt, "experts": _log(rng, 4, 128), "rows": rows, "cols": cols}
    if kind == "state":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f32"]), **_decoder(rng, rng.randint(1, 2))}
    if kind == "unstate":
        return {"kind": kind, **_decoder(rng, rng.randint(1, 2))}
    if kind == "act":
        return {"kind": kind, "dtype": dt, "tokens": tokens, "cols": 128 * _log(rng, 8, 96), "pow2": pow2}
    if kind == "kv":
        d = _decoder(rng, rng.randint(2, 16))
        return {"kind": kind, "dtype": dt, **{k: d[k] for k in ("hidden", "q", "kv", "layers")}}
    if kind == "loader":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), **_decoder(rng, rng.randint(1, 3)),
                "vocab": _log(rng, 1000, 60000)}
    if kind == "mlp":
        hidden = 128 * _log(rng, 8, 40)
        inter = 128 * _log(rng, hidden // 64, hidden // 32)
        return {"kind": kind, "dtype": dt, "tokens": min(tokens, _MOST_MACS // (3 * hidden * inter)),
                "hidden": hidden, "inter": inter, "pow2": pow2}
    cols, out = 128 * _log(rng, 8, 96), _log(rng, 512, 12288)
    if rng.random() < 0.75:  # most layers are a multiple of a head; a classifier's width is anything
        out = -(-out // 64) * 64
    return {"kind": kind, "dtype": dt, "tokens": min(tokens, _MOST_MACS // (cols * out)), "cols": cols, "out": out,
            "bias": rng.random() < 0.3, "pow2": pow2}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _linears(case):
    h, q, kv = case["hidden"], case["q"], case["kv"]
    qkv = [("self_attn.q_proj", q, h), ("self_attn.k_proj", kv, h), ("self_attn.v_proj", kv, h)]
    rest = []
    if "inter" in case:
        i = case["inter"]
        rest = [("self_attn.o_proj", h, q), ("mlp.gate_proj", i, h), ("mlp.up_proj", i, h), ("mlp.down_proj", h, i)]
    return [("layers.%d.%s.weight" % (n, name), r, c) for n in range(case["layers"]) for name, r, c in qkv + rest]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _weight(gen, dtype, *shape):
    """Trained weights: N(0, 0.02), one in a thousand an outlier."""
    w = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, 0.02, generator=gen)
    flat = w.view(-1)
    n = max(1, flat.numel() // 1000)
    at = torch.randint(0, flat.numel(), (n,), generator=gen, device="cuda")
    flat[at] *= 20.0
    return w.to(_DTYPES[dtype])


def _activation(gen, dtype, tokens, cols):
    """Normed hidden states: N(0, 1), a few channels many times larger."""
    x = torch.empty(tokens, cols, dtype=torch.float32, device="cuda").normal_(0.0, 1.0, generator=gen)
    at = torch.randint(0, cols, (max(1, cols // 500),), generator=gen, device="cuda")
    x[:, at] *= 30.0
    return x.to(_DTYPES[dtype])


class _Engine:
    """Takes the state dict that the loader hands over."""

    def update_weights(self, state_dict):
        self.weights = state_dict


class _Mlp(nn.Module):
    def __init__(self, gate, up, down):
        super().__init__()
        self.gate, self.up, self.down = gate, up, down

    def forward(self, x):
        return self.down(F.silu(self.gate(x)) * self.up(x))


def _module(gen, dtype, out, cols, bias):
    lin = nn.Linear(cols, out, bias=bias, device="meta")
    lin.weight = nn.Parameter(_weight(gen, dtype, out, cols), requires_grad=False)
    if bias:
        b = torch.empty(out, dtype=torch.float32, device="cuda").normal_(0.0, 0.5, generator=gen)
        lin.bias = nn.Parameter(b.to(_DTYPES[dtype]), requires_grad=False)
    return lin


def _patched(model, pow2):
    cfg = FP8Config(precision="fp8", use_deep_gemm=False, use_weight_pow2_scale=pow2, use_activation_pow2_scale=pow2)
    FP8RolloutQuantizer(cfg).quantize_model(model)
    return model


def _inputs(case, seed):
    """The floating inputs of a case, by name, from the seed alone."""
    gen, kind, dt = _gen(seed), case["kind"], case.get("dtype", "bf16")
    if kind == "tensor":
        return {"w": _weight(gen, dt, case["rows"], case["cols"])}
    if kind == "experts":
        return {"w": _weight(gen, dt, case["experts"], case["rows"], case["cols"])}
    if kind in ("plan", "state", "unstate", "kv", "loader"):
        sd = {n: _weight(gen, dt, r, c) for n, r, c in _linears(case)}
        if kind == "loader":
            sd["embed_tokens.weight"] = _weight(gen, dt, case["vocab"], case["hidden"])
            for n in range(case["layers"]):
                sd["layers.%d.input_layernorm.weight" % n] = 1.0 + _weight(gen, dt, case["hidden"])
            sd["norm.weight"] = 1.0 + _weight(gen, dt, case["hidden"])
        return sd
    if kind == "act":
        return {"x": _activation(gen, dt, case["tokens"], case["cols"])}
    if kind == "linear":
        return {"lin": _module(gen, dt, case["out"], case["cols"], case["bias"]),
                "x": _activation(gen, dt, case["tokens"], case["cols"])}
    h, i = case["hidden"], case["inter"]
    return {"gate": _module(gen, dt, i, h, False), "up": _module(gen, dt, i, h, False),
            "down": _module(gen, dt, h, i, False), "x": _activation(gen, dt, case["tokens"], h)}


def _plan_block(case):
    return (case["block"], 128) if case["fmt"] == "fp8_block" else (1, 32)


def prepare(case, seed):
    kind = case["kind"]
    ins = _inputs(case, seed)
    if kind == "tensor":
        return {"call": WeightQuantizer(FP8Config(use_weight_pow2_scale=case["pow2"])).quantize_tensor, "args": (ins["w"],)}
    if kind == "plan":
        return {"call": QuantPlan(list(ins.values()), case["fmt"], _plan_block(case)).run, "args": ()}
    if kind == "experts":
        return {"call": quantize_fp8_blockwise, "args": (ins["w"],)}
    if kind == "state":
        return {"call": WeightQuantizer(FP8Config()).quantize_state_dict, "args": (ins,)}
    if kind == "unstate":
        sd = {}
        for name, w in ins.items():
            codes, scales = _fp8_rows(w)
            sd[name], sd[name + "_fp8_scales"] = codes, scales.to(torch.bfloat16)
        return {"call": WeightQuantizer(FP8Config()).dequantize_state_dict, "args": (sd,)}
    if kind == "act":
        return {"x": ins["x"], "pow2": case["pow2"]}
    if kind == "kv":
        model, names = nn.Module(), []
        for n in range(case["layers"]):
            layer = nn.Module()
            for name in ("q_proj", "k_proj", "v_proj"):
                w = ins["layers.%d.self_attn.%s.weight" % (n, name)]
                lin = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
                lin.weight = nn.Parameter(w, requires_grad=False)
                setattr(layer, name, lin)
                names.append((lin, "_lumenrl_fp8_kv_scale_" + name))
            model.add_module("layer%d" % n, layer)
        return {"kv": FP8KVCacheQuantizer(FP8Config(precision="fp8")), "model": model, "buffers": names}
    if kind == "loader":
        return {"engine": _Engine(), "weights": ins}
    if kind == "linear":
        model = _patched(nn.Sequential(ins["lin"]), case["pow2"])
        return {"model": model, "x": ins["x"]}
    model = _patched(_Mlp(ins["gate"], ins["up"], ins["down"]), case["pow2"])
    return {"model": model, "x": ins["x"]}


def run(state):
    if "call" in state:
        out = state["call"](*state["args"])
        return {k: v for k, v in out.items() if not k.endswith("_fp8_meta")} if isinstance(out, dict) else out
    if "pow2" in state:
        return act_qdq(state["x"], 128, pow2=state["pow2"])
    if "kv" in state:
        state["kv"].recalibrate_scales(state["model"])
        return [getattr(lin, name) for lin, name in state["buffers"]]
    if "engine" in state:
        DynamicWeightLoader.load_weights(state["engine"], state["weights"], {"enabled": True})
        return state["engine"].weights
    with torch.no_grad():
        return state["model"](state["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far results may be off
# ---------------------------------------------------------------------------
def _esize(case):
    return 4 if case.get("dtype") == "f32" else 2


def _linear_work(tokens, cols, out, bias=False):
    """Weights in e4m3 with bf16 scales and 16-bit activations, each read once; 16-bit results."""
    return (out * cols + 2 * out * (cols // 128) + 2 * tokens * cols + 2 * tokens * out + 2 * out * bias,
            2 * tokens * cols * out)


def work(case):
    kind, e = case["kind"], _esize(case)
    flops = 0
    if kind == "tensor":
        n = case["rows"] * case["cols"]
        nbytes = n * (e + 1) + n // 128 * e
    elif kind == "experts":
        n = case["experts"] * case["rows"] * case["cols"]
        nbytes = n * (e + 1) + case["experts"] * -(-case["rows"] // 128) * -(-case["cols"] // 128) * 4
    elif kind == "act":
        nbytes = case["tokens"] * case["cols"] * (e + 4)
    elif kind == "linear":
        nbytes, flops = _linear_work(case["tokens"], case["cols"], case["out"], case["bias"])
    elif kind == "mlp":
        up, down = (_linear_work(case["tokens"], c, o) for c, o in ((case["hidden"], case["inter"]),
                                                                    (case["inter"], case["hidden"])))
        nbytes, flops = 2 * up[0] + down[0], 2 * up[1] + down[1]
    else:
        n = sum(r * c for _, r, c in _linears(case))
        if kind == "kv":
            nbytes = n * e + 4 * 3 * case["layers"]
        elif kind == "loader":
            nbytes = (n + case["hidden"] * (case["vocab"] + case["layers"] + 1)) * (e + 1)
        elif kind == "plan" and case["fmt"] == "mxfp4":
            nbytes = n * e + n // 2 + n // 32
        elif kind == "plan" and case["fmt"] == "mxfp8":
            nbytes = n * (e + 1) + n // 32
        elif kind == "plan":
            nbytes = n * (e + 1) + n // 128 // case["block"] * 4
        else:  # state and unstate: 1x128 blocks with bf16 scales
            nbytes = n * (e + 1) + n // 128 * 2
    return {"bytes": float(nbytes), "flops": float(flops)}


def tolerance(case):
    """Codes, scales and the elementwise paths are bytes that the format defines.
    A linear's sums may run in any order: about four times what the same float32
    product with its columns permuted showed (rel 1.3e-4 and one bf16 ulp over 1 to
    8192 tokens; 5.6e-5 and one fp16 ulp), and in an MLP, whose 16-bit
    intermediates round again, 5.1e-4 and 0.018 (1.3e-4 and 0.0028)."""
    if case["kind"] == "linear":
        return {"rel": 5e-4, "max": 0.032} if case["dtype"] == "bf16" else {"rel": 2.4e-4, "max": 0.004}
    if case["kind"] == "mlp":
        return {"rel": 2e-3, "max": 0.07} if case["dtype"] == "bf16" else {"rel": 5e-4, "max": 0.012}
    return "exact"


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _fp8_rows(w, pow2=False):
    """1x128 codes and float32 scales of a float32 weight, in torch: what a rollout linear keeps."""
    blocks = w.float().view(*w.shape[:-1], -1, 128)
    amax = blocks.abs().amax(-1)
    # a tensor divisor: torch on a GPU turns a division by a Python number into a product
    s = (amax / torch.full_like(amax, _MAX)).clamp_min(torch.finfo(torch.float32).tiny)
    s = _pow2_round(s) if pow2 else s
    return (blocks / s[..., None]).to(_E4M3).view(w.shape), s


def _pow2_round(s):
    return torch.exp2(torch.log2(s).round())


def _e4m3(q):
    return q.to(torch.float32).to(_E4M3).to(torch.float64)


def _rows64(w, pow2=False):
    b = w.double().view(-1, 128)
    s = (b.abs().amax(-1) / _MAX).clamp_min(torch.finfo(torch.float32).tiny)
    s = _pow2_round(s) if pow2 else s
    return _e4m3(b / s[:, None]).view(w.shape), s.view(*w.shape[:-1], -1)


def _tiles64(w):
    *lead, r, c = w.shape
    p = F.pad(w.double(), (0, -c % 128, 0, -r % 128))
    t = p.view(*lead, p.shape[-2] // 128, 128, p.shape[-1] // 128, 128)
    s = (t.abs().amax((-3, -1)) / _MAX).clamp_min(torch.finfo(torch.float32).tiny)
    q = _e4m3(t / s[..., :, None, :, None]).reshape(p.shape)[..., :r, :c]
    return q.contiguous(), s


def _mx64(w):
    """MXFP8 codes, and no value for their E8M0 scales, which are bytes."""
    b = w.double().view(-1, 32)
    e = torch.floor(torch.log2(b.abs().amax(-1))) - 8
    return _e4m3((b / torch.exp2(e)[:, None]).clamp(-_MAX, _MAX)).view(w.shape), None


def _linear64(lin, x, pow2):
    codes, s = _fp8_rows(lin.weight.data, pow2)
    s = s.to(torch.bfloat16).double()
    w = (codes.to(torch.float64).view(lin.out_features, -1, 128) * s[..., None]).view(lin.out_features, -1)
    # the activations' quantize -> dequantize keeps the quotient unrounded: x / s * s
    y = x @ w.T
    return y if lin.bias is None else y + lin.bias.data.double()


def exact(case, seed):
    kind = case["kind"]
    ins = _inputs(case, seed)
    if kind == "tensor":
        if case["dtype"] != "f32":  # quantize_tensor rounds each step to the weight's own 16 bits
            return None
        return _rows64(ins["w"], case["pow2"])
    if kind == "experts":
        return _tiles64(ins["w"])
    if kind == "plan":
        if case["fmt"] == "mxfp4":  # E2M1 codes packed two per byte, E8M0 scales
            return None
        if case["fmt"] == "mxfp8":
            return [_mx64(w) for w in ins.values()]
        return [_tiles64(w) if case["block"] == 128 else _rows64(w) for w in ins.values()]
    if kind == "state":
        out = {}
        for name, w in ins.items():
            out[name], out[name + "_fp8_scales"] = _rows64(w)
        return out
    if kind == "unstate":
        out = {}
        for name, w in ins.items():
            codes, s = _fp8_rows(w)
            out[name] = (codes.double().view(-1, 128) * s.to(torch.bfloat16).double().view(-1, 1)).view(w.shape)
        return out
    if kind == "act":  # x / s * s
        return ins["x"].double()
    if kind == "kv":
        order = ["layers.%d.self_attn.%s.weight" % (n, p) for n in range(case["layers"])
                 for p in ("q_proj", "k_proj", "v_proj")]
        return [ins[n].double().abs().max() / _MAX for n in order]
    if kind == "loader":
        return {n: _e4m3(w.float()) for n, w in ins.items()}
    x = ins["x"].double()
    if kind == "linear":
        return _linear64(ins["lin"], x, case["pow2"])
    gate, up = (_linear64(ins[n], x, case["pow2"]) for n in ("gate", "up"))
    return _linear64(ins["down"], F.silu(gate) * up, case["pow2"])
