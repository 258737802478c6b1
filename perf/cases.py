"""Workloads of the weight-only quantised linear and MoE path, for timing.

A case is one pass through the public entry points as a serving program makes it: the linears of a decoder layer
(`MarlinLinearKernel.apply_weights` for GPTQ-style checkpoints, `apply_awq_marlin_linear` for AWQ ones), an MoE block
(`fused_topk` + `fused_marlin_moe`), or the preparation of checkpoint weights at load time.  Shapes are those of the
repository's benchmark (a Llama-3-8B decoder layer, Mixtral-8x7B experts, a 128-expert top-8 layer) or generic ones.

  kind = "linear"  layers: "KxN,KxN,..." called one after the other on m rows each; graph: the calls were captured in a
                   HIP graph once and a pass replays it, as serving programs do for decode
  kind = "moe"     experts / hidden / inter / topk, tokens rows
  kind = "load"    experts = 0: the dense layers of `layers`; else the two stacked expert weights

fmt: gptq4 (uint4b8), gptq8 (uint8b128), awq4 (uint4 with zero points).  The fp8 and fp4 weight types are left out: this
card multiplies those natively, so a weight-only path is not what serves such checkpoints on it.
"""
import math

import torch

from vllm_amd import ops
from vllm_amd.fused_marlin_moe import fused_marlin_moe
from vllm_amd.fused_moe import fused_topk
from vllm_amd.marlin_utils import (apply_awq_marlin_linear, awq_to_marlin_zero_points, marlin_make_empty_g_idx,
                                   marlin_make_workspace_new, marlin_moe_permute_scales, marlin_permute_bias,
                                   marlin_permute_scales, moe_awq_to_marlin_zero_points)
from vllm_amd.mixed_precision import MarlinLinearKernel, MPLinearLayerConfig
from vllm_amd.scalar_type import scalar_types

DEV = "cuda"
LAYER_8B = "4096x6144,4096x4096,4096x28672,14336x4096"  # qkv, o, gate_up, down
WTYPES = {"gptq4": scalar_types.uint4b8, "gptq8": scalar_types.uint8b128, "awq4": scalar_types.uint4}
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
AWQ_ORDER = (0, 2, 4, 6, 1, 3, 5, 7)


def _linear(name, layers, m, fmt, dtype, group=128, act_order=False, bias=False, graph=False):
    c = {"kind": "linear", "layers": layers, "m": m, "fmt": fmt, "dtype": dtype, "group": group,
         "act_order": act_order, "bias": bias, "graph": graph}
    return {"name": name, **c} if name else c


def _moe(name, experts, hidden, inter, topk, tokens, fmt, dtype, group=128):
    c = {"kind": "moe", "experts": experts, "hidden": hidden, "inter": inter, "topk": topk, "tokens": tokens,
         "fmt": fmt, "dtype": dtype, "group": group}
    return {"name": name, **c} if name else c


def _load(name, experts, layers, fmt, dtype, group=128, act_order=False):
    c = {"kind": "load", "experts": experts, "layers": layers, "fmt": fmt, "dtype": dtype, "group": group,
         "act_order": act_order}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one sequence being decoded without graphs: a single projection, the smallest call there is
        _linear("o_proj_1_row", "4096x4096", 1, "gptq4", "fp16"),
        # decode of 16 sequences, captured: the whole decoder layer, the repository's headline workload
        _linear("decode_16_graph", LAYER_8B, 16, "gptq4", "fp16", graph=True),
        # decode of an odd number of sequences, called eagerly, AWQ checkpoint in bf16
        _linear("decode_37_awq", LAYER_8B, 37, "awq4", "bf16"),
        # 8-bit GPTQ checkpoint, decode
        _linear("decode_16_8bit", LAYER_8B, 16, "gptq8", "bf16"),
        # decode mixed with a chunk of a prompt; layers with a bias
        _linear("mixed_203", LAYER_8B, 203, "gptq4", "bf16", bias=True),
        # act-order checkpoint, the long-K projection, a chunk of a prompt
        _linear("act_order_down_300", "14336x4096", 300, "gptq4", "fp16", act_order=True),
        # a ragged batch of prompts on a fine-grouped checkpoint
        _linear("prefill_1501_g32", LAYER_8B, 1501, "gptq4", "fp16", group=32),
        # a full prefill chunk
        _linear("prefill_4096_awq", LAYER_8B, 4096, "awq4", "bf16"),
        # few, large experts: decode and a full prefill chunk
        _moe("mixtral_16", 8, 4096, 14336, 2, 16, "gptq4", "fp16"),
        _moe("mixtral_4096", 8, 4096, 14336, 2, 4096, "gptq4", "bf16"),
        # many, small experts with zero points, an odd number of tokens
        _moe("experts128_601_awq", 128, 2048, 768, 8, 601, "awq4", "bf16"),
        # what a server does with such a checkpoint when it starts
        _load("load_experts128", 128, "2048x1536,768x2048", "gptq4", "fp16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("linear", "moe", "load"), (6, 3, 1))[0]
    dtype = rng.choice(("fp16", "bf16"))
    group = rng.choice((128, 128, 128, 64, 32, -1))
    if kind == "linear":
        fmt = rng.choice(("gptq4", "gptq4", "awq4", "awq4", "gptq8"))
        if rng.random() < 0.3:
            layers = LAYER_8B
        else:
            layers = "%dx%d" % (128 * _log_int(rng, 8, 112), 64 * _log_int(rng, 16, 448))
        size = sum(int(s.split("x")[0]) * int(s.split("x")[1]) for s in layers.split(","))
        m = min(_log_int(rng, 1, 4096), int(9e11 / size))
        act = fmt != "awq4" and rng.random() < 0.2
        return _linear(None, layers, m, fmt, dtype, 128 if act else group, act, rng.random() < 0.2,
                       m <= 64 and rng.random() < 0.5)
    if kind == "moe":
        experts, hidden, inter, topk = rng.choice(
            ((8, 4096, 14336, 2), (128, 2048, 768, 8), (64, 2048, 1408, 6),
             (2 ** rng.randint(2, 7), 128 * _log_int(rng, 8, 32), 128 * _log_int(rng, 4, 32), rng.randint(1, 4))))
        return _moe(None, experts, hidden, inter, topk, _log_int(rng, 1, 4096), rng.choice(("gptq4", "awq4")), dtype,
                    rng.choice((128, 128, 64, 32)))
    fmt = rng.choice(("gptq4", "awq4"))
    if rng.random() < 0.5:
        k, n = 128 * _log_int(rng, 8, 112), 64 * _log_int(rng, 16, 448)
        return _load(None, 0, "%dx%d" % (k, n), fmt, dtype, 128, fmt == "gptq4" and rng.random() < 0.3)
    experts, hidden, inter = 2 ** rng.randint(3, 7), 128 * _log_int(rng, 8, 20), 128 * _log_int(rng, 4, 12)
    return _load(None, experts, "%dx%d,%dx%d" % (hidden, 2 * inter, inter, hidden), fmt, dtype)


# ------------------------------------------------------------------------------------------------ checkpoints
def _shapes(case):
    if case["kind"] == "moe":
        return [(case["hidden"], 2 * case["inter"]), (case["inter"], case["hidden"])]
    return [tuple(int(v) for v in s.split("x")) for s in case["layers"].split(",")]


def _groups(case, k):
    """Rows of the scales; one for channel-wise scales."""
    return 1 if case["group"] == -1 else k // case["group"]


def _quantise(case, k, n, gen):
    """Bell-shaped weights rounded to the nearest code -> (codes int32 [K, N], scales [G, N], zero points [G, N] or None)."""
    g = _groups(case, k)
    w = (torch.randn(g, k // g, n, device=DEV, dtype=torch.float16, generator=gen) * 0.02)
    if case["fmt"] == "awq4":
        lo, hi = w.amin(1, keepdim=True).float(), w.amax(1, keepdim=True).float()
        s = ((hi - lo) / 15).clamp(min=1e-5).to(DTYPES[case["dtype"]])
        z = (-lo / s).round().clamp(0, 15).int()
        q = (w / s).round().int().add_(z).clamp_(0, 15)
        return q.view(k, n), s.view(g, n), z.view(g, n)
    half = 127 if case["fmt"] == "gptq8" else 7
    s = (w.abs().amax(1, keepdim=True).float() / half).clamp(min=1e-5).to(DTYPES[case["dtype"]])
    q = (w / s).round().int().clamp_(-half - 1, half).add_(half + 1)
    return q.view(k, n), s.view(g, n), None


def _pack_rows(q, bits):
    """GPTQ packing: value i of word (r, n) is row r * 32 / bits + i."""
    per = 32 // bits
    v = q.view(q.shape[0] // per, per, q.shape[1])
    out = v[:, 0].clone()
    for i in range(1, per):
        out |= v[:, i] << (bits * i)
    return out


def _pack_cols(q, order):
    """Column packing: nibble t of word c is column 8 c + order[t]."""
    v = q.view(q.shape[0], q.shape[1] // 8, 8)
    out = v[:, :, order[0]].clone()
    for t in range(1, 8):
        out |= v[:, :, order[t]] << (4 * t)
    return out


def _checkpoint(case, k, n, gen):
    """One weight as its checkpoint stores it: (qweight, scales, qzeros or None)."""
    q, s, z = _quantise(case, k, n, gen)
    if case["fmt"] == "awq4":
        return _pack_cols(q, AWQ_ORDER), s, _pack_cols(z, AWQ_ORDER)
    return _pack_rows(q, 8 if case["fmt"] == "gptq8" else 4), s, None


def _g_idx(case, k, gen):
    """Act-order checkpoints number the group of every input row, in no order."""
    return (torch.randperm(k, device=DEV, generator=gen) // case["group"]).to(torch.int32)


def _gptq_layer(case, k, n, qweight, scales, g_idx, bias=None):
    """The layer as a model loader leaves it, and the kernel object that prepares and applies it."""
    config = MPLinearLayerConfig((k, n), (k, n), WTYPES[case["fmt"]], DTYPES[case["dtype"]], case["group"], False,
                                 g_idx is not None)
    kernel = MarlinLinearKernel(config, "qweight", "scales", None, "g_idx" if g_idx is not None else None)
    layer = torch.nn.Module()
    for name, t in (("qweight", qweight), ("scales", scales), ("g_idx", g_idx), ("bias", bias)):
        if t is not None:
            layer.register_parameter(name, torch.nn.Parameter(t, requires_grad=False))
    return kernel, layer


# ------------------------------------------------------------------------------------------------ linear
def _prepare_linear(case, gen):
    dtype, calls = DTYPES[case["dtype"]], []
    for k, n in _shapes(case):
        qweight, scales, qzeros = _checkpoint(case, k, n, gen)
        bias = torch.randn(n, device=DEV, dtype=dtype, generator=gen) if case["bias"] else None
        x = torch.randn(case["m"], k, device=DEV, dtype=dtype, generator=gen)
        if case["fmt"] == "awq4":
            empty = marlin_make_empty_g_idx(torch.device(DEV))
            layer = (ops.awq_marlin_repack(qweight, k, n, 4), marlin_permute_scales(scales, k, n, case["group"]),
                     awq_to_marlin_zero_points(qzeros, scales.shape[0], n, 4), empty, empty,
                     marlin_make_workspace_new(torch.device(DEV)), WTYPES["awq4"], n, k,
                     None if bias is None else marlin_permute_bias(bias))
            calls.append((None, layer, x))
        else:
            kernel, layer = _gptq_layer(case, k, n, qweight, scales, _g_idx(case, k, gen) if case["act_order"] else None, bias)
            kernel.process_weights_after_loading(layer)
            calls.append((kernel, layer, x))
    state = {"case": case, "calls": calls}
    if case["graph"]:
        _run_linear(calls)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = _run_linear(calls)
    return state


def _run_linear(calls):
    out = []
    for kernel, layer, x in calls:
        if kernel is None:
            out.append(apply_awq_marlin_linear(x, *layer))
        else:
            out.append(kernel.apply_weights(layer, x, getattr(layer, "bias", None)))
    return out


# ------------------------------------------------------------------------------------------------ MoE
def _expert_checkpoint(case, k, n, gen):
    parts = [_checkpoint(case, k, n, gen) for _ in range(case["experts"])]
    return tuple(None if p[0] is None else torch.stack(p) for p in zip(*parts))


def _load_experts(case, k, n, qweight, scales, qzeros):
    """Checkpoint tensors of all experts -> the operands of the MoE GEMM."""
    perm = torch.empty((case["experts"], 0), dtype=torch.int32, device=DEV)
    repack = ops.awq_marlin_moe_repack if case["fmt"] == "awq4" else ops.gptq_marlin_moe_repack
    w = repack(qweight, perm, k, n, 4)
    s = marlin_moe_permute_scales(scales, k, n, case["group"])
    z = None if qzeros is None else moe_awq_to_marlin_zero_points(qzeros, scales.shape[1], n, 4)
    return w, s, z


def _prepare_moe(case, gen):
    dtype = DTYPES[case["dtype"]]
    w = [_load_experts(case, k, n, *_expert_checkpoint(case, k, n, gen)) for k, n in _shapes(case)]
    return {"case": case, "w": w, "workspace": marlin_make_workspace_new(torch.device(DEV), 4),
            "x": torch.randn(case["tokens"], case["hidden"], device=DEV, dtype=dtype, generator=gen),
            "logits": torch.randn(case["tokens"], case["experts"], device=DEV, dtype=dtype, generator=gen)}


def _run_moe(s):
    case, ((w1, s1, z1), (w2, s2, z2)) = s["case"], s["w"]
    weights, ids, _ = fused_topk(s["x"], s["logits"], case["topk"], True)
    out = fused_marlin_moe(s["x"], w1, w2, None, None, s1, s2, s["logits"], weights, ids,
                           quant_type_id=WTYPES[case["fmt"]].id, global_num_experts=case["experts"], w1_zeros=z1,
                           w2_zeros=z2, workspace=s["workspace"])
    return {"out": out, "weights": weights, "ids": ids}


# ------------------------------------------------------------------------------------------------ load
def _prepare_load(case, gen):
    parts = []
    for k, n in _shapes(case):
        make = _expert_checkpoint if case["experts"] else _checkpoint
        parts.append((k, n) + make(case, k, n, gen) + (_g_idx(case, k, gen) if case["act_order"] else None,))
    return {"case": case, "parts": parts}


def _run_load(s):
    case, out = s["case"], []
    for k, n, qweight, scales, qzeros, g_idx in s["parts"]:
        if case["experts"]:
            out.append(_load_experts(case, k, n, qweight, scales, qzeros))
        elif case["fmt"] == "awq4":
            out.append((ops.awq_marlin_repack(qweight, k, n, 4), marlin_permute_scales(scales, k, n, case["group"]),
                        awq_to_marlin_zero_points(qzeros, scales.shape[0], n, 4)))
        else:
            kernel, layer = _gptq_layer(case, k, n, qweight, scales, g_idx)
            kernel.process_weights_after_loading(layer)
            out.append((layer.qweight, layer.scales, layer.g_idx, layer.g_idx_sort_indices))
    return out


# ------------------------------------------------------------------------------------------------ interface
def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return {"linear": _prepare_linear, "moe": _prepare_moe, "load": _prepare_load}[case["kind"]](case, gen)


def run(state):
    kind = state["case"]["kind"]
    if kind == "moe":
        return _run_moe(state)
    if kind == "load":
        return _run_load(state)
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _run_linear(state["calls"])


def _weight_bytes(case, k, n):
    g = _groups(case, k)
    return k * n * (8 if case["fmt"] == "gptq8" else 4) // 8 + g * n * 2 + (g * n // 2 if case["fmt"] == "awq4" else 0)


def work(case):
    shapes = _shapes(case)
    if case["kind"] == "load":
        return {"bytes": 2 * max(1, case["experts"]) * sum(_weight_bytes(case, k, n) for k, n in shapes), "flops": 0}
    if case["kind"] == "moe":
        t, e, topk = case["tokens"], case["experts"], case["topk"]
        hit = e * (1 - (1 - topk / e) ** t)  # experts that at least one token is expected to choose
        return {"bytes": hit * sum(_weight_bytes(case, k, n) for k, n in shapes) + t * (case["hidden"] * 4 + e * 2 + topk * 8),
                "flops": 2 * t * topk * sum(k * n for k, n in shapes)}
    m = case["m"]
    return {"bytes": sum(_weight_bytes(case, k, n) + m * (k + n) * 2 + (8 * k if case["act_order"] else 0) +
                         (2 * n if case["bias"] else 0) for k, n in shapes),
            "flops": 2 * m * sum(k * n for k, n in shapes)}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    # a weight may be rounded to 16 bits once, or stay exact and have its scale applied to the fp32 sum
    rel = 2e-3 if case["dtype"] == "fp16" else 1e-2
    return {"rel": rel} if case["kind"] == "linear" else {"rel": 2 * rel if case["dtype"] == "fp16" else rel, "differ": 1e-3}
