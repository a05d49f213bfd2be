"""The operator's workloads, as a serving program meets them, with their inputs, their necessary
work and their values in 64 bits.

Two geometries: "ds" (DeepSeek-V3: hidden 7168, intermediate 2048, 256 experts of which one rank
of eight holds 32, sigmoid routing limited to 4 of 8 groups) and "qwen3" (hidden 4096, intermediate
1536, 128 experts all local, softmax routing). Token counts are those of the operator's definition
(1 .. 14107 tokens, most of them decode batches, odd sizes among them) and of this repository's
benchmark configurations.

How a case reaches the operator ("entry"):
* "run": ``justgoal_amd.moe.run``, the output allocated by the call;
* "run_out": the same with the caller's output tensor;
* "bound": a ``justgoal_amd.moe.bind`` handle made once, then called (a decode loop);
* "layer": the layer as an engine calls it, bf16 activations quantised first, then ``run``;
* "quantize": the activation quantisation alone.
"""
import functools
import math

import torch

from justgoal_amd import moe
from justgoal_amd.geometry import DS_V3, QWEN3

BLOCK = 128
F8 = torch.float8_e4m3fn
GEOMETRY = {"ds": DS_V3, "qwen3": QWEN3}


def _case(name, geometry, tokens, entry, skew=False, offset=0, bias=True):
    case = {"geometry": geometry, "tokens": tokens, "entry": entry, "skew": skew, "offset": offset,
            "bias": bias}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest call: one sequence being decoded, eight experts streamed for one token.
        _case("qwen3_decode_1", "qwen3", 1, "run"),
        # A few sequences on one expert-parallel rank: most of the rank's experts stay idle.
        _case("ds_decode_7", "ds", 7, "run"),
        # A decode loop that keeps its buffers and calls through a bound handle.
        _case("ds_decode_16", "ds", 16, "bound"),
        # A decode batch as the layer of an engine: bf16 activations quantised, then the experts.
        _case("ds_layer_57", "ds", 57, "layer"),
        # A wide decode batch, or a short prompt, on another rank than the first.
        _case("ds_decode_193", "ds", 193, "run", offset=32),
        # A decode batch where every expert holds a few rows.
        _case("qwen3_decode_128", "qwen3", 128, "run"),
        # A ragged prefill chunk into the caller's output tensor.
        _case("ds_prefill_901", "ds", 901, "run_out"),
        # A prefill chunk with softmax routing: 64 rows on each of 128 experts.
        _case("qwen3_prefill_1024", "qwen3", 1024, "run"),
        # A usual prefill batch.
        _case("ds_prefill_4096", "ds", 4096, "run"),
        # The definition's longest batch.
        _case("ds_prefill_14107", "ds", 14107, "run_out"),
        # The largest batch with eight hot experts, the imbalance that load balancing fights.
        _case("ds_skewed_16384", "ds", 16384, "run", skew=True),
        # The producer of the operator's inputs at a prefill batch.
        _case("ds_quantize_4096", "ds", 4096, "quantize"),
    ]


def draw(rng):
    kind = rng.choice(("ds", "ds", "ds", "qwen3", "qwen3", "skew", "quantize"))
    top = {"ds": 14107, "qwen3": 2048, "skew": 16384, "quantize": 16384}[kind]
    low = 256 if kind == "skew" else 1
    tokens = int(round(math.exp(rng.uniform(math.log(low), math.log(top + 0.49)))))
    tokens = min(max(tokens, low), top)
    if kind == "quantize":
        return _case("", rng.choice(("ds", "qwen3")), tokens, "quantize")
    entry = rng.choice(("run", "run", "run_out", "bound", "layer"))
    if kind == "qwen3":
        return _case("", "qwen3", tokens, entry, bias=False)
    # the skewed batches' hot experts are those of the rank
    return _case("", "ds", tokens, entry, skew=kind == "skew", offset=32 * rng.randrange(8),
                 bias=rng.random() < 0.8)


def _generator(seed, part, device):
    return torch.Generator(device=device).manual_seed((int(seed) * 1000003 + part) & 0x7FFFFFFFFFFF)


def _routing_inputs(case, seed, device):
    """Router logits N(0, 1) and bias N(0, 0.1), the benchmark's distributions; a skewed batch's
    first eight local experts get +3."""
    geom = GEOMETRY[case["geometry"]]
    logits = torch.randn(case["tokens"], geom.num_experts, device=device,
                         generator=_generator(seed, 1, device))
    if case["skew"]:
        logits[:, case["offset"]:case["offset"] + 8] += 3.0
    bias = None
    if case["bias"]:
        bias = (torch.randn(geom.num_experts, device=device,
                            generator=_generator(seed, 2, device)) * 0.1).to(torch.bfloat16)
    return logits, bias


def _quantize_blocks(w):
    """[R, C] -> e4m3 codes and fp32 scales of its 128x128 blocks (scale = amax / 448)."""
    R, C = w.shape
    wb = w.view(R // BLOCK, BLOCK, C // BLOCK, BLOCK)
    s = wb.abs().amax(dim=(1, 3)) / 448.0
    return (wb / s[:, None, :, None]).clamp(-448, 448).to(F8).view(R, C), s


def _weights(geom, seed, device):
    """N(0, 0.02) expert weights in fp8 with 128x128 block scales."""
    E, H, I = geom.local_experts, geom.hidden, geom.intermediate
    g = _generator(seed, 3, device)
    w13 = torch.empty(E, 2 * I, H, dtype=F8, device=device)
    s13 = torch.empty(E, 2 * I // BLOCK, H // BLOCK, device=device)
    w2 = torch.empty(E, H, I, dtype=F8, device=device)
    s2 = torch.empty(E, H // BLOCK, I // BLOCK, device=device)
    for e in range(E):
        for w, s in ((w13, s13), (w2, s2)):
            q, sc = _quantize_blocks(torch.randn(w.shape[1:], device=device, generator=g) * 0.02)
            w[e].copy_(q)
            s[e].copy_(sc)
    return w13, s13, w2, s2


def _hidden(case, seed, device):
    geom = GEOMETRY[case["geometry"]]
    return torch.randn(case["tokens"], geom.hidden, device=device,
                       generator=_generator(seed, 4, device)).to(torch.bfloat16)


def _quantize_rows(x):
    """bf16 [T, H] -> e4m3 codes and transposed fp32 scales of its 1x128 blocks."""
    T, H = x.shape
    xb = x.float().view(T, H // BLOCK, BLOCK)
    amax = xb.abs().amax(dim=2)
    s = amax / torch.full_like(amax, 448.0)  # rounded division: many x / s fall on e4m3 ties
    s = torch.where(s > 0, s, torch.ones_like(s))
    q = (xb / s[:, :, None]).clamp(-448, 448).to(F8).view(T, H)
    return q, s.t().contiguous()


def _scaling(geom):
    return 2.5 if geom is DS_V3 else 1.0


def _inputs(case, seed, device):
    """The operator's ten arguments."""
    geom = GEOMETRY[case["geometry"]]
    logits, bias = _routing_inputs(case, seed, device)
    x = _hidden(case, seed, device)
    hs, hs_scale = _quantize_rows(x)
    args = [logits, bias, hs, hs_scale, *_weights(geom, seed, device), case["offset"], _scaling(geom)]
    return args, x


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def prepare(case, seed):
    geom = GEOMETRY[case["geometry"]]
    entry = case["entry"]
    if entry == "quantize":
        return {"entry": entry, "x": _hidden(case, seed, _device())}
    args, x = _inputs(case, seed, _device())
    state = {"entry": entry, "geometry": geom, "args": args}
    if entry == "run_out":
        state["out"] = torch.empty_like(x)
    elif entry == "bound":
        state["call"] = moe.bind(*args, geometry=geom)
    elif entry == "layer":
        state["x"] = x
    return state


def run(state):
    entry = state["entry"]
    if entry == "quantize":
        return moe.quantize_activations(state["x"])
    if entry == "bound":
        return state["call"]()
    args = state["args"]
    if entry == "run_out":
        return moe.run(*args, state["out"], geometry=state["geometry"])
    if entry == "layer":
        logits, bias = args[:2]
        hs, hs_scale = moe.quantize_activations(state["x"])
        return moe.run(logits, bias, hs, hs_scale, *args[4:], geometry=state["geometry"])
    return moe.run(*args, geometry=state["geometry"])


def _route64(geom, logits, bias, scaling):
    """Routing in 64 bits: (global expert ids [T, top_k], weights [T, top_k])."""
    x = logits.double()
    if geom is DS_V3:
        s = torch.sigmoid(x)
        v = s if bias is None else s + bias.double()
        T, E = v.shape
        groups = v.view(T, geom.n_group, E // geom.n_group)
        score = groups.topk(2, dim=2).values.sum(dim=2)
        kept = torch.zeros_like(score, dtype=torch.bool)
        kept.scatter_(1, score.topk(geom.topk_group, dim=1).indices, True)
        masked = torch.where(kept[:, :, None], groups, -math.inf).reshape(T, E)
        idx = masked.topk(geom.top_k, dim=1).indices
        w = s.gather(1, idx)
        return idx, w / (w.sum(dim=1, keepdim=True) + 1e-20) * scaling
    top = x.topk(geom.top_k, dim=1)
    return top.indices, torch.softmax(top.values, dim=1)


WORK_SEEDS = 5


@functools.lru_cache(maxsize=None)
def _routed(geometry, tokens, skew, offset, bias):
    """Mean (pairs, active local experts, tokens with a local pair) over a few routings."""
    case = _case("", geometry, tokens, "run", skew, offset, bias)
    geom = GEOMETRY[geometry]
    pairs = active = routed = 0.0
    for seed in range(WORK_SEEDS):
        logits, b = _routing_inputs(case, seed, torch.device("cpu"))
        idx, _ = _route64(geom, logits, b, 1.0)
        local = (idx >= offset) & (idx < offset + geom.local_experts)
        pairs += int(local.sum())
        active += idx[local].unique().numel()
        routed += int(local.any(dim=1).sum())
    return pairs / WORK_SEEDS, active / WORK_SEEDS, routed / WORK_SEEDS


def work(case):
    """Routed fp8 rows with their scales, the logits, the weights and scales of the experts that
    hold a pair, and the bf16 output, each once; 6 H I operations for each pair."""
    geom = GEOMETRY[case["geometry"]]
    T, H, I = case["tokens"], geom.hidden, geom.intermediate
    quant = T * H * 3 + 4 * T * (H // BLOCK)
    if case["entry"] == "quantize":
        return {"bytes": quant, "flops": 3 * T * H}
    pairs, active, routed = _routed(case["geometry"], T, case["skew"], case["offset"], case["bias"])
    expert = 3 * I * H + 4 * 3 * (I // BLOCK) * (H // BLOCK)
    bytes_ = (active * expert + routed * (H + 4 * (H // BLOCK)) + 4 * T * geom.num_experts
              + 2 * T * H)
    if case["entry"] == "layer":
        bytes_ += quant
    return {"bytes": int(bytes_), "flops": int(6 * H * I * pairs)}


def tolerance(case):
    if case["entry"] == "quantize":
        return "exact"
    # bf16 intermediate rows, one bf16 rounding per term of a token's sum, bf16 output: measured
    # 2.9e-3 of the 2-norm against 64 bits.
    return {"rel": 1e-2, "max": 1e-1}


def _dequant_rows(q, s):
    T, H = q.shape
    return (q.double().view(T, H // BLOCK, BLOCK) * s.double().t()[:, :, None]).view(T, H)


def _dequant_blocks(q, s):
    R, C = q.shape
    return (q.double().view(R // BLOCK, BLOCK, C // BLOCK, BLOCK)
            * s.double()[:, None, :, None]).view(R, C)


def exact(case, seed):
    device = _device()
    if case["entry"] == "quantize":
        x = _hidden(case, seed, device).double()
        xb = x.view(x.shape[0], -1, BLOCK)
        s = xb.abs().amax(dim=2) / 448.0
        return (xb / torch.where(s > 0, s, torch.ones_like(s))[:, :, None]).view_as(x), s.t()
    geom = GEOMETRY[case["geometry"]]
    args, _ = _inputs(case, seed, device)
    logits, bias, hs, hs_scale, w13, s13, w2, s2, offset, scaling = args
    I = geom.intermediate
    idx, weight = _route64(geom, logits, bias, scaling)
    out = torch.zeros(case["tokens"], geom.hidden, dtype=torch.float64, device=device)
    for e in range(geom.local_experts):
        tok, slot = (idx == offset + e).nonzero(as_tuple=True)
        if tok.numel() == 0:
            continue
        g = _dequant_rows(hs[tok], hs_scale[:, tok]) @ _dequant_blocks(w13[e], s13[e]).t()
        c = g[:, :I] * torch.nn.functional.silu(g[:, I:])
        out[tok] += weight[tok, slot][:, None] * (c @ _dequant_blocks(w2[e], s2[e]).t())
    return out
