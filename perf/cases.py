"""The workloads this package is measured on: block-FP8 linears, decoder layers, routed experts and the quantizer.

A case is a dict of plain values; ``prepare`` turns it into what a serving process holds before the call (quantized
weights, activations, routing), ``run`` is one pass through the public entry points.  ``kind`` selects the path:

  linear   the quantization method's ``apply`` (activation quantizer + GEMM) on ``layers`` weights of one shape
  decoder  the linears of ``layers`` dense decoder layers: qkv, o, gate_up, SiLU-mul, down (attention, norms and the
           residual stream are not this package's: what they hand over is an input here); with ``graph`` the pass is
           the replay of a captured HIP graph, as in decode loops
  moe      ``fused_experts`` of ``layers`` layers
  ep       ``masked_group_gemm``: one rank's experts on the padded layout of a low-latency dispatch
  quant    the standalone activation quantizer
"""
import math

import torch

from lightllm_amd.fused_moe import fused_experts, masked_group_gemm, silu_and_mul_fwd
from lightllm_amd.quantization import QUANTMETHODS, WeightPack, mm_weight_quant, per_token_group_quant_fp8

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# (N, K) of the linears of Llama-3-8B (qkv, o, gate_up, down), Llama-2 (gate_up, down) and DeepSeek-V3
# (dense gate_up, dense down, q_a+kv_a with its ragged last block, q_b)
LINEARS = ((6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (27648, 5120), (5120, 13824),
           (36864, 7168), (7168, 18432), (2112, 7168), (24576, 1536))
# experts, top-k, hidden, intermediate: DeepSeek-V3, Qwen3-30B-A3B, DeepSeek-V2-Lite, Mixtral
EXPERTS = ((256, 8, 7168, 2048), (128, 8, 2048, 768), (64, 6, 2048, 1408), (8, 2, 4096, 14336))
HIDDEN, QKV, INTER = 4096, 6144, 14336   # Llama-3-8B


def listed():
    return [
        # one sequence decoding, one linear per layer: the smallest call there is, launches and host work count;
        # each layer has its own weight, so that it comes from HBM as it does in a model
        {"name": "o_proj_1", "kind": "linear", "m": 1, "n": 4096, "k": 4096, "layers": 16, "dtype": "bf16"},
        # a few sequences decoding under a captured graph: how a server runs small decode batches
        {"name": "decoder_4_graph", "kind": "decoder", "m": 4, "layers": 4, "graph": True},
        # an ordinary decode batch, launched eagerly
        {"name": "decoder_48", "kind": "decoder", "m": 48, "layers": 3, "graph": False},
        # a short prompt with an odd number of tokens, float16 activations
        {"name": "gate_up_fp16_333", "kind": "linear", "m": 333, "n": 27648, "k": 5120, "layers": 1, "dtype": "fp16"},
        # a prefill chunk on a long K
        {"name": "down_640", "kind": "linear", "m": 640, "n": 7168, "k": 18432, "layers": 1, "dtype": "bf16"},
        # a longer chunk on a narrow weight whose last 128-row block is half empty
        {"name": "qkv_a_2047", "kind": "linear", "m": 2047, "n": 2112, "k": 7168, "layers": 1, "dtype": "bf16"},
        # a full prefill batch on the widest dense linear
        {"name": "gate_up_4096", "kind": "linear", "m": 4096, "n": 36864, "k": 7168, "layers": 1, "dtype": "bf16"},
        # small experts, a few sequences decoding: seven small steps per layer
        {"name": "moe_small_4", "kind": "moe", "t": 4, "experts": 128, "topk": 8, "hidden": 2048, "inter": 768,
         "zipf": 0.0, "layers": 4},
        # large experts, an ordinary decode batch: nearly every expert is read for one to a few rows
        {"name": "moe_decode_64", "kind": "moe", "t": 64, "experts": 256, "topk": 8, "hidden": 7168, "inter": 2048,
         "zipf": 0.0, "layers": 1},
        # large experts, a prefill batch with uneven popularity
        {"name": "moe_prefill_4096", "kind": "moe", "t": 4096, "experts": 256, "topk": 8, "hidden": 7168,
         "inter": 2048, "zipf": 1.1, "layers": 1},
        # one of eight expert-parallel ranks in decode: 64 tokens from each rank, padded to what could arrive
        {"name": "ep_512x16", "kind": "ep", "experts": 32, "padded": 512, "rows": 16, "hidden": 7168, "inter": 2048},
        # the quantizer by itself on a large prefill batch, heavy-tailed values
        {"name": "quant_16384", "kind": "quant", "m": 16384, "k": 7168, "dtype": "bf16", "columns": False},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "decoder", "decoder", "moe", "moe", "ep", "quant"))
    if kind == "linear":
        n, k = rng.choice(LINEARS)
        m = _log_int(rng, 1, 4096)
        layers = 1 if m > 128 else max(1, min(16, 300_000_000 // (n * k)))
        return {"kind": kind, "m": m, "n": n, "k": k, "layers": layers, "dtype": rng.choice(("bf16", "bf16", "fp16"))}
    if kind == "decoder":
        m = _log_int(rng, 1, 512)
        return {"kind": kind, "m": m, "layers": 2, "graph": m <= 128 and rng.random() < 0.5}
    if kind == "moe":
        experts, topk, hidden, inter = rng.choice(EXPERTS)
        t = _log_int(rng, 1, 4096)
        return {"kind": kind, "t": t, "experts": experts, "topk": topk, "hidden": hidden, "inter": inter,
                "zipf": rng.choice((0.0, 1.1)), "layers": 4 if t <= 64 and experts * hidden * inter < 500_000_000 else 1}
    if kind == "ep":
        rows = _log_int(rng, 1, 128)
        return {"kind": kind, "experts": rng.choice((16, 32)), "padded": rows * 32, "rows": rows, "hidden": 7168,
                "inter": 2048}
    return {"kind": kind, "m": _log_int(rng, 1, 16384), "k": 128 * rng.randint(8, 144) if rng.random() < 0.5 else 7168,
            "dtype": rng.choice(("bf16", "bf16", "fp16")), "columns": rng.random() < 0.5}


# ---- inputs

def _normal(gen, shape, dtype=torch.bfloat16, scale=1.0):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=dtype)
    return x if scale == 1.0 else x.mul_(scale)


def _pack(gen, n, k):
    return WeightPack(*mm_weight_quant(_normal(gen, (n, k), scale=0.02)))


def _expert_weights(gen, experts, n, k):
    w = torch.empty((experts, n, k), dtype=torch.float8_e4m3fn, device="cuda")
    s = torch.empty((experts, n // 128, k // 128), dtype=torch.float32, device="cuda")
    for e in range(experts):
        w[e], s[e] = mm_weight_quant(_normal(gen, (n, k), scale=0.02))
    return w, s


def _routing(case, seed):
    """topk_ids int32 [T, topk]: distinct experts per token, drawn by popularity (rank ** -zipf in a random order)."""
    gen = torch.Generator().manual_seed(seed)
    t, experts = case["t"], case["experts"]
    weight = torch.arange(1, experts + 1, dtype=torch.float32) ** -case["zipf"]
    weight = weight[torch.randperm(experts, generator=gen)]
    keys = weight.log() - torch.empty((t, experts)).exponential_(generator=gen).log()   # Gumbel top-k
    return keys.topk(case["topk"], dim=1).indices.to(torch.int32)


def _expert_rows(case, seed):
    """Rows that arrive for each expert of a rank: ``experts * rows`` in all, unevenly spread (popularity from 0 to 2
    times the mean, so that the padded size, 32 times the mean, is never reached)."""
    gen = torch.Generator().manual_seed(seed)
    share = torch.rand((case["experts"],), generator=gen)
    hits = torch.multinomial(share, case["experts"] * case["rows"], replacement=True, generator=gen)
    return torch.bincount(hits, minlength=case["experts"]).to(torch.int32)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind in ("linear", "decoder"):
        state["method"] = QUANTMETHODS.get("fp8w8a8-b128")
    if kind == "linear":
        m, n, k, layers = case["m"], case["n"], case["k"], case["layers"]
        state["x"] = [_normal(gen, (m, k), DTYPES[case["dtype"]]) for _ in range(layers)]
        state["w"] = [_pack(gen, n, k) for _ in range(layers)]
    elif kind == "decoder":
        m, layers = case["m"], case["layers"]
        state["x"] = [{name: _normal(gen, (m, HIDDEN)) for name in ("qkv", "o", "gate_up")} for _ in range(layers)]
        state["w"] = [{"qkv": _pack(gen, QKV, HIDDEN), "o": _pack(gen, HIDDEN, HIDDEN),
                       "gate_up": _pack(gen, 2 * INTER, HIDDEN), "down": _pack(gen, HIDDEN, INTER)}
                      for _ in range(layers)]
        if case["graph"]:
            _decoder(state)   # a server runs a shape once before it captures it
            torch.cuda.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["outputs"] = _decoder(state)
    elif kind == "moe":
        layers, t, hidden, inter = case["layers"], case["t"], case["hidden"], case["inter"]
        state["x"] = [_normal(gen, (t, hidden)) for _ in range(layers)]
        state["ids"] = [_routing(case, seed * 64 + i).cuda() for i in range(layers)]
        state["weights"] = [torch.softmax(_normal(gen, (t, case["topk"]), torch.float32), dim=-1) for _ in range(layers)]
        state["w1"] = [_expert_weights(gen, case["experts"], 2 * inter, hidden) for _ in range(layers)]
        state["w2"] = [_expert_weights(gen, case["experts"], hidden, inter) for _ in range(layers)]
    elif kind == "ep":
        experts, padded, hidden, inter = case["experts"], case["padded"], case["hidden"], case["inter"]
        rows = _expert_rows(case, seed)
        state["masked_m"] = rows.cuda()
        state["recv_x"] = per_token_group_quant_fp8(_normal(gen, (experts, padded, hidden)), 128)
        state["w1"] = _expert_weights(gen, experts, 2 * inter, hidden)
        state["w2"] = _expert_weights(gen, experts, hidden, inter)
        valid = torch.arange(padded)[None, :] < rows[:, None]
        state["arrived"] = valid.view(-1).nonzero().view(-1).cuda()   # the rows the combine step sends back
    else:
        x = _normal(gen, (case["m"], case["k"]), torch.float32)
        x = torch.where(torch.rand(x.shape, generator=gen, device="cuda") < 0.01, x * 50.0, x)
        if case["m"] > 1:
            x[0] = 0.0
        state["x"] = x.to(DTYPES[case["dtype"]])
    return state


# ---- one pass

def _decoder(state):
    method, outputs = state["method"], []
    for x, w in zip(state["x"], state["w"]):
        qkv = method.apply(x["qkv"], w["qkv"])
        o = method.apply(x["o"], w["o"])
        gate_up = method.apply(x["gate_up"], w["gate_up"])
        act = torch.empty((gate_up.shape[0], INTER), dtype=gate_up.dtype, device=gate_up.device)
        silu_and_mul_fwd(gate_up, act)
        outputs += [qkv, o, gate_up, act, method.apply(act, w["down"])]
    return outputs


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return [state["method"].apply(x, w) for x, w in zip(state["x"], state["w"])]
    if kind == "decoder":
        if "graph" not in state:
            return _decoder(state)
        state["graph"].replay()
        return state["outputs"]
    if kind == "moe":
        return [fused_experts(x, w1, w2, weights, ids, use_fp8_w8a8=True, w1_scale=s1, w2_scale=s2)
                for x, (w1, s1), (w2, s2), weights, ids in
                zip(state["x"], state["w1"], state["w2"], state["weights"], state["ids"])]
    if kind == "ep":
        (w1, s1), (w2, s2) = state["w1"], state["w2"]
        out = masked_group_gemm(state["recv_x"], state["masked_m"], torch.bfloat16, w1, s1, w2, s2, case["rows"])
        return out.view(-1, case["hidden"]).index_select(0, state["arrived"])
    x_q, x_s = per_token_group_quant_fp8(state["x"], 128, column_major_scales=case["columns"],
                                         scale_tma_aligned=case["columns"])
    return x_q.view(torch.uint8), x_s


# ---- what a pass cannot do without, and how far two correct results may be apart

def _linear_work(m, n, k):
    # activations in 16 bits, weights and their scales, output in 16 bits
    return 2 * m * k + n * k + 4 * -(-n // 128) * (k // 128) + 2 * m * n, 2 * m * n * k


def work(case):
    kind = case["kind"]
    if kind == "linear":
        nbytes, flops = _linear_work(case["m"], case["n"], case["k"])
        return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}
    if kind == "decoder":
        m = case["m"]
        parts = [_linear_work(m, n, k) for n, k in
                 ((QKV, HIDDEN), (HIDDEN, HIDDEN), (2 * INTER, HIDDEN), (HIDDEN, INTER))]
        nbytes, flops = sum(p[0] for p in parts) + 6 * m * INTER, sum(p[1] for p in parts)
        return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}
    if kind == "moe":
        t, hidden, inter = case["t"], case["hidden"], case["inter"]
        expert = 3 * hidden * inter   # elements of an expert's two weights
        hit = len(torch.unique(_routing(case, 0)))
        nbytes = hit * (expert + 4 * expert // 16384) + 4 * t * hidden + 8 * t * case["topk"]
        return {"bytes": nbytes * case["layers"], "flops": 2 * t * case["topk"] * expert * case["layers"]}
    if kind == "ep":
        rows = _expert_rows(case, 0)
        hidden, expert = case["hidden"], 3 * case["hidden"] * case["inter"]
        total = int(rows.sum())
        nbytes = int((rows > 0).sum()) * (expert + 4 * expert // 16384) + total * (hidden + hidden // 32 + 2 * hidden)
        return {"bytes": max(nbytes, 1), "flops": 2 * total * expert}
    m, k = case["m"], case["k"]
    return {"bytes": 3 * m * k + 4 * m * (k // 128), "flops": 0}


def tolerance(case):
    """About four times what the path shows against itself with its products and sums in float64 and the same roundings
    in between: a single linear 2.4e-4 / 7.8e-3 (one bf16 step; float16 8e-5 / 1e-3), a decoder layer 3.2e-3 / 2e-2
    (a bf16 step of the SiLU product can move an e4m3 byte of the next linear's input), experts 2.1e-3 / 4.5e-2."""
    kind = case["kind"]
    if kind == "quant":
        return "exact"   # bytes and scales are the closed form's
    if kind == "linear":
        return {"rel": 1e-3, "max": 3.2e-2} if case["dtype"] == "bf16" else {"rel": 3.2e-4, "max": 4e-3}
    if kind == "decoder":
        return {"rel": 1.2e-2, "max": 8e-2}
    return {"rel": 9e-3, "max": 1.8e-1}
