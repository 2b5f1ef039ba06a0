"""The work whose speed counts: what a program that serves, fine-tunes or converts a quantized mixture-of-experts
model has this package do, as a list of cases and a generator of more of the same ranges.

Three kinds of case, all through the package's public entry points:

``block``   one forward of the sparse MoE block (``SparseMoeBlock.forward`` / ``forward_residual``): router, top-k,
            dispatch, the three grouped products and the combine.  Decode batches, chunks of a few hundred tokens
            and prefill, even and skewed routing, 4- and 8-bit codes, group sizes 64 and 32 / 128.
``linear``  one quantized linear layer as the dense parts of the same models use it: forward
            (``quantized_linear``, codes along K) and the gradient with respect to the layer's input
            (``quantized_matmul`` with ``transpose=False``), in bfloat16, float16 and float32.
``codec``   a weight matrix quantised and dequantised again (``quantize``, ``dequantize``): what a checkpoint
            conversion or a merge of adapters does with every matrix.
"""
import math

import numpy as np
import torch

import mlx_rs_amd as m
from mlx_rs_amd import ops, synth

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def _block(name, config, tokens, zipf=0.0, residual=False, group=64):
    return {"name": name, "kind": "block", "config": config, "tokens": tokens, "zipf": zipf, "residual": residual, "group": group}


def _linear(name, way, rows, n, k, bits, group, dtype, bias=False):
    return {"name": name, "kind": "linear", "way": way, "rows": rows, "n": n, "k": k, "bits": bits, "group": group,
            "dtype": dtype, "bias": bias}


def listed():
    return [
        # one user's next token: four launches, a few microseconds each
        _block("decode 1", "qwen3_30b_a3b", 1),
        # a serving batch: every expert's weights are read for two or three tokens
        _block("decode 32", "qwen3_30b_a3b", 32),
        # a chunk of a prompt among running requests, in its decoder layer (norm before, residual behind); popular experts
        _block("chunk 203", "qwen3_30b_a3b", 203, zipf=1.1, residual=True),
        # a prompt, a few experts taking most of the tokens
        _block("prefill 4096", "qwen3_30b_a3b", 4096, zipf=1.1),
        # few wide experts, 8-bit codes: one token, then a prompt
        _block("wide decode 1", "mixtral_8x7b", 1),
        _block("wide prefill 2048", "mixtral_8x7b", 2048),
        # the largest layer and batch
        _block("large prefill 8192", "qwen3_235b_a22b", 8192, zipf=1.3),
        # the finer quantisation some checkpoints choose
        _block("group 32 chunk 512", "qwen3_30b_a3b", 512, group=32),
        # a projection of one token: the smallest call
        _linear("linear 1", "forward", 1, 4096, 2048, 4, 64, "bfloat16"),
        # a projection with a bias over a ragged prompt, in half precision
        _linear("linear f16 777", "forward", 777, 4096, 4096, 8, 64, "float16", bias=True),
        # fine-tuning on frozen quantized weights: the gradient with respect to the layer's input
        _linear("input gradient 1000", "backward", 1000, 2048, 4096, 4, 64, "bfloat16"),
        # a bank of expert matrices converted
        {"name": "codec", "kind": "codec", "rows": 98304, "cols": 2048, "bits": 4, "group": 64, "dtype": "bfloat16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "block", "block", "linear", "linear", "codec"])
    if kind == "block":
        group = rng.choice([64, 64, 64, 64, 32, 128])
        config = rng.choice(["qwen3_30b_a3b", "qwen3_30b_a3b", "mixtral_8x7b", "qwen3_235b_a22b"]) if group == 64 else "qwen3_30b_a3b"
        most = {"qwen3_30b_a3b": 8192, "mixtral_8x7b": 2048, "qwen3_235b_a22b": 8192}[config] if group == 64 else 512
        case = _block("", config, _log_int(rng, 2, most), rng.choice([0.0, 0.0, 1.1, 1.3]), rng.random() < 0.4, group)
    elif kind == "linear":
        way, dtype = rng.choice(["forward", "forward", "backward"]), rng.choice(["bfloat16", "bfloat16", "float16", "float32"])
        n, k = 128 * rng.randint(8, 32), 128 * rng.randint(8, 32)
        if way == "forward" and rng.random() < 0.5:
            n -= 16 * rng.randint(1, 7)  # an output that fills no whole tile
        case = _linear("", way, _log_int(rng, 1, 1000), n, k, rng.choice([4, 4, 8]), rng.choice([64, 64, 64, 32, 128]), dtype,
                       way == "forward" and rng.random() < 0.3)
    else:
        cols = 128 * rng.randint(6, 48)
        case = {"kind": "codec", "rows": _log_int(rng, 64, 2e8 / cols), "cols": cols, "bits": rng.choice([4, 4, 8]),
                "group": rng.choice([64, 64, 32, 128]), "dtype": rng.choice(["bfloat16", "bfloat16", "float16", "float32"])}
    case.pop("name", None)
    return case


def _config(case):
    c = synth.CONFIGS[case["config"]]
    return m.MoeConfig(c.hidden, c.n_experts, c.top_k, c.intermediate, c.bits, case["group"], c.score_mode)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * std

    if case["kind"] == "block":
        cfg = _config(case)
        block = synth.make_block(cfg, seed=seed, device="cuda", zipf_s=case["zipf"] or None, gen_device="cuda")
        x = normal(case["tokens"], cfg.hidden).to(torch.bfloat16)
        norm = (1.0 + normal(cfg.hidden, std=0.1)).to(torch.bfloat16) if case["residual"] else None
        return {"case": case, "block": block, "x": x, "norm": norm}
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "linear":
        # forward: w [N, K] quantised along K; backward: the same kind of matrix read the other way, w [K, N]
        rows, cols = (case["n"], case["k"]) if case["way"] == "forward" else (case["k"], case["n"])
        q, s, b = ops.quantize(normal(rows, cols, std=0.02), case["group"], case["bits"], dtype)
        x = normal(case["rows"], case["k"]).to(dtype)
        bias = normal(case["n"], std=0.5).to(dtype) if case["bias"] else None
        return {"case": case, "x": x, "q": q, "s": s, "b": b, "bias": bias}
    return {"case": case, "w": normal(case["rows"], case["cols"], std=0.02), "dtype": dtype}


def run(state):
    case = state["case"]
    if case["kind"] == "block":
        if case["residual"]:
            return state["block"].forward_residual(state["x"], state["norm"], 1e-6)
        return state["block"](state["x"])
    if case["kind"] == "linear":
        if case["way"] == "forward":
            return ops.quantized_linear(state["x"], state["q"], state["s"], state["b"], state["bias"],
                                        group_size=case["group"], bits=case["bits"])
        return ops.quantized_matmul(state["x"], state["q"], state["s"], state["b"], transpose=False,
                                    group_size=case["group"], bits=case["bits"])
    q, s, b = ops.quantize(state["w"], case["group"], case["bits"], state["dtype"])
    return q, s, b, ops.dequantize(q, s, b, case["group"], case["bits"])


def _active_experts(cfg, tokens, zipf):
    """Experts that at least one token picks, on average: counted over random logits of the layer's own spread."""
    rng = np.random.default_rng(0)
    spread = 0.02 * math.sqrt(cfg.hidden)  # x ~ N(0, 1), router ~ N(0, 0.02)
    bias = -zipf * np.log(np.arange(1, cfg.n_experts + 1))
    trials = max(1, 64 // tokens)
    seen = 0
    for _ in range(trials):
        logits = rng.standard_normal((min(tokens, 4096), cfg.n_experts)) * spread + bias
        seen += np.unique(np.argpartition(logits, -cfg.top_k, axis=1)[:, -cfg.top_k:]).size
    return seen / trials


def work(case):
    if case["kind"] == "block":
        cfg, t = _config(case), case["tokens"]
        codes = cfg.hidden * cfg.intermediate * cfg.bits // 8
        expert = 3 * (codes + 4 * cfg.hidden * cfg.intermediate // cfg.group_size)  # a bf16 scale and bias per group
        rows = 2 * t * cfg.hidden * 2  # x in, the result out
        return {"bytes": _active_experts(cfg, t, case["zipf"]) * expert + 2 * cfg.n_experts * cfg.hidden + rows,
                "flops": 6 * t * cfg.top_k * cfg.hidden * cfg.intermediate + 2 * t * cfg.hidden * cfg.n_experts}
    size = {"bfloat16": 2, "float16": 2, "float32": 4}[case["dtype"]]
    if case["kind"] == "linear":
        n, k, r = case["n"], case["k"], case["rows"]
        weights = n * k * case["bits"] // 8 + 2 * size * n * k // case["group"]
        return {"bytes": weights + size * (r * k + r * n + (n if case["bias"] else 0)), "flops": 2 * r * n * k}
    values = case["rows"] * case["cols"]
    packed = values * case["bits"] // 8 + 2 * size * values // case["group"]
    return {"bytes": 4 * values + 2 * packed + size * values, "flops": 8 * values}


def tolerance(case):
    if case["kind"] == "codec":
        return "exact"  # every step is one correctly rounded float32 operation
    if case["kind"] == "block":
        return {"rel": 1.2e-2, "max": 0.2}
    return {"bfloat16": {"rel": 1e-2, "max": 0.1}, "float16": {"rel": 1.2e-3, "max": 0.02},
            "float32": {"rel": 4e-6, "max": 1e-4}}[case["dtype"]]
