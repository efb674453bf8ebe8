"""The work that a user of this library has it do, as cases that can be measured.

Three kinds of case, all in the ggml activation mode unless a case says otherwise:

* ``block``  - the projections of `layers` transformer blocks for `rows` tokens, issued the way an engine walks its
  graph: norm -> q/k/v, the attention output's projection, norm -> gate/up -> swiglu -> down.  Every layer has its own
  weights and its own input rows (attention, rope and the residual adds between them are not this library's).
* ``matmul`` - one projection: `rows` x `k` against an `n` x `k` matrix.
* ``moe``    - one expert feed-forward: `tokens` tokens, `used` of `experts` experts each.

Weights are N(0, 0.02) in GGUF blocks, activations N(0, 1) with one channel in a hundred twenty times as large, as
hidden states have them.  One context serves the whole process, like the one executor thread of an engine.
"""
import math

import torch

from magnitude_amd import ACT_GGML, ACT_Q8X32, TYPE_Q4_K, TYPE_Q6_K, TYPE_Q8_0, Context, synth

TYPES = {"q8_0": TYPE_Q8_0, "q4_k": TYPE_Q4_K, "q6_k": TYPE_Q6_K}
BYTES_PER_WEIGHT = {"q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}
ACTS = {"ggml": ACT_GGML, "q8x32": ACT_Q8X32}
EPS = 1e-5

_context = None


def _ctx():
    global _context
    if _context is None:
        _context = Context(0)
    return _context


def _block(name, rows, layers, d, d_kv, d_ff, wtype, down):
    return {"name": name, "kind": "block", "rows": rows, "layers": layers, "d": d, "d_kv": d_kv, "d_ff": d_ff,
            "type": wtype, "down": down}


def _moe(name, tokens, experts=128, used=8, d=2048, d_ff=768, skew=0.0):
    return {"name": name, "kind": "moe", "tokens": tokens, "experts": experts, "used": used, "d": d, "d_ff": d_ff,
            "type": "q4_k", "skew": skew}


def listed():
    return [
        # the smallest call: one 4096 x 4096 Q8_0 matrix, one token
        {"name": "matvec-q8_0", "kind": "matmul", "type": "q8_0", "act": "ggml", "rows": 1, "k": 4096, "n": 4096},
        # a decoded token of an 8B-class model in Q4_K_M; enough layers that the weights come from HBM
        _block("decode-8b", 1, 8, 4096, 1024, 14336, "q4_k", "q6_k"),
        # a decoded token of a small model in Q8_0: launches of a few megabytes each
        _block("decode-small-q8_0", 1, 12, 2048, 512, 8192, "q8_0", "q8_0"),
        # speculative decoding: eight draft tokens verified at once
        _block("verify-8b", 8, 4, 4096, 1024, 14336, "q4_k", "q6_k"),
        # a serving step of 48 sequences, one token each
        _block("batch-8b", 48, 4, 4096, 1024, 14336, "q4_k", "q6_k"),
        # the last, ragged chunk of a prompt, another width, Q8_0
        _block("prompt-tail-q8_0", 187, 4, 3072, 1024, 8192, "q8_0", "q8_0"),
        # a full prompt batch of the engine (512 tokens)
        _block("prompt-8b", 512, 2, 4096, 1024, 14336, "q4_k", "q6_k"),
        # a long prompt's widest projection with per-32 activations
        {"name": "prefill-per32", "kind": "matmul", "type": "q4_k", "act": "q8x32", "rows": 4096, "k": 4096, "n": 14336},
        # a 128-expert, top-8 feed-forward: a decoded token, small and large serving batches, a prompt's last chunk
        _moe("moe-1", 1),
        _moe("moe-8", 8),
        _moe("moe-64", 64),
        _moe("moe-prompt", 500),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["block", "block", "block", "matmul", "moe", "moe"])
        if kind == "block":
            d = rng.choice([2048, 2560, 3072, 4096, 4096, 5120, 8192])
            wtype, down = rng.choice([("q4_k", "q6_k"), ("q4_k", "q6_k"), ("q4_k", "q4_k"), ("q8_0", "q8_0"), ("q6_k", "q6_k")])
            case = {"kind": kind, "rows": _log(rng, 1, 1024), "layers": rng.randint(1, 8), "d": d,
                    "d_kv": rng.choice([256, 512, 1024]), "d_ff": 256 * round(d * rng.uniform(2.5, 4.0) / 256),
                    "type": wtype, "down": down}
        elif kind == "matmul":
            case = {"kind": kind, "type": rng.choice(["q8_0", "q4_k", "q4_k", "q6_k"]), "act": "ggml",
                    "rows": _log(rng, 1, 4096), "k": 256 * _log(rng, 4, 64), "n": _log(rng, 512, 32000)}
            if case["type"] == "q4_k" and case["rows"] >= 256 and rng.random() < 0.5:
                case["act"] = "q8x32"
        else:
            experts = rng.choice([8, 32, 64, 128, 128, 256])
            case = {"kind": kind, "tokens": _log(rng, 1, 2048), "experts": experts,
                    "used": rng.choice([2, 4]) if experts <= 32 else rng.choice([4, 6, 8]),
                    "d": rng.choice([1024, 2048, 2048, 4096]), "d_ff": 256 * rng.randint(2, 8),
                    "type": "q4_k", "skew": rng.choice([0.0, 0.0, 1.0])}
        w = work(case)
        # what a pass or its weights may take: no more than the largest listed cases
        if w["flops"] / 6e14 + w["bytes"] / 4e12 <= 8e-4 and _weight_bytes(case) <= 1.2e9:
            return case


def _matrices(case):
    """(type, k, n) of every matrix of one layer"""
    if case["kind"] == "matmul":
        return [(case["type"], case["k"], case["n"])]
    d, d_ff = case["d"], case["d_ff"]
    if case["kind"] == "moe":
        return [(case["type"], d, d_ff), (case["type"], d, d_ff), (case["type"], d_ff, d)]
    t = case["type"]
    return [(t, d, d), (t, d, case["d_kv"]), (t, d, case["d_kv"]), (t, d, d), (t, d, d_ff), (t, d, d_ff), (case["down"], d_ff, d)]


def _weight_bytes(case):
    copies = case.get("layers", 1) * case.get("experts", 1)
    return copies * sum(BYTES_PER_WEIGHT[t] * k * n for t, k, n in _matrices(case))


def _rows(g, m, k):
    x = torch.randn((m, k), generator=g, device="cuda")
    x[:, torch.randperm(k, generator=g, device="cuda")[: max(1, k // 100)]] *= 20.0
    return x


def prepare(case, seed):
    ctx = _ctx()
    g = torch.Generator(device="cuda").manual_seed(seed)
    copies = case.get("experts", 1)
    count = 0

    def weight(t, k, n):
        nonlocal count
        count += 1
        blocks = synth.random_weight(TYPES[t], copies * n, k, seed * 1000 + count, "cuda", rows_per_pass=16384)
        return ctx.upload_from_device(TYPES[t], k, n, blocks, n_expert=copies)

    def out(m, n):
        return torch.empty((m, n), device="cuda")

    s = {"case": case, "layers": []}
    if case["kind"] == "matmul":
        m = case["rows"]
        s.update(w=weight(case["type"], case["k"], case["n"]), x=_rows(g, m, case["k"]), y=out(m, case["n"]))
    elif case["kind"] == "moe":
        b, d, experts, used = case["tokens"], case["d"], case["experts"], case["used"]
        gate, up, down = [weight(t, k, n) for t, k, n in _matrices(case)]
        popularity = case["skew"] * torch.randn(experts, generator=g, device="cuda")
        scores = popularity - torch.log(-torch.log(torch.rand((b, experts), generator=g, device="cuda").clamp(1e-9, 1 - 1e-6)))
        top, ids = scores.topk(used, dim=1)
        s.update(gate=gate, up=up, down=down, x=_rows(g, b, d), ids=ids.to(torch.int32).contiguous(),
                 weights=torch.softmax(top, dim=1).contiguous(), y=out(b, d))
    else:
        m, d, d_kv, d_ff = case["rows"], case["d"], case["d_kv"], case["d_ff"]
        for _ in range(case["layers"]):
            q, k, v, o, gate, up, down = [weight(*w) for w in _matrices(case)]
            s["layers"].append({
                "qkv": [q, k, v], "o": o, "gate": gate, "up": up, "down": down,
                "x": _rows(g, m, d), "attn": _rows(g, m, d), "h": _rows(g, m, d),
                "norm_attn": 1 + 0.1 * torch.randn(d, generator=g, device="cuda"),
                "norm_ffn": 1 + 0.1 * torch.randn(d, generator=g, device="cuda"),
                "y_qkv": [out(m, d), out(m, d_kv), out(m, d_kv)], "y_o": out(m, d), "y_ffn": out(m, d)})
    return s


def run(s):
    ctx, case = _ctx(), s["case"]
    if case["kind"] == "matmul":
        return ctx.mul_mat(s["w"], s["x"], ACTS[case["act"]], out=s["y"], sync=False)
    if case["kind"] == "moe":
        return ctx.moe_ffn(s["gate"], s["up"], s["down"], s["x"], s["ids"], s["weights"], out=s["y"], sync=False)
    outputs = []
    for l in s["layers"]:
        outputs += ctx.rms_norm_mul_mat(l["qkv"], l["x"], l["norm_attn"], EPS, outs=l["y_qkv"], sync=False)
        outputs.append(ctx.mul_mat(l["o"], l["attn"], out=l["y_o"], sync=False))
        outputs.append(ctx.ffn(l["gate"], l["up"], l["down"], l["h"], gamma=l["norm_ffn"], eps=EPS, out=l["y_ffn"], sync=False))
    return outputs


def work(case):
    """Weights, input rows and results once each; for experts, the expected number of distinct ones."""
    mats = _matrices(case)
    if case["kind"] == "moe":
        b, used, experts, d = case["tokens"], case["used"], case["experts"], case["d"]
        busy = experts * (1 - (1 - used / experts) ** b)
        return {"bytes": busy * sum(BYTES_PER_WEIGHT[t] * k * n for t, k, n in mats) + 8 * b * d + 8 * b * used,
                "flops": sum(2.0 * b * used * k * n for _, k, n in mats)}
    m, layers = case["rows"], case.get("layers", 1)
    io = case["k"] + case["n"] if case["kind"] == "matmul" else 6 * case["d"] + 2 * case["d_kv"]
    return {"bytes": layers * (sum(BYTES_PER_WEIGHT[t] * k * n for t, k, n in mats) + 4 * m * io),
            "flops": layers * sum(2.0 * m * k * n for _, k, n in mats)}


def tolerance(case):
    """Four times what the same rows differ by when they go through another kernel (one by one or in a batch): the
    integer dot products are exact and only the order of the fp32 sums differs, 6e-7 at most.  A feed-forward
    quantizes its intermediate rows again, and a value within a rounding of the middle between two codes may take
    either: 3.5e-4 at most over a result, 6.4e-3 in one output."""
    if case["kind"] == "matmul":
        return {"rel": 2.5e-6, "max": 2e-5}
    return {"rel": 1.4e-3, "max": 2.6e-2}
