"""Performance cases of the quantized-linear path: what a program that serves a model has it do.

Every case is one call, or one block of calls, of the package's prepared plans, with the buffers
that such a program keeps (outputs and workspaces). A case is a dict of plain values:

* ``linear``: a Q8 A16 projection (``upload_linear`` / ``prepare`` / ``run(x, out=)``);
* ``mlp``: a decode step's gated MLP over Q8 weights (RMSNorm, gate+up with SwiGLU, down, residual add);
* ``a8``: a W8A8 projection; ``norm`` says whether its activations come from the fused RMSNorm
  producer (the attention and gate+up inputs) or from the plan's own quantizer (o_proj and down);
* ``q4``: a Q4 W4A16 projection;
* ``moe``: the routed-expert Q4 MoE.

Weights are planes in the stored layout (Gaussian weights, rounded to nearest per group), made on the
GPU from the seed; activations are Gaussian.
"""

import math

import torch

from venturi_amd import Q8RowSplitWeight, create_backend, prepare_q8_dp4a
from venturi_amd.moe import MoEGeometry, Q4ExpertBank
from venturi_amd.rms_quant import prepare_rms_q8
from venturi_amd.weights import Q4RowSplitWeight

DEVICE = "cuda:0"
EPSILON = 1e-6
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}

# The dense model's projections (hidden 5120, intermediate 17408) as [out, in].
QKV, O_PROJ, GATE_UP, DOWN = (7168, 5120), (5120, 6144), (34816, 5120), (5120, 17408)


def listed():
    return [
        # The smallest call: one token through one square projection; launch and latency count.
        {"name": "linear_one_token", "kind": "linear", "tokens": 1, "n": 4096, "k": 4096, "dtype": "fp16"},
        # bf16 activations (the upload's default dtype) run the canonical-order kernel.
        {"name": "linear_bf16", "kind": "linear", "tokens": 4, "n": QKV[0], "k": QKV[1], "dtype": "bf16"},
        # A chat prompt of ordinary, ragged length through the fused QKV projection.
        {"name": "linear_prompt", "kind": "linear", "tokens": 200, "n": QKV[0], "k": QKV[1], "dtype": "fp16"},
        # A full prefill chunk through gate+up, called as the reference calls it (no workspace).
        {"name": "linear_prefill", "kind": "linear", "tokens": 2048, "n": GATE_UP[0], "k": GATE_UP[1], "dtype": "fp16"},
        # One layer's MLP in a decode step of a small batch, and of an odd one near the decode kernels' limit.
        {"name": "mlp_decode", "kind": "mlp", "tokens": 8, "hidden": 5120, "inter": 17408},
        {"name": "mlp_decode_batch", "kind": "mlp", "tokens": 29, "hidden": 5120, "inter": 17408},
        # A8 with residual compensation in a decode step: down, quantizer included.
        {"name": "a8_decode", "kind": "a8", "tokens": 8, "n": DOWN[0], "k": DOWN[1], "passes": 2, "norm": False},
        # A8 prefill: RMSNorm producer and the int8 GEMM of gate+up.
        {"name": "a8_prefill", "kind": "a8", "tokens": 2048, "n": GATE_UP[0], "k": GATE_UP[1], "passes": 1,
         "norm": True},
        # Q4 decode of a few sequences, and a Q4 prompt at the shape the reference quotes.
        {"name": "q4_decode", "kind": "q4", "tokens": 4, "n": DOWN[0], "k": DOWN[1]},
        {"name": "q4_prompt", "kind": "q4", "tokens": 128, "n": 5120, "k": 25600},
        # The routed-expert MoE (hidden 2048, 128 experts, top 8, intermediate 768): a prompt and a decode step.
        {"name": "moe_prompt", "kind": "moe", "tokens": 512, "hidden": 2048, "experts": 128, "top_k": 8, "inter": 768},
        {"name": "moe_decode", "kind": "moe", "tokens": 8, "hidden": 2048, "experts": 128, "top_k": 8, "inter": 768},
    ]


def _spread(rng, low, high):
    """An integer of [low, high], even over the logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _features(rng, low, high):
    """A feature count: mostly a multiple of 128, as models have it, else of 8."""
    step = rng.choice((128, 128, 128, 8))
    return max(step, _spread(rng, low, high) // step * step)


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "mlp", "a8", "a8", "q4", "q4", "moe"))
    if kind == "mlp":
        return {"kind": kind, "tokens": _spread(rng, 1, 32), "hidden": _features(rng, 1024, 5120),
                "inter": _features(rng, 2048, 17408)}
    if kind == "moe":
        experts = rng.choice((8, 32, 64, 128))
        return {"kind": kind, "tokens": _spread(rng, 1, 1024), "hidden": _features(rng, 1024, 4096),
                "experts": experts, "top_k": rng.choice((2, 4, 8)), "inter": _features(rng, 256, 1536)}
    n, k = _spread(rng, 1024, 34816), _features(rng, 1024, 25600)
    if rng.random() < 0.7:
        n = n // 64 * 64
    tokens = _spread(rng, 1, 2048)
    if n * k > GATE_UP[0] * GATE_UP[1]:  # no more than the largest listed weight
        n = GATE_UP[0] * GATE_UP[1] // k
    if kind == "a8":
        return {"kind": kind, "tokens": tokens, "n": n, "k": k, "passes": rng.choice((1, 1, 2)) if tokens <= 1024 else 1,
                "norm": rng.random() < 0.5}
    if kind == "q4":
        return {"kind": kind, "tokens": tokens, "n": n, "k": k}
    if rng.random() < 0.2:  # the canonical-order kernel: bf16, or a K that is not a multiple of 8
        odd = rng.random() < 0.3
        return {"kind": kind, "tokens": _spread(rng, 1, 32), "n": n, "k": k - 3 if odd else k,
                "dtype": "fp16" if odd else "bf16"}
    return {"kind": kind, "tokens": tokens, "n": n, "k": k, "dtype": "fp16"}


# ---------------------------------------------------------------- inputs


def _generator(seed, salt):
    return torch.Generator(device=DEVICE).manual_seed(1_000_003 * (seed + 1) + salt)


def _planes(gen, n, k, bits):
    """(codes, scales) of an n x k Gaussian matrix, as integers of the padded width and fp16 group scales."""
    group, top = (32, 127) if bits == 8 else (64, 7)
    padded = (k + 127) // 128 * 128
    codes = torch.empty(n, padded, dtype=torch.int8, device=DEVICE)
    scales = torch.empty(n, padded // group, dtype=torch.float16, device=DEVICE)
    rows = max(1, 2**26 // padded)
    for r in range(0, n, rows):
        w = torch.randn(min(rows, n - r), padded, generator=gen, device=DEVICE) * 0.02
        w[:, k:] = 0
        w = w.view(w.shape[0], padded // group, group)
        s = (w.abs().amax(-1) / top).clamp_min(2.0**-24).half()
        scales[r : r + rows] = s
        codes[r : r + rows] = (w / s.float().unsqueeze(-1)).round().clamp(-top, top).to(torch.int8).flatten(1)
    return codes, scales


def _q8(gen, n, k):
    codes, scales = _planes(gen, n, k, 8)
    return Q8RowSplitWeight(codes, scales, k)


def _nibbles(codes):
    low = codes.view(torch.uint8) & 15
    return low[:, 0::2] | (low[:, 1::2] << 4)


def _q4(gen, n, k):
    codes, scales = _planes(gen, n, k, 4)
    return Q4RowSplitWeight(_nibbles(codes), scales, k)


def _values(codes, scales, k):
    """The float64 weights of a pair of planes."""
    n, padded = codes.shape
    group = padded // scales.shape[1]
    return (codes.view(n, -1, group).double() * scales.double().unsqueeze(-1)).view(n, padded)[:, :k]


def _routing(case, seed):
    """Router output: distinct experts per token, softmax scores."""
    gen = _generator(seed, 2)
    logits = torch.randn(case["tokens"], case["experts"], generator=gen, device=DEVICE)
    top, ids = logits.topk(min(case["top_k"], case["experts"]), dim=-1)
    return ids.contiguous(), torch.softmax(top, -1).half().contiguous()


def _activations(case, seed, k, dtype=torch.float16):
    gen = _generator(seed, 1)
    return torch.randn(case["tokens"], k, generator=gen, device=DEVICE).to(dtype)


def _gamma(seed, features):
    return 1.0 + 0.1 * torch.randn(features, generator=_generator(seed, 3), device=DEVICE)


def _bytes(count):
    return torch.empty(count, dtype=torch.uint8, device=DEVICE)


def prepare(case, seed):
    backend = create_backend("hip")
    kind, tokens = case["kind"], case["tokens"]
    half = {"dtype": torch.float16, "device": DEVICE}
    if kind == "linear":
        dtype = DTYPES[case["dtype"]]
        resident = backend.upload_linear(_q8(_generator(seed, 0), case["n"], case["k"]), dtype=dtype, device=DEVICE)
        return {"kind": kind, "plan": resident.prepare(tokens=tokens),
                "x": _activations(case, seed, case["k"], dtype),
                "out": torch.empty(tokens, case["n"], dtype=dtype, device=DEVICE)}
    if kind == "q4":
        resident = backend.upload_linear(_q4(_generator(seed, 0), case["n"], case["k"]), **half)
        return {"kind": kind, "plan": resident.prepare(tokens=tokens), "x": _activations(case, seed, case["k"]),
                "out": torch.empty(tokens, case["n"], **half)}
    if kind == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        gen = _generator(seed, 0)
        gate_up = backend.upload_linear(_q8(gen, 2 * inter, hidden), residency="tiled-paired", **half)
        down = backend.upload_linear(_q8(gen, hidden, inter), residency="tiled", **half)
        norm = backend.upload_rmsnorm(_gamma(seed, hidden), epsilon=EPSILON, **half)
        return {"kind": kind, "norm": norm.prepare(tokens=tokens), "gate_up": gate_up.prepare_swiglu(tokens=tokens),
                "down": down.prepare(tokens=tokens), "add": backend.prepare_add(tokens=tokens, features=hidden, **half),
                "x": _activations(case, seed, hidden), "normed": torch.empty(tokens, hidden, **half),
                "h": torch.empty(tokens, inter, **half), "mlp": torch.empty(tokens, hidden, **half),
                "out": torch.empty(tokens, hidden, **half)}
    if kind == "a8":
        n, k = case["n"], case["k"]
        residual = case["passes"] == 2
        resident = backend.upload_linear(_q8(_generator(seed, 0), n, k), **half)
        plan = prepare_q8_dp4a(resident, tokens=tokens, residual_compensation=residual)
        state = {"kind": kind, "plan": plan, "x": _activations(case, seed, k), "out": torch.empty(tokens, n, **half),
                 "workspace": _bytes(plan.workspace_bytes), "norm": None}
        if case["norm"]:
            norm = backend.upload_rmsnorm(_gamma(seed, k), epsilon=EPSILON, **half)
            state["norm"] = prepare_rms_q8(norm, tokens=tokens, residual_compensation=residual)
        return state
    experts, hidden, inter = case["experts"], case["hidden"], case["inter"]
    gen = _generator(seed, 0)
    gate_up = _q4(gen, experts * 2 * inter, hidden)
    down = _q4(gen, experts * hidden, inter)
    bank = Q4ExpertBank.upload(
        backend, MoEGeometry(hidden, experts, min(case["top_k"], experts), inter),
        [(Q4RowSplitWeight(gate_up.codes[e * 2 * inter : (e + 1) * 2 * inter],
                           gate_up.scales[e * 2 * inter : (e + 1) * 2 * inter], hidden),
          Q4RowSplitWeight(down.codes[e * hidden : (e + 1) * hidden], down.scales[e * hidden : (e + 1) * hidden], inter))
         for e in range(experts)], device=DEVICE)
    plan = bank.prepare(tokens=tokens)
    ids, scores = _routing(case, seed)
    return {"kind": kind, "plan": plan, "x": _activations(case, seed, hidden), "ids": ids, "scores": scores,
            "out": torch.empty(tokens, hidden, **half), "workspace": _bytes(plan.workspace_bytes)}


# ---------------------------------------------------------------- one pass


def run(state):
    kind = state["kind"]
    if kind in ("linear", "q4"):
        return state["plan"].run(state["x"], out=state["out"])
    if kind == "mlp":
        state["norm"].run(state["x"], out=state["normed"])
        state["gate_up"].run(state["normed"], out=state["h"])
        state["down"].run(state["h"], out=state["mlp"])
        return state["add"].run(state["x"], state["mlp"], out=state["out"])
    if kind == "a8":
        if state["norm"] is None:
            return state["plan"].run(state["x"], out=state["out"], workspace=state["workspace"])
        state["norm"].run(state["x"], workspace=state["workspace"])
        return state["plan"].project(out=state["out"], workspace=state["workspace"])
    return state["plan"].run(state["x"], state["ids"], state["scores"], out=state["out"], workspace=state["workspace"])


# ---------------------------------------------------------------- work, tolerance, exact results


def _row_bytes(k, bits):
    padded = (k + 127) // 128 * 128
    return padded + padded // 32 * 2 if bits == 8 else padded // 2 + padded // 64 * 2


def work(case):
    tokens = case["tokens"]
    if case["kind"] == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        return {"bytes": 2 * inter * _row_bytes(hidden, 8) + hidden * _row_bytes(inter, 8) + 4 * tokens * hidden,
                "flops": 6 * tokens * hidden * inter}
    if case["kind"] == "moe":
        hidden, inter, experts = case["hidden"], case["inter"], case["experts"]
        top_k = min(case["top_k"], experts)
        touched = experts * (1.0 - (1.0 - top_k / experts) ** tokens)  # experts that some token selects
        expert = 2 * inter * _row_bytes(hidden, 4) + hidden * _row_bytes(inter, 4)
        return {"bytes": round(touched * expert) + 4 * tokens * hidden + 10 * tokens * top_k,
                "flops": 6 * tokens * top_k * hidden * inter}
    bits = 4 if case["kind"] == "q4" else 8
    n, k = case["n"], case["k"]
    return {"bytes": n * _row_bytes(k, bits) + 2 * tokens * (n + k),
            "flops": 2 * tokens * n * k * (case["passes"] if case["kind"] == "a8" else 1)}


def tolerance(case):
    # 16-bit outputs: one rounding is 2^-11 (fp16) or 2^-8 (bf16) of the value at most, and the sums before it
    # are fp32; against exact() the paths measure 2.1e-4 (fp16 projections), 1.7e-3 (bf16), 2.5e-4 (mlp, which
    # rounds between its stages), 1.4e-4 (moe) and 2.8e-4 (a8 behind the norm, where an activation may take a
    # neighbouring code when the norm's sum is associated otherwise). About four times that is allowed.
    if case["kind"] == "linear" and case["dtype"] == "bf16":
        return {"rel": 6e-3, "max": 2e-2}
    if case["kind"] == "mlp" or (case["kind"] == "a8" and case["norm"]):
        return {"rel": 1e-3, "max": 4e-3}
    return {"rel": 8e-4, "max": 4e-3}


def _matmul(x, codes, scales, k):
    """x [T, k] times the planes' matrix transposed, in float64, by chunks of rows."""
    n = codes.shape[0]
    out = torch.empty(x.shape[0], n, dtype=torch.float64, device=x.device)
    rows = max(1, 2**27 // codes.shape[1])
    for r in range(0, n, rows):
        out[:, r : r + rows] = x @ _values(codes[r : r + rows], scales[r : r + rows], k).T
    return out


def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPSILON) * gamma.double()


def _half(x):
    return x.half().double()


def _a8(x, passes):
    """The represented value of the group-32 int8 activations (one or two passes)."""
    tokens, k = x.shape
    padded = (k + 31) // 32 * 32
    rest = torch.zeros(tokens, padded, dtype=torch.float64, device=x.device)
    rest[:, :k] = x
    rest = rest.view(tokens, -1, 32)
    total = torch.zeros_like(rest)
    for _ in range(passes):
        top = rest.abs().amax(-1, keepdim=True)
        scale = (top / 127).float().double()
        code = (rest * torch.where(top > 0, 127 / top, 0.0)).round().clamp(-127, 127)
        total += code * scale
        rest = (rest - code * scale).float().double()
    return total.view(tokens, padded)[:, :k]


def exact(case, seed):
    kind = case["kind"]
    gen = _generator(seed, 0)
    if kind == "linear":
        x = _activations(case, seed, case["k"], DTYPES[case["dtype"]])
        return _matmul(x.double(), *_planes(gen, case["n"], case["k"], 8), case["k"])
    if kind == "q4":
        codes, scales = _planes(gen, case["n"], case["k"], 4)
        x = _activations(case, seed, case["k"]).double()
        n, k = case["n"], case["k"]
        out = torch.empty(case["tokens"], n, dtype=torch.float64, device=DEVICE)
        rows = max(1, 2**27 // codes.shape[1])
        for r in range(0, n, rows):  # the W4A16 weight is fp16(q * scale)
            out[:, r : r + rows] = x @ _half(_values(codes[r : r + rows], scales[r : r + rows], k)).T
        return out
    if kind == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        gate_up, down = _planes(gen, 2 * inter, hidden, 8), _planes(gen, hidden, inter, 8)
        x = _activations(case, seed, hidden).double()
        both = _half(_matmul(_half(_rms(x, _gamma(seed, hidden))), *gate_up, hidden))
        gate, up = both[:, :inter], both[:, inter:]
        return x + _half(_matmul(_half(gate * torch.sigmoid(gate) * up), *down, inter))
    if kind == "a8":
        x = _activations(case, seed, case["k"]).double()
        if case["norm"]:
            x = _half(_rms(x, _gamma(seed, case["k"])))
        return _matmul(_a8(x, case["passes"]), *_planes(gen, case["n"], case["k"], 8), case["k"])
    experts, hidden, inter = case["experts"], case["hidden"], case["inter"]
    gate_up, down = _planes(gen, experts * 2 * inter, hidden, 4), _planes(gen, experts * hidden, inter, 4)
    x = _activations(case, seed, hidden).double()
    ids, scores = _routing(case, seed)
    out = torch.zeros(case["tokens"], hidden, dtype=torch.float64, device=DEVICE)
    for e in range(experts):  # ascending expert order, fp16 at the reference's boundaries
        token, slot = (ids == e).nonzero(as_tuple=True)
        if token.numel() == 0:
            continue
        a, b = slice(e * 2 * inter, (e + 1) * 2 * inter), slice(e * hidden, (e + 1) * hidden)
        both = _half(x[token] @ _half(_values(gate_up[0][a], gate_up[1][a], hidden)).T)
        gate, up = both[:, :inter], both[:, inter:]
        h = _half(_half(gate * torch.sigmoid(gate)) * up)
        y = _half(h @ _half(_values(down[0][b], down[1][b], inter)).T)
        out[token] = _half(out[token] + _half(y * scores[token, slot].double().unsqueeze(-1)))
    return out
