"""Workloads of the quantized-linear library, as a program that uses it runs them.

A program loads a checkpoint (`make_linear` on each projection, `fuse_linears`
on those that read one input), prefills a prompt, then decodes: each step
runs every projection at a few rows, the `lm_head` over the vocabulary, and
the greedy token or the engine's sampling step.  Sizes are those of the
repository's benchmark and tests: hidden 2560 / FFN 9728 (the checkpoint),
hidden 4096 / FFN 12288 (the benchmark's stack), vocabulary 151936, and the
odd sizes of the test suite.

Kinds of case (`kind`):
  linear  one Int8Linear / DynamicInt8Linear forward on [M, K] activations
  fused   one FusedLinear forward over the eleven projections of a hybrid
          layer that read its normed input
  layer   one decode step through the projections of a hybrid layer (fused
          reads, the grouped lora and output pairs, gate+up, down), captured
          once in a HIP graph and replayed per step
  greedy  the lm_head and its greedy token in one pass (`forward_greedy`)
  sample  the sampling step over the logits (`sample_tokens`, or
          `greedy_tokens` at temperature 0)
  load    quantizing and packing one projection's checkpoint weight
"""
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "spikingbrain-cpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from sbq import quant  # noqa: E402

DEV = "cuda"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}

# the hybrid layer's projections of its normed input (heads 32, kv heads 8,
# head dim 128, lora 128, 4 partitions): sse_q/k/v, lora_q[0]/lora_k[0],
# sse_a/b/e, swa_q/k/v
READS_X = (4096, 4096, 4096, 128, 128, 64, 64, 4, 4096, 1024, 1024)

# no drawn case does more than the largest listed one
MOST_FLOPS = 2 * 8192 * 12288 * 4096


def listed():
    return [
        # one small projection of a decode step, called eagerly with the reference model's fp32 activations: latency
        {"name": "o_proj_m1", "kind": "linear", "fmt": "int8", "M": 1, "N": 2560, "K": 4096, "x": "f32"},
        # a batch of eight sequences through gate+up in the W8A8 format (decode, activations quantized per call)
        {"name": "gate_up_dyn_m8", "kind": "linear", "fmt": "int8-dyn", "M": 8, "N": 24576, "K": 4096, "x": "f16"},
        # every projection of one hybrid layer for one new token, as a serving loop replays it
        {"name": "layer_m1", "kind": "layer", "fmt": "int8", "M": 1, "H": 2560, "F": 9728, "x": "f32"},
        # the same for a batch of eight sequences in the W8A8 format
        {"name": "layer_dyn_m8", "kind": "layer", "fmt": "int8-dyn", "M": 8, "H": 2560, "F": 9728, "x": "f32"},
        # the logits and the greedy token of one decode step
        {"name": "lm_head_m1", "kind": "greedy", "fmt": "int8", "M": 1, "N": 151936, "K": 2560, "x": "f32"},
        # the engine's default sampling step (temperature 0.7, top_p 0.9) for one sequence
        {"name": "sample_m1", "kind": "sample", "M": 1, "V": 151936, "T": 0.7, "k": 0, "p": 0.9},
        # a batch of eight sequences sampled with top-k as well
        {"name": "sample_topk_m8", "kind": "sample", "M": 8, "V": 151936, "T": 0.7, "k": 50, "p": 0.95},
        # a short prompt on a layer whose sizes divide nothing (the test suite's odd sizes, scaled to a real layer)
        {"name": "ragged_m77", "kind": "linear", "fmt": "int8", "M": 77, "N": 2999, "K": 2500, "x": "f32"},
        # the reference's prompt chunk through the fused projections of a hybrid layer, fp32 in and out
        {"name": "fused_m512", "kind": "fused", "fmt": "int8", "M": 512, "H": 2560, "x": "f32"},
        # a long prompt in the W8A8 format
        {"name": "prefill_dyn_m2048", "kind": "linear", "fmt": "int8-dyn", "M": 2048, "N": 12288, "K": 4096, "x": "f16"},
        # the largest prefill of the benchmark: weight-only, fp16 activations
        {"name": "prefill_m8192", "kind": "linear", "fmt": "int8", "M": 8192, "N": 12288, "K": 4096, "x": "f16",
         "y": "f16"},
        # loading one FFN projection of a bf16 checkpoint (quantize, pack)
        {"name": "load_up", "kind": "load", "fmt": "int8-dyn", "N": 9728, "K": 2560, "w": "bf16"},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "fused", "layer", "greedy", "sample", "load"))
    fmt = rng.choice(("int8", "int8-dyn"))
    x = rng.choice(("f32", "f32", "f16", "bf16"))
    if kind == "linear":
        while True:
            M, N, K = _log(rng, 1, 8192), _log(rng, 128, 24576), _log(rng, 128, 12288)
            if rng.random() < 0.75:  # a real layer's sizes; the rest stay odd
                N, K = max(128, N // 64 * 64), max(128, K // 64 * 64)
            if 2 * M * N * K <= MOST_FLOPS:
                break
        c = {"kind": kind, "fmt": fmt, "M": M, "N": N, "K": K, "x": x, "bias": rng.random() < 0.3}
        if fmt == "int8-dyn" and rng.random() < 0.25:
            c["token"] = True
        if x == "f16" and rng.random() < 0.5:
            c["y"] = "f16"
        return c
    if kind == "fused":
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 1, 1024), "H": rng.choice((2560, 4096)), "x": x}
    if kind == "layer":
        H, F = rng.choice(((2560, 9728), (4096, 12288)))
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 1, 16), "H": H, "F": F, "x": x}
    if kind == "greedy":
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 1, 16), "N": _log(rng, 8192, 151936), "K": rng.choice((2560, 4096)),
                "x": x}
    if kind == "sample":
        return {"kind": kind, "M": _log(rng, 1, 16), "V": _log(rng, 4096, 151936),
                "T": rng.choice((0.0, 0.7, round(rng.uniform(0.3, 1.3), 2))), "k": rng.choice((0, 0, _log(rng, 5, 2000))),
                "p": rng.choice((1.0, 0.9, round(rng.uniform(0.5, 0.99), 3)))}
    return {"kind": kind, "fmt": fmt, "N": _log(rng, 128, 24576), "K": _log(rng, 128, 12288), "w": rng.choice(("bf16", "bf16", "f32", "f16"))}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _weight(g, N, K, dtype=torch.float32):
    return (torch.randn(N, K, generator=g, device=DEV) * 0.02).to(dtype)


def _act(g, M, K, x):
    """N(0, 1) activations (after a norm), 1% of the channels 20 times larger."""
    t = torch.randn(M, K, generator=g, device=DEV)
    t *= torch.where(torch.rand(K, generator=g, device=DEV) < 0.01, 20.0, 1.0)
    return t.to(DTYPES[x])


def _logits(g, M, V):
    """A language model's logits: a broad bulk and a few dozen likely tokens per row."""
    t = torch.randn(M, V, generator=g, device=DEV) * 2.5
    at = torch.randint(0, V, (M, 64), generator=g, device=DEV)
    return t.scatter_add_(1, at, torch.rand(M, 64, generator=g, device=DEV) * 8 + 4)


def _layer_inputs(case, g):
    """The raw weights and inputs of one hybrid layer's projections."""
    M, H, F, x = case["M"], case["H"], case["F"], case["x"]
    w = {"reads": [_weight(g, n, H) for n in READS_X], "lora": [_weight(g, 4096, 128) for _ in range(2)],
         "out": [_weight(g, H, 4096) for _ in range(2)], "gate_up": [_weight(g, F, H) for _ in range(2)],
         "down": [_weight(g, H, F)]}
    acts = {"reads": [_act(g, M, H, x)], "lora": [_act(g, M, 128, x) for _ in range(2)],
            "out": [_act(g, M, 4096, x) for _ in range(2)], "gate_up": [_act(g, M, H, x)], "down": [_act(g, M, F, x)]}
    return w, acts


def _inputs(case, seed):
    """(weight, bias, activations) of a linear / greedy case."""
    g = _gen(seed)
    w = _weight(g, case["N"], case["K"])
    b = torch.randn(case["N"], generator=g, device=DEV) if case.get("bias") else None
    return w, b, _act(g, case["M"], case["K"], case["x"])


def _fused_inputs(case, seed):
    g = _gen(seed)
    return [_weight(g, n, case["H"]) for n in READS_X], _act(g, case["M"], case["H"], case["x"])


def _sample_inputs(case, seed):
    g = _gen(seed)
    return _logits(g, case["M"], case["V"]), torch.rand(case["M"], generator=g, device=DEV)


def _layer_step(m, a):
    """One decode step's quantized linears of a hybrid layer on its inputs."""
    reads = m["reads"](a["reads"][0])
    lora = quant.grouped_forward(list(zip(m["lora"], a["lora"])))
    out = quant.grouped_forward(list(zip(m["out"], a["out"])))
    gate_up = m["gate_up"](a["gate_up"][0])
    return [*reads, *lora, *out, *gate_up, m["down"][0](a["down"][0])]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("linear", "greedy"):
        w, b, x = _inputs(case, seed)
        if case.get("token"):
            lin = quant.DynamicInt8Linear(w, b, granularity="token")
        else:
            lin = quant.make_linear(case["fmt"], w, b)
        if "y" in case:
            lin.out_dtype = DTYPES[case["y"]]
        return {"kind": kind, "lin": lin, "x": x}
    if kind == "fused":
        ws, x = _fused_inputs(case, seed)
        return {"kind": kind, "lin": quant.fuse_linears([quant.make_linear(case["fmt"], w) for w in ws]), "x": x}
    if kind == "layer":
        w, a = _layer_inputs(case, _gen(seed))
        m = {k: [quant.make_linear(case["fmt"], t) for t in v] for k, v in w.items()}
        m["reads"], m["gate_up"] = quant.fuse_linears(m["reads"]), quant.fuse_linears(m["gate_up"])
        del w
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # one eager step, then the capture
            _layer_step(m, a)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = _layer_step(m, a)
        return {"kind": kind, "m": m, "a": a, "graph": graph, "outs": outs}
    if kind == "sample":
        logits, u = _sample_inputs(case, seed)
        return {"kind": kind, "logits": logits, "u": u, "T": case["T"], "k": case["k"], "p": case["p"]}
    g = _gen(seed)
    return {"kind": kind, "fmt": case["fmt"], "w": _weight(g, case["N"], case["K"], DTYPES[case["w"]])}


def run(s):
    kind = s["kind"]
    if kind in ("linear", "fused"):
        return s["lin"](s["x"])
    if kind == "greedy":
        return s["lin"].forward_greedy(s["x"])
    if kind == "layer":
        s["graph"].replay()
        return s["outs"]
    if kind == "sample":
        if s["T"] == 0.0:
            return quant.greedy_tokens(s["logits"])
        return quant.sample_tokens(s["logits"], s["T"], s["p"], s["k"], u=s["u"])
    lin = quant.make_linear(s["fmt"], s["w"])
    if s["fmt"] == "int8":
        return {"qweight": lin.qweight, "scale": lin.scale, "packed": lin.packed}
    return {"packed": lin.packed, "scale": lin.scale, "colsum": lin.colsum}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _size(name):
    return 4 if name == "f32" else 2


def _linear_work(M, N, K, x, y="f32"):
    return N * K + 4 * N + M * K * _size(x) + M * N * _size(y), 2 * M * N * K


def work(case):
    kind = case["kind"]
    if kind in ("linear", "greedy"):
        b, f = _linear_work(case["M"], case["N"], case["K"], case["x"], case.get("y", "f32"))
    elif kind == "fused":
        b, f = _linear_work(case["M"], sum(READS_X), case["H"], case["x"])
    elif kind == "layer":
        H, F, M, x = case["H"], case["F"], case["M"], case["x"]
        shapes = [(sum(READS_X), H), (4096, 128), (4096, 128), (H, 4096), (H, 4096), (2 * F, H), (H, F)]
        b, f = (sum(t) for t in zip(*(_linear_work(M, n, k, x) for n, k in shapes)))
    elif kind == "sample":
        b, f = case["M"] * case["V"] * 4 + case["M"] * 8, 0
    else:
        # the weight in; the packed tiles (and the int8 rows the state_dict keeps), scales and column sums out
        n = case["N"] * case["K"]
        b, f = n * _size(case["w"]) + n * (2 if case["fmt"] == "int8" else 1) + case["N"] * (4 if case["fmt"] == "int8" else 8), 0
    return {"bytes": b, "flops": f}


def tolerance(case):
    """int8-dyn, tokens and packed weights are defined bit for bit.  Weight-only
    results differ by summation order with fp16 / bf16 activations (measured
    1e-7 ... 3e-6), by the 16-bit split of fp32 activations at decode sizes
    (about 4e-6), and by the 11-bit staging of fp32 activations in the prefill
    GEMM (2.9e-4)."""
    kind = case["kind"]
    if kind in ("sample", "load") or case["fmt"] == "int8-dyn":
        return "exact"
    if case.get("y") == "f16":
        return {"rel": 3e-4}  # a few outputs one fp16 rounding apart
    if case["x"] != "f32":
        return {"rel": 1.2e-5}
    return {"rel": 2e-5} if case["M"] <= 16 else {"rel": 1e-3}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _div32(a, b):
    """fp32 quotients rounded once (a double quotient of floats rounds to them)."""
    return (a.double() / b.double()).float()


def _quantize(w):
    w = w.float()
    scale = _div32(w.abs().amax(1).clamp_min(1e-8), torch.tensor(127.0, device=DEV))
    return torch.round(_div32(w, scale[:, None])).clamp(-127, 127), scale


def _qparams(x):
    """(scale, zero point) of the dynamic uint8 quantization of x."""
    lo, hi = min(0.0, float(x.min())), max(0.0, float(x.max()))
    s = (hi - lo) / 255.0  # the activations here are far from its tiny-scale branch
    from_min, from_max = 0.0 - lo / s, 255.0 - hi / s
    z = from_min if -abs(lo / s) < 255.0 - abs(hi / s) else from_max
    return float(torch.tensor(s, dtype=torch.float32)), int(min(255, max(0, round(z))))


def _linear64(case_fmt, w, b, x, token=False):
    q, scale = _quantize(w)
    x32 = x.float()
    if case_fmt == "int8":
        y = (x32.double() @ q.double().t()) * scale.double()
    elif token:
        xq, st = _quantize(x32)
        y = (xq.double() @ q.double().t()) * (st.double()[:, None] * scale.double())
    else:
        s, zp = _qparams(x32)
        inv = float(torch.tensor(1.0, dtype=torch.float32) / torch.tensor(s, dtype=torch.float32))
        # one rounding to fp32 (the fused multiply-add), then to an integer
        xq = torch.round((x32.double() * inv + zp).float()).clamp(0, 255) - zp
        y = (xq.double() @ q.double().t()) * (s * scale.double())
    return y if b is None else y + b.double()


def _pack64(q):
    """The packed tile order: [N/16][K/64] tiles, lane (g, r) holding row r's
    bytes g*16 .. g*16+15, offset binary."""
    N, K = q.shape
    Nt, Kc = (N + 15) // 16, (K + 63) // 64
    t = torch.full((Nt * 16, Kc * 64), 0, dtype=torch.int16, device=q.device)
    t[:N, :K] = q.to(torch.int16)
    t = t.view(Nt, 16, Kc, 4, 16).permute(0, 2, 3, 1, 4)
    return ((t + 128) & 255).to(torch.uint8).reshape(-1)


def _sample64(logits, u, T, p, k):
    z = (logits / T).double() if T != 0.0 else logits.double()
    if T == 0.0:
        return z.argmax(-1)
    if 0 < k < z.shape[1]:
        z = z.masked_fill(z < z.topk(k, dim=-1).values[:, -1:], float("-inf"))
    e = torch.softmax(z, -1)
    if 0.0 < p < 1.0:
        s, at = e.sort(dim=-1, descending=True, stable=True)
        s = s * ((s.cumsum(-1) - s) < p)
        e = torch.zeros_like(e).scatter_(1, at, s)
    c = e.cumsum(-1)
    return torch.searchsorted(c, (u.double()[:, None] * c[:, -1:]), right=True)[:, 0].clamp_max(z.shape[1] - 1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("linear", "greedy"):
        w, b, x = _inputs(case, seed)
        y = _linear64(case["fmt"], w, b, x, case.get("token", False))
        return (y, y.argmax(-1)) if kind == "greedy" else y
    if kind == "fused":
        ws, x = _fused_inputs(case, seed)
        return tuple(_linear64(case["fmt"], w, None, x) for w in ws)
    if kind == "layer":
        w, a = _layer_inputs(case, _gen(seed))
        f = case["fmt"]
        return [*(_linear64(f, t, None, a["reads"][0]) for t in w["reads"]),
                *(_linear64(f, t, None, x) for t, x in zip(w["lora"], a["lora"])),
                *(_linear64(f, t, None, x) for t, x in zip(w["out"], a["out"])),
                *(_linear64(f, t, None, a["gate_up"][0]) for t in w["gate_up"]),
                _linear64(f, w["down"][0], None, a["down"][0])]
    if kind == "sample":
        return _sample64(*_sample_inputs(case, seed), case["T"], case["p"], case["k"])
    g = _gen(seed)
    q, scale = _quantize(_weight(g, case["N"], case["K"], DTYPES[case["w"]]))
    if case["fmt"] == "int8":
        return {"qweight": q.to(torch.int8), "scale": scale.double(), "packed": _pack64(q)}
    return {"packed": _pack64(q), "scale": scale.double(), "colsum": q.sum(1).to(torch.int32)}
