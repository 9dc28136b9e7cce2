"""The quantized-linear workloads that users of this package run, for timing.

Four kinds of call, each over the sizes, bit widths and group sizes it is used with:

* ``linear``  one ``quantized_matmul`` from the host program: decode (M = 1), speculative
              verify and batched decode (M up to a few dozen), prompt chunks and prefill
              (M up to 2048);
* ``stack``   the seven projections of a few Llama-shaped layers for M concurrent
              sequences, captured once in a HIP graph and replayed for every token;
* ``moe``     the router and the expert layer (with the shared expert) of a
              mixture-of-experts model: decode steps as a replayed graph, larger token
              counts as plain calls;
* ``requant`` the load-time pass over an attention band: dequantize, then quantize.

Weights and activations follow the distributions of the repository's benchmark: x ~ N(0, 1);
4-bit scales uniform in [0.002, 0.02] with biases near -8 scale; 8-bit scales uniform in
[1e-4, 2e-3] with biases -128 scale.
"""
import math

import torch

from fastmlx_amd import ops

DEV = "cuda"

# Expert layers: experts, experts per token, width, expert width, router.
QWEN = {"E": 512, "k": 10, "D": 2048, "I": 512, "router": "softmax"}
DEEPSEEK = {"E": 256, "k": 8, "D": 7168, "I": 2048, "router": "group"}


def listed():
    return [
        # One small projection of a decode step called from the host: launch latency.
        dict(name="linear_decode_2048", kind="linear", M=1, N=2048, K=2048, bits=4, group=64),
        # Single-sequence decode through 8B-sized layers: weight streaming, launch count.
        dict(name="stack_decode_m1", kind="stack", M=1, D=4096, KV=1024, F=14336, layers=4, bits=4,
             group=64),
        # The same layers serving an odd number of concurrent sequences.
        dict(name="stack_decode_m13", kind="stack", M=13, D=4096, KV=1024, F=14336, layers=4,
             bits=4, group=64),
        # Batched decode / draft verify of a checkpoint quantized with groups of 32.
        dict(name="linear_g32_m24", kind="linear", M=24, N=14336, K=4096, bits=4, group=32),
        # A short prompt (or the rest of a chunked one) through a down projection.
        dict(name="linear_prompt_m200", kind="linear", M=200, N=4096, K=14336, bits=4, group=64),
        # A ragged prompt chunk on an 8-bit checkpoint.
        dict(name="linear_8bit_m509", kind="linear", M=509, N=14336, K=4096, bits=8, group=64),
        # Prefill of a long prompt chunk through a gate/up projection.
        dict(name="linear_prefill_m2048", kind="linear", M=2048, N=14336, K=4096, bits=4, group=64),
        # One token through many-expert layers: the latency of a decode step.
        dict(name="moe_decode_t1", kind="moe", T=1, layers=4, graph=True, bits=4, group=64, **QWEN),
        # Batched decode on an 8-bit many-expert checkpoint.
        dict(name="moe_8bit_t24", kind="moe", T=24, layers=1, graph=False, bits=8, group=64, **QWEN),
        # A larger decode batch or a short prompt on the 4-bit one.
        dict(name="moe_t100", kind="moe", T=100, layers=1, graph=False, bits=4, group=64, **QWEN),
        # A prompt chunk through a wide expert layer with skewed expert popularity.
        dict(name="moe_prefill_t1024", kind="moe", T=1024, layers=1, graph=False, bits=4, group=64,
             **DEEPSEEK),
        # Weight absorption at load: a band of an attention projection requantized.
        dict(name="requant_band", kind="requant", rows=32768, K=512, bits=4, group=64),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step):
    return max(lo, _logint(rng, lo, hi) // step * step)


def _quant(rng):
    bits = rng.choice((4, 4, 4, 8))
    group = rng.choice((64, 64, 64, 64, 32, 128))
    return bits, group


def _seconds(case):
    """A rough estimate of a pass, to keep drawn cases below the largest listed one."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 1e15


def draw(rng):
    most = max(_seconds(c) for c in listed())
    while True:
        kind = rng.choice(("linear", "linear", "linear", "stack", "moe", "moe", "requant"))
        bits, group = _quant(rng)
        if kind == "linear":
            # Model widths are multiples of 256 almost always, of the group in any case.
            step = rng.choice((256, 256, 256, 128))
            c = dict(kind=kind, M=_logint(rng, 1, 2048), N=_width(rng, 512, 28672, step),
                     K=_width(rng, 512, 16384, step), bits=bits, group=group)
        elif kind == "stack":
            D = _width(rng, 2048, 5120, 512)
            c = dict(kind=kind, M=_logint(rng, 1, 64), D=D, KV=rng.choice((512, 1024, D)),
                     F=_width(rng, 2 * D, 4 * D, 256), layers=rng.randint(1, 4), bits=bits,
                     group=group)
        elif kind == "moe":
            shape = rng.choice((QWEN, DEEPSEEK, None))
            if shape is None:
                shape = {"E": rng.choice((16, 64, 128)), "k": rng.randint(2, 8),
                         "D": _width(rng, 1024, 4096, 256), "I": _width(rng, 512, 2048, 256),
                         "router": "softmax"}
            graph = rng.random() < 0.5
            T = _logint(rng, 1, 32) if graph else _logint(rng, 2, 2048)
            c = dict(kind=kind, T=T, layers=rng.randint(1, 2) if graph else 1, graph=graph,
                     bits=bits, group=group, **shape)
        else:
            c = dict(kind=kind, rows=_logint(rng, 256, 65536), K=_width(rng, 256, 2048, 128),
                     bits=bits, group=group)
        if _seconds(c) <= most:
            return c


# ---- inputs -------------------------------------------------------------------


def _packed(gen, lead, K, bits, group):
    """A random quantized weight [*lead, K]: (words, scales, biases)."""
    w = torch.randint(-2**31, 2**31, (*lead, K * bits // 32), dtype=torch.int32, device=DEV,
                      generator=gen)
    lo, hi, mid = (0.002, 0.02, 8) if bits == 4 else (1e-4, 2e-3, 128)
    s = torch.empty(*lead, K // group, device=DEV).uniform_(lo, hi, generator=gen).bfloat16()
    b = -mid * s.float()
    if bits == 4:
        b += torch.empty_like(b).normal_(0.0, 1e-3, generator=gen)
    return w, s, b.bfloat16()


def _normal(gen, *shape):
    return torch.empty(*shape, device=DEV).normal_(generator=gen).bfloat16()


def _logits(c, gen):
    T, E = c["T"], c["E"]
    if c["router"] == "softmax":
        return _normal(gen, T, E)
    # Top-k of log-popularity plus Gumbel noise is a draw without replacement from
    # Zipf(1.1) popularities, spread over the expert ids.
    rank = torch.randperm(E, device=DEV, generator=gen).float() + 1
    u = torch.empty(T, E, device=DEV).uniform_(1e-6, 1 - 1e-6, generator=gen)
    return (-1.1 * rank.log() - (-u.log()).log()).bfloat16()


def _inputs(c, seed):
    """The tensors of a case, made on the GPU from the seed alone."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    bits, group = c["bits"], c["group"]
    if c["kind"] == "linear":
        return {"x": _normal(gen, c["M"], c["K"]),
                "w": _packed(gen, (c["N"],), c["K"], bits, group)}
    if c["kind"] == "stack":
        D, KV, F, M = c["D"], c["KV"], c["F"], c["M"]
        layers = []
        for _ in range(c["layers"]):
            dims = (("x", D, D), ("x", KV, D), ("x", KV, D), ("a", D, D), ("m", F, D), ("m", F, D),
                    ("h", D, F))
            layers.append([(act, _packed(gen, (n,), k, bits, group)) for act, n, k in dims])
        acts = {"x": _normal(gen, M, D), "a": _normal(gen, M, D), "m": _normal(gen, M, D),
                "h": _normal(gen, M, F)}
        return {"acts": acts, "layers": layers}
    if c["kind"] == "moe":
        E, D, I = c["E"], c["D"], c["I"]
        layers = []
        for _ in range(c["layers"]):
            experts = [_packed(gen, (E, I), D, bits, group), _packed(gen, (E, I), D, bits, group),
                       _packed(gen, (E, D), I, bits, group)]
            shared = [_packed(gen, (1, I), D, bits, group), _packed(gen, (1, I), D, bits, group),
                      _packed(gen, (1, D), I, bits, group)]
            gate = _normal(gen, c["T"]) if c["router"] == "softmax" else None
            layers.append({"logits": _logits(c, gen), "experts": experts, "shared": shared,
                           "gate": gate, "x": _normal(gen, c["T"], D)})
        return {"layers": layers}
    return {"w": _packed(gen, (c["rows"],), c["K"], bits, group)}


# ---- one pass -----------------------------------------------------------------


def _linear(c, x, w):
    return ops.quantized_matmul(x, *w, True, c["group"], c["bits"])


def _moe_layer(c, p):
    if c["router"] == "softmax":
        inds, weights = ops.route_softmax_topk(p["logits"], c["k"])
    else:
        inds, weights = ops.route_group_topk(p["logits"], None, c["k"], 8, 4, 2.5,
                                             weights_dtype=torch.bfloat16)
    y = ops.moe_layer(p["x"], inds, *p["experts"], weights, p["shared"], p["gate"], c["group"],
                      c["bits"])
    return {"y": y, "inds": inds, "weights": weights}


def _calls(c, p):
    if c["kind"] == "linear":
        return _linear(c, p["x"], p["w"])
    if c["kind"] == "stack":
        return [_linear(c, p["acts"][act], w) for layer in p["layers"] for act, w in layer]
    if c["kind"] == "moe":
        return [_moe_layer(c, layer) for layer in p["layers"]]
    d = ops.dequantize(*p["w"], c["group"], c["bits"])
    return [d, *ops.quantize(d, c["group"], c["bits"])]


def prepare(case, seed):
    p = _inputs(case, seed)
    state = {"case": case, "inputs": p}
    if case["kind"] == "stack" or case.get("graph"):
        # A decode loop captures its step once and replays it for every token.
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _calls(case, p)
        stream.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=stream):
            state["out"] = _calls(case, p)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _calls(state["case"], state["inputs"])


# ---- what a pass cannot do without ----------------------------------------------


def _weight_bytes(N, K, bits, group):
    return N * K * bits // 8 + N * (K // group) * 4


def _linear_work(M, N, K, bits, group):
    return _weight_bytes(N, K, bits, group) + 2 * M * K + 2 * M * N, 2 * M * N * K


def work(case):
    c, bits, group = case, case["bits"], case["group"]
    if c["kind"] == "linear":
        b, f = _linear_work(c["M"], c["N"], c["K"], bits, group)
    elif c["kind"] == "stack":
        D, KV, F = c["D"], c["KV"], c["F"]
        b = f = 0
        for n, k in ((D, D), (KV, D), (KV, D), (D, D), (F, D), (F, D), (D, F)):
            bb, ff = _linear_work(c["M"], n, k, bits, group)
            b, f = b + c["layers"] * bb, f + c["layers"] * ff
    elif c["kind"] == "moe":
        T, E, k, D, I = c["T"], c["E"], c["k"], c["D"], c["I"]
        if c["router"] == "softmax":
            hit = E * (1 - (1 - k / E) ** T)
        else:
            # Distinct experts under Zipf(1.1), independent draws.
            p = [r ** -1.1 for r in range(1, E + 1)]
            s = sum(p)
            hit = sum(1 - (1 - q / s) ** (T * k) for q in p)
        per = 2 * _weight_bytes(I, D, bits, group) + _weight_bytes(D, I, bits, group)
        b = c["layers"] * ((hit + 1) * per + 4 * T * D + 2 * T * E + 6 * T * k)
        f = c["layers"] * 6 * T * (k + 1) * D * I
    else:
        n = c["rows"] * c["K"]
        b, f = 2 * (n * 2 + n * bits // 8 + n // group * 4), 0
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    if case["kind"] == "requant":
        return "exact"
    if case["kind"] == "moe":
        return {"rel": 1.6e-2, "max": 0.1, "differ": 1e-3}
    return {"rel": 8e-3, "max": 0.04}


# ---- the same in 64 bits --------------------------------------------------------


def _unpacked(w, c):
    words, s, b = w
    bits, group = c["bits"], c["group"]
    at = torch.arange(0, 32, bits, device=DEV, dtype=torch.int32)
    q = (words.unsqueeze(-1) >> at) & ((1 << bits) - 1)
    q = q.reshape(*s.shape, group).double()
    v = q * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)
    return v.reshape(*words.shape[:-1], -1)


def _exact_linear(c, x, w):
    return x.double() @ _unpacked(w, c).T


def _exact_route(c, logits):
    g = logits.double()
    if c["router"] == "softmax":
        g = torch.softmax(g, -1)
        score = g
    else:
        g = torch.sigmoid(g)
        T, E = g.shape
        best = g.reshape(T, 8, E // 8).sort(dim=-1, descending=True).values[..., :2].sum(-1)
        kept = best.sort(dim=-1, descending=True, stable=True).indices[:, :4]
        keep = torch.zeros(T, 8, dtype=torch.bool, device=DEV).scatter_(1, kept, True)
        score = torch.where(keep.repeat_interleave(E // 8, dim=1), g, torch.zeros_like(g))
    inds = score.sort(dim=-1, descending=True, stable=True).indices[:, : c["k"]]
    w = g.gather(1, inds)
    w = w / w.sum(-1, keepdim=True)
    return inds, w if c["router"] == "softmax" else 2.5 * w


def _exact_mlp(c, x, mats, e):
    g, u, d = (tuple(t[e] for t in m) for m in mats)
    gate = _exact_linear(c, x, g)
    h = gate * torch.sigmoid(gate) * _exact_linear(c, x, u)
    return h @ _unpacked(d, c).T


def _exact_moe(c, p):
    inds, w = _exact_route(c, p["logits"])
    x = p["x"].double()
    y = _exact_mlp(c, x, p["shared"], 0)
    if p["gate"] is not None:
        y = y * torch.sigmoid(p["gate"].double()).unsqueeze(-1)
    for e in inds.unique().tolist():
        t, j = (inds == e).nonzero(as_tuple=True)
        y.index_add_(0, t, _exact_mlp(c, x[t], p["experts"], e) * w[t, j].unsqueeze(-1))
    return {"y": y, "inds": None, "weights": w}


def exact(case, seed):
    c, p = case, _inputs(case, seed)
    if c["kind"] == "linear":
        return _exact_linear(c, p["x"], p["w"])
    if c["kind"] == "stack":
        return [_exact_linear(c, p["acts"][act], w) for layer in p["layers"] for act, w in layer]
    if c["kind"] == "moe":
        return [_exact_moe(c, layer) for layer in p["layers"]]
    return [_unpacked(p["w"], c), None, None, None]
