"""The work this library is asked for, as cases that can be timed.

A serving program holds a model's expert stacks, router rows and norms on the card, keeps a scratch for each layer shape, and
calls the library in three ways:

  * decode: the tokens of a few running requests go through every layer, router and experts, as one captured graph that is
    replayed step after step;
  * prefill: a prompt's tokens (whole, or a chunk with a ragged end) go through a layer at a time, enqueued as they come;
  * single matrices: a few f32 columns against one quantized matrix or a few, enqueued as they come.

Shapes are the repository's two layers (hidden 2048, 128 experts of 768, top-8; hidden 7168, 256 experts of 2048, top-8 and a
shared expert) and sizes between and around the tests'. Weights are random legal blocks whose values have about the spread of
a trained layer's (sigma 0.02); the router's logits come out near N(0, 1) plus a bias an expert, so some experts are popular
and a few get nothing, as in a real batch.
"""
import math

import torch

import bloomery_amd as bm

TYPES = {"Q3_K": bm.Q3_K, "Q4_K": bm.Q4_K, "Q5_K": bm.Q5_K, "Q6_K": bm.Q6_K, "IQ2_XXS": bm.IQ2_XXS, "IQ3_XXS": bm.IQ3_XXS,
         "IQ4_XS": bm.IQ4_XS}
BLOCK_BYTES = {"Q3_K": 110, "Q4_K": 144, "Q5_K": 176, "Q6_K": 210, "IQ2_XXS": 66, "IQ3_XXS": 98, "IQ4_XS": 136}
# where a block keeps its f16 scale, and the scale at which its values have a standard deviation of about 0.02
SCALE_AT = {"Q3_K": (108, 4.8e-4), "Q4_K": (0, 9e-5), "Q5_K": (0, 4.5e-5), "Q6_K": (208, 1.5e-5), "IQ2_XXS": (0, 4e-4),
            "IQ3_XXS": (0, 2e-4), "IQ4_XS": (0, 1.5e-5)}
RULES = {"silu": (bm.ACT_SILU_MUL, 0.0), "clamp": (bm.ACT_SWIGLU_CLAMP, 7.0), "oai": (bm.ACT_SWIGLU_OAI, 7.0)}
EPS = 1e-6
GRAPH_TOKENS = 64  # batches up to this are decode steps: captured once, replayed


def _layers(name, tokens, layers, gate, down, hidden=2048, ff=768, experts=128, top_k=8, mode="exact", rule="silu", skew=0.5,
            shared=False):
    c = {"kind": "layers", "tokens": tokens, "layers": layers, "gate": gate, "down": down, "hidden": hidden, "ff": ff,
         "experts": experts, "top_k": top_k, "mode": mode, "rule": rule, "skew": skew, "shared": shared}
    return dict(c, name=name) if name else c


def _matrix(name, wtype, rows, k, columns, matrices=1):
    c = {"kind": "matrix", "type": wtype, "rows": rows, "k": k, "columns": columns, "matrices": matrices}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest calls: one token's row against two expert-sized matrices (a gate and an up), quantizer included
        _matrix("matrix_768x2048", "Q4_K", 768, 2048, 1, 2),
        # four columns against a down matrix of the larger layer's shared expert
        _matrix("matrix_7168x2048_4", "Q6_K", 7168, 2048, 4),
        # one request being decoded: eight layers from residual row to residual row
        _layers("decode_1", 1, 8, "Q4_K", "Q6_K"),
        # a batch of running requests, the usual serving load
        _layers("decode_16", 16, 4, "Q4_K", "Q6_K"),
        # a full batch of running requests, on the stacks of a five-bit file
        _layers("decode_64", 64, 2, "Q5_K", "Q6_K"),
        # a few requests on a three-bit file of the importance types, with the clamped gate rule
        _layers("decode_5_iq", 5, 4, "IQ3_XXS", "IQ4_XS", rule="clamp"),
        # the large layer with its shared expert, four requests
        _layers("decode_large_4", 4, 2, "IQ2_XXS", "IQ2_XXS", 7168, 2048, 256, 8, shared=True),
        # a short prompt with a ragged length, in the order of sums that a decode of the same tokens would have
        _layers("prefill_333", 333, 1, "Q4_K", "Q6_K", skew=1.0),
        # a long prompt's chunk, the same
        _layers("prefill_2048", 2048, 1, "Q4_K", "Q6_K", skew=1.0),
        # the longest chunk in the tolerance mode of the sums
        _layers("prefill_4096_fast", 4096, 1, "Q4_K", "Q6_K", mode="fast", skew=1.0),
        # a ragged prompt on a four-bit file of the importance types
        _layers("prefill_777_iq4", 777, 1, "IQ4_XS", "IQ4_XS", skew=1.0),
        # a prompt's chunk through the large layer and its shared expert
        _layers("prefill_large_1024_fast", 1024, 1, "IQ2_XXS", "IQ2_XXS", 7168, 2048, 256, 8, mode="fast", skew=1.0, shared=True),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if rng.random() < 0.15:
        return _matrix(None, rng.choice(sorted(TYPES)), spread(256, 8192), 256 * spread(2, 28), rng.randint(1, 8), rng.randint(1, 3))
    gate, down = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q6_K"), ("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q6_K", "Q6_K"),
                             ("Q3_K", "Q4_K"), ("IQ4_XS", "IQ4_XS"), ("IQ3_XXS", "IQ4_XS"), ("IQ2_XXS", "IQ2_XXS")])
    hidden, ff, experts = 256 * spread(4, 28), 256 * spread(2, 8), spread(8, 256)
    top_k = rng.randint(1, 8)
    tokens = spread(1, 4096)
    while experts * hidden * ff > 2 << 30:
        experts = max(8, experts // 2)
    cost = 6.0 * top_k * hidden * ff
    tokens = max(1, min(tokens, int(4e11 / cost), 40960 // top_k))
    layers = 1 if tokens > GRAPH_TOKENS or experts * hidden * ff > 1 << 29 else 2
    return _layers(None, tokens, layers, gate, down, hidden, ff, experts, top_k,
                   "fast" if tokens > GRAPH_TOKENS and rng.random() < 0.5 else "exact", rng.choice(["silu", "silu", "clamp", "oai"]),
                   1.0 if tokens > GRAPH_TOKENS else 0.5, rng.random() < 0.2)


_contexts = {}


def _gpu(mode):
    """A program's context for each order of sums, made once."""
    if mode not in _contexts:
        gpu = bm.Gpu(0)
        gpu.set_gemm_mode(bm.GEMM_FAST if mode == "fast" else bm.GEMM_EXACT)
        _contexts[mode] = gpu
    return _contexts[mode]


def _stack(gen, wtype, rows, k):
    """rows x k values of random legal blocks on the card."""
    bb, n = BLOCK_BYTES[wtype], rows * (k // 256)
    # 16 bytes behind the last row, as the library's own loader leaves
    words = torch.randint(-(1 << 62), 1 << 62, ((n * bb + 16 + 7) // 8,), dtype=torch.int64, device="cuda", generator=gen)
    raw = words.view(torch.uint8)
    blocks = raw[:n * bb].view(n, bb)
    at, d = SCALE_AT[wtype]
    scale = (torch.rand(n, device="cuda", generator=gen) * (0.5 * d) + 0.75 * d).to(torch.float16)
    blocks[:, at:at + 2] = scale.view(torch.uint8).view(n, 2)
    if wtype in ("Q4_K", "Q5_K"):
        # minimum = scale code x 7.5 (15.5) steps, so the values lie around zero: the mins' six bits are the scales'
        half = 7.5 if wtype == "Q4_K" else 15.5
        blocks[:, 2:4] = (scale.float() * half).to(torch.float16).view(torch.uint8).view(n, 2)
        blocks[:, 4:8] |= 32  # the trained scales lie in the upper half of their range
        blocks[:, 8:12] = blocks[:, 4:8]
        blocks[:, 12:16] = (blocks[:, 12:16] & 15) * 17
    return raw


class _State:
    """What a program keeps for a layer stack or a matrix. Freed with the last reference."""

    def __init__(self):
        self.gpu, self.held, self.graph, self.keep = None, [], None, []

    def own(self, h):
        self.held.append(h)
        return h

    def weights(self, gen, wtype, rows, k):
        raw = _stack(gen, wtype, rows, k)
        self.keep.append(raw)
        return self.own(bm.DeviceTensor(self.gpu, TYPES[wtype], rows, k, dev_ptr=raw.data_ptr()))

    def __del__(self):
        if self.gpu is None:
            return
        if self.graph is not None:
            self.gpu.graph_destroy(self.graph)
        for h in self.held:
            h.free()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    normal = lambda *shape: torch.randn(*shape, device="cuda", generator=gen)  # noqa: E731
    s = _State()
    s.case = case
    if case["kind"] == "matrix":
        s.gpu = _gpu("exact")
        s.w = [s.weights(gen, case["type"], case["rows"], case["k"]) for _ in range(case["matrices"])]
        s.x = normal(case["columns"], case["k"])
        s.y = [torch.zeros(case["rows"], case["columns"], device="cuda") for _ in s.w]
        s.act = s.own(s.gpu.act(TYPES[case["type"]], case["k"], case["columns"]))
        torch.cuda.synchronize()
        return s
    m, hidden, ff, n, top_k = case["tokens"], case["hidden"], case["ff"], case["experts"], case["top_k"]
    s.gpu = _gpu(case["mode"])
    s.layers = []
    for _ in range(case["layers"]):
        layer = {"gate": s.weights(gen, case["gate"], n * ff, hidden), "up": s.weights(gen, case["gate"], n * ff, hidden),
                 "down": s.weights(gen, case["down"], n * hidden, ff)}
        layer["router"] = normal(n, hidden) * math.sqrt((1.0 + case["skew"] ** 2) / hidden)
        layer["norm"] = 1.0 + 0.1 * normal(hidden)
        if case["shared"]:
            layer["shared"] = [s.weights(gen, "Q6_K", ff, hidden), s.weights(gen, "Q6_K", ff, hidden), s.weights(gen, "Q6_K", hidden, ff)]
        s.layers.append(layer)
    # the residual rows: the tokens of a batch have a part in common, which is what makes some experts popular
    x = normal(m, hidden) + case["skew"] * normal(hidden)
    s.rows = [x] + [torch.zeros(m, hidden, device="cuda") for _ in s.layers]
    s.normed, s.logits = torch.zeros(m, hidden, device="cuda"), torch.zeros(m, n, device="cuda")
    s.ids = [torch.zeros(m, top_k, dtype=torch.int32, device="cuda") for _ in s.layers]
    s.wts = [torch.zeros(m, top_k, device="cuda") for _ in s.layers]
    s.scratch = s.own(s.gpu.scratch(TYPES[case["gate"]], TYPES[case["down"]], hidden, ff, n, top_k, m))
    if case["shared"]:
        s.shared_scratch = s.own(s.gpu.scratch(bm.Q6_K, bm.Q6_K, hidden, ff, 1, 1, m))
        s.shared_rows = torch.zeros(m, hidden, device="cuda")
        s.zero, s.one = torch.zeros(m, dtype=torch.int32, device="cuda"), torch.ones(m, device="cuda")
    s.rule = None if case["rule"] == "silu" else RULES[case["rule"]]
    torch.cuda.synchronize()
    if m <= GRAPH_TOKENS:
        s.gpu.capture_begin()
        _enqueue(s)
        s.graph = s.gpu.capture_end()
    return s


def _enqueue(s):
    """Every layer from its residual rows: norm and router, the shared expert where there is one, the routed experts."""
    c, gpu = s.case, s.gpu
    m = c["tokens"]
    for i, layer in enumerate(s.layers):
        x, y = s.rows[i].data_ptr(), s.rows[i + 1].data_ptr()
        ids, wts, normed = s.ids[i].data_ptr(), s.wts[i].data_ptr(), s.normed.data_ptr()
        gpu.enqueue_norm_route(layer["router"].data_ptr(), x, layer["norm"].data_ptr(), EPS, m, c["experts"], c["hidden"], c["top_k"], True,
                               normed, s.logits.data_ptr(), None, ids, wts)
        if c["shared"]:
            gate, up, down = layer["shared"]
            gpu.enqueue_moe_forward(s.shared_scratch, gate, up, down, normed, s.zero.data_ptr(), s.one.data_ptr(), x, m,
                                    s.shared_rows.data_ptr(), rule=s.rule)
            x = s.shared_rows.data_ptr()
        gpu.enqueue_moe_forward(s.scratch, layer["gate"], layer["up"], layer["down"], normed, ids, wts, x, m, y, rule=s.rule)


def run(s):
    if s.case["kind"] == "matrix":
        x, m = s.x.data_ptr(), s.case["columns"]
        if m == 1:
            for w, y in zip(s.w, s.y):
                s.gpu.enqueue_gemv_x(w, x, 1, y.data_ptr())
        else:
            s.gpu.enqueue_quantize(x, m, s.act)
            for w, y in zip(s.w, s.y):
                s.gpu.enqueue_gemv(w, s.act, m, y.data_ptr())
        return s.y
    if s.graph is not None:
        s.gpu.graph_launch(s.graph)
    else:
        _enqueue(s)
    return {"rows": s.rows[1:], "ids": s.ids, "weights": s.wts}


def work(case):
    if case["kind"] == "matrix":
        rows, k, m, n = case["rows"], case["k"], case["columns"], case["matrices"]
        return {"bytes": n * (rows * (k // 256) * BLOCK_BYTES[case["type"]] + 4 * m * rows) + 4 * m * k, "flops": 2 * n * m * rows * k}
    m, hidden, ff, n, top_k = case["tokens"], case["hidden"], case["ff"], case["experts"], case["top_k"]
    expert = hidden * ff // 256 * (2 * BLOCK_BYTES[case["gate"]] + BLOCK_BYTES[case["down"]])
    # the experts that m tokens hit when every expert is as likely (a skewed router hits somewhat fewer)
    hit = n * (1.0 - (1.0 - top_k / n) ** m)
    nbytes = hit * expert + 4 * n * hidden + 8 * m * hidden
    flops = 2 * m * hidden * n + 6 * m * top_k * hidden * ff
    if case["shared"]:
        nbytes += hidden * ff // 256 * 3 * BLOCK_BYTES["Q6_K"]
        flops += 6 * m * hidden * ff
    return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * flops}


def tolerance(case):
    # The order of the f32 sums is part of the library's contract, and every path but the tolerance mode's GEMM keeps it.
    # There the sums differ by f32 rounding, and now and then one tips an eight-bit code of h by a step.
    if case["kind"] == "layers" and case["mode"] == "fast":
        return {"rel": 1e-4}
    return "exact"
