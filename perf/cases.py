"""What the performance of this framework is measured on: the MoE layer from
one decode token to a 16K prefill, the Q4_0 / Q4_1 projections around it and
the router, each through its public entry point, plus one captured pipeline
of all of them.

Weights, activations and routes follow the distributions of workloads.py,
made on the GPU from the seed.  `exact` restates the arithmetic in float64
with torch alone: the Q8_1 codes and the fp16 block fields are part of the
formats and are formed as the formats define them (float32 scales, the
pairwise raw sum), everything between them is float64.
"""
import importlib.util
import math
import os
import sys

import torch

TOP_K, EXPERTS = 10, 512
Q4_0, Q4_1 = 2, 3
BLOCK = {Q4_0: 18, Q4_1: 20}


def _package():
    """The binding of the tree the program runs in (its folder's name is no
    Python identifier)."""
    if "moe_ffn" not in sys.modules:
        path = os.path.join(os.getcwd(), "gfx906-qwen3.8fn_amd", "moe_ffn.py")
        spec = importlib.util.spec_from_file_location("moe_ffn", path)
        module = importlib.util.module_from_spec(spec)
        sys.modules["moe_ffn"] = module
        spec.loader.exec_module(module)
    return sys.modules["moe_ffn"]


# ----------------------------------------------------------------- cases ---
def _layer(tokens, hidden=2048, intermediate=512, q41=False, routing="uniform", s=0.0, gate=False):
    return {"kind": "layer", "tokens": tokens, "hidden": hidden, "intermediate": intermediate, "q41": q41,
            "routing": routing, "s": s, "gate": gate}


def _linear(type_, inputs, outputs, columns, q8=False):
    return {"kind": "linear", "q41": type_ == Q4_1, "input": inputs, "output": outputs, "columns": columns, "q8": q8}


def listed():
    return [
        # One user's decode step as a server runs it: projection, router
        # matrix, device top-10 and MoE layer of four layers, replayed from a graph.
        dict({"kind": "pipeline", "layers": 4, "tokens": 1}, name="pipeline_decode_1"),
        # A decode batch of eight on one layer, the benchmark's headline shape.
        dict(_layer(8), name="layer_decode_8"),
        # A few users on the checkpoint's own expert shape: Q4_1 downs, gated shared expert.
        dict(_layer(5, 2560, 640, q41=True, gate=True), name="layer_decode_5_q41"),
        # A larger continuous batch: most experts get one or two tokens.
        dict(_layer(72, gate=True), name="layer_batch_72"),
        # Decode tokens beside a 1,024-token prefill chunk, skewed routing.
        dict(_layer(1032, routing="zipf", s=1.3), name="layer_mixed_1032"),
        # A 4K prompt with Zipf routing.
        dict(_layer(4096, routing="zipf", s=1.1), name="layer_prefill_4096"),
        # A 16K prompt with balanced routing: the largest work here.
        dict(_layer(16384), name="layer_prefill_16384"),
        # An odd-sized prompt on the checkpoint's expert shape, Q4_1 downs and the shared gate.
        dict(_layer(3001, 2560, 640, q41=True, routing="zipf", s=1.1, gate=True), name="layer_prefill_3001_q41"),
        # A dense projection in a decode batch, its input quantised by an earlier step.
        dict(_linear(Q4_0, 8192, 8192, 8, q8=True), name="linear_decode_8"),
        # A hidden-size projection over a prefill chunk, from fp32 activations.
        dict(_linear(Q4_0, 2048, 2048, 1032), name="linear_prefill_1032"),
        # The checkpoint's Q4_1 matrices over a prompt of 128 tokens.
        dict(_linear(Q4_1, 640, 2560, 128), name="linear_q41_128"),
        # Router selection for a 4K prompt.
        dict({"kind": "router", "tokens": 4096}, name="router_4096"),
    ]


def _spread(rng, lo, hi):
    """A whole number, evenly over the logarithm of lo..hi."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


LINEAR_SHAPES = [(2048, 2048), (2048, 512), (2560, 640), (640, 2560), (2560, 2560), (1024, 4096), (2048, 8192),
                 (8192, 2048), (8192, 8192), (2080, 1000), (512, 2047)]


def draw(rng):
    kind = rng.choice(["layer"] * 7 + ["linear"] * 5 + ["pipeline", "router"])
    if kind == "layer":
        routing = rng.choice(["uniform", "zipf", "zipf"])
        s = rng.choice([1.1, 1.3]) if routing == "zipf" else 0.0
        if rng.random() < 0.6:
            return _layer(_spread(rng, 1, 16000), routing=routing, s=s, gate=rng.random() < 0.5)
        return _layer(_spread(rng, 1, 8192), 2560, 640, q41=rng.random() < 0.5, routing=routing, s=s,
                      gate=rng.random() < 0.5)
    if kind == "linear":
        inputs, outputs = rng.choice(LINEAR_SHAPES)
        return _linear(rng.choice([Q4_0, Q4_0, Q4_1]), inputs, outputs, _spread(rng, 1, 1500), q8=rng.random() < 0.5)
    if kind == "pipeline":
        return {"kind": "pipeline", "layers": rng.choice([2, 3, 4]), "tokens": _spread(rng, 1, 600)}
    return {"kind": "router", "tokens": _spread(rng, 1, 16384)}


# ---------------------------------------------------------------- inputs ---
def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + stream * 7919 + 17) % (1 << 62))
    return g


def _blocks(n, type_, g):
    """n canonical weight blocks, uint8 [n][18 or 20]."""
    out = torch.empty((n, BLOCK[type_]), dtype=torch.uint8, device="cuda")
    d = (torch.randn(n, generator=g, device="cuda") * 0.02).abs().half()
    out[:, :2] = d.view(torch.uint8).view(n, 2)
    if type_ == Q4_1:
        m = (-8.0 * d.float() * (0.75 + 0.5 * torch.rand(n, generator=g, device="cuda"))).half()
        out[:, 2:4] = m.view(torch.uint8).view(n, 2)
    codes = torch.empty((n, 16), dtype=torch.uint8, device="cuda").random_(0, 256, generator=g)
    out[:, BLOCK[type_] - 16:] = codes
    return out


def _bank(experts, hidden, intermediate, q41, g):
    """Canonical experts, uint8 [experts][bytes]: gate, up, down blocks."""
    n = hidden // 32 * intermediate
    gate_up = _blocks(experts * 2 * n, Q4_0, g).view(experts, -1)
    down = _blocks(experts * n, Q4_1 if q41 else Q4_0, g).view(experts, -1)
    return torch.cat([gate_up, down], dim=1)


def _routes(c, g):
    """(ids, weights): top-10 by Gumbel keys, strongest first."""
    n = c["tokens"]
    logp = torch.zeros(EXPERTS, device="cuda", dtype=torch.float64)
    if c["routing"] == "zipf":
        perm = torch.randperm(EXPERTS, generator=g, device="cuda")
        logp[perm] = -c["s"] * torch.log(torch.arange(1, EXPERTS + 1, device="cuda", dtype=torch.float64))
    u = torch.rand((n, EXPERTS), generator=g, device="cuda", dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
    ids = (logp - torch.log(-torch.log(u))).topk(TOP_K, dim=1).indices.to(torch.int32).contiguous()
    return ids, torch.softmax(torch.randn((n, TOP_K), generator=g, device="cuda"), dim=1).contiguous()


def _layer_inputs(c, seed):
    g = _generator(seed, 1)
    x = torch.randn((c["tokens"], c["hidden"]), generator=g, device="cuda")
    ids, weights = _routes(c, g)
    gate = torch.randn(c["tokens"], generator=g, device="cuda") if c["gate"] else None
    return x, ids, weights, gate


def _layer_bank(c, seed):
    g = _generator(seed, 2)
    return (_bank(EXPERTS, c["hidden"], c["intermediate"], c["q41"], g),
            _bank(1, c["hidden"], c["intermediate"], c["q41"], g))


def _make_layer(c, bank, shared, max_tokens):
    m = _package()
    return m.MoeLayer(c["hidden"], c["intermediate"], EXPERTS, TOP_K, True, max_tokens, experts_q4=bank.view(-1),
                      shared_q4=shared.view(-1), down_type=m.DOWN_Q4_1 if c["q41"] else m.DOWN_Q4_0)


def _pipeline_part(c, seed, layer):
    """One pipeline layer's canonical weights and input batch."""
    g = _generator(seed, 10 + layer)
    shape = _layer(c["tokens"])
    h = shape["hidden"]
    return {"shape": shape, "bank": _bank(EXPERTS, h, shape["intermediate"], False, g),
            "shared": _bank(1, h, shape["intermediate"], False, g), "proj": _blocks(h * h // 32, Q4_0, g),
            "router": _blocks(EXPERTS * h // 32, Q4_0, g),
            "x": torch.randn((c["tokens"], h), generator=g, device="cuda")}


def _linear_inputs(c, seed):
    g = _generator(seed, 3)
    type_ = Q4_1 if c["q41"] else Q4_0
    w = _blocks(c["input"] // 32 * c["output"], type_, g)
    return w, torch.randn((c["columns"], c["input"]), generator=g, device="cuda")


def prepare(case, seed):
    m = _package()
    kind = case["kind"]
    if kind == "layer":
        x, ids, weights, gate = _layer_inputs(case, seed)
        layer = _make_layer(case, *_layer_bank(case, seed), case["tokens"])
        return {"kind": kind, "layer": layer, "args": (x, ids, weights, gate)}
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        matrix = m.MoeLinear(Q4_1 if case["q41"] else Q4_0, case["input"], case["output"], w, max_columns=case["columns"])
        if case["q8"]:
            return {"kind": "linear_q8", "matrix": matrix, "x": m.quantize_q8_1(x)[0], "columns": case["columns"]}
        return {"kind": kind, "matrix": matrix, "x": x}
    if kind == "router":
        return {"kind": kind, "logits": torch.randn((case["tokens"], EXPERTS), generator=_generator(seed, 4), device="cuda") * 2.0}
    layers, projections, routers, xs = [], [], [], []
    for l in range(case["layers"]):
        p = _pipeline_part(case, seed, l)
        h = p["shape"]["hidden"]
        layers.append(_make_layer(p["shape"], p["bank"], p["shared"], case["tokens"]))
        projections.append(m.MoeLinear(Q4_0, h, h, p["proj"], max_columns=case["tokens"]))
        routers.append(m.MoeLinear(Q4_0, h, EXPERTS, p["router"], max_columns=case["tokens"]))
        xs.append(p["x"])
    stack = m.MoeStack(layers, projections, routers)
    stack.bind(xs)
    stack.capture()
    return {"kind": kind, "stack": stack}


# ------------------------------------------------------------------ runs ---
def run(state):
    kind = state["kind"]
    if kind == "layer":
        x, ids, weights, gate = state["args"]
        return state["layer"].forward(x, ids, weights, shared_gate=gate)
    if kind == "linear":
        return state["matrix"].apply(state["x"])
    if kind == "linear_q8":
        return state["matrix"].forward_q8(state["x"], state["columns"])
    if kind == "router":
        ids, weights, _, error = _package().router_select(state["logits"], top_k=TOP_K)
        return ids, weights, error
    stack = state["stack"]
    stack.replay()
    return [{"h": st["h"], "logits": st["logits"], "ids": st["ids"], "y": st["y"]} for st in stack.steps]


def _expert_bytes(c):
    return c["hidden"] // 32 * c["intermediate"] * (36 + BLOCK[Q4_1 if c["q41"] else Q4_0])


def _touched(c):
    """Experts that a batch reaches, on average: expert i is among a token's
    ten with probability 1 - exp(-r p_i), r such that they add up to ten."""
    n = c["tokens"]
    p = [(i + 1.0) ** -c["s"] if c["routing"] == "zipf" else 1.0 for i in range(EXPERTS)]
    lo, hi = 0.0, 1e9
    for _ in range(80):
        r = (lo + hi) / 2
        lo, hi = (r, hi) if sum(1 - math.exp(-r * q) for q in p) < TOP_K else (lo, r)
    return sum(1 - math.exp(-lo * q * n) for q in p)


def work(case):
    kind = case["kind"]
    if kind == "layer":
        n = case["tokens"]
        return {"bytes": (_touched(case) + 1) * _expert_bytes(case) + n * case["hidden"] * 8 + n * TOP_K * 8,
                "flops": 6.0 * case["hidden"] * case["intermediate"] * n * (TOP_K + 1)}
    if kind == "linear":
        k, m, n = case["input"], case["output"], case["columns"]
        x = n * (k // 32 * 36 if case["q8"] else 4 * k)
        return {"bytes": k // 32 * m * BLOCK[Q4_1 if case["q41"] else Q4_0] + x + 4.0 * n * m, "flops": 2.0 * k * m * n}
    if kind == "router":
        return {"bytes": case["tokens"] * (EXPERTS * 4.0 + TOP_K * 8), "flops": case["tokens"] * EXPERTS * 4.0}
    n, one = case["tokens"], _layer(case["tokens"])
    h = one["hidden"]
    layer = work(one)
    matrices = h // 32 * (h + EXPERTS) * 18
    return {"bytes": case["layers"] * (layer["bytes"] + matrices + n * (h + EXPERTS) * 8.0),
            "flops": case["layers"] * (layer["flops"] + 2.0 * h * (h + EXPERTS) * n)}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times the distance from `exact` that the paths show.  Linear and
# router outputs are plain float32 sums (1e-7 measured).  A layer rounds its
# middle to Q8 codes: where a float32 sum in any order and the float64 sum fall
# on different sides of a rounding boundary, one code of 512 or 640 changes
# and its token moves by about 1e-2 rms; a batch holds a few such codes (8e-8
# without one, 7e-5 to 2.7e-4 with; the pipeline's router input is quantised
# likewise).
TOLERANCE = {"layer": {"rel": 1e-3}, "linear": {"rel": 5e-7}, "router": {"rel": 3e-7}, "pipeline": {"rel": 1e-3}}


# ----------------------------------------------------------------- exact ---
def _q8(x):
    """float rows -> (codes, half d, half s) of their Q8_1 blocks, float64."""
    b = x.float().view(x.shape[0], -1, 32)
    d = b.abs().amax(dim=2) / 127.0
    v = (b / torch.where(d > 0, d, 1.0)[..., None]).double()
    codes = torch.sign(v) * torch.floor(v.abs() + 0.5)
    s = b
    while s.shape[2] > 1:
        s = s[..., 0::2] + s[..., 1::2]
    return codes, d.half().double(), s[..., 0].half().double()


def _unpack(blocks, rows, type_):
    """Canonical blocks -> (q [rows][nb][32], d, m) float64."""
    b = blocks.reshape(rows, -1, BLOCK[type_])
    field = lambda o: b[:, :, o:o + 2].contiguous().view(torch.float16)[..., 0].double()  # noqa: E731
    c = b[:, :, BLOCK[type_] - 16:]
    q = torch.cat([c & 15, c >> 4], dim=2).double()
    return q, field(0), field(2) if type_ == Q4_1 else None


def _project(blocks, rows, type_, q8):
    """One matrix over Q8_1 rows: [columns][rows] float64."""
    codes, d8, s8 = q8
    q, d, m = _unpack(blocks, rows, type_)
    n = codes.shape[0]
    if type_ == Q4_0:
        return (codes * d8[..., None]).view(n, -1) @ (q * d[..., None]).view(rows, -1).T - 8.0 * (s8 @ d.T)
    y = torch.zeros((n, rows), dtype=torch.float64, device=codes.device)
    for b in range(q.shape[1]):   # the format rounds both block products to fp16
        dd = (d8[:, b, None] * d[None, :, b]).float().half().double()
        y += dd * (codes[:, b] @ q[:, b].T) + (s8[:, b, None] * m[None, :, b]).float().half().double()
    return y


def _expert(blob, c, q8):
    n = c["hidden"] // 32 * c["intermediate"] * 18
    g = _project(blob[:n], c["intermediate"], Q4_0, q8)
    u = _project(blob[n:2 * n], c["intermediate"], Q4_0, q8)
    return _project(blob[2 * n:], c["hidden"], Q4_1 if c["q41"] else Q4_0, _q8(g / (1.0 + torch.exp(-g)) * u))


def _layer_exact(c, bank, shared, x, ids, weights, gate):
    n = x.shape[0]
    q8 = _q8(x)
    y = torch.zeros((n, c["hidden"]), dtype=torch.float64, device=x.device)
    flat = ids.reshape(-1).long()
    order = torch.argsort(flat)
    counts = torch.bincount(flat, minlength=EXPERTS).tolist()
    at = 0
    for e in range(EXPERTS):
        if not counts[e]:
            continue
        pairs = order[at:at + counts[e]]
        at += counts[e]
        t = pairs // TOP_K
        out = _expert(bank[e], c, tuple(v[t] for v in q8))
        y.index_add_(0, t, out * weights.reshape(-1)[pairs].double()[:, None])
    scale = 1.0 if gate is None else torch.sigmoid(gate.double())[:, None]
    return y + scale * _expert(shared[0], c, q8)


def _flag():
    return torch.zeros(1, dtype=torch.int32)


def _select(logits):
    p = torch.softmax(logits.double(), dim=1)
    w, ids = torch.sort(p, dim=1, descending=True, stable=True)
    w, ids = w[:, :TOP_K], ids[:, :TOP_K].to(torch.int32)
    return ids, w / w.sum(dim=1, keepdim=True).clamp_min(1.0 / 16384)


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        bank, shared = _layer_bank(case, seed)
        return _layer_exact(case, bank, shared, *_layer_inputs(case, seed)), _flag()
    if kind == "linear":
        w, x = _linear_inputs(case, seed)
        y = _project(w, case["output"], Q4_1 if case["q41"] else Q4_0, _q8(x))
        return y if case["q8"] else (y, _flag())
    if kind == "router":
        logits = torch.randn((case["tokens"], EXPERTS), generator=_generator(seed, 4), device="cuda") * 2.0
        return (*_select(logits), _flag())
    out = []
    for l in range(case["layers"]):
        p = _pipeline_part(case, seed, l)
        h = _project(p["proj"], p["shape"]["hidden"], Q4_0, _q8(p["x"]))
        logits = _project(p["router"], EXPERTS, Q4_0, _q8(h))
        ids, w = _select(logits)
        out.append({"h": h, "logits": logits, "ids": ids,
                    "y": _layer_exact(p["shape"], p["bank"], p["shared"], h, ids, w, None)})
    return out
