"""What a program spends its time on in this framework: MoE layer calls from one decoded token to a
long prefill, single EXL3 linears from one row to thousands, the router and the weight decode, each
through its public entry point, with the sizes of the benchmark's configurations and of the runners'
default checkpoint, and a generator of further cases over the same ranges.

Kinds of case:

- ``moe``      ``ops.moe_forward`` on a ``MoeWorkspace``: one eager call, or a hipGraph of a few
               stacked layers updating a bf16 residual stream, as a decode loop keeps it;
- ``runner``   ``CoopRunner3072.run`` with given routes;
- ``chain``    a hipGraph of alternating up and down ``ELinear`` calls (a decode step's dense layers);
- ``linear``   one eager ``ELinear`` call;
- ``route``    ``ops.route``: the gate product and the top-k of a batch;
- ``dequant``  ``ops.exl3_dequant`` of one projection.
"""
from __future__ import annotations

import functools
import math

import torch

from eva_amd import ops, verification
from eva_amd.coop import CoopRunner3072
from eva_amd.linear import build_linear

LIMIT = 10.0                 # SwiGLU limit
CHAIN_PAIRS = 8              # up/down pairs of a chain
STACK_DOWN = 0.25            # scale of a stack's down projections: its residual stream stays O(1)
RATES = (1.5, 2.0, 2.5, 3.0, 3.5, 4.0, 5.0)


def _moe(name, rows, bits, **kw):
    case = {"name": name, "kind": "moe", "rows": rows, "bits": float(bits), "mixed": False, "hidden": 7168,
            "inter": 2048, "experts": 256, "topk": 8, "shared": True, "gated": False, "routing": "normal",
            "layers": 1, "graph": False}
    case.update(kw)
    return case


def listed():
    return [
        # one token of a decode loop: four resident layers in one graph, routed from logits (the
        # layers' weights together exceed the caches, as a model's do)
        _moe("decode_1", 1, 4, layers=4, graph=True),
        # a speculative verification batch at the default bound: every row keeps its one-row bits
        _moe("verify_8", 8, 2.5, layers=2, graph=True),
        # a decode batch past the bound with hot experts that every token picks
        _moe("batch_16", 16, 4, layers=2, graph=True, routing="skewed"),
        # a serving batch of mixed sequences, routed by the router weight in the same call, the
        # shared expert gated
        _moe("batch_100", 100, 3, routing="gate", gated=True),
        # a prefill chunk: Zipf expert loads, a rate of its own for each expert
        _moe("prefill_512", 512, 4, mixed=True, routing="gate_zipf"),
        # a long prefill with a ragged number of tokens
        _moe("prefill_3001", 3001, 4),
        # the capacity runner at its default checkpoint's shape, routes given
        {"name": "runner_333", "kind": "runner", "rows": 333, "bits": 3.0, "hidden": 5120, "inter": 2304, "experts": 384,
         "topk": 6},
        # a decode step's dense linears at one token: launches and latency
        {"name": "chain_1", "kind": "chain", "rows": 1, "bits": 4.0, "in": 2048, "out": 7168},
        # the same for an odd-sized batch of tokens
        {"name": "chain_13", "kind": "chain", "rows": 13, "bits": 4.0, "in": 2048, "out": 7168},
        # a dense linear on a short prompt, at a half-integer rate
        {"name": "linear_200", "kind": "linear", "rows": 200, "bits": 3.5, "in": 7168, "out": 2048},
        # a dense linear on a long prompt
        {"name": "linear_8192", "kind": "linear", "rows": 8192, "bits": 4.0, "in": 2048, "out": 7168},
        # decoding one projection to fp16, at a half-integer rate
        {"name": "dequant", "kind": "dequant", "bits": 2.5, "in": 7168, "out": 2048},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "runner", "chain", "linear", "linear", "route", "dequant"])
    bits = rng.choice(RATES)
    if kind in ("moe", "runner"):
        hidden, inter, experts, topk = rng.choice([(7168, 2048, 256, 8), (5120, 2304, 384, 6), (4096, 1536, 128, 8),
                                                   (2048, 768, 64, 6), (1024, 512, 16, 4), (640, 384, 40, 3)])
        rows = _log_int(rng, 1, 512 if kind == "runner" else 3000)
        if kind == "runner":
            return {"kind": kind, "rows": rows, "bits": bits, "hidden": hidden, "inter": inter, "experts": experts, "topk": topk}
        graph = rows <= 16 and rng.random() < 0.7
        shared = rng.random() < 0.8
        return {"kind": kind, "rows": rows, "bits": bits, "mixed": rng.random() < 0.3, "hidden": hidden, "inter": inter,
                "experts": experts, "topk": topk, "shared": shared, "gated": shared and rng.random() < 0.3,
                "routing": rng.choice(["normal", "skewed", "zipf"] if graph else ["normal", "skewed", "zipf", "gate", "gate_zipf"]),
                "layers": 2 if graph else 1, "graph": graph}
    if kind == "route":
        return {"kind": kind, "rows": _log_int(rng, 1, 8192), "hidden": 128 * rng.randint(8, 56),
                "experts": rng.choice([64, 128, 160, 256, 384]), "topk": rng.choice([4, 6, 8]),
                "score": rng.choice(["sigmoid", "sqrt_softplus"])}
    a, b = 128 * _log_int(rng, 4, 56), 128 * _log_int(rng, 4, 56)
    if kind == "chain":
        return {"kind": kind, "rows": rng.randint(1, 16), "bits": bits, "in": a, "out": b}
    if kind == "linear":
        return {"kind": kind, "rows": _log_int(rng, 1, 4096), "bits": bits, "in": a, "out": b}
    return {"kind": "dequant", "bits": rng.choice(RATES + (1.0, 6.0, 8.0)), "in": a, "out": b}


# ---- inputs -----------------------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _tile(bits):
    return int(round(16 * bits))


def _codes(g, n):
    t = torch.empty(n, dtype=torch.int16, device="cuda")
    for s in range(0, n, 1 << 28):
        t[s:s + (1 << 28)].random_(-32768, 32768, generator=g)
    return t


def _signs(g, *shape):
    return (torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1).half()


def _scales(g, *shape, scale=1.0):
    mag = (torch.rand(shape, generator=g, device="cuda") + 0.5) * scale
    return (mag * (torch.randint(0, 2, shape, generator=g, device="cuda") * 2 - 1)).half()


def _projection(g, n_in, n_out, bits):
    t = _codes(g, (n_in // 16) * (n_out // 16) * _tile(bits)).view(n_in // 16, n_out // 16, _tile(bits))
    return t, _signs(g, n_in), _scales(g, n_out, scale=n_in ** -0.5)


class _Layer:
    """One MoE layer's experts (the shared one last): packed weights, scales and pointer tables."""

    def __init__(self, g, hidden, inter, experts, bits, mixed, shared, down):
        n = experts + (1 if shared else 0)
        self.rates = [bits] * n
        if mixed:
            pick = torch.randint(0, 4, (n,), generator=g, device="cuda").tolist()
            self.rates = [(2.0, 3.0, 4.0, 5.0)[i] for i in pick]
        tiles = (hidden // 16) * (inter // 16)
        self.hidden, self.inter, self.tiles = hidden, inter, tiles
        self.offs, total = [], 0
        for r in self.rates:
            self.offs.append(total)
            total += 3 * tiles * _tile(r)
        self.codes = _codes(g, total)
        vec = max(hidden, inter)
        self.suh = _signs(g, n, 3, vec)
        self.svh = _scales(g, n, 3, vec, scale=hidden ** -0.5)
        self.svh[:, 2] *= down
        rows = []
        for e in range(n):
            step = 2 * tiles * _tile(self.rates[e])
            rows.append([v for p in range(3) for v in (self.codes.data_ptr() + 2 * self.offs[e] + p * step,
                                                       self.suh[e, p].data_ptr(), self.svh[e, p].data_ptr())])
        self.shared = rows[experts] if shared else None
        self.table = torch.tensor(rows[:experts], dtype=torch.int64).t().contiguous().cuda()
        self.k2 = torch.tensor([int(2 * r) for r in self.rates[:experts]], dtype=torch.uint8).cuda() if mixed else None

    def parts(self, e, p):
        """Codes, suh and svh of projection p (gate, up, down) of expert e."""
        n_in, n_out = (self.inter, self.hidden) if p == 2 else (self.hidden, self.inter)
        size = self.tiles * _tile(self.rates[e])
        codes = self.codes[self.offs[e] + p * size:][:size]
        return codes.view(n_in // 16, n_out // 16, _tile(self.rates[e])), self.suh[e, p, :n_in], self.svh[e, p, :n_out]


def _zipf_log(g, experts):
    lp = -1.1 * torch.log(torch.arange(1, experts + 1, dtype=torch.float64, device="cuda"))
    return lp[torch.randperm(experts, generator=g, device="cuda")]


def _logits(g, rows, experts, routing):
    z = torch.randn(rows, experts, generator=g, device="cuda")
    if routing == "skewed":      # two experts that every token picks, six that about half do
        order = torch.randperm(experts, generator=g, device="cuda")
        z[:, order[:2]] += 6.0
        z[:, order[2:8]] += 3.0 * torch.randint(0, 2, (rows, order[2:8].numel()), generator=g, device="cuda")
    elif routing == "zipf":      # picks without replacement, Zipf(1.1) over the experts
        u = torch.rand(rows, experts, generator=g, device="cuda", dtype=torch.float64).clamp_(1e-300, 1.0)
        z = (_zipf_log(g, experts) - torch.log(-torch.log(u))).float()
    return z


def _moe_inputs(case, seed):
    g = _gen(seed)
    rows, hidden, experts = case["rows"], case["hidden"], case["experts"]
    layers = [_Layer(g, hidden, case["inter"], experts, case["bits"], case["mixed"], case["shared"],
                     STACK_DOWN if case["graph"] else 1.0) for _ in range(case["layers"])]
    s = {"layers": layers, "x": torch.randn(rows, hidden, generator=g, device="cuda").bfloat16()}
    s["gated"] = (torch.randn(hidden, generator=g, device="cuda") * hidden ** -0.5).half() if case["gated"] else None
    if case["routing"].startswith("gate"):
        s["gate_w"] = torch.randn(experts, hidden, generator=g, device="cuda") * hidden ** -0.5
        s["bias"] = (0.16 * _zipf_log(g, experts)).float() if case["routing"] == "gate_zipf" else None
    else:
        s["logits"] = [_logits(g, rows, experts, case["routing"]) for _ in layers]
    return s


def _moe_args(case, s, l):
    """Keyword arguments of layer l's call."""
    layer = s["layers"][l]
    kw = {"limit": LIMIT, "sel": s["sel"][l], "weights": s["weights"][l], "shared_gate_w": s["gated"]}
    kw.update({"k2_per_expert": layer.k2} if case["mixed"] else {"bits": case["bits"]})
    kw.update({"gate_w": s["gate_w"], "sel_bias": s["bias"]} if "gate_w" in s else {"logits": s["logits"][l]})
    if case["shared"]:
        kw.update(shared_ptrs=layer.shared, shared_bits=layer.rates[-1])
    return kw


def _prepare_moe(case, seed):
    s = _moe_inputs(case, seed)
    rows, topk = case["rows"], case["topk"]
    ws = ops.MoeWorkspace("cuda:0", rows_max=rows, hidden=case["hidden"], inter=case["inter"], topk=topk,
                          n_local=case["experts"], has_shared=case["shared"],
                          strict_rows=verification.moe_strict_rows(rows, topk))
    s["ws"], n = ws, case["layers"]
    s["sel"] = torch.empty(n, rows, topk, dtype=torch.int64, device="cuda")
    s["weights"] = torch.empty(n, rows, topk, dtype=torch.float32, device="cuda")
    if not case["graph"]:
        s["out"] = torch.empty(rows, case["hidden"], dtype=torch.float32, device="cuda")
        s["kw"] = _moe_args(case, s, 0)
        return s
    s["h"] = torch.empty_like(s["x"])
    s["graph"] = _capture(lambda: _step(case, s))
    return s


def _step(case, s):
    torch.mul(s["x"], 1.0, out=s["h"])          # the step's residual stream
    for l, layer in enumerate(s["layers"]):
        ops.moe_forward(s["ws"], s["h"], layer.table, None, residual=s["h"], **_moe_args(case, s, l))


def _capture(step):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _runner_inputs(case, seed):
    g = _gen(seed)
    layer = _Layer(g, case["hidden"], case["inter"], case["experts"], case["bits"], False, False, 1.0)
    x = torch.randn(case["rows"], case["hidden"], generator=g, device="cuda").bfloat16()
    sel = _logits(g, case["rows"], case["experts"], "zipf").topk(case["topk"], dim=1).indices
    w = torch.rand(case["rows"], case["topk"], generator=g, device="cuda") + 0.1
    return {"layer": layer, "x": x, "sel": sel.contiguous(), "w": w / w.sum(1, keepdim=True)}


def _chain_inputs(case, seed):
    g = _gen(seed)
    parts = [_projection(g, *((case["in"], case["out"]) if i % 2 == 0 else (case["out"], case["in"])), case["bits"])
             for i in range(2 * CHAIN_PAIRS)]
    return {"parts": parts, "x": torch.randn(case["rows"], case["in"], generator=g, device="cuda").half()}


def _linear_inputs(case, seed):
    g = _gen(seed)
    return {"parts": _projection(g, case["in"], case["out"], case["bits"]),
            "x": torch.randn(case["rows"], case["in"], generator=g, device="cuda").half()}


def _route_inputs(case, seed):
    g = _gen(seed)
    return {"x": torch.randn(case["rows"], case["hidden"], generator=g, device="cuda").bfloat16(),
            "gate_w": torch.randn(case["experts"], case["hidden"], generator=g, device="cuda") * case["hidden"] ** -0.5,
            "bias": 0.1 * torch.randn(case["experts"], generator=g, device="cuda")}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "moe":
        s = _prepare_moe(case, seed)
    elif kind == "runner":
        s = _runner_inputs(case, seed)
        s["runner"] = CoopRunner3072("cuda:0", topk=case["topk"], hidden=case["hidden"], inter=case["inter"])
        s["k"] = case["bits"]
    elif kind == "chain":
        s = _chain_inputs(case, seed)
        s["mods"] = [build_linear(su, sv, t) for t, su, sv in s["parts"]]

        def step():
            y = s["x"]
            s["y"] = [y := m(y) for m in s["mods"]][-2:]

        s["graph"] = _capture(step)
    elif kind == "linear":
        s = _linear_inputs(case, seed)
        t, su, sv = s["parts"]
        s["mod"] = build_linear(su, sv, t)
    elif kind == "route":
        s = _route_inputs(case, seed)
        s.update(topk=case["topk"], score=case["score"])
    else:
        s = {"codes": _projection(_gen(seed), case["in"], case["out"], case["bits"])[0], "bits": case["bits"]}
    s["kind"] = kind
    return s


def run(s):
    kind = s["kind"]
    if kind == "moe":
        if "graph" in s:
            s["graph"].replay()
            return {"h": s["h"], "sel": s["sel"], "weights": s["weights"]}
        ops.moe_forward(s["ws"], s["x"], s["layers"][0].table, s["out"], **s["kw"])
        return {"out": s["out"], "sel": s["sel"], "weights": s["weights"]}
    if kind == "runner":
        return s["runner"].run(s["x"], s["sel"], s["w"], s["layer"].table, s["k"], LIMIT, check_bounds=False)
    if kind == "chain":
        s["graph"].replay()
        return s["y"]
    if kind == "linear":
        return s["mod"](s["x"])
    if kind == "route":
        return ops.route(s["x"], s["gate_w"], s["bias"], s["topk"], score_fn=s["score"])
    return ops.exl3_dequant(s["codes"], s["bits"])


# ---- what a pass cannot do without --------------------------------------------------------------


def _projection_bytes(n_in, n_out, bits):
    return n_in * n_out * bits / 8 + 2 * (n_in + n_out)


@functools.lru_cache(maxsize=None)
def _touched(rows, experts, topk, routing):
    """Experts that at least one of the rows picks, as one draw of this routing has it."""
    g = torch.Generator()
    g.manual_seed(1)
    z = torch.randn(rows, experts, generator=g)
    if routing == "skewed":
        z[:, :2] += 6.0
        z[:, 2:8] += 3.0 * torch.randint(0, 2, (rows, min(6, experts - 2)), generator=g)
    elif "zipf" in routing:
        z = -1.1 * torch.log(torch.arange(1, experts + 1.0)) - torch.log(-torch.log(torch.rand(rows, experts, generator=g)))
    return int(z.topk(topk, dim=1).indices.unique().numel())


def work(case):
    kind = case["kind"]
    if kind in ("moe", "runner"):
        h, i, rows, shared = case["hidden"], case["inter"], case["rows"], int(case.get("shared", False))
        bits = 3.5 if case.get("mixed") else case["bits"]
        n = _touched(rows, case["experts"], case["topk"], case.get("routing", "zipf")) + shared
        b = n * (2 * _projection_bytes(h, i, bits) + _projection_bytes(i, h, bits))
        b += rows * (2 * h + (2 if case.get("graph") else 4) * h + 4 * case["experts"] + 12 * case["topk"])
        f = 6.0 * rows * (case["topk"] + shared) * h * i
        if case.get("routing", "").startswith("gate"):
            b += 4 * h * case["experts"]
            f += 2.0 * rows * h * case["experts"]
        return {"bytes": b * case.get("layers", 1), "flops": f * case.get("layers", 1)}
    if kind == "route":
        return {"bytes": 2 * case["rows"] * case["hidden"] + 4 * case["experts"] * case["hidden"] + 12 * case["rows"] * case["topk"],
                "flops": 2.0 * case["rows"] * case["hidden"] * case["experts"]}
    a, b = case["in"], case["out"]
    if kind == "dequant":
        return {"bytes": a * b * (case["bits"] / 8 + 2), "flops": 0}
    n = 2 * CHAIN_PAIRS if kind == "chain" else 1
    return {"bytes": n * (_projection_bytes(a, b, case["bits"]) + 2 * case["rows"] * (a + b)),
            "flops": 2.0 * n * case["rows"] * a * b}


def tolerance(case):
    """About four times what the same rounding points show with the sums in another order: strict
    against automatic splits for the MoE, the one- to sixteen-row against the larger path for the
    linears (relative 5e-4 and 9e-5, 1.3e-3 over a stack's bf16 stream, 2.1e-3 over a chain's sixteen
    fp16 layers), another fp32 product for the router, where a near tie may go the other way."""
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "route":
        return {"rel": 1.5e-5, "max": 1.6e-3, "differ": 5e-4}
    if kind == "linear":
        return {"rel": 4e-4, "max": 1e-2}
    if kind == "chain":
        return {"rel": 8e-3, "max": 6e-2}
    return {"rel": 5e-3 if case.get("graph") else 2e-3, "max": 6e-2 if case.get("graph") else 3e-2, "differ": 1e-3}


# ---- the same results in 64 bits ----------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def _codebook():
    """The value of each 16-bit state: fp16(k * (1024 + sum of the bytes of state * 0x83DCD12D) + b)."""
    p = (torch.arange(65536, dtype=torch.int64) * 0x83DCD12D) & 0xFFFFFFFF
    total = sum((p >> (8 * i)) & 0xFF for i in range(4)) + 1024
    return (total.double() * 0.00676727294921875 - 10.3828125).half().double().cuda()


@functools.lru_cache(maxsize=None)
def _windows(bits):
    """For each of a tile's 256 codes: the two words its 16-bit window lies in, its shift, and its row and column."""
    words = int(8 * bits)
    p = torch.arange(256)
    if bits == int(bits):
        end = (p + 1) * int(bits)
    else:
        b = int(bits)
        end = torch.where(p % 2 == 1, (p + 1) // 2 * (2 * b + 1), p // 2 * (2 * b + 1) + b)
    end = end + 32 * words
    lo = (end - 1) // 32
    lane, j = p >> 3, p & 7
    k = 2 * (lane & 3) + (j & 1) + 8 * ((j >> 1) & 1)
    n = (lane >> 2) + 8 * (j >> 2)
    order = torch.argsort(16 * k + n)                  # codes in row-major order of the tile
    return [t[order].cuda() for t in (((end - 16) // 32) % words, lo % words, 32 * (lo + 1) - end)]


def _decode(codes):
    kt, nt, t16 = codes.shape
    words = (codes.view(torch.int32).long() & 0xFFFFFFFF)
    hi, lo, shift = _windows(t16 / 16)
    state = ((words[..., hi] << (32 - shift)) | (words[..., lo] >> shift)) & 0xFFFF
    return _codebook()[state].view(kt, nt, 16, 16).transpose(1, 2).reshape(16 * kt, 16 * nt)


@functools.lru_cache(maxsize=None)
def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (h / math.sqrt(128.0)).cuda()


def _rotate(x):
    return (x.reshape(-1, 128) @ _hadamard()).view(x.shape)


def _linear(x, codes, suh, svh):
    return _rotate(_rotate(x * suh.double()) @ _decode(codes)) * svh.double()


def _expert(x, layer, e, shared):
    g = _linear(x, *layer.parts(e, 0))
    u = _linear(x, *layer.parts(e, 1)).clamp(-LIMIT, LIMIT)
    g = torch.nn.functional.silu(g.clamp(max=LIMIT)) if shared else torch.nn.functional.silu(g).clamp(max=LIMIT)
    return _linear(g * u, *layer.parts(e, 2))


def _routes(z, bias, topk, score):
    s = torch.sigmoid(z) if score == "sigmoid" else torch.nn.functional.softplus(z).sqrt()
    key = z if bias is None and score == "sigmoid" else s if bias is None else s + bias.double()
    idx = key.sort(dim=1, descending=True, stable=True).indices[:, :topk]
    w = s.gather(1, idx)
    return idx, w / w.sum(1, keepdim=True)


def _routed(x, layer, idx, w):
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        r, k = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, r, w[r, k, None] * _expert(x[r], layer, e, False))
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        s = _moe_inputs(case, seed)
        h, ws = s["x"].double(), []
        for l, layer in enumerate(s["layers"]):
            x = h.half().double()
            z = x @ s["gate_w"].double().t() if "gate_w" in s else s["logits"][l].double()
            idx, w = _routes(z, s.get("bias"), case["topk"], "sigmoid")
            y = _routed(x, layer, idx, w)
            if case["shared"]:
                sh = _expert(x, layer, case["experts"], True)
                y += sh if s["gated"] is None else torch.sigmoid(x @ s["gated"].double())[:, None] * sh
            ws.append(w)
            h = h + y
        return {"h" if case["graph"] else "out": h if case["graph"] else y, "sel": None, "weights": torch.stack(ws)}
    if kind == "runner":
        s = _runner_inputs(case, seed)
        return _routed(s["x"].double(), s["layer"], s["sel"], s["w"].double())
    if kind == "chain":
        s = _chain_inputs(case, seed)
        ys = [s["x"].double()]
        for t, su, sv in s["parts"]:
            ys.append(_linear(ys[-1], t, su, sv))
        return ys[-2:]
    if kind == "linear":
        s = _linear_inputs(case, seed)
        return _linear(s["x"].double(), *s["parts"])
    if kind == "route":
        s = _route_inputs(case, seed)
        return _routes(s["x"].double() @ s["gate_w"].double().t(), s["bias"], case["topk"], case["score"])[1], None
    return _decode(_projection(_gen(seed), case["in"], case["out"], case["bits"])[0])
