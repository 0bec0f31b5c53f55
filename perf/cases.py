"""What a user of this framework has it compute, as cases that can be timed.

The user is a server of a hybrid MoE model whose linears, hyper-connection
mixers, router gates and heads are the packed-weight products of
fp4x_kernels.  It captures its decode step into graphs, one per batch size, so
a decoder layer's linears and a step's int8 work are captured here and a pass
replays the capture; single calls, the heads and the weight preparation run
eagerly, as the plugin runs them.

A case is a dict with a "kind":

  linear  one eager call of a packed linear
  layer   the linears of `layers` decoder layers, one graph replay: attention
          qkv, its small gate projection, attention output, shared expert up
          and down, router gate; `fmt` is the served format (lowbit: NVFP4 qkv,
          W6 elsewhere; mx8; w8)
  step    a step's int8 work, one graph replay: every router gate as one
          layer-batched call, then `mixers` hyper-connection mixers
  head    the target LM head: INT2 coarse logits, their top C, exact MXFP8
          rescore in place
  draft   the draft head over a token subset: INT2 coarse, top C, exact NVFP4
          rescore scattered into the full vocabulary
  prep    load-time weight preparation of one matrix
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "qwen3.8-flash-next-fp4-local-spark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import fp4patch  # noqa: E402
import fp4x_kernels as F  # noqa: E402

DEV = "cuda:0"
_SERVED = {"hidden": 2560, "qkv": 16384, "attn": 6144, "inter": 640, "experts": 512}


def listed():
    return [
        # one router gate for one token, outside any graph: launch latency
        {"name": "gate_one_row", "kind": "linear", "fmt": "w8", "m": 1, "n": 512, "k": 2560, "out": "f32"},
        # one sequence without drafting, the plugin's default dense mode
        {"name": "layer_mx8_m1", "kind": "layer", "fmt": "mx8", "m": 1, "layers": 6, **_SERVED, "gate": "w8"},
        # one sequence with two draft rows in the shipped low-bit mode: the tuned shape
        {"name": "layer_lowbit_m3", "kind": "layer", "fmt": "lowbit", "m": 3, "layers": 6, **_SERVED, "gate": "w8"},
        # the widest single launch, full-attention qkv
        {"name": "layer_mx8_m16", "kind": "layer", "fmt": "mx8", "m": 16, "layers": 6,
         **{**_SERVED, "qkv": 13312}, "gate": "bf16"},
        # eight sequences of the int8 draft layer with two draft rows each
        {"name": "layer_w8_m24", "kind": "layer", "fmt": "w8", "m": 24, "layers": 6,
         **{**_SERVED, "qkv": 13312}, "gate": "w8"},
        # thirteen sequences with two draft rows each
        {"name": "layer_lowbit_m39", "kind": "layer", "fmt": "lowbit", "m": 39, "layers": 6, **_SERVED, "gate": "w8"},
        # a full batch, or a prefill chunk
        {"name": "layer_mx8_m256", "kind": "layer", "fmt": "mx8", "m": 256, "layers": 6, **_SERVED, "gate": "w8"},
        # all 48 router gates and 20 mixers at the served shape
        {"name": "step_int8_m3", "kind": "step", "m": 3, "hidden": 2560, "experts": 512, "gates": 48, "lr": 320,
         "mixers": 20, "scales": "f32"},
        # the target head of one sequence with two draft rows
        {"name": "head_m3", "kind": "head", "m": 3, "v": 248320, "k": 2560, "c": 512, "g": 16},
        # the draft head over its token subset
        {"name": "draft_m2", "kind": "draft", "m": 2, "v": 248320, "subset": 65197, "k": 2560, "c": 64},
        # a layer's NVFP4 copy and the head's INT2 copy, made when the model is loaded
        {"name": "prep_nv4", "kind": "prep", "src": "mx8", "to": "nv4", "n": 16384, "k": 2560},
        {"name": "prep_head_int2", "kind": "prep", "src": "mx8", "to": "int2", "n": 248320, "k": 2560},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("linear", "layer", "step", "head", "draft", "prep"), (4, 6, 2, 2, 2, 3))[0]
    hidden = 64 * rng.randint(16, 44)
    if kind == "linear":
        return {"kind": kind, "fmt": rng.choice(("mx8", "w8", "w6", "nv4", "bf16")), "m": _log(rng, 1, 256),
                "n": _log(rng, 64, 20000), "k": 64 * rng.randint(8, 96), "out": rng.choice(("bf16", "f32"))}
    if kind == "layer":
        return {"kind": kind, "fmt": rng.choice(("lowbit", "mx8", "w8")), "m": _log(rng, 1, 256),
                "layers": rng.randint(2, 6), "hidden": hidden, "qkv": _log(rng, 1500, 16000),
                "attn": 64 * rng.randint(16, 96), "inter": 64 * rng.randint(4, 16),
                "experts": rng.choice((64, 128, 256, 512)), "gate": rng.choice(("w8", "bf16"))}
    if kind == "step":
        return {"kind": kind, "m": rng.randint(1, 16), "hidden": hidden, "experts": rng.choice((128, 256, 512)),
                "gates": rng.randint(8, 48), "lr": 64 * rng.randint(3, 10), "mixers": rng.randint(4, 20),
                "scales": rng.choice(("f32", "f16"))}
    if kind == "head":
        return {"kind": kind, "m": rng.randint(1, 16), "v": _log(rng, 30000, 248320), "k": hidden,
                "c": rng.choice((128, 256, 512, 1024)), "g": rng.choice((16, 32))}
    if kind == "draft":
        v = _log(rng, 60000, 248320)
        return {"kind": kind, "m": rng.randint(1, 16), "v": v, "subset": _log(rng, 8000, v // 2), "k": hidden,
                "c": rng.choice((32, 64, 128))}
    return {"kind": kind, "src": rng.choice(("mx8", "bf16")), "to": rng.choice(("w8", "w6", "nv4", "int2", "f32")),
            "n": _log(rng, 300, 20000), "k": hidden}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _x(g, *shape):
    return torch.randn(shape, generator=g, device=DEV).to(torch.bfloat16)


def _planes(fmt, n, k, g):
    """A packed [n, k] weight of about N(0, 0.02) in the format's own layout."""
    def normal(std):
        return torch.randn((n, k), generator=g, device=DEV) * std

    def near(cols, mean):
        return mean * (0.75 + 0.5 * torch.rand((n, cols), generator=g, device=DEV))

    if fmt == "bf16":
        return (normal(0.02).to(torch.bfloat16),)
    if fmt == "mx8":
        codes = normal(100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
        return codes, torch.randint(113, 116, (n, k // 32), generator=g, device=DEV, dtype=torch.uint8)
    if fmt in ("w8", "w8_f16"):
        q = normal(42.0).round_().clamp_(-127, 127).to(torch.int8)
        s = near(k // 64, 0.02 / 42)
        return q, s.half() if fmt == "w8_f16" else s
    if fmt == "w6":
        c = normal(12.0).round_().clamp_(-32, 31).to(torch.int32) + 32
        lo, hi = c & 15, c >> 4
        L = (lo[:, 0::2] | (lo[:, 1::2] << 4)).to(torch.uint8)
        H = (hi[:, 0::4] | (hi[:, 2::4] << 2) | (hi[:, 1::4] << 4) | (hi[:, 3::4] << 6)).to(torch.uint8)
        return L, H, near(k // 32, 0.02 / 12).half()
    v = normal(2.4)
    mids = torch.tensor([.25, .75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    c = torch.bucketize(v.abs(), mids, out_int32=True) | ((v < 0).to(torch.int32) << 3)
    P = (c[:, 0::2] | (c[:, 1::2] << 4)).to(torch.uint8)
    return P, near(k // 16, 8.0).to(torch.float8_e4m3fn), 0.02 / 2.4 / 8.0


def _call(fmt, x, planes, out=torch.bfloat16):
    """The linear as the plugin calls it: its tile table's entry, else one K slice."""
    tables = {"mx8": fp4patch.CFG_MX8, "w6": fp4patch.CFG_W6, "w8": fp4patch.CFG_W8, "bf16": fp4patch.CFG_BG}
    n, k = planes[0].shape[0], x.shape[1]
    if fmt == "nv4":
        return F.nv4_linear(x, *planes, (32, 64, 4), out)
    cfg = tables[fmt].get((n, k)) or (32, 64, 1, 4)
    fn = {"mx8": F.mx8_linear, "w6": F.w6_linear, "w8": F.w8_linear, "bf16": F.bf16_linear}[fmt]
    return fn(x, *planes, cfg, out)


def _layer_shapes(c):
    """(input, fmt, n, k) of one decoder layer's linears."""
    low = {"lowbit": "w6"}.get(c["fmt"], c["fmt"])
    h = c["hidden"]
    return [("h", "nv4" if c["fmt"] == "lowbit" else low, c["qkv"], h), ("h", low, 96, h), ("a", low, h, c["attn"]),
            ("h", low, 2 * c["inter"], h), ("i", low, h, c["inter"]), ("h", c["gate"], c["experts"], h)]


def _capture(fn):
    """fn's launches as a graph and its outputs, after one eager run."""
    fn()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return {"graph": graph, "out": out, "fn": fn}


def _inputs(c, seed):
    """Everything that the seed makes."""
    g, kind = _gen(seed), c["kind"]
    if kind == "linear":
        return {"x": _x(g, c["m"], c["k"]), "w": _planes(c["fmt"], c["n"], c["k"], g)}
    if kind == "layer":
        width = {"h": c["hidden"], "a": c["attn"], "i": c["inter"]}
        layers = []
        for _ in range(c["layers"]):
            x = {name: _x(g, c["m"], w) for name, w in width.items()}
            layers.append([(fmt, x[name], _planes(fmt, n, k, g)) for name, fmt, n, k in _layer_shapes(c)])
        return {"layers": layers}
    if kind == "step":
        h, fmt = c["hidden"], "w8" if c["scales"] == "f32" else "w8_f16"
        gates = [_planes(fmt, c["experts"], h, g) for _ in range(c["gates"])]
        d = {"gx": _x(g, c["gates"], c["m"], h), "gq": torch.stack([q for q, _ in gates]),
             "gs": torch.stack([s for _, s in gates]), "mixers": []}
        for _ in range(c["mixers"]):
            d["mixers"].append((_x(g, c["m"], 4 * h), _planes(fmt, c["lr"] + 16, 4 * h, g),
                                _planes(fmt, 4 * h, c["lr"], g)))
        return d
    if kind == "head":
        q, s = _planes("mx8", c["v"], c["k"], g)
        s[torch.randperm(c["v"], generator=g, device=DEV)[:64]] += 2      # a few frequent tokens' rows are larger
        return {"w": (q, s), "x": _x(g, c["m"], c["k"])}
    if kind == "draft":
        ids = torch.sort(torch.randperm(c["v"], generator=g, device=DEV)[:c["subset"]]).values
        return {"w": _planes("nv4", c["subset"], c["k"], g), "ids": ids, "x": _x(g, c["m"], c["k"])}
    return {"w": _planes(c["src"], c["n"], c["k"], g)}


# ------------------------------------------------------------------ the passes
def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "layer":
        return {"case": case, **_capture(lambda: [[_call(fmt, x, w) for fmt, x, w in layer] for layer in d["layers"]])}
    if kind == "step":
        lr = case["lr"]
        fx = F.HCFused(torch.device(DEV), n_down=max(336, lr + 16))
        mixers = [(x, *down, *F.HCFused.interleave_up(*up, 4, 8)) for x, down, up in d["mixers"]]

        def step():
            gates = F.w8_linear_layers(d["gx"], d["gq"], d["gs"], torch.float32)
            return [gates, [fx.mix(x, qd, sd, lr, 4, qi, si, x, fp4patch.HC_DOWN_CFG, fp4patch.HC_UP_CFG)
                            for x, qd, sd, qi, si in mixers]]
        return {"case": case, **_capture(step)}
    if kind == "head":
        d["coarse"] = F.requantize_mx8(*d["w"], "int2", group=case["g"])
    if kind == "draft":
        d["coarse"] = F.requantize_nv4(*d["w"], "int2", group=16)
    return {"case": case, **d}


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind in ("layer", "step"):
        state["graph"].replay()
        return state["out"]
    if kind == "linear":
        return _call(c["fmt"], state["x"], state["w"], torch.float32 if c["out"] == "f32" else torch.bfloat16)
    if kind == "head":
        coarse, idx = F.int2_topk(state["x"], *state["coarse"], c["v"], c["c"], sorted=False)
        return F.refine_mx8_(coarse, state["x"], idx, *state["w"])
    if kind == "draft":
        _, cand = F.int2_topk(state["x"], *state["coarse"], c["subset"], c["c"], out_dtype=torch.float32, sorted=False)
        return F.draft_nv4(state["x"], cand, *state["w"], state["ids"], c["v"])
    if c["to"] == "f32":
        return F.mx8_dequant(*state["w"]) if c["src"] == "mx8" else F.quantize_w8(*state["w"])
    if c["src"] == "mx8":
        return F.requantize_mx8(*state["w"], c["to"])
    return {"w8": F.quantize_w8, "w6": F.quantize_w6, "nv4": F.quantize_nv4, "int2": F.quantize_int2}[c["to"]](
        *state["w"])


# ------------------------------------------------------------------ what a pass needs
_BITS = {"bf16": 16, "mx8": 8 + 8 / 32, "w8": 8 + 32 / 64, "w8_f16": 8 + 16 / 64, "w6": 6 + 16 / 32,
         "nv4": 4 + 8 / 16, "f32": 32}


def _linear_work(fmt, m, n, k, out_bytes):
    return n * k * _BITS[fmt] / 8 + m * k * 2 + m * n * out_bytes, 2 * m * n * k


def work(case):
    c, kind = case, case["kind"]
    if kind == "linear":
        parts = [_linear_work(c["fmt"], c["m"], c["n"], c["k"], 4 if c["out"] == "f32" else 2)]
    elif kind == "layer":
        parts = [_linear_work(fmt, c["m"], n, k, 2) for _, fmt, n, k in _layer_shapes(c)] * c["layers"]
    elif kind == "step":
        fmt, h, lr = "w8" if c["scales"] == "f32" else "w8_f16", c["hidden"], c["lr"]
        parts = [_linear_work(fmt, c["m"], c["experts"], h, 4)] * c["gates"]
        down, up = _linear_work(fmt, c["m"], lr + 16, 4 * h, 2), _linear_work(fmt, c["m"], 4 * h, lr, 0)
        parts += [down, up, (c["m"] * h * 2, 0)] * c["mixers"]
    elif kind == "head":
        coarse = c["v"] * c["k"] * (2 + 16 / c["g"]) / 8 + c["m"] * c["k"] * 2 + c["m"] * c["v"] * 2
        parts = [(coarse, 2 * c["m"] * c["v"] * c["k"]),
                 (c["m"] * c["c"] * c["k"] * _BITS["mx8"] / 8, 2 * c["m"] * c["c"] * c["k"])]
    elif kind == "draft":
        coarse = c["subset"] * c["k"] * 3 / 8 + c["m"] * c["k"] * 2
        parts = [(coarse, 2 * c["m"] * c["subset"] * c["k"]),
                 (c["m"] * c["c"] * c["k"] * _BITS["nv4"] / 8 + c["m"] * c["v"] * 2, 2 * c["m"] * c["c"] * c["k"])]
    else:
        to = 3.0 if c["to"] == "int2" else _BITS["w8"] if c["to"] == "f32" and c["src"] == "bf16" else _BITS[c["to"]]
        parts = [(c["n"] * c["k"] * (_BITS[c["src"]] + to) / 8, c["n"] * c["k"])]
    return {"bytes": sum(b for b, _ in parts), "flops": sum(f for _, f in parts)}


def tolerance(case):
    """About four times what the kernels' two summation orders (their streaming
    and few-rows paths against their MFMA core) differ by."""
    kind = case["kind"]
    if kind == "prep":
        return "exact"                       # codes, scales and exact dequants
    if kind == "linear" and case["out"] == "f32":
        return {"rel": 1e-6, "max": 1e-5}    # fp32 sums of exact products: 1.7e-7, 6e-7
    if kind == "linear" or kind == "layer":
        return {"rel": 4e-4, "max": 0.03}    # some sums round to the neighbouring bf16 value: 1e-4, 0.0078
    if kind == "step":
        return {"rel": 1e-3, "max": 0.03}    # two products and bf16 epilogues in a row: a neighbour in the first
    return {"rel": 1e-3, "max": 0.5}         # as layer, and a tie in the coarse logits may swap a candidate


# ------------------------------------------------------------------ 64 bits
_E2M1 = (0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6)


def _dense(fmt, p):
    """The operand that the format defines, in 64 bits: scaled codes, rounded
    to bf16 where the format's product takes a bf16 operand."""
    def scaled(codes, s):
        n, k = codes.shape
        return (codes.float().view(n, s.shape[1], -1) * s.float().unsqueeze(-1)).view(n, k)

    if fmt == "bf16":
        return p[0].double()
    if fmt == "mx8":
        return scaled(p[0], torch.exp2(p[1].float() - 127)).double()
    if fmt in ("w8", "w8_f16"):
        return scaled(p[0], p[1]).to(torch.bfloat16).double()
    if fmt == "w6":
        L, H, s = p
        c = torch.stack([L & 15, L >> 4], -1).view(L.shape[0], -1)
        hi = torch.stack([H & 3, (H >> 4) & 3, (H >> 2) & 3, H >> 6], -1).view(H.shape[0], -1)
        return scaled((c | (hi << 4)).float() - 32, s).to(torch.bfloat16).double()
    P, s, gs = p
    lut = torch.tensor(_E2M1, device=DEV)
    v = torch.stack([lut[(P & 15).long()], lut[(P >> 4).long()]], -1).view(P.shape[0], -1)
    return scaled(v, s).double() * gs


def _int2(w, group):
    """The INT2 coarse operand of fp32 rows (four levels per group, fp16 scale)."""
    g = w.view(w.shape[0], -1, group)
    s = (g.abs().amax(-1, keepdim=True).clamp_min(1e-8) / 1.5).half().float()
    code = (torch.floor(g / s) + 2).clamp_(0, 3) - 1.5
    return (code * s).to(torch.bfloat16).view_as(w).double()


def _rows(planes, r0, r1):
    return tuple(t[r0:r1] if torch.is_tensor(t) else t for t in planes)


def _head_logits(d, fmt, group, c, dtype):
    """Coarse logits in 64 bits, the top c of them as dtype (ties to the lower
    index) and the exact logits of those."""
    x, n = d["x"].double(), d["w"][0].shape[0]
    coarse = []
    for r0 in range(0, n, 16384):
        w = _dense(fmt, _rows(d["w"], r0, r0 + 16384)).float()
        coarse.append(x @ _int2(w, group).T)
    coarse = torch.cat(coarse, 1)
    idx = torch.sort(coarse.to(dtype), dim=1, descending=True, stable=True).indices[:, :c]
    vals = torch.stack([_dense(fmt, tuple(t[i] if torch.is_tensor(t) else t for t in d["w"])) @ x[m]
                        for m, i in enumerate(idx)])
    return coarse, idx, vals


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    if kind == "linear":
        return d["x"].double() @ _dense(case["fmt"], d["w"]).T
    if kind == "layer":
        return [[x.double() @ _dense(fmt, w).T for fmt, x, w in layer] for layer in d["layers"]]
    if kind == "step":
        gates = torch.stack([x.double() @ _dense("w8", (q, s)).T for x, q, s in zip(d["gx"], d["gq"], d["gs"])])
        mixed = []
        for x, down, up in d["mixers"]:
            x = x.double()
            di = x @ _dense("w8", down).T
            sc = di[:, :case["lr"]] / 4
            bot = sc * torch.sigmoid(sc)
            gate = torch.sigmoid(bot @ _dense("w8", up).T)
            mixed.append([di, bot, (x * gate).view(case["m"], 4, -1).mean(1)])
        return [gates, mixed]
    if kind == "head":
        coarse, idx, vals = _head_logits(d, "mx8", case["g"], case["c"], torch.bfloat16)
        return coarse.scatter_(1, idx, vals)
    if kind == "draft":
        _, idx, vals = _head_logits(d, "nv4", 16, case["c"], torch.float32)
        full = torch.full((case["m"], case["v"]), -math.inf, dtype=torch.float64, device=DEV)
        return full.scatter_(1, d["ids"][idx], vals)
    w, to = _dense(case["src"], d["w"]), case["to"]
    if to == "f32" and case["src"] == "mx8":
        return w

    def amax(group):
        return w.view(w.shape[0], -1, group).abs().amax(-1)
    if to in ("w8", "f32"):
        return [None, amax(64) / 127]
    if to == "w6":
        return [None, None, amax(32) / 31]
    if to == "int2":
        return [None, amax(16) / 1.5]
    gs = float(w.abs().max()) / 6 / 448
    return [None, amax(16) / 6 / gs, gs]
