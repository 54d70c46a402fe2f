"""The measured cases: the work that a program using this framework has it do, through
`Context`'s entry points (moe-680m_amd/__init__.py), at the layer shape of the repository's
configurations (hidden 2048, expert intermediate 512, up to 256 routed experts + 1 shared).

A case is a dict of plain values:
  kind     "ffn":    one MoE layer from given router logits (ffn_route): the layer of a decode
                     step (M = 1..8), of a short or batched prompt, of a long prefill
           "layer":  one MoE layer from its activations: the router GEMV, then the expert FFN
                     into the residual -- what a model's forward pass calls per layer
           "router": the router gate product and top-8 alone (router_gemv_topk)
           "stack":  one token through consecutive layers in one call (decode_stack)
  M        tokens
  E        routed experts
  wmode    0 (softmax weights, scale 1/9) or 1 (renormalised over the 8)
  routing  logits "uniform" N(0,1), "zipf" (a Zipf(1.1) bias over the experts: a prompt on one
           subject) or "hot" (5 % of the tokens forced onto one expert)
  gate     element type of the router gate matrix: "iq4", "f16" or "f32" (kinds that have one;
           "" otherwise)
  layers   layers of a stack (else 1)
  residual 1: y += FFN(RMSNorm(x)), the residual update; 0: y = FFN(RMSNorm(x))

Inputs come from torch generators alone (quant blocks of random nibbles and 6-bit scales,
d = |N(0,1)| * 2e-3; activations N(0,1)), so the f64 references need nothing of this package.
"""
import importlib.util
import math
import os
import sys

import torch

H, I = 2048, 512
QK, SB = 256, 136
SLOTS, TOPK = 9, 8
KVALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
MATRIX_BYTES = H * I // QK * SB
EXPERT_BYTES = 3 * MATRIX_BYTES
ZIPF_S, HOT_SHARE, HOT_LOGIT = 1.1, 0.05, 1000.0
GATE_BYTES = {"iq4": SB / QK, "f16": 2.0, "f32": 4.0}


def _package():
    """The package directory moe-680m_amd/ (not an importable name) as moe680m_amd."""
    if "moe680m_amd" in sys.modules:
        return sys.modules["moe680m_amd"]
    here = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "moe-680m_amd")
    spec = importlib.util.spec_from_file_location("moe680m_amd", os.path.join(here, "__init__.py"),
                                                  submodule_search_locations=[here])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["moe680m_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


# ---------------------------------------------------------------- the cases
def _case(name, kind, M, E=256, wmode=1, routing="uniform", gate="", layers=1, residual=0):
    c = {"kind": kind, "M": M, "E": E, "wmode": wmode, "routing": routing, "gate": gate, "layers": layers,
         "residual": residual}
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one layer of a decode step, one sequence: the smallest call, all latency
        _case("ffn_m1", "ffn", 1),
        # one layer, a few tokens verified together (odd size), softmax weights, into the residual
        _case("ffn_m3", "ffn", 3, wmode=0, residual=1),
        # one layer, the widest small-batch decode
        _case("ffn_m8", "ffn", 8),
        # one layer, a batch of sequences decoding together
        _case("ffn_m21", "ffn", 21),
        # one layer, a short prompt or a large decode batch; fewer experts, a ragged size
        _case("ffn_m100_e128", "ffn", 100, E=128, wmode=0),
        # one layer, prompt prefill with skewed load (some experts receive no token)
        _case("ffn_m512_zipf", "ffn", 512, routing="zipf"),
        # one layer, long prefill with one hot expert: the largest call
        _case("ffn_m4096_hot", "ffn", 4096, routing="hot"),
        # one layer of a forward pass from the activations: a decode step ...
        _case("layer_m1_iq4", "layer", 1, gate="iq4", residual=1),
        # ... and a prompt (GGUF files keep the gate matrix in f32)
        _case("layer_m1000_f32", "layer", 1000, gate="f32", residual=1),
        # the router of a long prefill
        _case("router_m4096_f16", "router", 4096, gate="f16"),
        # a whole decode token: 40 layers, seeded router logits
        _case("stack_40", "stack", 1, layers=40),
        # the same as a forward pass, every layer routed from its own input
        _case("stack_40_routed", "stack", 1, gate="iq4", layers=40),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("ffn", "layer", "router", "stack"), (6, 2, 2, 1))[0]
    E = rng.choice((256, 256, 256, 128, 64))
    wmode = rng.choice((0, 1))
    gate = rng.choice(("iq4", "f16", "f32"))
    if kind == "ffn":
        return _case("", kind, _log_uniform(rng, 1, 4096), E, wmode, rng.choice(("uniform", "zipf", "hot")),
                     residual=rng.choice((0, 1)))
    if kind == "layer":
        return _case("", kind, _log_uniform(rng, 1, 2048), E, wmode, gate=gate, residual=1)
    if kind == "router":
        return _case("", kind, _log_uniform(rng, 1, 4096), E, wmode, gate=gate)
    return _case("", kind, 1, 256, wmode, gate=rng.choice(("", gate)), layers=rng.randint(1, 40))


# ---------------------------------------------------------------- inputs (torch only)
def _gen(seed, tag, layer=0, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed((int(seed) * 1000003 + layer * 131 + tag) & (2**63 - 1))
    return g


def _blocks(n, g, scale):
    """n IQ4_XS super-blocks: random nibbles and 6-bit scales, d = f16(|N(0,1)| * scale)."""
    b = torch.randint(0, 256, (n, SB), dtype=torch.uint8, device="cuda", generator=g)
    d = (torch.randn(n, device="cuda", generator=g).abs_() * scale).half()
    b[:, :2] = d.view(torch.uint8).view(n, 2)
    return b


def _layer_blocks(case, seed, layer):
    n = (case["E"] + 1) * EXPERT_BYTES // SB
    return _blocks(n, _gen(seed, 1, layer), 2e-3)


def _gate_matrix(case, seed, layer):
    """[E][H] gate matrix whose logits over N(0,1) activations have a deviation of about 1."""
    g, E = _gen(seed, 2, layer), case["E"]
    if case["gate"] == "iq4":
        return _blocks(E * H // QK, g, 2e-5)
    w = torch.randn(E, H, device="cuda", generator=g) * (1.0 / math.sqrt(H))
    return w.half() if case["gate"] == "f16" else w


def _x(case, seed):
    return torch.randn(case["M"], H, device="cuda", generator=_gen(seed, 3))


def _make_logits(routing, M, E, g):
    dev = g.device
    lg = torch.randn(M, E, device=dev, generator=g)
    if routing == "zipf":
        rank = torch.randperm(E, device=dev, generator=g).float() + 1.0
        lg -= ZIPF_S * rank.log()
    elif routing == "hot":
        hot = torch.rand(M, device=dev, generator=g) < HOT_SHARE
        e = torch.randint(0, E, (1,), device=dev, generator=g)
        lg[:, e] = torch.where(hot[:, None], torch.full_like(lg[:, e], HOT_LOGIT), lg[:, e])
    return lg


def _logits(case, seed):
    rows = case["layers"] if case["kind"] == "stack" else case["M"]
    return _make_logits(case["routing"], rows, case["E"], _gen(seed, 4))


# ---------------------------------------------------------------- the program
def prepare(case, seed):
    """The context with its bound layers (and routers), the activations and the output buffers."""
    pkg = _package()
    M, E, n = case["M"], case["E"], case["layers"]
    s = {"case": case, "x": _x(case, seed)}
    s["ctx"] = ctx = pkg.Context(H, I, E, n, max(M, 16), case["wmode"])
    if case["kind"] != "router":
        for l in range(n):
            ctx.bind_packed(l, _layer_blocks(case, seed, l))
    if case["gate"]:
        s["wg"] = [_gate_matrix(case, seed, l) for l in range(n)]
    if case["kind"] == "stack":
        if case["gate"]:
            for l in range(n):
                ctx.bind_router(l, s["wg"][l])
        else:
            s["logits"] = _logits(case, seed)
    elif case["kind"] == "ffn":
        s["logits"] = _logits(case, seed)
    rows = n if case["kind"] == "stack" else M
    s["ids"] = torch.empty((rows, SLOTS), dtype=torch.uint16, device="cuda")
    s["w"] = torch.empty((rows, SLOTS), dtype=torch.float32, device="cuda")
    s["y"] = torch.empty_like(s["x"])
    s["lg"] = torch.empty((M, E), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    """One pass; returns y, the routing (ids as int16, weights) and the logits it computed."""
    c, ctx, x, y, ids, w = s["case"], s["ctx"], s["x"], s["y"], s["ids"], s["w"]
    out = {"ids": ids.view(torch.int16), "w": w}
    if c["kind"] == "stack":
        out["y"] = ctx.decode_stack(0, x, s.get("logits"), y=y, ids=ids, w=w, rmsnorm=True, n_layers=c["layers"])
        return out
    if c["kind"] in ("layer", "router"):
        ctx.router_gemv_topk(s["wg"][0], x, rmsnorm=True, logits=s["lg"], ids=ids, w=w)
        out["logits"] = s["lg"]
        if c["kind"] == "router":
            return out
    if c["residual"]:
        y.copy_(x)  # the residual stream of this pass
    if c["kind"] == "ffn":
        ctx.ffn_route(0, x, s["logits"], y=y, ids=ids, w=w, accumulate=bool(c["residual"]), rmsnorm=True)
    else:
        ctx.ffn(0, x, ids, w, y=y, accumulate=bool(c["residual"]), rmsnorm=True)
    out["y"] = y
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def _distinct_experts(case):
    """Experts (the shared one included) that the case's tokens select, on one seeded sample."""
    g = _gen(0, 5, device="cpu")
    top = _make_logits(case["routing"], case["M"], case["E"], g).topk(TOPK, dim=1).indices
    return int(top.unique().numel()) + 1


def work(case):
    M, E, n = case["M"], case["E"], case["layers"]
    ffn_flops = 2 * SLOTS * 3 * H * I
    gate = int(E * H * GATE_BYTES.get(case["gate"], 0.0))
    gate_flops = 2 * H * E if case["gate"] else 0
    route_io = E * 4 + SLOTS * 6  # logits read or written, ids and weights
    if case["kind"] == "stack":
        return {"bytes": n * (SLOTS * EXPERT_BYTES + gate + (0 if gate else E * 4) + SLOTS * 6) + 2 * H * 4,
                "flops": n * (ffn_flops + gate_flops)}
    if case["kind"] == "router":
        return {"bytes": gate + M * (H * 4 + route_io), "flops": M * gate_flops}
    y_io = H * 4 * (2 if case["residual"] else 1)
    return {"bytes": _distinct_experts(case) * EXPERT_BYTES + gate + M * (H * 4 + y_io + route_io),
            "flops": M * (ffn_flops + gate_flops)}


def tolerance(case):
    if case["kind"] == "router":
        # f32 sums of 2048 terms in another order; near ties may swap two ids
        return {"rel": 1e-5, "differ": 1e-3}
    if case["kind"] == "stack":
        # int8-plane activations, 40 chained layers
        return {"rel": 1e-3, "differ": 0.0}
    if case["M"] <= 8:
        # 16-bit activations (two int8 planes per 32 elements), f32 sums
        return {"rel": 1.5e-4, "differ": 0.0}
    # f16 operands, f32 sums; a near tie in computed logits may swap two ids
    return {"rel": 3e-3, "differ": 1e-3 if case["gate"] else 0.0}


# ---------------------------------------------------------------- f64 reference (torch only)
def _dequant(blocks, rows):
    """IQ4_XS super-blocks [n][136] -> f64 matrix of `rows` rows."""
    n = blocks.shape[0]
    b = blocks.to(torch.int32)
    d = blocks[:, :2].contiguous().view(torch.float16).double()                    # [n][1]
    sh = b[:, 2] | (b[:, 3] << 8)
    ib = torch.arange(8, device=b.device)
    lo = (b[:, 4 + ib // 2] >> (4 * (ib % 2))) & 15
    ls = lo | (((sh[:, None] >> (2 * ib)) & 3) << 4)
    q = b[:, 8:].view(n, 8, 16)
    kv = torch.tensor(KVALUES, dtype=torch.float64, device=b.device)
    v = kv[torch.cat((q & 15, q >> 4), dim=2)]                                     # [n][8][32]
    return (v * (d * (ls - 32).double())[:, :, None]).view(rows, -1)


def _expert(blocks, e):
    nb = MATRIX_BYTES // SB
    b = blocks[e * 3 * nb:(e + 1) * 3 * nb]
    return _dequant(b[:nb], I), _dequant(b[nb:2 * nb], I), _dequant(b[2 * nb:], H)


def _rms(x):
    return x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + 1e-6)


def _route(logits, wmode):
    """(ids [M][9], w [M][9]) of f64 logits: top-8, lower index first among equals, + shared."""
    M, E = logits.shape
    order = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :TOPK]
    p = torch.softmax(logits, dim=1).gather(1, order)
    if wmode == 1:
        p = p / p.sum(dim=1, keepdim=True)
    ids = torch.cat((order, torch.full((M, 1), E, device=logits.device, dtype=order.dtype)), dim=1)
    return ids, torch.cat((p, torch.ones(M, 1, dtype=p.dtype, device=p.device)), dim=1)


def _ffn(blocks, xin, ids, w, wmode):
    y = torch.zeros_like(xin)
    for e in ids.unique().tolist():
        t, s = (ids == e).nonzero(as_tuple=True)
        w1, w3, w2 = _expert(blocks, e)
        g = xin[t] @ w1.T
        h = g * torch.sigmoid(g) * (xin[t] @ w3.T)
        y.index_add_(0, t, (h @ w2.T) * w[t, s][:, None])
    return y * (1.0 if wmode == 1 else 1.0 / 9.0)


def _gate64(case, seed, layer):
    g = _gate_matrix(case, seed, layer)
    return _dequant(g, case["E"]) if case["gate"] == "iq4" else g.double()


def exact(case, seed):
    """What run returns, in f64; None for the routed stack (one swapped near tie in any of its
    layers changes everything after it)."""
    if case["kind"] == "stack" and case["gate"]:
        return None
    x = _x(case, seed).double()
    if case["kind"] == "stack":
        logits = _logits(case, seed).double()
        ids, w = _route(logits, case["wmode"])
        for l in range(case["layers"]):
            x = x + _ffn(_layer_blocks(case, seed, l), _rms(x), ids[l:l + 1], w[l:l + 1], case["wmode"])
        return {"ids": ids.to(torch.int16), "w": w, "y": x}
    if case["kind"] == "ffn":
        logits = _logits(case, seed).double()
    else:
        logits = _rms(x) @ _gate64(case, seed, 0).T
    ids, w = _route(logits, case["wmode"])
    out = {"ids": ids.to(torch.int16), "w": w}
    if case["kind"] != "ffn":
        out["logits"] = logits
        if case["kind"] == "router":
            return out
    y = _ffn(_layer_blocks(case, seed, 0), _rms(x), ids, w, case["wmode"])
    out["y"] = x + y if case["residual"] else y
    return out
