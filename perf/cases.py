"""Layer calls that stand for the use of this framework, with their inputs,
their work, their tolerances and a float64 restatement of their results.

Every case is one call (or one decode step over several layers) of MoELayer:
a decode step runs `layers` independent layers, each with its own weights and
rows, captured in a HIP graph as a serving loop captures it, so that no
layer's weights are still in the memory-side cache when they are read again;
a prefill (or the tiny layer) is a plain call of MoELayer.forward.

Weights are centred as mlx's affine quantiser leaves them, so that outputs
are of order one. Rows whose k-th and (k+1)-th router scores lie within the
rounding of a 16-bit logit are not used: which expert they take is not
defined by the real-valued function.
"""
import math

import torch

from ffai_amd import _lib
from ffai_amd.layer import MoEGatingMode, MoELayer, MoERouter, StackedExperts

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
GATINGS = {"softmax_topk": MoEGatingMode.softmaxThenTopK, "topk_softmax": MoEGatingMode.topKThenSoftmax,
           "sigmoid": MoEGatingMode.sigmoidTopK}
ACTIVATIONS = {"swiglu": _lib.MOE_ACT_SWIGLU, "gptoss": _lib.MOE_ACT_GPTOSS, "geglu": _lib.MOE_ACT_GEGLU,
               "relu2": _lib.MOE_ACT_RELU2}
ALPHA, LIMIT, EPS = 1.702, 7.0, 1e-6
ZIPF_BETA = 0.33  # router-bias strength: the hottest expert gets about 10x the median load

# Fields of a case: T rows, H hidden, E experts, k per token, I intermediate,
# SI shared intermediate (0: none), gu / dn bits of gate-up / down, gs group
# size, sb scale dtype, dt activation dtype, act, gating, rb router bias
# ("none", "normal", "zipf"), ob per-expert output biases, rq router bits
# (0: dense), split (the router reads its own rows), entry ("forward" or
# "residual"), layers, graph.
BASE = dict(SI=0, gu=4, dn=4, gs=64, sb="bf16", dt="bf16", act="swiglu", gating="softmax_topk", rb="none",
            ob=False, rq=0, split=False, entry="forward", layers=1, graph=False)
TINY = dict(BASE, H=256, E=8, k=2, I=512, sb="f16", dt="f16")
GPTOSS = dict(BASE, H=2880, E=32, k=4, I=2880, act="gptoss", gating="topk_softmax", rb="normal", ob=True)
QWEN3 = dict(BASE, H=2048, E=128, k=8, I=768, sb="f16")
MIXED = dict(BASE, H=2048, E=256, k=8, I=512, SI=512, gu=3, dn=6)
NEMOTRON = dict(BASE, H=2688, E=128, k=6, I=1856, SI=3712, act="relu2", gating="sigmoid")
GEMMA4 = dict(BASE, H=1024, E=64, k=8, I=384, act="geglu", gating="topk_softmax", split=True)
Q8 = dict(BASE, H=1024, E=64, k=8, I=384, gu=8, dn=8, gs=32, sb="f16", dt="f16", rq=8)


def listed():
    return [
        # the smallest call: a tiny f16 layer, where launches and host work are all there is
        dict(TINY, name="tiny_t16", T=16),
        # one token of a 4-bit GPT-OSS-20B-shaped model: a decode step over eight of its layers
        dict(GPTOSS, name="gptoss_decode_t1", T=1, layers=8, graph=True),
        # one token of a Qwen3-MoE-shaped model, with the decoder's residual add and norm around the block
        dict(QWEN3, name="qwen3_step_t1", T=1, layers=16, graph=True, entry="residual"),
        # batched decode of 16 and 64 sequences
        dict(QWEN3, name="qwen3_decode_t16", T=16, layers=4, graph=True),
        dict(QWEN3, name="qwen3_decode_t64", T=64, layers=4, graph=True),
        # an odd batch on few large experts
        dict(GPTOSS, name="gptoss_decode_t37", T=37, layers=2, graph=True),
        # a large decode batch of a mixed-width layer with a gated shared expert
        dict(MIXED, name="mixed_decode_t100", T=100, layers=2, graph=True),
        # 8-bit experts, quantised router, f16, small groups: a medium batch
        dict(Q8, name="q8_decode_t48", T=48, layers=8, graph=True),
        # a short ragged prompt through sigmoid-routed squared-ReLU experts and a large shared one
        dict(NEMOTRON, name="nemotron_prefill_t333", T=333),
        # a prompt on few large experts
        dict(GPTOSS, name="gptoss_prefill_t1000", T=1000),
        # a prompt through 256 small mixed-width experts and a shared one
        dict(MIXED, name="mixed_prefill_t2048", T=2048),
        # a long prompt with skewed expert loads
        dict(QWEN3, name="qwen3_prefill_t4096", T=4096, rb="zipf"),
    ]


def draw(rng):
    while True:
        c = dict(rng.choice([TINY, GPTOSS, GPTOSS, QWEN3, QWEN3, MIXED, MIXED, NEMOTRON, GEMMA4, Q8]))
        c["T"] = max(1, round(math.exp(rng.uniform(0, math.log(4096)))))
        if rng.random() < 0.4:  # another width of the same kind
            c["H"] = 64 * rng.randint(8, 46)
            c["I"] = 64 * rng.randint(5, 46)
            c["E"] = max(2 * c["k"], rng.choice([16, 24, 32, 60, 64, 96, 128, 160]))
            c["SI"] = c["SI"] and c["I"] * rng.choice([1, 2])
        if rng.random() < 0.3:
            c["gu"], c["dn"] = rng.choice([(4, 4), (3, 4), (2, 4), (5, 5), (6, 6), (8, 8), (4, 6)])
            c["gs"] = rng.choice([32, 64]) if c["H"] % 128 or c["I"] % 128 else rng.choice([32, 64, 128])
        if rng.random() < 0.15:
            c["dt"] = "f16"
        if c["T"] <= 128:
            c["layers"], c["graph"] = rng.choice([1, 2, 4, 8]), True
        if not c["split"] and rng.random() < 0.2:
            c["entry"] = "residual"
        w = work(c)
        if w["flops"] <= 300e9 and w["bytes"] <= 900e6:
            return c


# ---------------------------------------------------------------- inputs --

def _centred(gen, E, N, K, bits, gs, sb, ob_dt=None):
    """A stacked projection: uniform codes, biases about -scale * (2^bits - 1) / 2,
    scales sized so that a row of unit-variance values gives order one."""
    w = torch.randint(0, 256, (E, N, K * bits // 8), dtype=torch.uint8, device="cuda", generator=gen)
    top = 2 ** bits - 1
    s0 = math.sqrt(12.0 / K) / top
    s = torch.empty(E, N, K // gs, device="cuda").uniform_(0.8 * s0, 1.2 * s0, generator=gen).to(DTYPES[sb])
    b = torch.randn(E, N, K // gs, device="cuda", generator=gen).mul_(0.05).sub_(top / 2).mul_(s.float())
    ob = None if ob_dt is None else (0.1 * torch.randn(E, N, device="cuda", generator=gen)).to(ob_dt)
    return StackedExperts(w.view(torch.int32), s, b.to(DTYPES[sb]), bits, gs, out_bias=ob)


def _zipf_bias(gen, E):
    p = (torch.randperm(E, device="cuda", generator=gen).double() + 1) ** -1.1
    return ZIPF_BETA * torch.log(p / p.sum())


def _layer(c, gen):
    """The tensors of one layer and the layer over them."""
    H, E, I, dt = c["H"], c["E"], c["I"], DTYPES[c["dt"]]
    ob = dt if c["ob"] else None
    gated = c["act"] != "relu2"

    def proj(n_e, n, k, bits, out_bias=None):
        return _centred(gen, n_e, n, k, bits, c["gs"], c["sb"], out_bias)

    if c["rq"]:
        rw = proj(1, E, H, c["rq"])
    else:
        scale = 1.0 if c["split"] else H ** -0.5
        rw = (scale * torch.randn(E, H, device="cuda", generator=gen)).to(dt)
    rb = None
    if c["rb"] == "normal":
        rb = (0.1 * torch.randn(E, device="cuda", generator=gen)).to(dt)
    elif c["rb"] == "zipf":
        rb = _zipf_bias(gen, E).to(dt)
    ebias = escale = None
    if c["gating"] == "sigmoid":
        ebias = torch.empty(E, device="cuda").uniform_(-0.05, 0.05, generator=gen)
    if c["split"]:
        escale = torch.empty(E, device="cuda").uniform_(0.5, 1.5, generator=gen)
    router = MoERouter(E, c["k"], GATINGS[c["gating"]], True, ebias, float(H ** -0.5) if c["split"] else 1.0,
                       2.5 if c["gating"] == "sigmoid" else 1.0, escale)
    shared = sgw = None
    if c["SI"]:
        shared = (proj(1, c["SI"], H, c["gu"]) if gated else None, proj(1, c["SI"], H, c["gu"]),
                  proj(1, H, c["SI"], c["dn"]))
        if gated:
            sgw = (H ** -0.5 * torch.randn(1, H, device="cuda", generator=gen)).to(dt)
    return MoELayer(router_weight=rw, router=router, gate=proj(E, I, H, c["gu"], ob) if gated else None,
                    up=proj(E, I, H, c["gu"], ob), down=proj(E, H, I, c["dn"], ob), hidden=H, act_dtype=dt,
                    router_bias=rb, activation=ACTIVATIONS[c["act"]], alpha=ALPHA, limit=LIMIT, shared=shared,
                    shared_gate_weight=sgw)


def _logits(layer, x):
    """Router logits of rows x in float64."""
    rw = layer.router_weight
    w = _dequantised(rw, 0) if isinstance(rw, StackedExperts) else rw.double()
    logits = x.double() @ w.t()
    return logits if layer.router_bias is None else logits + layer.router_bias.double()


def _scores(layer, logits):
    """What the top-k is taken of, and how far two scores have to be apart
    for 16-bit logits to keep their order: two bf16 ulps of the row's largest."""
    apart = logits.abs().amax(1) * 2.0 ** -6
    if layer.router.gatingMode == MoEGatingMode.sigmoidTopK:
        return torch.sigmoid(logits) + layer.router.expertBias.double(), apart / 4
    return logits, apart


def _add_norm(h, m, w, dt):
    """round(h + m) and its RMS norm times w, the way the block computes them."""
    r = (h.double() + m.double()).to(dt).double()
    return r, r / torch.sqrt((r * r).mean(1, keepdim=True) + EPS) * w.double()


def _rows(c, layer, gen):
    """T rows (h, mixer output, norm weight for the residual entry; x and the
    router's own rows otherwise) whose routing 16-bit logits decide."""
    T, H, k, dt = c["T"], c["H"], c["k"], DTYPES[c["dt"]]
    if c["entry"] == "residual":
        norm = torch.empty(H, device="cuda").uniform_(0.5, 1.5, generator=gen).to(dt)
    kept, have = [], 0
    while have < T:
        n = 3 * (T - have) + 64
        x = torch.randn(n, H, device="cuda", generator=gen).to(dt)
        if c["entry"] == "residual":
            other = (0.5 * torch.randn(n, H, device="cuda", generator=gen)).to(dt)
            logits = _logits(layer, _add_norm(x, other, norm, dt)[1])
        else:
            other = torch.randn(n, H, device="cuda", generator=gen).to(dt) if c["split"] else x
            logits = _logits(layer, other)
        scores, apart = _scores(layer, logits)
        top = scores.topk(k + 1, dim=1).values
        fine = (top[:, k - 1] - top[:, k] >= apart).nonzero().flatten()[:T - have]
        kept.append((x[fine], other[fine]))
        have += fine.numel()
    a, b = (torch.cat([p[i] for p in kept]).contiguous() for i in (0, 1))
    if c["entry"] == "residual":
        return dict(h=a, m=b, norm=norm)
    return dict(x=a, rx=b if c["split"] else None)


def _inputs(c, seed):
    """(layer, rows) of each of the case's layers, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000 * seed + 17)
    out = []
    for _ in range(c["layers"]):
        layer = _layer(c, gen)
        out.append((layer, _rows(c, layer, gen)))
    return out


def _call(layer, rows, out=None, residual_out=None):
    if "h" in rows:
        y = layer.forward_residual(rows["h"], rows["m"], rows["norm"], EPS, out=out, residual_out=residual_out)
        return (y, residual_out)
    return (layer.forward(rows["x"], out=out, router_x=rows["rx"]),)


def prepare(case, seed):
    c = case
    state = dict(case=c, inputs=_inputs(c, seed), graph=None)
    for layer, _ in state["inputs"]:
        layer.workspace(c["T"])
    # the residual stream is the caller's own buffer
    state["res"] = [torch.empty_like(r["h"]) if "h" in r else None for _, r in state["inputs"]]
    if c["graph"]:
        outs = [torch.empty_like(r["h"] if "h" in r else r["x"]) for _, r in state["inputs"]]
        bufs = list(zip(state["inputs"], outs, state["res"]))
        _call(*bufs[0][0], *bufs[0][1:])  # the library's one-time set-up happens outside the capture
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            for (layer, rows), y, r in bufs:
                _call(layer, rows, y, r)
        state["outs"] = [(y,) if r is None else (y, r) for _, y, r in bufs]
    return state


def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["outs"]
    return [_call(layer, rows, residual_out=r) for (layer, rows), r in zip(state["inputs"], state["res"])]


# ------------------------------------------------------------------ work --

def work(case):
    c = case
    T, H, E, k, I, SI = (c[n] for n in ("T", "H", "E", "k", "I", "SI"))
    used = E * (1 - (1 - k / E) ** T)  # distinct experts under even routing
    gated = 1 if c["act"] == "relu2" else 2
    side = 4.0 / c["gs"]  # scale and bias bytes per weight

    def weights(i):
        return gated * i * H * (c["gu"] / 8 + side) + i * H * (c["dn"] / 8 + side)

    router = E * H * (c["rq"] / 8 + side if c["rq"] else 2)
    rows = {"forward": 3 if c["split"] else 2, "residual": 4}[c["entry"]]
    nbytes = used * weights(I) + weights(SI) + router + rows * T * H * 2
    flops = 2 * T * H * ((gated + 1) * (k * I + SI) + E)
    return {"bytes": c["layers"] * nbytes, "flops": c["layers"] * flops}


def tolerance(case):
    # Logits, activations between the products and per-expert outputs are 16-bit:
    # up to 8e-3 (bf16) and 9e-4 (f16) from exact(), so that two correct
    # implementations lie up to sqrt(2) times that apart.
    return {"rel": 1.5e-2, "max": 0.15} if case["dt"] == "bf16" else {"rel": 3e-3, "max": 3e-2}


# ----------------------------------------------------------------- exact --

def _dequantised(p, e):
    """Expert e of a stacked projection as [n, k] float64."""
    words = p.weight[e].long() & 0xFFFFFFFF
    words = torch.cat([words, torch.zeros_like(words[:, :1])], 1)
    bit = torch.arange(p.k, device=words.device) * p.bits
    at, off = bit // 32, bit % 32
    q = ((words[:, at] >> off) | (words[:, at + 1] << (32 - off))) & (2 ** p.bits - 1)
    s, b = (t[e].double().repeat_interleave(p.group_size, 1) for t in (p.scales, p.biases))
    return q.double() * s + b


def _act(c, g, u):
    if c["act"] == "relu2":
        return torch.relu(u) ** 2
    if c["act"] == "gptoss":
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        return g * torch.sigmoid(ALPHA * g) * (u + 1)
    if c["act"] == "geglu":
        return torch.nn.functional.gelu(g, approximate="tanh") * u
    return g * torch.sigmoid(g) * u


def _ffn(c, gate, up, down, e, x):
    def product(p, a):
        y = a @ _dequantised(p, e).t()
        return y if p.out_bias is None else y + p.out_bias[e].double()

    u = product(up, x)
    return product(down, _act(c, None if gate is None else product(gate, x), u))


def _routing(layer, logits):
    r = layer.router
    if r.gatingMode == MoEGatingMode.sigmoidTopK:
        idx = _scores(layer, logits)[0].topk(r.topK, dim=1).indices
        w = torch.sigmoid(logits).gather(1, idx)
        w = w / w.sum(1, keepdim=True)
    else:  # softmax over all, renormalised over the picks, is softmax over the picks
        val, idx = logits.topk(r.topK, dim=1)
        w = torch.softmax(val * r.logitScale, 1)
    w = w * r.routedScale
    return idx, w if r.expertScale is None else w * r.expertScale.double()[idx]


def _exact_layer(c, layer, rows):
    if "h" in rows:
        r, x = _add_norm(rows["h"], rows["m"], rows["norm"], DTYPES[c["dt"]])
        rx = x
    else:
        x = rows["x"].double()
        rx = x if rows["rx"] is None else rows["rx"].double()
    idx, w = _routing(layer, _logits(layer, rx))
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        t, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, t, w[t, slot, None] * _ffn(c, layer.gate, layer.up, layer.down, e, x[t]))
    if layer.shared is not None:
        s = _ffn(c, *layer.shared, 0, x)
        if layer.shared_gate_weight is not None:
            s = s * torch.sigmoid(x @ layer.shared_gate_weight.double().t())
        y = y + s
    return (y + r, r) if "h" in rows else (y,)


def exact(case, seed):
    return [_exact_layer(case, layer, rows) for layer, rows in _inputs(case, seed)]
