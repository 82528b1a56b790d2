"""The layer calls whose speed counts, as data: which calls, their inputs, their results.

Every case is one pass through the public modules of layerbatch_amd.moe with the weights, the
activations and (where one is kept) the workspace or the captured graph that an engine holds
before the call. ``listed`` names a dozen of them, ``draw`` takes one more out of the same
ranges: the three layers of layerbatch_amd.synth.SHAPES and generic layers around them, 1 to
8192 tokens in bf16 (4096 for the 512-expert layer) and 1 to 16384 in fp8.

A case is a dict of

    call      "block" (router + experts + shared expert), "norm" (the same behind the residual
              add and RMSNorm), "experts" (routed experts on given indices), "shared" (the
              dense SwiGLU MLP) or "router"
    H E k I Is    the layer's sizes
    T         tokens
    fp8       e4m3 weights with 128x128 block scales
    zipf      Zipf(1.2) router bias: a few experts get most of the tokens
    tiled     weights also held in the prefill GEMMs' tiled layout (pack_tiled_)
    layers    layers of one pass, each with weights and input of its own. A model's decode step
              goes through tens of layers, so a layer's weights come from HBM even where one
              layer's would stay in the caches: small batches run four
    graph     replayed from a captured graph, as the engine's decode buckets are
"""
import math

import numpy as np
import torch
from torch import nn

from layerbatch_amd.moe import Qwen3_5SparseMoeBlock
from layerbatch_amd.synth import SHAPES

WEIGHT_STD = 0.02
NORM_EPS = 1e-6


def _case(call, shape, T, **kw):
    s = SHAPES[shape] if isinstance(shape, str) else shape
    H, E, k, I, Is = s if isinstance(s, tuple) else (
        s.hidden_size, s.num_experts, s.top_k, s.moe_intermediate_size,
        s.shared_expert_intermediate_size)
    c = {"call": call, "H": H, "E": E, "k": k, "I": I, "Is": Is, "T": T, "fp8": False,
         "zipf": False, "tiled": False, "layers": 1, "graph": False}
    c.update(kw)
    return c


def listed():
    cases = {
        # one user, one token at a time, launched eagerly: latency of the smallest call
        "decode-1": _case("block", "qwen3-30b-a3b", 1, layers=4),
        # a decode bucket of the engine, replayed from its captured graph
        "decode-16-graph": _case("block", "qwen3-30b-a3b", 16, layers=4, graph=True),
        # the decoder layer's MLP half at an odd batch between two buckets
        "norm-decode-45": _case("norm", "qwen3-30b-a3b", 45),
        # the headline decode batch of bench.py
        "decode-128": _case("block", "qwen3-30b-a3b", 128),
        # decode of the 512-expert layer with its shared expert
        "e512-decode-128": _case("block", "qwen3-next-e512", 128),
        # the same layer with fp8 weights, an odd batch
        "e512-fp8-decode-75": _case("block", "qwen3-next-e512", 75, fp8=True),
        # the routed experts alone, on a router's int64 indices: the largest decode batches, and
        # a short prompt's prefill
        "experts-509": _case("experts", "qwen3-30b-a3b", 509),
        # the shared expert as a module of its own (a dense SwiGLU MLP), a ragged prefill chunk
        "shared-777": _case("shared", "qwen3-next-e512", 777),
        # the router as a module of its own, prefill
        "router-2048": _case("router", "qwen3-next-e512", 2048),
        # the headline prefill of bench.py: skewed expert loads
        "prefill-8192-zipf": _case("block", "qwen3-30b-a3b", 8192, zipf=True),
        # prefill of the 512-expert layer: many experts with few tokens each
        "e512-prefill-4096": _case("block", "qwen3-next-e512", 4096),
        # the largest: fp8 prefill of the 512-expert layer
        "e512-fp8-prefill-16384": _case("block", "qwen3-next-e512", 16384, fp8=True),
    }
    return [{"name": n, **c} for n, c in cases.items()]


def _tokens(rng, hi):
    """1..hi, spread over the logarithm."""
    return min(hi, int(math.exp(rng.uniform(0.0, math.log(hi + 1)))))


def draw(rng):
    while True:
        call = rng.choices(["block", "norm", "experts", "shared", "router"], [10, 3, 4, 2, 2])[0]
        fp8 = call != "router" and rng.random() < 0.3
        if rng.random() < 0.6:
            shape = rng.choice(["small-h1024-e16", "qwen3-30b-a3b", "qwen3-next-e512"])
        else:
            E = rng.choice([4, 8, 16, 20, 32, 48, 64, 96, 100, 128, 160, 256, 512])
            shape = (rng.choice([512, 1024, 2048] if fp8 else [512, 1024, 1536, 2048]), E,
                     rng.randint(1, min(E, 12)),
                     rng.choice([256, 512, 768] if fp8 else [128, 256, 384, 512, 768]),
                     rng.choice([0, 256, 512]))
        c = _case(call, shape, 1, fp8=fp8)
        if call == "shared" and not c["Is"]:
            c["Is"] = c["I"]
        c["T"] = _tokens(rng, 16384 if fp8 else 8192 if c["E"] <= 128 or call in ("shared", "router")
                         else 4096)
        if call in ("block", "norm"):
            c["zipf"] = rng.random() < 0.25
            c["tiled"] = not fp8 and c["H"] % 256 == 0 and c["T"] > 256 and rng.random() < 0.25
            c["graph"] = c["T"] <= 512 and rng.random() < 0.5
        if c["T"] <= 16 and call not in ("shared", "router"):
            c["layers"] = 4
        w = work(c)
        if w["bytes"] <= 3.3e9 and w["flops"] <= (1.1e12 if fp8 else 6.0e11):
            return c


# --- inputs -----------------------------------------------------------------------------------

def _randn(g, *shape, std=1.0):
    t = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    return t.normal_(0.0, std, generator=g)


def _inputs(case, seed):
    """Weights ~N(0, 0.02^2) and activations ~N(0, 1) of each layer, drawn in a fixed order."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    H, E, k, I, Is, T = (case[n] for n in ("H", "E", "k", "I", "Is", "T"))
    out = []
    for _ in range(case["layers"]):
        d = {"x": _randn(g, T, H)}
        if case["call"] in ("block", "norm", "router"):
            d["gate"] = _randn(g, E, H, std=WEIGHT_STD)
        if case["call"] in ("block", "norm", "experts"):
            d["gate_up"] = _randn(g, E, 2 * I, H, std=WEIGHT_STD)
            d["down"] = _randn(g, E, H, I, std=WEIGHT_STD)
        if case["call"] == "shared" or (Is and case["call"] in ("block", "norm")):
            d["sh_gate"] = _randn(g, Is, H, std=WEIGHT_STD)
            d["sh_up"] = _randn(g, Is, H, std=WEIGHT_STD)
            d["sh_down"] = _randn(g, H, Is, std=WEIGHT_STD)
            d["sh_gate_w"] = _randn(g, 1, H, std=WEIGHT_STD)
        if case["zipf"]:
            p = torch.arange(1, E + 1, dtype=torch.float64, device="cuda").pow(-1.2)
            p = p / p.sum()
            d["bias"] = torch.log(p[torch.randperm(E, generator=g, device="cuda")]).float()
        if case["call"] == "norm":
            d["residual"] = _randn(g, T, H)
            d["norm_w"] = _randn(g, H, std=0.1)
        if case["call"] == "experts":
            z = torch.randn(T, E, generator=g, device="cuda", dtype=torch.float32)
            top, d["idx"] = torch.topk(z, k, dim=-1)
            d["topw"] = torch.softmax(top, dim=-1).to(torch.bfloat16)
        out.append(d)
    return out


class _Norm:
    """What forward_norm takes of a Qwen3_5RMSNorm: its weight and its eps."""

    def __init__(self, weight):
        self.weight, self.eps = weight, NORM_EPS


def _param(t):
    return nn.Parameter(t, requires_grad=False)


def _module(case, d):
    """The block with the drawn weights in place; only the part that the call uses has any."""
    H, E, k, I, Is = (case[n] for n in ("H", "E", "k", "I", "Is"))
    with torch.device("meta"):
        b = Qwen3_5SparseMoeBlock(H, E, k, I, Is if "sh_gate" in d else 0)
    if "gate" in d:
        b.gate.weight = _param(d["gate"])
        b.gate.logit_bias = d.get("bias")
    if "gate_up" in d:
        b.experts.gate_up_proj = _param(d["gate_up"])
        b.experts.down_proj = _param(d["down"])
    if "sh_gate" in d:
        b.shared_expert.gate_proj.weight = _param(d["sh_gate"])
        b.shared_expert.up_proj.weight = _param(d["sh_up"])
        b.shared_expert.down_proj.weight = _param(d["sh_down"])
        b.shared_expert_gate.weight = _param(d["sh_gate_w"])
    if case["fp8"]:
        if case["call"] == "shared":
            # the module is used alone: the routed experts beside it are the smallest there are
            b.experts.num_experts, b.experts.intermediate_size = 1, 128
            b.experts.gate_up_proj = _param(_zeros(1, 256, H))
            b.experts.down_proj = _param(_zeros(1, H, 128))
        b.quantize_fp8_()
    elif case["tiled"]:
        b.pack_tiled_()
    if case["call"] == "router":
        return b.gate
    if case["call"] == "experts":
        return b.experts
    if case["call"] == "shared":
        return b.shared_expert
    return b


def _zeros(*shape):
    return torch.zeros(shape, dtype=torch.bfloat16, device="cuda")


def prepare(case, seed):
    layers = []
    for d in _inputs(case, seed):
        keep = {n: d[n] for n in ("x", "idx", "topw", "residual") if n in d}
        if "norm_w" in d:
            keep["norm"] = _Norm(d["norm_w"])
        layers.append((_module(case, d), keep))
    state = {"call": case["call"], "layers": layers, "workspace": None, "replay": None}
    if case["graph"] or case["call"] == "norm":
        # one workspace for all layers of a stream, as the engine keeps it
        n = layers[0][0].workspace_size(case["T"])
        state["workspace"] = torch.empty(n, dtype=torch.uint8, device="cuda")
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _eager(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = _eager(state)
        state["replay"] = (graph, out)
    return state


def _eager(state):
    call, out = state["call"], []
    for m, d in state["layers"]:
        if call == "block":
            out.append(m(d["x"], workspace=state["workspace"]))
        elif call == "norm":
            out.append(m.forward_norm(d["x"], d["residual"], d["norm"],
                                      workspace=state["workspace"]))
        elif call == "experts":
            out.append(m(d["x"], d["idx"], d["topw"]))
        else:
            out.append(m(d["x"]))
    return out


def run(state):
    if state["replay"] is not None:
        graph, out = state["replay"]
        graph.replay()
        return out
    return _eager(state)


# --- what a pass cannot do without --------------------------------------------------------------

def _hit_experts(case):
    """Experts with at least one token: routing on logits of the inputs' distribution."""
    E, k, T = case["E"], case["k"], case["T"]
    rng = np.random.default_rng(0)
    n = min(T, 4096)
    z = rng.standard_normal((n, E), dtype=np.float32)
    if case["zipf"]:
        p = np.arange(1, E + 1, dtype=np.float64) ** -1.2
        z = z * (WEIGHT_STD * math.sqrt(case["H"])) + np.log(p / p.sum())
    return len(np.unique(np.argpartition(-z, min(k, E) - 1, axis=1)[:, :k]))


def work(case):
    H, E, k, I, Is, T = (case[n] for n in ("H", "E", "k", "I", "Is", "T"))
    call, wb = case["call"], 1.0 + 4.0 / 16384 if case["fp8"] else 2.0
    nbytes = flops = 0.0
    if call in ("block", "norm", "router"):
        nbytes += 2.0 * E * H
        flops += 2.0 * T * E * H
    if call in ("block", "norm", "experts"):
        nbytes += _hit_experts(case) * 3.0 * H * I * wb
        flops += 6.0 * T * k * H * I
    if call == "shared" or (Is and call in ("block", "norm")):
        nbytes += 3.0 * H * Is * wb
        flops += 6.0 * T * H * Is
    nbytes += 2.0 * T * H                           # x
    if call == "router":
        nbytes += T * k * 10.0                      # bf16 weights, int64 indices
    else:
        nbytes += 2.0 * T * H                       # y
    if call == "norm":
        nbytes += 4.0 * T * H                       # residual in and out
    if call == "experts":
        nbytes += T * k * 10.0
    return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}


# --- results in 64 bits -------------------------------------------------------------------------

def _codes(b, amax):
    """The values b (fp32) as e4m3 codes with the fp32 scale amax / 448. Divided in 64 bits and
    rounded to 32, which are the correctly rounded 32-bit quotients: many values lie on the
    boundary of two codes, and torch divides by a number as a product with its reciprocal."""
    s = (amax.double() / torch.full_like(amax, 448.0, dtype=torch.float64)).float().double()
    s = torch.where(s > 0, s, torch.ones_like(s))
    return (b.double() / s).float().to(torch.float8_e4m3fn).double() * s


def _q_blocks(w):
    """The values that bf16 weights [N, K] hold as e4m3 codes with 128x128 block scales."""
    N, K = w.shape
    b = w.float().view(N // 128, 128, K // 128, 128)
    return _codes(b, b.abs().amax(dim=(1, 3), keepdim=True)).view(N, K)


def _q_groups(a):
    """The values that bf16 rows hold as e4m3 codes with one scale per 128 channels."""
    R, C = a.shape
    b = a.float().view(R, C // 128, 128)
    return _codes(b, b.abs().amax(dim=2, keepdim=True)).view(R, C)


def _swiglu(x, gate, up, down, fp8):
    """down(silu(gate x) * up x) of bf16 x and weights. With fp8, of what their codes hold; the
    intermediate is a bf16 value that is quantised in its turn, by definition of that format."""
    if not fp8:
        x = x.double()
        a = torch.nn.functional.silu(x @ gate.double().t()) * (x @ up.double().t())
        return a @ down.double().t()
    x = _q_groups(x)
    a = torch.nn.functional.silu(x @ _q_blocks(gate).t()) * (x @ _q_blocks(up).t())
    return _q_groups(a.to(torch.bfloat16)) @ _q_blocks(down).t()


def _route(case, d, x):
    """(weights in 64 bits, indices): the router's logits are bf16 values by definition, and
    ties go to the lower expert."""
    z = (x.double() @ d["gate"].double().t()).to(torch.bfloat16).float()
    if "bias" in d:
        z = z + d["bias"]
    z, idx = torch.sort(z, dim=-1, descending=True, stable=True)
    return torch.softmax(z[:, :case["k"]].double(), dim=-1), idx[:, :case["k"]]


def _experts(case, d, x, idx, w):
    y = torch.zeros(x.shape, dtype=torch.float64, device=x.device)
    I = case["I"]
    for e in range(case["E"]):
        t, s = torch.nonzero(idx == e, as_tuple=True)
        if t.numel():
            o = _swiglu(x[t], d["gate_up"][e, :I], d["gate_up"][e, I:], d["down"][e], case["fp8"])
            y.index_add_(0, t, o * w[t, s].double()[:, None])
    return y


def exact(case, seed):
    out = []
    for d in _inputs(case, seed):
        x, call = d["x"], case["call"]
        if call == "router":
            out.append(_route(case, d, x))
            continue
        if call == "shared":
            out.append(_swiglu(x, d["sh_gate"], d["sh_up"], d["sh_down"], case["fp8"]))
            continue
        if call == "experts":
            out.append(_experts(case, d, x, d["idx"], d["topw"]))
            continue
        if call == "norm":
            total = d["residual"].double() + x.double()
            h = total.to(torch.bfloat16).double()
            h = h * torch.rsqrt(h.square().mean(dim=-1, keepdim=True) + NORM_EPS)
            x = (h * (1.0 + d["norm_w"].double())).to(torch.bfloat16)
        w, idx = _route(case, d, x)
        y = _experts(case, d, x, idx, w)
        if "sh_gate" in d:
            g = torch.sigmoid(x.double() @ d["sh_gate_w"].double().t())
            y += g * _swiglu(x, d["sh_gate"], d["sh_up"], d["sh_down"], case["fp8"])
        out.append((y, total) if call == "norm" else y)
    return out


def tolerance(case):
    # The 2-norm against the 64-bit result, measured (0.002 to 0.004), times about four. A block
    # may differ by a little more: a token's k-th and next expert change places where a logit lies
    # on the other side of a bf16 rounding boundary.
    if case["call"] == "router":
        return {"rel": 7e-3, "differ": 5e-3}
    return {"rel": 1e-2 if case["call"] in ("experts", "shared") else 1.5e-2}
