"""The work that a serving program has this package do, as timed cases.

A case is one call chain of a decoder layer (or the LM head) through the
package's public modules, at one number of tokens:

  linear       LinearW8A8(x): one projection
  norm_linear  RMSNorm.forward_quant(x, residual) -> gemm_quantized: the fused
               residual add, norm and quantization in front of a QKV projection
  mlp          GatedMLP(x): gate_up, activation, down
  layer        the linears and norms of one decoder layer (attention's output is
               an input), captured in a graph and replayed, as a decode loop does
  head         LMHead(hidden[:, -1]): the vocabulary projection of the last tokens
  moe          SparseMoE(x): router, sorted grouped expert GEMMs, combine

Weights are per-row int8 (`bits` 8) or grouped int4 (`bits` 4, `group` columns a
scale).  `tokens` is small in decode (one row per sequence) and large in prefill.
The shapes are those of Qwen3-0.6B, Qwen3-8B and Qwen3-30B-A3B, and generic ones.
"""
import importlib.util
import math
import os
import sys

import torch


def _package():
    """The package in the directory `fni8-serve_amd`, imported as fni8serve_amd."""
    name = "fni8serve_amd"
    if name not in sys.modules:
        home = os.path.join(os.getcwd(), "fni8-serve_amd")
        spec = importlib.util.spec_from_file_location(
            name, os.path.join(home, "__init__.py"), submodule_search_locations=[home])
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


def _case(kind, tokens, hidden, **more):
    c = {"kind": kind, "tokens": tokens, "hidden": hidden, "inter": 0, "out": 0, "bits": 8,
         "group": 0, "bias": False, "act": "silu", "experts": 0, "top_k": 0}
    c.update(more)
    return c


def listed():
    cases = [
        # single-stream decode, one projection called eagerly: the smallest call
        ("o_1tok", _case("linear", 1, 4096, out=4096)),
        # a small decode batch through the MLP, eagerly
        ("mlp_16tok", _case("mlp", 16, 4096, inter=12288)),
        # a larger decode batch: one whole layer's linears replayed from a graph
        ("layer_48tok_graph", _case("layer", 48, 4096, inter=12288, out=6144)),
        # a short ragged prompt: norm + quantization feeding a QKV with bias
        ("qkv_333tok", _case("norm_linear", 333, 4096, out=6144, bias=True)),
        # a ragged prompt through one of eight tensor-parallel shards of a GELU MLP:
        # the shard's width is no multiple of 64
        ("mlp_shard_777tok", _case("mlp", 777, 4096, inter=1376, act="gelu_pytorch_tanh")),
        # a full prefill chunk through the MLP: the largest work
        ("mlp_4096tok", _case("mlp", 4096, 4096, inter=12288)),
        # logits of eight sequences
        ("head_8tok", _case("head", 8, 4096, out=151936)),
        # MoE decode: few rows per expert, weights dominate
        ("moe_16tok", _case("moe", 16, 2048, inter=768, experts=128, top_k=8)),
        # MoE prefill: ragged segments of many rows
        ("moe_3000tok", _case("moe", 3000, 2048, inter=768, experts=128, top_k=8)),
        # int4 weights: a small decode batch
        ("mlp_int4_6tok", _case("mlp", 6, 4096, inter=12288, bits=4, group=128)),
        # int4 weights: a ragged prefill chunk
        ("mlp_int4_1500tok", _case("mlp", 1500, 4096, inter=12288, bits=4, group=128)),
        # int4 experts: a large decode batch or a short prompt
        ("moe_int4_200tok", _case("moe", 200, 2048, inter=768, experts=128, top_k=8, bits=4,
                                  group=128)),
    ]
    return [dict(c, name=n) for n, c in cases]


# hidden, inter, qkv width: the repository's model shapes and generic ones; the last
# two are shards (widths that are no multiple of 64) and run fewer tokens
_DENSE = ((1024, 3072, 4096), (1536, 4608, 2560), (4096, 12288, 6144), (4096, 1376, 768),
          (2080, 5472, 3130))


def _tokens(rng, most):
    """1..most, even over the logarithm."""
    return max(1, min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1.0))))))


def draw(rng):
    kind = rng.choice(("linear", "norm_linear", "mlp", "mlp", "layer", "head", "moe", "mlp4",
                       "mlp4", "moe4"))
    act = rng.choice(("silu", "silu", "gelu_pytorch_tanh"))
    if kind in ("moe", "moe4"):
        experts, top_k = rng.choice(((128, 8), (64, 6), (16, 2)))
        more = {"bits": 4, "group": rng.choice((64, 128))} if kind == "moe4" else {}
        return _case("moe", _tokens(rng, 2048 if more else 3000), rng.choice((1024, 2048)),
                     inter=768, act=act, experts=experts, top_k=top_k, **more)
    if kind == "mlp4":
        hidden, inter, _ = rng.choice(_DENSE[:3])
        return _case("mlp", _tokens(rng, 1500), hidden, inter=inter, act=act, bits=4,
                     group=rng.choice((32, 64, 128, 128)), bias=rng.random() < 0.2)
    hidden, inter, qkv = rng.choice(_DENSE)
    most = 4096 if inter % 64 == 0 else 777 if hidden % 64 == 0 else 48
    if kind == "head":
        hidden = rng.choice((1024, 1536, 4096))
        return _case("head", rng.randint(1, 64), hidden, out=rng.choice((32000, 50257, 151936)))
    if kind == "layer":
        return _case("layer", rng.randint(1, min(most, 128)), hidden, inter=inter, out=qkv,
                     act=act)
    if kind == "mlp":
        return _case("mlp", _tokens(rng, most), hidden, inter=inter, act=act,
                     bias=rng.random() < 0.2)
    return _case(kind, _tokens(rng, most), hidden, out=rng.choice((qkv, hidden, 2 * inter)),
                 bias=rng.random() < 0.3)


# ---- inputs ------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _activations(g, *shape):
    """N(0, 1) with 1% outliers of twenty times the size, as hidden states have."""
    x = torch.randn(*shape, generator=g, device="cuda")
    out = torch.rand(*shape, generator=g, device="cuda") < 0.01
    return torch.where(out, 20 * x, x).half()


def _weight(g, n, k, bits, group):
    """Codes of a normal weight of variance 1/k and their scales: int8 [n, k] and
    fp32 [n], or two int4 codes a byte [n, k/2] (low nibble first) and fp32 [n, k/group]."""
    w = torch.randn(n, k, generator=g, device="cuda")
    if bits == 8:
        s = (0.8 + 0.4 * torch.rand(n, generator=g, device="cuda")) / (35 * math.sqrt(k))
        return w.mul_(35).round_().clamp_(-127, 127).to(torch.int8), s
    s = (0.8 + 0.4 * torch.rand(n, k // group, generator=g, device="cuda")) / (2.7 * math.sqrt(k))
    c = w.mul_(2.7).round_().clamp_(-8, 7).to(torch.int32) & 15
    return (c[:, 0::2] | (c[:, 1::2] << 4)).to(torch.uint8), s


def _vector(g, n, centre, spread):
    return (centre + spread * torch.randn(n, generator=g, device="cuda")).half()


def _inputs(case, seed):
    """Every tensor of the case in plain torch, made from the seed."""
    g = _gen(seed)
    m, h, i, n = case["tokens"], case["hidden"], case["inter"], case["out"]
    bits, group, kind = case["bits"], case["group"], case["kind"]

    def weight(rows, cols):
        return _weight(g, rows, cols, bits, group)

    t = {}
    if kind == "linear":
        t = {"x": _activations(g, m, h), "w": weight(n, h)}
    elif kind == "norm_linear":
        t = {"x": _activations(g, m, h), "res": _activations(g, m, h), "w": weight(n, h),
             "norm": _vector(g, h, 1.0, 0.1)}
    elif kind == "head":
        t = {"x": _activations(g, m, 3, h), "w": weight(n, h)}
    elif kind == "moe":
        e = case["experts"]
        t = {"x": _activations(g, 1, m, h),
             "gate": (torch.randn(e, h, generator=g, device="cuda") / math.sqrt(h)).half(),
             "experts": [(weight(2 * i, h), weight(h, i)) for _ in range(e)]}
    else:
        t = {"x": _activations(g, m, h), "gate_up": weight(2 * i, h), "down": weight(h, i)}
        if kind == "layer":
            t.update(res=_activations(g, m, h), attn=_activations(g, m, h), qkv=weight(n, h),
                     o=weight(h, h), norm=_vector(g, h, 1.0, 0.1), norm2=_vector(g, h, 1.0, 0.1))
    if case["bias"]:
        t["bias"] = _vector(g, n or 2 * i, 0.0, 0.5)
        t["bias_down"] = _vector(g, h, 0.0, 0.5)
    return t


def prepare(case, seed):
    pkg = _package()
    t = _inputs(case, seed)
    kind, h, act = case["kind"], case["hidden"], case["act"]
    scheme = {"scheme": "per_row_i8"} if case["bits"] == 8 else {
        "scheme": "per_group_i4", "group_size": case["group"], "codebook": "int4"}

    def qt(w):
        return pkg.QTensor(w[0], w[1], **scheme)

    def norm(w):
        return pkg.RMSNorm(h, 1e-6, w).requires_grad_(False)

    def mlp():
        return pkg.GatedMLP(qt(t["gate_up"]), qt(t["down"]), act=act,
                            bias_gate_up=t.get("bias"), bias_down=t.get("bias_down"))

    state = {"kind": kind, "pkg": pkg, "x": t["x"]}
    if kind == "linear":
        state["module"] = pkg.LinearW8A8(qt(t["w"]), t.get("bias"))
    elif kind == "norm_linear":
        state.update(res=t["res"], norm=norm(t["norm"]), w=qt(t["w"]), bias=t.get("bias"))
    elif kind == "mlp":
        state["module"] = mlp()
    elif kind == "head":
        state["module"] = pkg.LMHead(qt(t["w"]))
    elif kind == "moe":
        state["module"] = pkg.SparseMoE(
            gate=t["gate"], experts=[(qt(a), qt(b)) for a, b in t["experts"]],
            top_k=case["top_k"], act=act).requires_grad_(False)
    else:
        parts = {"norm": norm(t["norm"]), "norm2": norm(t["norm2"]), "mlp": mlp(),
                 "qkv": qt(t["qkv"]), "o": pkg.LinearW8A8(qt(t["o"]))}

        def step():
            xq, xs, res = parts["norm"].forward_quant(t["x"], t["res"])
            qkv = pkg.gemm_quantized(xq, xs, parts["qkv"])
            y, res = parts["norm2"](parts["o"](t["attn"]), res)
            return qkv, res, parts["mlp"](y)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = step()
        state.update(graph=graph, out=out, keep=(t, parts))
    return state


def run(state):
    kind = state["kind"]
    if kind == "layer":
        state["graph"].replay()
        return state["out"]
    if kind == "norm_linear":
        xq, xs, res = state["norm"].forward_quant(state["x"], state["res"])
        return state["pkg"].gemm_quantized(xq, xs, state["w"], state["bias"]), res
    if kind == "head":
        return state["module"](state["x"][:, -1])
    return state["module"](state["x"])


# ---- what a pass cannot do without -------------------------------------------

def _linear_work(case, m, n, k):
    size = n * k if case["bits"] == 8 else n * k // 2
    scales = 4 * n if case["bits"] == 8 else 4 * n * (k // case["group"])
    return size + scales + (2 * n if case["bias"] else 0), 2.0 * m * n * k


def work(case):
    m, h, i, n = case["tokens"], case["hidden"], case["inter"], case["out"]
    kind = case["kind"]
    if kind == "moe":
        e, k = case["experts"], case["top_k"]
        active = e * (1.0 - (1.0 - k / e) ** m)
        up, f1 = _linear_work(case, m * k, 2 * i, h)
        down, f2 = _linear_work(case, m * k, h, i)
        return {"bytes": active * (up + down) + 2 * e * h + 4 * m * h,
                "flops": f1 + f2 + 2.0 * m * e * h}
    shapes = {"linear": [(n, h)], "norm_linear": [(n, h)], "head": [(n, h)],
              "mlp": [(2 * i, h), (h, i)],
              "layer": [(n, h), (h, h), (2 * i, h), (h, i)]}[kind]
    parts = [_linear_work(case, m, a, b) for a, b in shapes]
    io = {"linear": h + n, "norm_linear": 3 * h + n, "head": h + n, "mlp": 2 * h,
          "layer": 5 * h + n}[kind]
    norms = {"norm_linear": 2 * h, "layer": 4 * h}.get(kind, 0)
    return {"bytes": sum(p[0] for p in parts) + norms + 2 * m * io,
            "flops": sum(p[1] for p in parts)}


# ---- the same in 64 bits -----------------------------------------------------

def _w64(w, bits, group):
    codes, s = w
    if bits == 8:
        return codes.double(), s.double()
    c = torch.stack([codes & 15, codes >> 4], -1).reshape(codes.shape[0], -1).double()
    c = torch.where(c >= 8, c - 16, c)
    full = (c.reshape(c.shape[0], -1, group) * s.double().unsqueeze(-1)).reshape(c.shape)
    return full, torch.ones(c.shape[0], dtype=torch.float64, device=c.device)


def _linear64(x, w, case, bias=None):
    s = x.abs().amax(-1, keepdim=True).clamp_min(1e-6) / 127
    q = torch.round(x / s).clamp(-127, 127)
    codes, ws = _w64(w, case["bits"], case["group"])
    y = (q @ codes.t()) * s * ws
    return y if bias is None else y + bias.double()


def _norm64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w.double()


def _mlp64(x, up, down, case, b1=None, b2=None):
    gate, value = _linear64(x, up, case, b1).chunk(2, -1)
    if case["act"] == "silu":
        a = gate * torch.sigmoid(gate)
    else:
        a = torch.nn.functional.gelu(gate, approximate="tanh")
    return _linear64(a * value, down, case, b2)


def _moe64(x, t, case):
    scores = torch.softmax(x @ t["gate"].double().t(), -1)
    topw, topi = torch.topk(scores, case["top_k"], -1)
    topw = topw / topw.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e, (up, down) in enumerate(t["experts"]):
        row, slot = (topi == e).nonzero(as_tuple=True)
        if row.numel():
            out.index_add_(0, row, _mlp64(x[row], up, down, case) * topw[row, slot].unsqueeze(-1))
    return out


def exact(case, seed):
    t = _inputs(case, seed)
    kind, b1, b2 = case["kind"], t.get("bias"), t.get("bias_down")
    x = t["x"].double()
    if kind == "linear":
        return _linear64(x, t["w"], case, b1)
    if kind == "head":
        return _linear64(x[:, -1], t["w"], case)
    if kind == "norm_linear":
        x = x + t["res"].double()
        return _linear64(_norm64(x, t["norm"]), t["w"], case, b1), x
    if kind == "mlp":
        return _mlp64(x, t["gate_up"], t["down"], case, b1, b2)
    if kind == "moe":
        return _moe64(x[0], t, case).unsqueeze(0)
    x = x + t["res"].double()
    qkv = _linear64(_norm64(x, t["norm"]), t["qkv"], case)
    x = x + _linear64(t["attn"].double(), t["o"], case)
    return qkv, x, _mlp64(_norm64(x, t["norm2"]), t["gate_up"], t["down"], case)


def tolerance(case):
    # fp16 results of exact integer sums; behind a norm or an activation a value
    # next to a rounding boundary may take the neighbouring int8 code, and in a
    # layer these add up over the chain.  About four times what the present code
    # shows against 64 bits (2.1e-4, 4.5e-3, 2.2e-2).
    return {"rel": {"linear": 1e-3, "head": 1e-3, "layer": 8e-2}.get(case["kind"], 1.8e-2)}
