"""The work a user of this framework has it do, as cases that can be timed and compared.

One case is one pass through the public entry points of `functional`, on operands that live on the GPU:

  layer    the four linear layers of a decoder layer (qkv, o_proj, gate_up, down) on `m` rows, `layers` layers one
           behind the other with weights of their own: W4A16 with group or per-channel scales, W8A16, W4A8
           (W4A8: the two norms in front of qkv and gate_up included, which is where its activations become fp8)
  experts  the two expert matmuls of a mixture-of-experts layer (gate_up with SwiGLU, down) on the rows that `m` tokens
           send to their two experts each
  call     one matmul, called by itself

Decode passes (up to 256 rows) are replayed from a HIP graph that captured the entry points, which is how a serving
loop runs them; prefill passes and the single call go through the entry points each time.  Weights are quantized from
normally distributed ones and laid out by `preprocess_weights_for_mixed_gemm`, as a loader does it.
"""
import math

import torch

from __graft_entry__ import import_package

SHAPES = {  # hidden size, qkv columns, intermediate size (gate_up has twice as many columns)
    "llama3-8b": (4096, 6144, 14336),
    "llama3-70b": (8192, 10240, 28672),
    "mixtral-8x7b": (4096, 0, 14336),
}
LARGEST_FLOPS = 2.0 * 8192 * (4096 * 6144 + 4096 * 4096 + 3 * 4096 * 14336)


def _layer(name, shape, m, fmt, group, dtype, zero=False, smooth=False, bias=False, layers=1):
    hidden, qkv, inter = SHAPES[shape]
    return dict(name=name, kind="layer", m=m, hidden=hidden, qkv=qkv, inter=inter, fmt=fmt, group=group, dtype=dtype,
                zero=zero, smooth=smooth, bias=bias, layers=layers, graph=m <= 256)


def _experts(name, m, fmt, group, dtype, zero=False):
    hidden, _, inter = SHAPES["mixtral-8x7b"]
    return dict(name=name, kind="experts", m=m, hidden=hidden, inter=inter, experts=8, fmt=fmt, group=group,
                dtype=dtype, zero=zero, graph=m <= 128)


def listed():
    return [
        # one matmul called from Python outside a graph, smallest common size: what a call costs by itself
        dict(name="call-int8-1row", kind="call", m=1, k=4096, n=4096, fmt="int8", dtype="float16"),
        # one user decoding: the headline workload, GPTQ-style weights (scales and zeros per 128 rows of K)
        _layer("decode-1row", "llama3-8b", 1, "int4", 128, "bfloat16", zero=True, layers=2),
        # a small batch on AWQ-style weights (smoothing vector, symmetric), half precision
        _layer("decode-4row-awq", "llama3-8b", 4, "int4", 128, "float16", smooth=True, layers=2),
        # a medium batch on a large model with the finer group size
        _layer("decode-16row-g64", "llama3-70b", 16, "int4", 64, "bfloat16", zero=True),
        # a large decode batch (or a short chunk of prompt tokens), where reading weights and multiplying weigh alike
        _layer("decode-48row", "llama3-8b", 48, "int4", 128, "bfloat16", zero=True, layers=2),
        # the largest decode batches, on the large model
        _layer("decode-160row", "llama3-70b", 160, "int4", 128, "bfloat16", zero=True),
        # a ragged prompt on per-channel int8 weights, half precision
        _layer("prefill-333row-int8", "llama3-8b", 333, "int8", 0, "float16"),
        # the largest chunk of prompt tokens a server packs into one pass
        _layer("prefill-8192row", "llama3-8b", 8192, "int4", 128, "bfloat16", zero=True),
        # fp8 activations: decode, with the norms that produce them
        _layer("w4a8-decode-8row", "llama3-70b", 8, "w4a8", 128, "bfloat16", smooth=True),
        # fp8 activations: a ragged prompt
        _layer("w4a8-prefill-1990row", "llama3-8b", 1990, "w4a8", 128, "bfloat16", smooth=True),
        # mixture of experts while decoding: a handful of rows per expert
        _experts("experts-24token", 24, "int4", 128, "bfloat16", zero=True),
        # mixture of experts on a prompt chunk, per-channel scales as the reference's expert layers have them
        _experts("experts-300token", 300, "int4", 0, "float16"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["layer"] * 8 + ["experts"] * 2 + ["call"])
    dtype = rng.choice(["bfloat16", "float16"])
    if kind == "call":
        k, n = 128 * _log_int(rng, 8, 64), 16 * _log_int(rng, 64, 640)
        return dict(kind="call", m=rng.randint(1, 8), k=k, n=n, fmt=rng.choice(["int8", "int4"]), dtype=dtype)
    fmt = rng.choice(["int4"] * 5 + ["int8"] * 2 + (["w4a8"] * 3 if kind == "layer" else []))
    group = {"int4": [128, 128, 128, 64, 64, 0], "int8": [0, 0, 128], "w4a8": [128]}[fmt]
    group = rng.choice(group)
    zero = group != 0 and fmt == "int4" and rng.random() < 0.6
    if kind == "experts":
        hidden, inter = 128 * rng.randint(16, 32), 128 * rng.randint(40, 112)
        m = _log_int(rng, 1, 2048)
        return dict(kind="experts", m=m, hidden=hidden, inter=inter, experts=8, fmt=fmt, group=group, dtype=dtype,
                    zero=zero, graph=m <= 128)
    if rng.random() < 0.5:
        hidden, qkv, inter = SHAPES[rng.choice(["llama3-8b", "llama3-70b"])]
    else:
        hidden = 128 * _log_int(rng, 16, 64)
        qkv = 16 * int(hidden * rng.choice([1.25, 1.5, 3.0]) / 16 + rng.randint(0, 8))
        inter = 128 * int(hidden * rng.uniform(2.0, 3.5) / 128)
    weights = hidden * (qkv + hidden + 3 * inter)
    m = _log_int(rng, 1, max(2, min(8192, int(LARGEST_FLOPS / 2 / weights))))
    smooth = fmt == "w4a8" or (fmt == "int4" and group != 0 and rng.random() < 0.3)
    return dict(kind="layer", m=m, hidden=hidden, qkv=qkv, inter=inter, fmt=fmt, group=group, dtype=dtype, zero=zero,
                smooth=smooth, bias=group != 0 and rng.random() < 0.2, layers=2 if weights < 3e8 and m <= 256 else 1,
                graph=m <= 256)


class _Maker:
    """Operands from one seed, on the GPU; `plain`: each weight as its values in 64 bits instead of laid out."""

    def __init__(self, case, seed, plain=False):
        self.plain = plain
        self.pkg = None if plain else import_package()
        self.dev = torch.device("cuda:0")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)
        self.fmt, self.group, self.zero = case["fmt"], case.get("group", 0), case.get("zero", False)
        self.dtype = getattr(torch, case["dtype"])
        self.bits = 8 if self.fmt == "int8" else 4

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device=self.dev)

    def activations(self, m, k):
        # a few channels carry larger values, as they do in trained models
        channels = torch.where(torch.rand(k, generator=self.gen, device=self.dev) < 0.01, 6.0, 1.0)
        return (self.normal(m, k) * channels).to(self.dtype)

    def gated(self, m, k):
        return (torch.nn.functional.silu(self.normal(m, k)) * self.normal(m, k)).to(self.dtype)

    def quantized(self, k, n):
        """(laid-out weight on the GPU, scales, zeros or None) of one [k, n] matrix."""
        w = self.normal(k, n) * 0.02
        scale_type = torch.float16 if self.fmt == "w4a8" else self.dtype
        rows = self.group or k
        grouped = w.view(-1, rows, n)
        half = 1 << (self.bits - 1)
        if self.zero:
            low, high = grouped.amin(1), grouped.amax(1)
            scales = ((high - low) / (2 * half - 1)).to(scale_type)
            point = torch.round(-low / scales.float()).clamp(0, 2 * half - 1)
            q = (torch.round(grouped / scales.float()[:, None]) + point[:, None]).clamp(0, 2 * half - 1) - half
            zeros = ((half - point) * scales.float()).to(scale_type)
        else:
            scales = (grouped.abs().amax(1) / (half - 0.5)).to(scale_type)
            q = torch.round(grouped / scales.float()[:, None]).clamp(-half, half - 1)
            zeros = None
        if self.plain:
            w = q.double() * scales.double()[:, None] + (zeros.double()[:, None] if zeros is not None else 0.0)
            return (_e4m3(w) if self.fmt == "w4a8" else w).view(k, n), None, None
        q = q.view(k, n).to(torch.int8)
        if not self.group:
            scales = scales.view(n)
        if self.bits == 4:
            q = (q[:, 0::2] & 0xF) | (q[:, 1::2] << 4)
        kind = torch.int8 if self.bits == 8 else torch.quint4x2
        return self.pkg.ops.preprocess_weights_for_mixed_gemm(q.cpu(), kind, self.dtype).to(self.dev), scales, zeros

    def linear(self, k, n, smooth=False, bias=False):
        weight, scales, zeros = self.quantized(k, n)
        vector = (self.normal(k).abs() * 0.3 + 0.6).to(self.dtype) if smooth else None
        return dict(weight=weight, scales=scales, zeros=zeros, smooth=vector,
                    bias=self.normal(n).to(self.dtype) if bias else None, k=k, n=n)


def _linear(state, lin, x, smooth=True):
    """One linear layer through the functional interface."""
    F, case = state["F"], state["case"]
    if not case.get("group", 0):
        return F.weight_only_quant_matmul(x, lin["weight"], lin["scales"], F.INT8 if case["fmt"] == "int8" else F.INT4,
                                          case["dtype"])
    vector = lin["smooth"] if smooth else None
    algo = (F.ZERO if lin["zeros"] is not None else 0) | (F.BIAS if lin["bias"] is not None else 0) \
        | (F.PRE_QUANT_SCALE if vector is not None else 0) | (F.INT8_WEIGHT if case["fmt"] == "int8" else 0) \
        | (F.FP8_ALPHA if case["fmt"] == "w4a8" else 0)
    return F.weight_only_groupwise_quant_matmul(x, vector, lin["weight"], lin["scales"], lin["zeros"], lin["bias"],
                                                state["alpha"], algo, case["group"], case["dtype"])


def _pass(state):
    F, case = state["F"], state["case"]
    if case["kind"] == "call":
        return [_linear(state, state["linear"], state["x"])]
    if case["kind"] == "experts":
        rows, out = state["rows_before"], []
        algo = (F.ZERO if case["zero"] else 0) | (F.INT8_WEIGHT if case["fmt"] == "int8" else 0)
        x = state["x"]
        for lin, activation in ((state["fc1"], "swiglu"), (state["fc2"], "identity")):
            x = F.woq_grouped_matmul_raw(x, lin["weight"], lin["scales"], lin["zeros"], None, rows, n=lin["n"],
                                         k=lin["k"], group_size=case["group"], quant_algo=algo, activation=activation)
            out.append(x)
        return out
    out = []
    for qkv, o_proj, gate_up, down, norms in state["layers"]:
        x, x2, fp8 = state["x"], state["x2"], case["fmt"] == "w4a8"
        if fp8:  # the norm smooths and casts in the same pass
            x = F.rmsnorm_prequant(x, norms[0], qkv["smooth"], 1e-5, None, torch.float8_e4m3fn)
            x2 = F.rmsnorm_prequant(x2, norms[1], gate_up["smooth"], 1e-5, None, torch.float8_e4m3fn)
        out += [_linear(state, qkv, x, not fp8), _linear(state, o_proj, state["attended"]),
                _linear(state, gate_up, x2, not fp8), _linear(state, down, state["gated"])]
    return out


def _operands(mk, case):
    m = case["m"]
    state = dict(case=case, alpha=0.75)
    if case["kind"] == "call":
        state["linear"] = mk.linear(case["k"], case["n"])
        state["x"] = mk.activations(m, case["k"])
    elif case["kind"] == "experts":
        experts, hidden, inter = case["experts"], case["hidden"], case["inter"]
        # every token goes to its two best experts; some experts are more popular than others
        liking = mk.normal(m, experts) + 0.4 * mk.normal(experts)
        counts = torch.bincount(liking.topk(2, dim=1).indices.view(-1), minlength=experts)
        state["rows_before"] = counts.cumsum(0).to(torch.int64)
        state["x"] = mk.activations(2 * m, hidden)
        for name, k, n in (("fc1", hidden, 2 * inter), ("fc2", inter, hidden)):
            each = [mk.quantized(k, n) for _ in range(experts)]
            state[name] = dict(k=k, n=n, weight=torch.stack([e[0] for e in each]),
                               scales=None if mk.plain else torch.stack([e[1] for e in each]),
                               zeros=torch.stack([e[2] for e in each]) if case["zero"] and not mk.plain else None)
    else:
        hidden, qkv, inter = case["hidden"], case["qkv"], case["inter"]
        sizes = ((hidden, qkv), (hidden, hidden), (hidden, 2 * inter), (inter, hidden))
        state["layers"] = []
        for _ in range(case["layers"]):
            linears = [mk.linear(k, n, case["smooth"], case["bias"]) for k, n in sizes]
            norms = [(1.0 + 0.1 * mk.normal(hidden)).to(mk.dtype) for _ in range(2)]
            state["layers"].append((*linears, norms))
        state["x"], state["x2"] = mk.activations(m, hidden), mk.activations(m, hidden)
        state["attended"], state["gated"] = mk.normal(m, hidden).to(mk.dtype), mk.gated(m, inter)
    return state


def prepare(case, seed):
    mk = _Maker(case, seed)
    state = _operands(mk, case)
    state["F"] = mk.pkg.functional
    if case.get("graph"):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            _pass(state)  # first use of every kernel, outside the capture
            stream.synchronize()
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"], stream=stream):
                state["out"] = _pass(state)
        torch.cuda.current_stream().wait_stream(stream)
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


def _e4m3(x):
    return x.float().to(torch.float8_e4m3fn).double()


def exact(case, seed):
    """The outputs of `run` in 64 bits.  Where activations and weights become e4m3, that rounding is part of what is
    asked for and is kept; every other rounding is left out."""
    mk = _Maker(case, seed, plain=True)
    st = _operands(mk, case)
    fp8 = case["fmt"] == "w4a8"

    def linear(lin, x, ready=False):
        x = x.double()
        if lin["smooth"] is not None and not ready:
            x = x * lin["smooth"].double()
            x = _e4m3(x.to(mk.dtype)) if fp8 else x
        y = x @ lin["weight"] * (st["alpha"] if fp8 else 1.0)
        return y if lin["bias"] is None else y + lin["bias"].double()

    def norm(x, gamma, smooth):
        x = x.double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * gamma.double()
        return _e4m3((x.to(mk.dtype).double() * smooth.double()).to(mk.dtype))

    if case["kind"] == "call":
        return [linear(st["linear"], st["x"])]
    if case["kind"] == "experts":
        ends = st["rows_before"].tolist()
        pick = [slice(begin, end) for begin, end in zip([0] + ends[:-1], ends)]
        x = st["x"].double()
        both = torch.cat([x[rows] @ w for rows, w in zip(pick, st["fc1"]["weight"])])
        value, gate = both.chunk(2, dim=1)
        hidden = value * torch.nn.functional.silu(gate)
        return [hidden, torch.cat([hidden[rows] @ w for rows, w in zip(pick, st["fc2"]["weight"])])]
    out = []
    for qkv, o_proj, gate_up, down, norms in st["layers"]:
        x, x2 = st["x"], st["x2"]
        if fp8:
            x, x2 = norm(x, norms[0], qkv["smooth"]), norm(x2, norms[1], gate_up["smooth"])
        out += [linear(qkv, x, fp8), linear(o_proj, st["attended"]), linear(gate_up, x2, fp8), linear(down, st["gated"])]
    return out


def _matmul_work(case, m, k, n, n_out=None, matrices=1.0):
    bits, group = (8 if case["fmt"] == "int8" else 4), case.get("group", 0)
    tables = (2 if case.get("zero") else 1) * ((k // group) if group else 1) * n * 2
    extra = (k * 2 if case.get("smooth") else 0) + (n * 2 if case.get("bias") else 0)
    return matrices * (k * n * bits / 8 + tables) + extra + m * k * 2 + m * (n_out or n) * 2, 2.0 * m * n * k


def work(case):
    m = case["m"]
    if case["kind"] == "call":
        parts = [_matmul_work(case, m, case["k"], case["n"])]
    elif case["kind"] == "experts":
        hidden, inter, e = case["hidden"], case["inter"], case["experts"]
        used = e * (1.0 - (1.0 - 2.0 / e) ** m)  # experts that some token chose, on average
        parts = [_matmul_work(case, 2 * m, hidden, 2 * inter, inter, used),
                 _matmul_work(case, 2 * m, inter, hidden, hidden, used)]
    else:
        hidden, qkv, inter = case["hidden"], case["qkv"], case["inter"]
        sizes = ((hidden, qkv), (hidden, hidden), (hidden, 2 * inter), (inter, hidden))
        parts = [_matmul_work(case, m, k, n) for k, n in sizes] * case["layers"]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # Against a float64 product of the same operands the outputs differ by the rounding of the weights to the
    # activation type (which kernels that keep the scale out of the weight skip) and by their own rounding:
    # measured 1.7e-3 ... 2.2e-3 (largest value 1.1e-2) in bfloat16, 2e-4 ... 3.6e-4 (4.5e-3) in float16.
    # Four times that.
    return {"rel": 9e-3, "max": 0.045} if case["dtype"] == "bfloat16" else {"rel": 1.5e-3, "max": 0.018}
