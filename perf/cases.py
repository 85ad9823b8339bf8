"""The work this framework is timed on, through its public entry points.

Two families, as the package has them: the Arctic-embed-xs encoder (whole
calls, the feed-forward block, the attention core, int8-weight linears) and
the lazy expressions of `tenzor_amd.expr` (elementwise chains, reductions,
softmax, LayerNorm, matmul).  Sizes are those of the benchmark's workloads
(batch 256 x 512 ragged, batch 32 x 128, one sequence of 128 tokens, the
65 536-row linear, the 16384 x 16384 chain) and of the tests (4097-token
feed-forward, linears with k = 1000 and n = 1537), or generic.

`listed()` names the cases; `draw(rng)` gives further ones of the same
ranges; `prepare` builds what a program holds before the call, `run` is one
call, `exact` the same result from plain torch in 64 bits.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import tenzor_amd
from tenzor_amd import _abi, synth
from tenzor_amd.arctic import ModelWeights, feedForward, forwardBatch
from tenzor_amd.expr import BinaryExpr, LayerNormExpr, MatmulExpr, ReduceExpr, SoftmaxExpr, Tensor, evalInto

H, HEADS, INTER, LAYERS = 384, 12, 1536, 6
EPS = 1e-12  # arctic.Config.layer_norm_eps
_WEIGHTS_SEED = 1
_FFN_LAYER = 2


def listed():
    return [
        # a search query embedded alone: the smallest call, all latency
        dict(name="embed_1x128", kind="embed", batch=1, smin=128, smax=128, dtype="float32"),
        # document indexing: the headline batch of ragged sequences
        dict(name="embed_256x512", kind="embed", batch=256, smin=16, smax=512, dtype="float32"),
        # one encoder layer's feed-forward block of a mid-sized ragged batch
        dict(name="ffn_4097", kind="ffn", tokens=4097),
        # the attention core of a ragged batch in the default arithmetic
        dict(name="attention_f32_b64", kind="attention", batch=64, smin=16, smax=512, dtype="float32"),
        # and of the headline batch with the opt-in f16 activations
        dict(name="attention_f16_b256", kind="attention", batch=256, smin=16, smax=512, dtype="float16"),
        # caller-owned int8 weights: the wide linear with GELU at 65 536 rows
        dict(name="linear_gelu_65536", kind="linear", m=65536, k=384, n=1536, dtype="float32", epilogue="gelu"),
        # f16 activations, residual + LayerNorm epilogue, batch 32 x 128 rows
        dict(name="linear_ln_f16_4096", kind="linear", m=4096, k=1536, n=384, dtype="float16", epilogue="ln"),
        # a general W8A32 matmul of a model that is not Arctic: ragged in m, k and n
        dict(name="linear_odd_197", kind="linear", m=197, k=1000, n=1537, dtype="float32", epilogue="bias"),
        # a memory-sized elementwise chain: exp((A + b) * c)
        dict(name="chain_16384", kind="chain", rows=16384, cols=16384, form="scale_bias_exp", dtype="float32"),
        # mean pooling over the sequence axis of [batch, seq, hidden]
        dict(name="reduce_mean_pool", kind="reduce", outer=256, length=512, inner=384, axis="mid", op="mean",
             dtype="float32"),
        # attention probabilities of batch 32 x 12 heads x 128 queries x 128 keys
        dict(name="softmax_49152x128", kind="softmax", outer=49152, length=128, inner=1, dtype="float32"),
        # a dense layer as an expression: gelu(X W + b), the fused matmul epilogue
        dict(name="matmul_gelu_4096", kind="matmul", batch=1, m=4096, k=384, n=1536, epilogue="gelu",
             dtype="float32"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["embed", "ffn", "attention", "linear", "linear", "chain", "reduce", "softmax", "layernorm",
                       "matmul"])
    if kind in ("embed", "attention"):
        smax = _log_int(rng, 16, 512)
        smin = rng.choice([smax, max(1, smax // 4), min(16, smax)])
        dtype = rng.choice(["float32", "float32", "float16"])
        return dict(kind=kind, batch=_log_int(rng, 1, 256), smin=smin, smax=smax, dtype=dtype)
    if kind == "ffn":
        return dict(kind=kind, tokens=_log_int(rng, 16, 65536))
    if kind == "linear":
        dtype = rng.choice(["float32", "float32", "float16"])
        epilogue = rng.choice(["bias", "gelu", "ln"])
        m, k, n = _log_int(rng, 1, 65536), rng.choice([384, 1536, _log_int(rng, 17, 2048)]), rng.choice([384, 1152, 1536])
        if epilogue == "ln":
            n = 384
        elif dtype == "float32" and rng.random() < 0.5:
            n = _log_int(rng, 17, 2048)
        return dict(kind=kind, m=m, k=k, n=n, dtype=dtype, epilogue=epilogue)
    dtype = rng.choice(["float32", "float32", "float32", "float64"])
    if kind == "chain":
        return dict(kind=kind, rows=_log_int(rng, 1, 8192), cols=_log_int(rng, 1, 16384),
                    form=rng.choice(["scale_bias_exp", "gelu_bias", "axpby", "row_center"]), dtype=dtype)
    if kind == "reduce":
        axis, op = rng.choice(["last", "mid", "all"]), rng.choice(["sum", "mean", "reduce_max"])
        outer, length = _log_int(rng, 1, 4096), _log_int(rng, 8, 4096)
        inner = _log_int(rng, 256, 4096) if axis != "last" else 1
        while outer * length * inner > 1 << 26:
            outer = max(1, outer // 3)
            length = max(8, length // 2)
        return dict(kind=kind, outer=outer, length=length, inner=inner, axis=axis, op=op, dtype=dtype)
    if kind == "softmax":
        outer, length = _log_int(rng, 1, 65536), _log_int(rng, 8, 4096)
        inner = rng.choice([1, 1, _log_int(rng, 2, 512)])
        while outer * length * inner > 1 << 26:
            outer = max(1, outer // 3)
            inner = max(1, inner // 2)
        return dict(kind=kind, outer=outer, length=length, inner=inner, dtype=dtype)
    if kind == "layernorm":
        rows, cols = _log_int(rng, 1, 65536), rng.choice([384, 768, 1024, _log_int(rng, 17, 4096)])
        while rows * cols > 1 << 26:
            rows //= 2
        return dict(kind=kind, rows=rows, cols=cols, dtype=dtype)
    m, k, n = _log_int(rng, 1, 8192), _log_int(rng, 16, 2048), _log_int(rng, 16, 2048)
    batch = rng.choice([1, 1, _log_int(rng, 2, 64)])
    while batch * m * k * n > 1 << 34:
        m = max(1, m // 2)
    return dict(kind=kind, batch=batch, m=m, k=k, n=n, epilogue=rng.choice(["none", "bias", "gelu"]), dtype=dtype)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=1)
def _weights():
    """The model file's content: int8 linears, LayerNorm parameters around 1 and 0."""
    return synth.quantize(synth.make_arctic_f32(_WEIGHTS_SEED, synth.Config(), ln_random=True))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) + 1)


def _lengths(case):
    """The batch's sequence lengths, part of the case as every other size is."""
    rng = np.random.default_rng([7, case["batch"], case["smin"], case["smax"]])
    return rng.integers(case["smin"], case["smax"] + 1, size=case["batch"]).astype(np.int32)


def _dt(case):
    return getattr(torch, case["dtype"])


def _qkv(case, seed, lengths):
    T = int(lengths.sum())
    return torch.randn(T, 3 * H, device="cuda", generator=_generator(seed)).to(_dt(case))


def _embed_inputs(case, seed):
    lengths = _lengths(case)
    rng = np.random.default_rng([8, int(seed)])
    S = case["smax"]
    ids = rng.integers(1000, 30522, size=(case["batch"], S)).astype(np.int32)
    ids[:, 0] = 101
    ids[np.arange(S)[None, :] >= lengths[:, None]] = 0  # padding, as a tokenizer leaves it
    return ids, lengths


def _linear_inputs(case, seed):
    """Activations of a LayerNorm'd row, codes and scales of N(0, 0.02) weights."""
    g = _generator(seed)
    m, k, n = case["m"], case["k"], case["n"]
    a = torch.randn(m, k, device="cuda", generator=g).to(_dt(case))
    q = (torch.randn(n, k, device="cuda", generator=g) * 35.0).round().clamp(-127, 127).to(torch.int8)
    s = (torch.rand(n, device="cuda", generator=g) * 3e-4 + 4e-4).to(torch.float16)
    bias = torch.randn(n, device="cuda", generator=g) * 0.02
    d = dict(a=a, q=q, s=s, bias=bias)
    if case["epilogue"] == "ln":
        d["res"] = torch.randn(m, n, device="cuda", generator=g).to(_dt(case))
        d["gamma"] = 1.0 + 0.1 * torch.randn(n, device="cuda", generator=g)
        d["beta"] = 0.1 * torch.randn(n, device="cuda", generator=g)
    return d


def _eval_inputs(case, seed):
    g, dt, kind = _generator(seed), _dt(case), case["kind"]

    def randn(*shape):
        return torch.randn(*shape, device="cuda", generator=g, dtype=dt)

    if kind == "chain":
        r, c, form = case["rows"], case["cols"], case["form"]
        if form == "scale_bias_exp":
            return [torch.rand(*s, device="cuda", generator=g, dtype=dt) * 2 - 1 for s in ((r, c), (c,), (r, c))]
        if form == "gelu_bias":
            return [randn(r, c), randn(c)]
        if form == "axpby":
            return [randn(r, c), randn(r, c)]
        return [randn(r, c), randn(r, 1), randn(r, 1).abs() + 0.5]
    if kind == "reduce":
        shape = (case["outer"], case["length"]) + (() if case["axis"] == "last" else (case["inner"],))
        return [randn(*shape) for _ in range(2 if case["op"] == "sum" else 1)]
    if kind == "softmax":
        return [randn(case["outer"], case["length"], case["inner"]) * 3]
    if kind == "layernorm":
        c = case["cols"]
        return [randn(case["rows"], c) + 0.5, 1.0 + 0.1 * randn(c), 0.1 * randn(c)]
    m, k, n = case["m"], case["k"], case["n"]
    lead = (case["batch"],) if case["batch"] > 1 else ()
    return [randn(*lead, m, k), randn(*lead, k, n) / math.sqrt(k), randn(n) * 0.1]


def _expression(case, leaves):
    """The lazy expression of an eval case over its leaves."""
    t, kind = [Tensor(x) for x in leaves], case["kind"]
    if kind == "chain":
        form = case["form"]
        if form == "scale_bias_exp":
            return BinaryExpr("add", t[0], t[1]).mul(t[2]).exp()
        if form == "gelu_bias":
            return t[0].add(t[1]).gelu()
        if form == "axpby":
            return t[0].mul(0.75).add(t[1].mul(0.25))
        return t[0].sub(t[1]).mul(t[2])
    if kind == "reduce":
        axes = () if case["axis"] == "all" else (1,)
        if case["op"] == "sum":  # squared distances
            d = t[0].sub(t[1])
            return ReduceExpr("sum", d.mul(d), axes)
        if case["op"] == "mean":  # pooling of activations
            return ReduceExpr("mean", t[0].relu() if axes == () else t[0], axes)
        return ReduceExpr("reduce_max", t[0].abs(), axes)
    if kind == "softmax":
        return SoftmaxExpr(t[0], 1)
    if kind == "layernorm":
        return LayerNormExpr(t[0], t[1], t[2])
    e = MatmulExpr(t[0], t[1])
    if case["epilogue"] != "none":
        e = e.add(t[2])
    return e.gelu() if case["epilogue"] == "gelu" else e


def prepare(case, seed):
    kind = case["kind"]
    ctx = tenzor_amd.Context(0)
    st = dict(case=case, ctx=ctx)
    if kind in ("embed", "ffn"):
        st["model"] = ModelWeights.fromHost(ctx, _weights(), synth.Config())
    if kind == "embed":
        st["model"].set_precision(case["dtype"])
        ids, st["lengths"] = _embed_inputs(case, seed)
        st["ids"] = torch.from_numpy(ids).cuda()
        st["out"] = torch.empty(case["batch"], H, device="cuda")
    elif kind == "ffn":
        st["x"] = torch.randn(case["tokens"], H, device="cuda", generator=_generator(seed))
        st["out"] = torch.empty_like(st["x"])
    elif kind == "attention":
        lengths = _lengths(case)
        st["qkv"] = _qkv(case, seed, lengths)
        st["cu"] = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)).cuda()
        st["out"] = torch.empty(int(lengths.sum()), H, device="cuda", dtype=_dt(case))
    elif kind == "linear":
        st.update(_linear_inputs(case, seed))
        st["out"] = torch.empty(case["m"], case["n"], device="cuda", dtype=_dt(case))
    else:
        st["leaves"] = _eval_inputs(case, seed)
        st["expr"] = _expression(case, st["leaves"])
        st["out"] = torch.empty(st["expr"].shape, device="cuda", dtype=_dt(case))
    return st


def run(st):
    case, out, ctx = st["case"], st["out"], st["ctx"]
    kind = case["kind"]
    lib = tenzor_amd.lib()
    if kind == "embed":
        forwardBatch(out, st["ids"], st["lengths"], st["model"])
    elif kind == "ffn":
        feedForward(out, st["x"], st["model"], _FFN_LAYER, case["tokens"])
    elif kind == "attention":
        code = _abi.F32 if case["dtype"] == "float32" else _abi.F16
        tenzor_amd.check(lib.tzh_attention_varlen(ctx.handle, st["qkv"].data_ptr(), out.data_ptr(), code,
                                                  st["cu"].data_ptr(), case["batch"], HEADS, H))
    elif kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        w = (st["q"].data_ptr(), st["s"].data_ptr(), st["bias"].data_ptr(), out.data_ptr())
        if case["dtype"] == "float32" and case["epilogue"] == "bias":
            tenzor_amd.check(lib.tzh_matmul_w8a32(ctx.handle, st["a"].data_ptr(), *w, m, k, n))
            return out
        code = _abi.F32 if case["dtype"] == "float32" else _abi.F16
        epi = {"bias": _abi.EPI_BIAS, "gelu": _abi.EPI_BIAS_GELU, "ln": _abi.EPI_BIAS_RES_LN}[case["epilogue"]]
        extra = ((st["res"].data_ptr(), code, st["gamma"].data_ptr(), st["beta"].data_ptr()) if epi == _abi.EPI_BIAS_RES_LN
                 else (None, code, None, None))
        tenzor_amd.check(lib.tzh_linear_w8(ctx.handle, st["a"].data_ptr(), code, *w, code, m, k, n, epi, *extra, EPS))
    else:
        evalInto(st["expr"], out, ctx)
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("embed", "attention"):
        lengths = _lengths(case).astype(np.float64)
        T = float(lengths.sum())
        attn = 4.0 * float((lengths ** 2).sum()) * H
        if kind == "attention":
            es = 4 if case["dtype"] == "float32" else 2
            return {"bytes": T * 4 * H * es, "flops": attn}
        linears = H * 3 * H + H * H + 2 * H * INTER
        # ids and the rows of the word table they name, the layers' int8 weights, the embeddings
        return {"bytes": T * 4 + T * H * 4 + LAYERS * linears + case["batch"] * H * 4,
                "flops": LAYERS * (2.0 * T * linears + attn)}
    if kind == "ffn":
        return {"bytes": case["tokens"] * H * 8 + 2 * H * INTER, "flops": 4.0 * case["tokens"] * H * INTER}
    es = {"float16": 2, "float32": 4, "float64": 8}[case["dtype"]]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        res = m * n * es if case["epilogue"] == "ln" else 0
        return {"bytes": m * k * es + n * k + n * 6 + m * n * es + res, "flops": 2.0 * m * k * n}
    if kind == "chain":
        r, c = case["rows"], case["cols"]
        n, small = {"scale_bias_exp": (3, c), "gelu_bias": (2, c), "axpby": (3, 0), "row_center": (2, 2 * r)}[case["form"]]
        return {"bytes": (n * r * c + small) * es, "flops": 3.0 * r * c}
    if kind in ("reduce", "softmax"):
        n = case["outer"] * case["length"] * case["inner"]
        if kind == "softmax":
            return {"bytes": 2 * n * es, "flops": 5.0 * n}
        out = 1 if case["axis"] == "all" else n // case["length"]
        ins = 2 if case["op"] == "sum" else 1
        return {"bytes": (ins * n + out) * es, "flops": 2.0 * n}
    if kind == "layernorm":
        n = case["rows"] * case["cols"]
        return {"bytes": (2 * n + 2 * case["cols"]) * es, "flops": 8.0 * n}
    b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
    return {"bytes": (b * (m * k + k * n + m * n) + n) * es, "flops": 2.0 * b * m * k * n}


# Four times the largest relative error against `exact` that the listed sizes
# and the ends of the drawn ranges (sums of up to 4096 terms) showed, per kind
# and element type.
_REL = {
    "embed": {"float32": 1.1e-6, "float16": 3e-3},
    "ffn": {"float32": 4e-7},
    "attention": {"float32": 1.2e-6, "float16": 1.2e-3},
    "linear": {"float32": 1.8e-6, "float16": 9e-4},
    "chain": {"float32": 2.2e-7, "float64": 4e-16},
    "reduce": {"float32": 4.8e-6, "float64": 9e-15},
    "softmax": {"float32": 6.5e-7, "float64": 8e-15},
    "layernorm": {"float32": 3.2e-7, "float64": 6e-16},
    "matmul": {"float32": 3.6e-6, "float64": 4.8e-15},
}


def tolerance(case):
    if case["kind"] == "reduce" and case["op"] == "reduce_max":
        return "exact"
    return {"rel": _REL[case["kind"]][case.get("dtype", "float32")]}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _gelu(x):
    """The tanh form (arctic.zig:750-756)."""
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _layer_norm(x, gamma, beta, eps):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + eps) * gamma + beta


def _w64(name):
    """A weight of the model in 64 bits, int8 codes times their row scale."""
    w = _weights()
    a = torch.from_numpy(w[name]).cuda().double()
    if w[name].dtype == np.int8:
        s = torch.from_numpy(w[name + ".scale"].view(np.float16)).cuda().double()
        a = a * s[:, None]
    return a


def _linear64(x, prefix):
    return x @ _w64(prefix + ".weight").t().contiguous() + _w64(prefix + ".bias")


def _ffn64(x, layer):
    p = f"encoder.layer.{layer}."
    y = _linear64(_gelu(_linear64(x, p + "intermediate.dense")), p + "output.dense")
    return _layer_norm(x + y, _w64(p + "output.LayerNorm.weight"), _w64(p + "output.LayerNorm.bias"), EPS)


def _attention64(qkv, lengths):
    out = torch.empty(qkv.shape[0], H, device="cuda", dtype=torch.float64)
    d = H // HEADS
    s0 = 0
    for L in lengths:
        L = int(L)
        q, k, v = (qkv[s0:s0 + L, i * H:(i + 1) * H].reshape(L, HEADS, d).permute(1, 0, 2).contiguous() for i in range(3))
        p = torch.softmax(torch.bmm(q, k.permute(0, 2, 1).contiguous()) / math.sqrt(d), -1)
        out[s0:s0 + L] = torch.bmm(p, v).permute(1, 0, 2).reshape(L, H)
        s0 += L
    return out


def _embed64(case, seed):
    ids, lengths = _embed_inputs(case, seed)
    flat = np.concatenate([ids[b, :L] for b, L in enumerate(lengths)]).astype(np.int64)
    pos = np.concatenate([np.arange(L) for L in lengths])
    e = "embeddings."
    x = (_w64(e + "word_embeddings.weight")[torch.from_numpy(flat).cuda()]
         + _w64(e + "position_embeddings.weight")[torch.from_numpy(pos).cuda()]
         + _w64(e + "token_type_embeddings.weight")[0])
    x = _layer_norm(x, _w64(e + "LayerNorm.weight"), _w64(e + "LayerNorm.bias"), EPS)
    for layer in range(LAYERS):
        p = f"encoder.layer.{layer}.attention."
        qkv = torch.cat([_linear64(x, p + "self." + n) for n in ("query", "key", "value")], 1)
        a = _linear64(_attention64(qkv, lengths), p + "output.dense")
        x = _layer_norm(x + a, _w64(p + "output.LayerNorm.weight"), _w64(p + "output.LayerNorm.bias"), EPS)
        x = _ffn64(x, layer)
    first = np.concatenate([[0], np.cumsum(lengths)[:-1]]).astype(np.int64)
    cls = x[torch.from_numpy(first).cuda()]
    return cls / cls.norm(dim=-1, keepdim=True)


def exact(case, seed):
    kind = case["kind"]
    if kind == "embed":
        return _embed64(case, seed)
    if kind == "ffn":
        return _ffn64(torch.randn(case["tokens"], H, device="cuda", generator=_generator(seed)).double(), _FFN_LAYER)
    if kind == "attention":
        lengths = _lengths(case)
        return _attention64(_qkv(case, seed, lengths).double(), lengths)
    if kind == "linear":
        d = {key: v.double() for key, v in _linear_inputs(case, seed).items()}
        y = d["a"] @ (d["q"] * d["s"][:, None]).t().contiguous() + d["bias"]
        if case["epilogue"] == "gelu":
            return _gelu(y)
        return _layer_norm(d["res"] + y, d["gamma"], d["beta"], EPS) if case["epilogue"] == "ln" else y
    t = [x.double() for x in _eval_inputs(case, seed)]
    if kind == "chain":
        form = case["form"]
        if form == "scale_bias_exp":
            return torch.exp((t[0] + t[1]) * t[2])
        if form == "gelu_bias":
            return _gelu(t[0] + t[1])
        return t[0] * 0.75 + t[1] * 0.25 if form == "axpby" else (t[0] - t[1]) * t[2]
    if kind == "reduce":
        dim = (0, 1, 2) if case["axis"] == "all" else 1
        if case["op"] == "sum":
            return ((t[0] - t[1]) ** 2).sum(dim)
        if case["op"] == "mean":
            return (torch.relu(t[0]) if case["axis"] == "all" else t[0]).mean(dim)
        return t[0].abs().amax(dim)
    if kind == "softmax":
        z = torch.exp(t[0] - t[0].amax(1, keepdim=True))
        return z / z.sum(1, keepdim=True)
    if kind == "layernorm":
        return _layer_norm(t[0], t[1], t[2], float(np.float32(1e-5)))
    y = t[0] @ t[1]
    if case["epilogue"] != "none":
        y = y + t[2]
    return _gelu(y) if case["epilogue"] == "gelu" else y
