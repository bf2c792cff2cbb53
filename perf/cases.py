"""Timed cases of the dense ML-ops path: what a program that uses this package has it do.

Each case is one call (or one block of calls) through a public entry point:
the Python op API (Tensor, fused_mlp, TensorSession) and, where a serving loop
holds its own buffers, the C ABI through the ctypes binding.  Inputs are
seeded torch tensors; the ops' outputs are returned as views of the buffers
that the package wrote, without a copy.

Kinds:
  matmul     C[m, n] = A[m, k] B[k, n]                 Tensor.matmul, or bch_sgemm (api "c")
  batched    C[b] = A[b] B[b]                          Tensor.batch_matmul
  mlp        act(act(x W1^T + b1) W2^T + b2)           fused_mlp, weights [out, in]
  attention  softmax(Q K^T / sqrt(D)) V, [B, H, S, D]  Tensor.causal_attention / attention
  decode     the same for a few query rows over a long
             cache, H / Hkv query heads a cache head   bch_sdpa_fwd_ex
  block      pre-norm transformer block                TensorSession.run
  rows       row softmax / layer norm / GELU           Tensor.softmax_dim / layer_norm_wgsl / gelu_wgsl
  gemm64     C = A B in float64, either transposed     bch_dgemm
"""
import ctypes
import math

import torch

from barracuda_amd import Activation, AttentionDims, Tensor, TensorSession, fused_mlp, get_device
from barracuda_amd import _native

LN_EPS = 1e-5


def listed():
    return [
        # one small product, the size of the reference's CPU-path matmul: launch latency counts
        {"name": "matmul_256", "kind": "matmul", "api": "c", "m": 256, "n": 256, "k": 256},
        # the square f32 product that bench.py reports
        {"name": "matmul_4096", "kind": "matmul", "api": "tensor", "m": 4096, "n": 4096, "k": 4096},
        # a product whose sizes divide by nothing: rows and columns of a data set as they come
        {"name": "matmul_ragged", "kind": "matmul", "api": "tensor", "m": 2047, "n": 3001, "k": 1537},
        # bench.py's batch of products
        {"name": "batched_16x1024", "kind": "batched", "batch": 16, "m": 1024, "n": 1024, "k": 1024},
        # one projection of a decode step with eight sequences in flight, weights [in, out]
        {"name": "decode_matmul_m8", "kind": "matmul", "api": "c", "m": 8, "n": 11008, "k": 4096},
        # the MLP of a decode step with 32 sequences in flight, weights [out, in]
        {"name": "mlp_decode_m32", "kind": "mlp", "m": 32, "d": 4096, "hidden": 11008, "act": "GELU"},
        # the same MLP over a prompt of 512 tokens
        {"name": "mlp_prefill_m512", "kind": "mlp", "m": 512, "d": 4096, "hidden": 11008, "act": "GELU"},
        # prefill attention, bench.py's shape
        {"name": "attention_causal", "kind": "attention", "b": 4, "h": 32, "sq": 2048, "skv": 2048, "d": 128,
         "causal": True},
        # one decode step's attention: a query row per sequence over a cache of 4096 keys, 8 cache heads
        {"name": "attention_decode", "kind": "decode", "b": 8, "h": 32, "hkv": 8, "sq": 1, "skv": 4096, "d": 128},
        # a small transformer block recorded once and run per batch: many short launches
        {"name": "session_block", "kind": "block", "s": 256, "h": 8, "d": 64},
        # row softmax, bench.py's shape
        {"name": "softmax_rows", "kind": "rows", "op": "softmax", "rows": 65536, "cols": 2048},
        # double-precision product
        {"name": "gemm_f64", "kind": "gemm64", "m": 2048, "n": 2048, "k": 2048, "ta": False, "tb": False},
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of lo .. hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng, lo, hi):
    """_log, half of the time rounded to a multiple of 64 as layer widths are."""
    v = _log(rng, lo, hi)
    return max(64, v // 64 * 64) if rng.random() < 0.5 else v


def draw(rng):
    """A case of the listed ones' ranges that takes no longer than the largest of them."""
    while True:
        case = _draw(rng)
        if work(case)["flops"] <= (7e10 if case["kind"] == "matmul" else 3.5e10):
            return case


def _draw(rng):
    kind = rng.choice(["matmul", "matmul", "batched", "decode_matmul", "mlp", "mlp", "attention", "attention",
                       "decode", "block", "rows", "gemm64"])
    if kind == "matmul":
        return {"kind": "matmul", "api": rng.choice(["tensor", "c"]), "m": _dim(rng, 65, 4096),
                "n": _dim(rng, 65, 4096), "k": _dim(rng, 65, 4096)}
    if kind == "decode_matmul":
        return {"kind": "matmul", "api": "c", "m": _log(rng, 1, 64), "n": _dim(rng, 1024, 11008),
                "k": _dim(rng, 1024, 11008)}
    if kind == "batched":
        return {"kind": "batched", "batch": _log(rng, 2, 32), "m": _dim(rng, 65, 1024), "n": _dim(rng, 65, 1024),
                "k": _dim(rng, 65, 1024)}
    if kind == "mlp":
        return {"kind": "mlp", "m": _log(rng, 1, 1024), "d": _dim(rng, 512, 4096),
                "hidden": _dim(rng, 1024, 11008), "act": rng.choice(["GELU", "ReLU"])}
    if kind == "attention":
        causal = rng.random() < 0.5
        sq = _log(rng, 64, 2048)
        return {"kind": "attention", "b": rng.randint(1, 4), "h": rng.choice([4, 8, 12, 16, 32]), "sq": sq,
                "skv": sq if causal else _log(rng, 64, 2048), "d": rng.choice([32, 64, 80, 96, 128, 128]),
                "causal": causal}
    if kind == "decode":
        hkv = rng.choice([1, 4, 8, 32])
        return {"kind": "decode", "b": _log(rng, 1, 32), "h": 32, "hkv": hkv, "sq": rng.choice([1, 1, 1, 4]),
                "skv": _log(rng, 256, 8192), "d": rng.choice([64, 128])}
    if kind == "block":
        return {"kind": "block", "s": _log(rng, 64, 1024), "h": rng.choice([4, 8, 12, 16]),
                "d": rng.choice([32, 64, 128])}
    if kind == "rows":
        cols = _log(rng, 64, 16384)
        return {"kind": "rows", "op": rng.choice(["softmax", "layer_norm", "gelu"]),
                "rows": _log(rng, 64, max(65, (1 << 27) // cols)), "cols": cols}
    return {"kind": "gemm64", "m": _dim(rng, 65, 2048), "n": _dim(rng, 65, 2048), "k": _dim(rng, 65, 2048),
            "ta": rng.random() < 0.25, "tb": rng.random() < 0.5}


# ---- inputs -------------------------------------------------------------------


def _inputs(case, seed):
    """The case's inputs as torch tensors on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, sigma=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype) * sigma

    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        # a decode step's weights have the spread of a trained layer's
        return {"a": normal(m, k), "b": normal(k, n, sigma=0.02 if m <= 64 else 1.0)}
    if kind == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"a": normal(b, m, k), "b": normal(b, k, n)}
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["hidden"]
        return {"x": normal(m, d), "w1": normal(f, d, sigma=0.02), "b1": normal(f, sigma=0.02),
                "w2": normal(d, f, sigma=0.02), "b2": normal(d, sigma=0.02)}
    if kind == "attention":
        b, h, sq, skv, d = (case[x] for x in ("b", "h", "sq", "skv", "d"))
        return {"q": normal(b, h, sq, d), "k": normal(b, h, skv, d), "v": normal(b, h, skv, d)}
    if kind == "decode":
        b, h, hkv, sq, skv, d = (case[x] for x in ("b", "h", "hkv", "sq", "skv", "d"))
        return {"q": normal(b, h, sq, d), "k": normal(b, hkv, skv, d), "v": normal(b, hkv, skv, d)}
    if kind == "block":
        s, w = case["s"], case["h"] * case["d"]
        r = 1.0 / math.sqrt(w)
        return {"x": normal(s, w), "wq": normal(w, w, sigma=r), "wk": normal(w, w, sigma=r),
                "wv": normal(w, w, sigma=r), "wo": normal(w, w, sigma=r), "w1": normal(w, 4 * w, sigma=r),
                "w2": normal(4 * w, w, sigma=0.5 * r)}
    if kind == "rows":
        return {"x": normal(case["rows"], case["cols"], sigma=3.0)}
    m, n, k = case["m"], case["n"], case["k"]
    return {"a": normal(*((k, m) if case["ta"] else (m, k)), dtype=torch.float64),
            "b": normal(*((n, k) if case["tb"] else (k, n)), dtype=torch.float64)}


class _Span:
    """Device memory that another object owns, for torch.as_tensor."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (ptr, False), "version": 2}


def _view(t):
    """A Tensor's (or SessionTensor's) buffer as a torch tensor, without a copy."""
    return torch.as_tensor(_Span(t.ptr, t.shape(), getattr(t, "_session", t)), device="cuda")


def _tensor(x):
    """A Tensor that holds a copy of a torch tensor."""
    t = Tensor.empty(list(x.shape), get_device())
    _view(t).copy_(x)
    return t


def _p(x):
    return ctypes.c_void_p(x.data_ptr())


def _dense(h, s, d):
    return _native.AttnLayout(h * s * d, s * d, d)


def _session(case, t):
    """The block recorded in a session: x + attention(norm(x)), then the MLP the same way."""
    dims = AttentionDims(1, case["h"], case["s"], case["d"])
    w = case["h"] * case["d"]
    ses = TensorSession.with_device(get_device())
    i = {k: ses.import_(v) for k, v in t.items()}
    n1 = ses.layer_norm(i["x"], w)
    q, k, v = (ses.head_split(ses.matmul(n1, i[x]), dims) for x in ("wq", "wk", "wv"))
    o = ses.reshape(ses.head_concat(ses.attention(q, k, v, dims), dims), [case["s"], w])
    h = ses.add(i["x"], ses.matmul(o, i["wo"]))
    up = ses.gelu(ses.matmul(ses.layer_norm(h, w), i["w1"]))
    return ses, ses.add(h, ses.matmul(up, i["w2"]))


def prepare(case, seed):
    """Inputs, weights and handles in HBM; the C calls' outputs too, which a serving loop holds."""
    x = _inputs(case, seed)
    state = {"case": case}
    kind = case["kind"]
    if kind == "matmul" and case["api"] == "c":
        state.update(x, c=torch.empty(case["m"], case["n"], device="cuda"))
    elif kind == "decode":
        state.update(x, o=torch.empty_like(x["q"]))
    elif kind == "gemm64":
        state.update(x, c=torch.empty(case["m"], case["n"], device="cuda", dtype=torch.float64))
    elif kind == "block":
        ses, out = _session(case, {k: _tensor(v) for k, v in x.items()})
        get_device().sync()
        state.update(ses=ses, out=out)
    else:
        state.update({k: _tensor(v) for k, v in x.items()})
    state.update(dev=get_device(), lib=_native.load())
    torch.cuda.synchronize()
    return state


def run(state):
    case, dev, lib = state["case"], state["dev"], state["lib"]
    kind = case["kind"]
    if kind == "matmul":
        if case["api"] == "tensor":
            return _view(state["a"].matmul(state["b"]))
        m, n, k = case["m"], case["n"], case["k"]
        dev.check(lib.bch_sgemm(dev.ctx, m, n, k, _p(state["a"]), k, _p(state["b"]), n, _p(state["c"]), n), "matmul")
        return state["c"]
    if kind == "batched":
        return _view(state["a"].batch_matmul(state["b"]))
    if kind == "mlp":
        return _view(fused_mlp(state["x"], [state["w1"], state["w2"]], [state["b1"], state["b2"]],
                               Activation[case["act"]]))
    if kind == "attention":
        q, k, v = state["q"], state["k"], state["v"]
        return _view(q.causal_attention(k, v) if case["causal"] else q.attention(k, v))
    if kind == "decode":
        b, h, hkv, sq, skv, d = (case[x] for x in ("b", "h", "hkv", "sq", "skv", "d"))
        kv = _dense(hkv, skv, d)
        dev.check(lib.bch_sdpa_fwd_ex(dev.ctx, b, h, hkv, sq, skv, d, 1.0 / math.sqrt(d), 0,
                                      _p(state["q"]), _dense(h, sq, d), _p(state["k"]), kv, _p(state["v"]), kv,
                                      _p(state["o"]), _dense(h, sq, d)), "attention")
        return state["o"]
    if kind == "block":
        state["ses"].run()
        return _view(state["out"])
    if kind == "rows":
        x = state["x"]
        if case["op"] == "softmax":
            return _view(x.softmax_dim(1))
        return _view(x.layer_norm_wgsl(LN_EPS) if case["op"] == "layer_norm" else x.gelu_wgsl())
    m, n, k, ta, tb = case["m"], case["n"], case["k"], case["ta"], case["tb"]
    dev.check(lib.bch_dgemm(dev.ctx, int(ta), int(tb), 1, m, n, k, 1.0, _p(state["a"]), m if ta else k, m * k,
                            _p(state["b"]), k if tb else n, k * n, 0.0, _p(state["c"]), n, m * n), "gemm_f64")
    return state["c"]


# ---- what a pass cannot do without ------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"bytes": 4 * b * (m * k + k * n + m * n), "flops": 2 * b * m * n * k}
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["hidden"]
        return {"bytes": 4 * (2 * m * d + 2 * d * f + d + f), "flops": 4 * m * d * f}
    if kind == "attention":
        b, h, sq, skv, d = (case[x] for x in ("b", "h", "sq", "skv", "d"))
        pairs = sq * (sq + 1) // 2 if case["causal"] else sq * skv
        return {"bytes": 4 * b * h * d * (2 * sq + 2 * skv), "flops": 4 * b * h * pairs * d}
    if kind == "decode":
        b, h, hkv, sq, skv, d = (case[x] for x in ("b", "h", "hkv", "sq", "skv", "d"))
        return {"bytes": 4 * b * d * (2 * h * sq + 2 * hkv * skv), "flops": 4 * b * h * sq * skv * d}
    if kind == "block":
        s, w = case["s"], case["h"] * case["d"]
        return {"bytes": 4 * (2 * s * w + 12 * w * w), "flops": 24 * s * w * w + 4 * s * s * w}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n, "flops": 5 * n}
    m, n, k = case["m"], case["n"], case["k"]
    return {"bytes": 8 * (m * k + k * n + m * n), "flops": 2 * m * n * k}


def tolerance(case):
    """About four times the error against 64 bits that the float32 sums (2.3e-6 at most) and the float64 ones
    (1.1e-15 at k = 2048) show over these ranges."""
    return {"rel": 1e-14} if case["kind"] == "gemm64" else {"rel": 1e-5}


# ---- the same in 64 bits, in plain torch ----------------------------------------------


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x * x * x)))


def _norm(x):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + LN_EPS)


def _attend(q, k, v, causal=False):
    """Attention one (batch, head) at a time."""
    out = torch.empty_like(q)
    group = q.shape[1] // k.shape[1]
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = q[b, h] @ k[b, h // group].T.contiguous() / math.sqrt(q.shape[-1])
            if causal:
                s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -math.inf)
            out[b, h] = torch.softmax(s, -1) @ v[b, h // group]
    return out


def exact(case, seed):
    x = {k: v.double() for k, v in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "matmul":
        return x["a"] @ x["b"]
    if kind == "batched":
        return torch.stack([a @ b for a, b in zip(x["a"], x["b"])])
    if kind == "mlp":
        act = _gelu if case["act"] == "GELU" else torch.relu
        h = act(x["x"] @ x["w1"].T.contiguous() + x["b1"])
        return act(h @ x["w2"].T.contiguous() + x["b2"])
    if kind == "attention":
        return _attend(x["q"], x["k"], x["v"], case["causal"])
    if kind == "decode":
        return _attend(x["q"], x["k"], x["v"])
    if kind == "block":
        s, h, d = case["s"], case["h"], case["d"]
        n1 = _norm(x["x"])
        q, k, v = ((n1 @ x[w]).reshape(s, h, d).transpose(0, 1)[None].contiguous() for w in ("wq", "wk", "wv"))
        o = _attend(q, k, v)[0].transpose(0, 1).reshape(s, h * d)
        r = x["x"] + o @ x["wo"]
        return r + _gelu(_norm(r) @ x["w1"]) @ x["w2"]
    if kind == "rows":
        if case["op"] == "softmax":
            return torch.softmax(x["x"], -1)
        return _norm(x["x"]) if case["op"] == "layer_norm" else _gelu(x["x"])
    a = x["a"].T.contiguous() if case["ta"] else x["a"]
    b = x["b"].T.contiguous() if case["tb"] else x["b"]
    return a @ b
