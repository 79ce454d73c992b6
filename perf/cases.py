"""The work that programs give this backend, as measurable cases.

Three kinds of entry point are called the way programs call them: the direct
ops on device tensors (gomlx_hip.ops), the graph API (Builder -> Compile ->
Execute, gomlx_hip.backend) and the ready-made model graphs (gomlx_hip.graphs).
A graph is compiled once for its sizes and kept while any prepared state uses
it; inputs are device buffers filled from the seed, and Execute's output buffers
come back as tensors over the same device memory.

`listed` names the fixed cases, `draw` gives more from the same ranges, and
`exact` evaluates a case in float64 with plain torch.
"""
import math
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "go-darwinml_amd"))

from gomlx_hip import graphs, ops  # noqa: E402
from gomlx_hip.backend import ActivationType, AxesLayout, Backend, dtypes, make_shape  # noqa: E402

DEV = "cuda"
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
ACT = {"none": ActivationType.NONE, "gelu": ActivationType.GELU, "relu": ActivationType.RELU,
       "silu": ActivationType.SILU, "tanh": ActivationType.TANH}
EPS = 1e-6


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # A decoding step's normalisation of 16 sequences: the smallest call.
        {"name": "rmsnorm_decode", "kind": "norm", "op": "rms", "rows": 16, "n": 4096, "dtype": "bf16"},
        # Normalisation over a training batch's tokens (the benchmark's headline size).
        {"name": "rmsnorm_train", "kind": "norm", "op": "rms", "rows": 8192, "n": 4096, "dtype": "f32"},
        # Token log-probabilities over a vocabulary whose rows do not divide into vectors.
        {"name": "log_softmax_vocab", "kind": "softmax", "rows": 2048, "n": 32003, "log": True, "dtype": "f32"},
        # The batched product the benchmark quotes.
        {"name": "dot_batched", "kind": "dot", "B": 8, "M": 2048, "K": 4096, "N": 4096, "ta": False, "tb": False,
         "dtype": "bf16"},
        # A feed-forward layer with bias and activation on a ragged batch of tokens.
        {"name": "dense_ragged", "kind": "dense", "M": 1000, "K": 1531, "N": 776, "act": "gelu", "dtype": "bf16"},
        # Prefill: causal self-attention (the benchmark's size).
        {"name": "attn_prefill", "kind": "attn", "B": 4, "H": 16, "Hkv": 16, "Sq": 2048, "Sk": 2048, "D": 128,
         "mask": "causal", "dtype": "bf16"},
        # Encoder attention over padded sequences of a ragged length, with a key padding mask.
        {"name": "attn_padded", "kind": "attn", "B": 8, "H": 12, "Hkv": 12, "Sq": 1000, "Sk": 1000, "D": 64,
         "mask": "padding", "dtype": "f16"},
        # Decoding: one query per sequence over a long KV cache, grouped-query heads.
        {"name": "attn_decode", "kind": "attn", "B": 8, "H": 32, "Hkv": 8, "Sq": 1, "Sk": 8192, "D": 128,
         "mask": "none", "dtype": "bf16"},
        # A decoding step of one decoder block for 16 sequences through the graph API.
        {"name": "decode_step", "kind": "decode", "B": 16, "cache": 4096, "d": 4096, "H": 32, "Hkv": 8, "ffn": 14336},
        # Prefill of one decoder block through the graph API.
        {"name": "block_prefill", "kind": "block", "B": 8, "S": 1024, "d": 2048, "H": 16, "ffn": 8192},
        # A training step's gradients of a text classifier in float32: embedding lookup,
        # mean over the tokens, two dense layers, cross-entropy, and back to the table.
        {"name": "classifier_grads", "kind": "classifier", "B": 256, "L": 50, "V": 32000, "E": 256, "H": 512, "C": 10},
        # A training step's gradients of a decoder block's feed-forward half (RMSNorm,
        # SwiGLU, residual) in bfloat16.
        {"name": "ffn_grads", "kind": "ffn", "T": 4096, "d": 2048, "ffn": 8192},
    ]


def _size(rng, lo, hi, step=1):
    """A size in [lo, hi], spread over the logarithm; a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["norm", "softmax", "dot", "dense", "attn", "attn", "attn_decode", "decode", "block",
                       "classifier", "ffn"])
    if kind == "norm":
        n = _size(rng, 64, 8192, rng.choice([1, 8, 128]))
        return {"kind": kind, "op": rng.choice(["rms", "layer"]), "rows": _size(rng, 1, 8192), "n": n,
                "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "softmax":
        n = _size(rng, 10, 65536, rng.choice([1, 8]))
        return {"kind": kind, "rows": _size(rng, 1, max(1, min(8192, (1 << 26) // n))), "n": n,
                "log": rng.random() < 0.5, "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "dot":
        B = rng.choice([1, 1, 2, 4, 8, 16])
        dt = rng.choice(["f32", "bf16", "bf16", "f16"])
        hi = 2048 if dt == "f32" else 4096
        step = rng.choice([1, 8, 64, 256])
        if step == 1:
            hi //= 2
        M, K, N = (_size(rng, 16, hi, step) for _ in range(3))
        return {"kind": kind, "B": min(B, max(1, (1 << 34) // (M * K * N))), "M": M, "K": K, "N": N,
                "ta": rng.random() < 0.3, "tb": rng.random() < 0.3, "dtype": dt}
    if kind == "dense":
        step = rng.choice([1, 8, 64])
        hi = 2048 if step == 1 else 8192
        return {"kind": kind, "M": _size(rng, 1, 8192), "K": _size(rng, 32, hi, step), "N": _size(rng, 16, hi, step),
                "act": rng.choice(["none", "gelu", "relu", "silu", "tanh"]), "dtype": rng.choice(["f32", "bf16", "bf16", "f16"])}
    if kind == "attn":
        D = rng.choice([64, 64, 128, 128, 128, 80, 96, 256])
        Hkv = rng.choice([1, 2, 4, 8])
        H = Hkv * rng.choice([1, 1, 2, 4])
        dt = rng.choice(["bf16", "bf16", "f16", "f32"]) if D in (64, 128) else rng.choice(["bf16", "f16"])
        S = _size(rng, 32, 1024 if dt == "f32" else 4096, rng.choice([1, 64]))
        B = _size(rng, 1, max(1, min(16, (1 << 28) // (H * S * S))))
        return {"kind": "attn", "B": B, "H": H, "Hkv": Hkv, "Sq": S, "Sk": S, "D": D,
                "mask": rng.choice(["causal", "causal", "none", "padding", "additive"]), "dtype": dt}
    if kind == "attn_decode":
        Hkv = rng.choice([1, 4, 8])
        return {"kind": "attn", "B": _size(rng, 1, 32), "H": Hkv * rng.choice([1, 4, 8]), "Hkv": Hkv,
                "Sq": rng.choice([1, 1, 1, 4]), "Sk": _size(rng, 128, 16384), "D": rng.choice([64, 128, 128]),
                "mask": "none", "dtype": rng.choice(["bf16", "f16"])}
    if kind == "decode":
        Hkv = rng.choice([4, 8])
        H = Hkv * rng.choice([1, 2, 4])
        return {"kind": kind, "B": _size(rng, 1, 32), "cache": _size(rng, 256, 4096), "d": _size(rng, 512, 4096, 128),
                "H": H, "Hkv": Hkv, "ffn": _size(rng, 1024, 14336, 256)}
    if kind == "block":
        H = rng.choice([4, 8, 16])
        S = _size(rng, 64, 2048, rng.choice([1, 64]))
        return {"kind": kind, "B": _size(rng, 1, max(1, 8192 // S)), "S": S, "d": H * 128, "H": H,
                "ffn": H * rng.choice([352, 512])}
    if kind == "classifier":
        return {"kind": kind, "B": _size(rng, 16, 1024), "L": _size(rng, 4, 64), "V": _size(rng, 1000, 64000),
                "E": _size(rng, 32, 512, rng.choice([1, 8, 64])), "H": _size(rng, 32, 1024, rng.choice([1, 8, 64])),
                "C": _size(rng, 2, 1000)}
    return {"kind": kind, "T": _size(rng, 64, 4096), "d": _size(rng, 512, 2048, 128), "ffn": _size(rng, 1024, 8192, 256)}


def work(case):
    c, k = case, case["kind"]
    es = 4 if c.get("dtype") == "f32" else 2
    if k == "norm":
        params = c["n"] * (2 if c["op"] == "layer" else 1)
        return {"bytes": (2 * c["rows"] * c["n"] + params) * es, "flops": 5 * c["rows"] * c["n"]}
    if k == "softmax":
        return {"bytes": 2 * c["rows"] * c["n"] * es, "flops": 4 * c["rows"] * c["n"]}
    if k == "dot":
        B, M, K, N = c["B"], c["M"], c["K"], c["N"]
        return {"bytes": B * (M * K + K * N + M * N) * es, "flops": 2 * B * M * K * N}
    if k == "dense":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": (M * K + K * N + N + M * N) * es, "flops": 2 * M * K * N}
    if k == "attn":
        B, H, Hkv, Sq, Sk, D = (c[x] for x in ("B", "H", "Hkv", "Sq", "Sk", "D"))
        pairs = Sq * (Sq + 1) // 2 if c["mask"] == "causal" else Sq * Sk
        mask = B * Sk if c["mask"] == "padding" else Sq * Sk * es if c["mask"] == "additive" else 0
        return {"bytes": 2 * B * D * (H * Sq + Hkv * Sk) * es + mask, "flops": 4 * B * H * D * pairs}
    if k == "decode":
        cfg = _decode_cfg(c)
        weights = sum(math.prod(s.dims) for n, s in cfg.param_shapes() if n not in ("x", "k_cache", "v_cache", "g_attn", "g_ffn"))
        return {"bytes": cfg.bytes(), "flops": c["B"] * (2 * weights + 4 * c["H"] * 128 * c["cache"])}
    if k == "block":
        T, d, S = c["B"] * c["S"], c["d"], c["S"]
        n = sum(math.prod(s.dims) for name, s in _block_cfg(c).param_shapes() if name not in ("ids", "embedding"))
        attn = 4 * c["B"] * c["H"] * 128 * (S * (S + 1) // 2)
        return {"bytes": 2 * (n + 2 * T * d) + 4 * T, "flops": 2 * T * (4 * d * d + 3 * d * c["ffn"]) + attn}
    if k == "classifier":
        B, L, V, E, H, C = (c[x] for x in "BLVEHC")
        return {"bytes": 4 * (2 * B * L * E + V * E + 2 * (E * H + H * C + H + C) + B * L + B * C),
                "flops": 6 * B * (E * H + H * C)}
    T, d, f = c["T"], c["d"], c["ffn"]
    return {"bytes": 2 * (4 * T * d + 2 * (3 * d * f + d)), "flops": 18 * T * d * f}


def tolerance(case):
    """Relative (2-norm) and largest differences that another evaluation at the same
    precision shows: about four times the distance between this library's results and
    float64 ones."""
    k, dt = case["kind"], case.get("dtype", "bf16")
    if k in ("norm", "softmax"):
        return {"f32": {"rel": 1e-6, "max": 1e-5}, "f16": {"rel": 1e-3, "max": 4e-3},
                "bf16": {"rel": 8e-3, "max": 3e-2}}[dt]
    if k in ("dot", "attn"):
        return {"f32": {"rel": 5e-6, "max": 2e-4}, "f16": {"rel": 1.2e-3, "max": 1e-2},
                "bf16": {"rel": 1e-2, "max": 6e-2}}[dt]
    if k == "dense":  # the bias and each step of the activation round once more
        return {"f32": {"rel": 5e-6, "max": 2e-4}, "f16": {"rel": 2.5e-3, "max": 2e-2},
                "bf16": {"rel": 1.5e-2, "max": 0.15}}[dt]
    if k == "classifier":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 2e-2, "max": 0.3}


# ---------------------------------------------------------------- inputs
def _normal(gen, shape, dtype, std=1.0):
    """N(0, std^2) values rounded to `dtype`."""
    return (torch.randn(shape, generator=gen, device=DEV) * std).to(dtype)


def _zipf(gen, shape, V):
    """Token ids in [0, V) with frequencies falling as 1 / rank, as in text."""
    u = torch.rand(shape, generator=gen, device=DEV, dtype=torch.float64)
    return (torch.pow(float(V), u) - 1).to(torch.int32).clamp_(0, V - 1)


def _decode_cfg(c):
    return graphs.DecodeStepConfig(batch=c["B"], cache=c["cache"], d_model=c["d"], heads=c["H"], kv_heads=c["Hkv"],
                                   head_dim=128, ffn=c["ffn"], eps=EPS)


def _block_cfg(c):
    return graphs.TransformerBlockConfig(batch=c["B"], seq=c["S"], d_model=c["d"], heads=c["H"], head_dim=128,
                                         ffn=c["ffn"], eps=EPS)


def _inputs(case, seed):
    """The case's input tensors by name, made from the seed alone."""
    c, k = case, case["kind"]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    dt = TORCH.get(c.get("dtype"), torch.bfloat16)
    if k == "norm":
        t = {"x": _normal(g, (c["rows"], c["n"]), dt),
             "gamma": (0.5 + torch.rand(c["n"], generator=g, device=DEV)).to(dt)}
        if c["op"] == "layer":
            t["beta"] = _normal(g, (c["n"],), dt, 0.1)
        return t
    if k == "softmax":
        return {"x": _normal(g, (c["rows"], c["n"]), dt, 2.0)}
    if k == "dot":
        std = c["K"] ** -0.25
        a = _normal(g, (c["B"], c["K"], c["M"]) if c["ta"] else (c["B"], c["M"], c["K"]), dt, std)
        b = _normal(g, (c["B"], c["N"], c["K"]) if c["tb"] else (c["B"], c["K"], c["N"]), dt, std)
        return {"a": a, "b": b}
    if k == "dense":
        return {"x": _normal(g, (c["M"], c["K"]), dt), "w": _normal(g, (c["K"], c["N"]), dt, c["K"] ** -0.5),
                "bias": _normal(g, (c["N"],), dt, 0.1)}
    if k == "attn":
        t = {"q": _normal(g, (c["B"], c["H"], c["Sq"], c["D"]), dt),
             "k": _normal(g, (c["B"], c["Hkv"], c["Sk"], c["D"]), dt),
             "v": _normal(g, (c["B"], c["Hkv"], c["Sk"], c["D"]), dt)}
        if c["mask"] == "padding":  # each sequence keeps its first half or more
            keep = c["Sk"] // 2 + torch.randint(0, c["Sk"] - c["Sk"] // 2 + 1, (c["B"], 1), generator=g, device=DEV)
            keep = keep.clamp_(min=1)
            t["mask"] = (torch.arange(c["Sk"], device=DEV)[None] < keep).view(c["B"], 1, 1, c["Sk"])
        elif c["mask"] == "additive":  # a position bias shared by all heads
            t["mask"] = _normal(g, (c["Sq"], c["Sk"]), dt)
        return t
    if k == "classifier":
        B, L, V, E, H, C = (c[x] for x in "BLVEHC")
        f = torch.float32
        return {"ids": _zipf(g, (B, L), V),
                "labels": torch.randint(0, C, (B,), generator=g, device=DEV, dtype=torch.int32),
                "table": _normal(g, (V, E), f), "w1": _normal(g, (E, H), f, E ** -0.5), "b1": _normal(g, (H,), f, 0.1),
                "w2": _normal(g, (H, C), f, H ** -0.5), "b2": _normal(g, (C,), f, 0.1)}
    if k == "ffn":
        T, d, f = c["T"], c["d"], c["ffn"]
        return {"x": _normal(g, (T, d), dt), "dy": _normal(g, (T, d), dt),
                "gamma": (0.5 + torch.rand(d, generator=g, device=DEV)).to(dt),
                "w_gate": _normal(g, (d, f), dt, d ** -0.5), "w_up": _normal(g, (d, f), dt, d ** -0.5),
                "w_down": _normal(g, (f, d), dt, f ** -0.5)}
    cfg = _decode_cfg(c) if k == "decode" else _block_cfg(c)
    t = {}
    for name, shape in cfg.param_shapes():
        if name == "ids":
            t[name] = _zipf(g, shape.dims, cfg.vocab)
        elif name.startswith("g_"):
            t[name] = (0.5 + torch.rand(shape.dims, generator=g, device=DEV)).to(dt)
        elif name in ("x", "embedding", "k_cache", "v_cache"):
            t[name] = _normal(g, shape.dims, dt)
        else:
            t[name] = _normal(g, shape.dims, dt, shape.dims[0] ** -0.5)
    return t


# ---------------------------------------------------------------- graphs
def _classifier_graph(f, p, c):
    """Loss and gradients of the classifier, as the primitives and fused ops that a
    differentiated graph program sends to the backend."""
    B, L, V, E, H, C = (c[x] for x in "BLVEHC")
    F32 = dtypes.Float32

    def scalar(v, *dims):
        return f.BroadcastInDim(f.Constant(np.array(v, np.float32), dtype=F32), make_shape(F32, *dims), [])

    idx = f.Reshape(p["ids"], B, L, 1)
    emb = f.Gather(p["table"], idx, 2, [2], [0], [0], [1, E], False)          # [B, L, E]
    mean = f.Mul(f.ReduceSum(emb, 1), scalar(1.0 / L, B, E))
    act = f.FusedDense(mean, p["w1"], p["b1"], ActivationType.RELU)           # [B, H]
    logits = f.FusedDense(act, p["w2"], p["b2"], ActivationType.NONE)         # [B, C]
    logp = graphs.log_softmax_chain(f, logits)
    classes = f.Iota(make_shape(dtypes.Int32, B, C), 1)
    hot = f.ConvertDType(f.Equal(classes, f.BroadcastInDim(p["labels"], make_shape(dtypes.Int32, B, C), [0])), F32)
    loss = f.Neg(f.Mul(f.ReduceSum(f.Mul(hot, logp), 0, 1), f.Constant(np.array(1.0 / B, np.float32), dtype=F32)))
    dlogits = f.Mul(f.Sub(f.Exp(logp), hot), scalar(1.0 / B, B, C))
    dw2 = f.DotGeneral(act, [0], [], dlogits, [0], [])
    db2 = f.ReduceSum(dlogits, 0)
    dact = f.DotGeneral(dlogits, [1], [], p["w2"], [1], [])
    dz = f.Where(f.GreaterThan(act, scalar(0.0, B, H)), dact, scalar(0.0, B, H))
    dw1 = f.DotGeneral(mean, [0], [], dz, [0], [])
    db1 = f.ReduceSum(dz, 0)
    dmean = f.Mul(f.DotGeneral(dz, [1], [], p["w1"], [1], []), scalar(1.0 / L, B, E))
    demb = f.BroadcastInDim(dmean, make_shape(F32, B, L, E), [0, 2])
    dtable = f.ScatterSum(scalar(0.0, V, E), idx, demb, 2, [2], [0], [0])
    return [loss, logits, dtable, dw1, db1, dw2, db2]


def _ffn_graph(f, p, c):
    """y = x + (silu(h Wg) * (h Wu)) Wd with h = RMSNorm(x) gamma, and the gradients of
    <y, dy>, as primitives."""
    T, d, n = c["T"], c["d"], c["ffn"]
    BF = dtypes.BFloat16
    xs, fs, rows = make_shape(BF, T, d), make_shape(BF, T, n), make_shape(BF, T)

    def scalar(v, shape):
        return f.BroadcastInDim(f.Constant(np.array(v, np.float32), dtype=BF), shape, [])

    def row_mean(v):
        return f.Mul(f.ReduceSum(v, 1), scalar(1.0 / d, rows))

    x, dy = p["x"], p["dy"]
    gamma = f.BroadcastInDim(p["gamma"], xs, [1])
    r = f.BroadcastInDim(f.Rsqrt(f.Add(row_mean(f.Mul(x, x)), scalar(EPS, rows))), xs, [0])
    xhat = f.Mul(x, r)
    h = f.Mul(xhat, gamma)
    gate, up = graphs.dense(f, h, p["w_gate"]), graphs.dense(f, h, p["w_up"])
    s = f.Logistic(gate)
    silu = f.Mul(gate, s)
    act = f.Mul(silu, up)
    y = f.Add(x, graphs.dense(f, act, p["w_down"]))
    dw_down = f.DotGeneral(act, [0], [], dy, [0], [])
    dact = f.DotGeneral(dy, [1], [], p["w_down"], [1], [])
    dup = f.Mul(dact, silu)
    one = scalar(1.0, fs)
    dgate = f.Mul(f.Mul(dact, up), f.Mul(s, f.Add(one, f.Mul(gate, f.Sub(one, s)))))
    dw_gate = f.DotGeneral(h, [0], [], dgate, [0], [])
    dw_up = f.DotGeneral(h, [0], [], dup, [0], [])
    dh = f.Add(f.DotGeneral(dgate, [1], [], p["w_gate"], [1], []), f.DotGeneral(dup, [1], [], p["w_up"], [1], []))
    dgamma = f.ReduceSum(f.Mul(dh, xhat), 0)
    dxhat = f.Mul(dh, gamma)
    m = f.BroadcastInDim(row_mean(f.Mul(dxhat, xhat)), xs, [0])
    dx = f.Add(dy, f.Mul(r, f.Sub(dxhat, f.Mul(xhat, m))))
    return [y, dx, dgamma, dw_gate, dw_up, dw_down]


class Program:
    """A compiled graph: input names in parameter order and the executable."""

    def __init__(self, case, shapes):
        c, k = case, case["kind"]
        be = _backend()
        if k == "decode":
            self.ex = graphs.decode_step(be, _decode_cfg(c))
        elif k == "block":
            self.ex = graphs.transformer_block(be, _block_cfg(c))
        else:
            b = be.Builder(k)
            f = b.Main()
            p = {n: f.Parameter(n, s) for n, s in shapes}
            if k == "dense":
                outs = [f.FusedDense(p["x"], p["w"], p["bias"], ACT[c["act"]])]
            else:
                outs = (_classifier_graph if k == "classifier" else _ffn_graph)(f, p, c)
            f.Return(outs)
            self.ex = b.Compile()
        self.shapes = shapes
        self.outputs = [(s.dims, s.dtype) for s in self.ex.Outputs()]

    def __del__(self):
        if getattr(self, "ex", None) is not None:
            self.ex.Finalize()


_BACKEND = []
_PROGRAMS = weakref.WeakValueDictionary()  # a program lives while a prepared state holds it


def _backend():
    if not _BACKEND:
        _BACKEND.append(Backend(""))
    return _BACKEND[0]


_NP_TYPE = {dtypes.Float32: "<f4", dtypes.BFloat16: "<i2", dtypes.Float16: "<f2", dtypes.Int32: "<i4"}


class _DeviceArray:
    """Device memory of a backend buffer, for torch: keeps the buffer alive."""

    def __init__(self, buf, dims, dtype):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(dims), "typestr": _NP_TYPE[dtype], "version": 2,
                                         "data": (buf.device_ptr(), False)}


def _tensor(buf, dims, dtype):
    t = torch.as_tensor(_DeviceArray(buf, dims, dtype), device=DEV)
    return t.view(torch.bfloat16) if dtype == dtypes.BFloat16 else t


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    c, k = case, case["kind"]
    t = _inputs(case, seed)
    s = {"case": dict(case), "in": t}
    if k in ("norm", "softmax"):
        s["out"] = torch.empty_like(t["x"])
    elif k == "dot":
        s["a"] = t["a"].transpose(1, 2) if c["ta"] else t["a"]
        s["b"] = t["b"].transpose(1, 2) if c["tb"] else t["b"]
        s["out"] = torch.empty((c["B"], c["M"], c["N"]), dtype=t["a"].dtype, device=DEV)
        s["ws"] = ops.gemm_workspace(t["a"].dtype, t["a"].dtype, c["B"], c["M"], c["N"], c["K"], DEV)
    elif k == "attn":
        s["out"] = torch.empty_like(t["q"])
        s["ws"] = ops.sdpa_workspace(t["q"], c["Hkv"], c["Sk"], c["mask"] == "causal")
    else:
        gdt = {torch.float32: dtypes.Float32, torch.bfloat16: dtypes.BFloat16, torch.float16: dtypes.Float16,
               torch.int32: dtypes.Int32}
        shapes = [(n, make_shape(gdt[v.dtype], *v.shape)) for n, v in t.items()]
        key = tuple(sorted((n, v) for n, v in case.items() if n != "name"))
        prog = _PROGRAMS.get(key)
        if prog is None:
            prog = _PROGRAMS[key] = Program(case, shapes)
        be = _backend()
        s["prog"], s["bufs"] = prog, []
        for n, shape in shapes:
            buf = be.NewSharedBuffer(0, shape)
            _tensor(buf, shape.dims, shape.dtype).copy_(t[n])
            s["bufs"].append(buf)
        s["in"] = None
        torch.cuda.synchronize()  # the copies ran on torch's stream, Execute runs on the backend's
    return s


def run(state):
    c, t = state["case"], state["in"]
    k = c["kind"]
    if k == "norm":
        if c["op"] == "rms":
            return ops.rmsnorm(t["x"], t["gamma"], EPS, out=state["out"])
        return ops.layernorm(t["x"], t["gamma"], t["beta"], EPS, out=state["out"])
    if k == "softmax":
        return ops.softmax(t["x"], log=c["log"], out=state["out"])
    if k == "dot":
        return ops.gemm(state["a"], state["b"], out=state["out"], workspace=state["ws"])
    if k == "attn":
        return ops.sdpa_masked(t["q"], t["k"], t["v"], t.get("mask"), c["D"] ** -0.5, c["mask"] == "causal",
                               out=state["out"], workspace=state["ws"])
    prog = state["prog"]
    outs = prog.ex.Execute(state["bufs"])
    return [_tensor(b, dims, dt) for b, (dims, dt) in zip(outs, prog.outputs)]


# ---------------------------------------------------------------- float64
def _rms(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma


def _attention(q, k, v, scale, causal, mask=None):
    """Attention of q [B,H,Sq,D] over k, v [B,Hkv,Sk,D], one batch row at a time."""
    B, H, Sq, _ = q.shape
    g, Sk = H // k.shape[1], k.shape[2]
    out = torch.empty_like(q)
    tri = torch.ones((Sq, Sk), dtype=torch.bool, device=q.device).tril() if causal else None
    for b in range(B):
        kb = k[b].repeat_interleave(g, 0)
        vb = v[b].repeat_interleave(g, 0)
        s = torch.matmul(q[b], kb.transpose(1, 2).contiguous()) * scale
        if mask is not None:
            m = mask[b, 0] if mask.dim() == 4 else mask
            s = s.masked_fill(~m, -math.inf) if m.dtype == torch.bool else s + m.double()
        if causal:
            s = s.masked_fill(~tri, -math.inf)
        out[b] = torch.matmul(torch.softmax(s, -1), vb)
    return out


def _activation(z, act):
    if act == "gelu":
        return 0.5 * z * (1 + torch.tanh(0.7978845608 * (z + 0.044715 * z ** 3)))
    return {"none": lambda v: v, "relu": torch.relu, "silu": lambda v: v * torch.sigmoid(v), "tanh": torch.tanh}[act](z)


def exact(case, seed):
    c, k = case, case["kind"]
    raw = _inputs(case, seed)
    t = {n: v.double() if v.is_floating_point() else v for n, v in raw.items()
         if n != "embedding"}
    if k == "norm":
        if c["op"] == "rms":
            return _rms(t["x"], t["gamma"])
        x = t["x"]
        d = x - x.mean(-1, keepdim=True)
        return d * torch.rsqrt((d * d).mean(-1, keepdim=True) + EPS) * t["gamma"] + t["beta"]
    if k == "softmax":
        return torch.log_softmax(t["x"], -1) if c["log"] else torch.softmax(t["x"], -1)
    if k == "dot":
        a = t["a"].transpose(1, 2).contiguous() if c["ta"] else t["a"]
        b = t["b"].transpose(1, 2).contiguous() if c["tb"] else t["b"]
        return torch.matmul(a, b)
    if k == "dense":
        return [_activation(t["x"] @ t["w"] + t["bias"], c["act"])]
    if k == "attn":
        return _attention(t["q"], t["k"], t["v"], c["D"] ** -0.5, c["mask"] == "causal", t.get("mask"))
    if k == "classifier":
        B, L, V, E = c["B"], c["L"], c["V"], c["E"]
        ids, labels = t["ids"].long(), t["labels"].long()
        mean = t["table"][ids].mean(1)
        act = torch.relu(mean @ t["w1"] + t["b1"])
        logits = act @ t["w2"] + t["b2"]
        logp = torch.log_softmax(logits, -1)
        hot = torch.nn.functional.one_hot(labels, c["C"]).double()
        loss = -(hot * logp).sum() / B
        dlogits = (logp.exp() - hot) / B
        dz = torch.where(act > 0, dlogits @ t["w2"].t(), 0.0)
        demb = (dz @ t["w1"].t() / L)[:, None].expand(B, L, E).reshape(B * L, E)
        dtable = torch.zeros((V, E), dtype=torch.float64, device=DEV).index_add_(0, ids.reshape(-1), demb)
        return [loss, logits, dtable, mean.t() @ dz, dz.sum(0), act.t() @ dlogits, dlogits.sum(0)]
    if k == "ffn":
        x, dy, gamma = t["x"], t["dy"], t["gamma"]
        r = torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
        xhat = x * r
        h = xhat * gamma
        gate, up = h @ t["w_gate"], h @ t["w_up"]
        s = torch.sigmoid(gate)
        silu = gate * s
        act = silu * up
        y = x + act @ t["w_down"]
        dact = dy @ t["w_down"].t()
        dup = dact * silu
        dgate = dact * up * s * (1 + gate * (1 - s))
        dh = dgate @ t["w_gate"].t() + dup @ t["w_up"].t()
        dxhat = dh * gamma
        dx = dy + r * (dxhat - xhat * (dxhat * xhat).mean(-1, keepdim=True))
        return [y, dx, (dh * xhat).sum(0), h.t() @ dgate, h.t() @ dup, act.t() @ dy]
    if k == "decode":
        B, H, Hkv = c["B"], c["H"], c["Hkv"]
        qkv = _rms(t["x"], t["g_attn"]) @ t["w_qkv"]
        a = _attention(qkv[:, :H * 128].reshape(B, H, 1, 128), t["k_cache"], t["v_cache"], 128 ** -0.5, False)
        x2 = t["x"] + a.reshape(B, H * 128) @ t["wo"]
        h2 = _rms(x2, t["g_ffn"])
        gate = h2 @ t["w_gate"]
        return [x2 + (gate * torch.sigmoid(gate) * (h2 @ t["w_up"])) @ t["w_down"], qkv]
    B, S, d, H = c["B"], c["S"], c["d"], c["H"]
    x = raw["embedding"][t["ids"].long()].double().reshape(B * S, d)
    h = _rms(x, t["g_attn"])
    q, kk, v = ((h @ t[w]).reshape(B, S, H, 128).transpose(1, 2).contiguous() for w in ("wq", "wk", "wv"))
    a = _attention(q, kk, v, 128 ** -0.5, True).transpose(1, 2).reshape(B * S, d)
    x2 = x + a @ t["wo"]
    h2 = _rms(x2, t["g_ffn"])
    gate = h2 @ t["w_gate"]
    return [(x2 + (gate * torch.sigmoid(gate) * (h2 @ t["w_up"])) @ t["w_down"]).reshape(B, S, d)]
