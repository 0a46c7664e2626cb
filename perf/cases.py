"""Performance cases of the framework's main path: rew's layers as one lazy call.

A case is one layer or block of rew (``rew_amd.nn``) traced by ``rew_amd.jit.lazy`` and
called on tensors that are already on the device, the way an inference program runs it:
the layer is traced once per shape, its weights stay on the device, and every call is one
module execution whose outputs are read in place as torch tensors.  The sizes are those of
the decoder layer, SwiGLU, MoE, MNIST and row-op workloads of bench.py, a small float32
decoder, and what lies between and beside them (decode batches, ragged sequences).

Kinds:

* ``classifier``  float32 MLP, softmax and argmax;
* ``rows``        float32 elementwise chain, reductions, softmax and rmsNorm over rows;
* ``linear``      one Linear (bfloat16 or float32), up to a language model's head;
* ``ffn``         the SwiGLU feed-forward block;
* ``attention``   grouped-query scaled-dot-product attention, prefill and decode;
* ``decoder``     token ids -> embedding -> one whole decoder layer;
* ``moe``         the DeepSeek-style routed mixture of experts.
"""
from __future__ import annotations

import functools
import math

import torch

from rew_amd import eager as E
from rew_amd import jit as J
from rew_amd import nn
from rew_amd import ops as O
from rew_amd.eager import DType

# (hidden, heads, kv heads, head dim, intermediate, vocabulary, rope theta)
MODELS = {"large": (4096, 32, 8, 128, 14336, 128256, 500000.0),
          "small": (1024, 16, 4, 64, 2816, 32000, 10000.0)}
EPS = 1e-5


def listed():
    return [
        # the smallest call: one batch of digits through the MNIST MLP
        {"name": "classifier_128", "kind": "classifier", "rows": 128, "inputs": 784,
         "hidden": 128, "classes": 10},
        # the row operations of a float32 model at a prefill's size
        {"name": "rows_8192x4096", "kind": "rows", "rows": 8192, "cols": 4096},
        # the logits of a decode step: 16 sequences against the whole vocabulary
        {"name": "head_16", "kind": "linear", "rows": 16, "inputs": 4096, "outputs": 128256,
         "dtype": "bfloat16"},
        # the feed-forward block of a decode step with 8 sequences
        {"name": "ffn_8", "kind": "ffn", "tokens": 8, "hidden": 4096, "inner": 14336,
         "dtype": "bfloat16"},
        # one short prompt (a ragged token count)
        {"name": "ffn_300", "kind": "ffn", "tokens": 300, "hidden": 4096, "inner": 14336,
         "dtype": "bfloat16"},
        # a full prefill batch
        {"name": "ffn_4096", "kind": "ffn", "tokens": 4096, "hidden": 4096, "inner": 14336,
         "dtype": "bfloat16"},
        # one decode step of 16 sequences over cached keys and values
        {"name": "attention_decode_4000", "kind": "attention", "batch": 16, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "queries": 1, "keys": 4000, "causal": False,
         "dtype": "bfloat16"},
        # a prefill whose prompt is no multiple of any tile
        {"name": "attention_prefill_1500", "kind": "attention", "batch": 2, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "queries": 1500, "keys": 1500, "causal": True,
         "dtype": "bfloat16"},
        # the headline workload: one decoder layer over 4 prompts of 2048 tokens
        {"name": "decoder_4x2048", "kind": "decoder", "model": "large", "batch": 4, "seq": 2048,
         "norm": "rms", "dtype": "bfloat16"},
        # rew's own default precision and norm: a small float32 model's layer
        {"name": "decoder_f32_4x500", "kind": "decoder", "model": "small", "batch": 4,
         "seq": 500, "norm": "layer", "dtype": "float32"},
        # the routed experts of a decode step with 40 sequences
        {"name": "moe_40", "kind": "moe", "tokens": 40, "hidden": 2048, "inner": 1408,
         "routed": 64, "shared": 2, "top_k": 6},
        # the routed experts of a prefill
        {"name": "moe_8192", "kind": "moe", "tokens": 8192, "hidden": 2048, "inner": 1408,
         "routed": 64, "shared": 2, "top_k": 6},
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["classifier", "rows", "linear", "linear", "ffn", "ffn", "attention",
                       "attention", "decoder", "decoder", "moe"])
    if kind == "classifier":
        return {"kind": kind, "rows": _log(rng, 1, 4096), "inputs": rng.choice([784, 256, 1000]),
                "hidden": rng.choice([64, 128, 300, 512]), "classes": rng.choice([10, 26, 100])}
    if kind == "rows":
        cols = _log(rng, 200, 8192)
        return {"kind": kind, "rows": _log(rng, 64, min(16384, (8192 * 4096) // cols)),
                "cols": cols}
    if kind == "linear":
        if rng.random() < 0.5:
            k, n = rng.choice([(784, 128), (1024, 1024), (1024, 2816), (2816, 1024),
                               (1000, 3000), (2048, 64), (1024, 32000)])
            most = min(4096, int(3.5e10 / (2 * k * n)))
            return {"kind": kind, "rows": _log(rng, 1, most), "inputs": k, "outputs": n,
                    "dtype": "float32"}
        k, n = rng.choice([(4096, 4096), (4096, 1024), (4096, 14336), (14336, 4096),
                           (2048, 1408), (1408, 2048), (1000, 3000), (4096, 128256)])
        return {"kind": kind, "rows": _log(rng, 1, 8192 if n < 100000 else 256), "inputs": k,
                "outputs": n, "dtype": "bfloat16"}
    if kind == "ffn":
        h, i = rng.choice([(4096, 14336), (4096, 14336), (2048, 1408), (1024, 2816)])
        f32 = h == 1024 and rng.random() < 0.5
        return {"kind": kind, "tokens": _log(rng, 1, 2048 if f32 else 4096), "hidden": h,
                "inner": i, "dtype": "float32" if f32 else "bfloat16"}
    if kind == "attention":
        h, kv, d = rng.choice([(32, 8, 128), (32, 32, 128), (16, 4, 64)])
        if rng.random() < 0.5:
            return {"kind": kind, "batch": _log(rng, 1, 32), "heads": h, "kv_heads": kv,
                    "head_dim": d, "queries": rng.choice([1, 1, 4]), "keys": _log(rng, 100, 8192),
                    "causal": False, "dtype": "bfloat16"}
        f32 = d == 64 and rng.random() < 0.5
        s = _log(rng, 16, 512 if f32 else 2048)
        return {"kind": kind, "batch": rng.choice([1, 2, 3]), "heads": h, "kv_heads": kv,
                "head_dim": d, "queries": s, "keys": s, "causal": rng.random() < 0.75,
                "dtype": "float32" if f32 else "bfloat16"}
    if kind == "decoder":
        model = rng.choice(["large", "small"])
        f32 = model == "small" and rng.random() < 0.5
        b, s = rng.choice([1, 2, 3, 4]), _log(rng, 16, 500 if f32 else 2048)
        return {"kind": kind, "model": model, "batch": b, "seq": s,
                "norm": rng.choice(["rms", "layer"]), "dtype": "float32" if f32 else "bfloat16"}
    e, k = rng.choice([(64, 6), (64, 6), (16, 2)])
    return {"kind": kind, "tokens": _log(rng, 1, 8192), "hidden": 2048, "inner": 1408,
            "routed": e, "shared": rng.choice([1, 2]), "top_k": k}


# ---- inputs ----------------------------------------------------------------------------

_DT = {"bfloat16": (DType.BFLOAT16, torch.bfloat16, "<i2"),
       "float32": (DType.FLOAT32, torch.float32, "<f4"),
       "int32": (DType.INT32, torch.int32, "<i4")}
_BY_DTYPE = {d: (t, s) for d, t, s in _DT.values()}


class _Memory:
    """A backend tensor's device memory under the array interface torch reads."""

    __slots__ = ("__cuda_array_interface__", "tensor")


def _view(t):
    """The backend tensor's memory as a torch tensor (no copy; it keeps `t` alive)."""
    dt, typestr = _BY_DTYPE[t.dtype]
    m = _Memory()
    m.tensor = t
    m.__cuda_array_interface__ = {"shape": t.shape, "typestr": typestr, "version": 2,
                                  "data": (E.devicePtr(t), False)}
    v = torch.as_tensor(m, device="cuda")
    return v.view(torch.bfloat16) if dt is torch.bfloat16 else v


class _Maker:
    """Makes a case's inputs from its seed, in a fixed order: backend tensors for
    `prepare`, plain torch tensors of the same values for `exact`."""

    def __init__(self, seed, plain):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.plain = plain

    def _new(self, shape, dtype):
        if self.plain:
            t = torch.empty(shape, dtype=_DT[dtype][1], device="cuda")
            return t, t
        t = E.empty(_DT[dtype][0], shape)
        return t, _view(t)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        t, v = self._new(shape, dtype)
        v.normal_(mean, std, generator=self.gen)
        return t

    def uniform(self, shape, dtype, lo, hi):
        t, v = self._new(shape, dtype)
        v.uniform_(lo, hi, generator=self.gen)
        return t

    def ids(self, shape, limit):
        t, v = self._new(shape, "int32")
        v.random_(0, limit, generator=self.gen)
        return t

    def of(self, data):
        """A float32 table computed on the host (the rotary angles)."""
        return torch.from_numpy(data).cuda() if self.plain else E.fromHost(data)

    def linear(self, k, n, dtype, std=0.02):
        return [self.normal((k, n), dtype, std), self.normal((n,), dtype, 0.02)]


def _inputs(c, make):
    """The arguments of the case's traced function, in order."""
    kind = c["kind"]
    if kind == "classifier":
        d, h, n = c["inputs"], c["hidden"], c["classes"]
        xavier = lambda a, b: make.uniform((a, b), "float32", -math.sqrt(6 / (a + b)),  # noqa: E731
                                           math.sqrt(6 / (a + b)))
        return [make.uniform((c["rows"], d), "float32", 0.0, 1.0), xavier(d, h),
                make.normal((h,), "float32", 0.02), xavier(h, n),
                make.normal((n,), "float32", 0.02)]
    if kind == "rows":
        return [make.normal((c["rows"], c["cols"]), "float32"),
                make.normal((c["cols"],), "float32", 0.1, 1.0)]
    if kind == "linear":
        return [make.normal((c["rows"], c["inputs"]), c["dtype"]),
                *make.linear(c["inputs"], c["outputs"], c["dtype"])]
    if kind == "ffn":
        h, i, dt = c["hidden"], c["inner"], c["dtype"]
        return [make.normal((1, c["tokens"], h), dt), *make.linear(h, i, dt),
                *make.linear(h, i, dt), *make.linear(i, h, dt)]
    if kind == "attention":
        b, d, dt = c["batch"], c["head_dim"], c["dtype"]
        return [make.normal((b, c["heads"], c["queries"], d), dt),
                make.normal((b, c["kv_heads"], c["keys"], d), dt),
                make.normal((b, c["kv_heads"], c["keys"], d), dt)]
    if kind == "decoder":
        H, nh, nkv, hd, I, V, theta = MODELS[c["model"]]
        dt = c["dtype"]
        cos, sin = _tables(hd, c["seq"], theta)
        args = [make.ids((c["batch"] * c["seq"],), V), make.normal((V, H), dt, 1.0)]
        for k, n in ((H, nh * hd), (H, nkv * hd), (H, nkv * hd), (nh * hd, H), (H, I), (H, I),
                     (I, H)):
            args += make.linear(k, n, dt)
        args += [make.of(cos), make.of(sin)]
        for _ in range(2):
            args += [make.normal((H,), "float32", 0.1, 1.0), make.normal((H,), "float32", 0.1)]
        return args
    H, I = c["hidden"], c["inner"]
    args = [make.normal((c["tokens"], H), "bfloat16"), *make.linear(H, c["routed"], "float32")]
    for _ in range(c["shared"] + c["routed"]):
        for k, n in ((H, I), (H, I), (I, H)):
            args += make.linear(k, n, "bfloat16")
    return args


@functools.lru_cache(maxsize=None)
def _tables(head_dim, seq, theta):
    return nn.rope_tables(head_dim, seq, theta)


# ---- the traced layers ----------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _traced(key):
    """The case's layer as one lazy function of its arguments."""
    c = dict(key)
    kind = c["kind"]

    def classifier(a):
        hidden = nn.relu(nn.Linear(a[1], a[2]).forward(a[0]))
        return [nn.softmax(nn.Linear(a[3], a[4]).forward(hidden), 1)]

    def rows(a):
        x, g = a
        y = nn.relu(O.add(x, x))
        return [y, O.reduceSum(y, [1]), O.reduceMean(y, [1]), O.reduceMax(y, [1]),
                nn.softmax(x, 1), nn.rmsNorm(x, g, EPS)]

    def linear(a):
        return [nn.Linear(a[1], a[2]).forward(a[0])]

    def ffn(a):
        return [nn.GatedFeedForward(nn.Linear(a[1], a[2]), nn.Linear(a[3], a[4]),
                                    nn.Linear(a[5], a[6])).forward(a[0])]

    def attention(a):
        b, h, kv, s, d = c["batch"], c["heads"], c["kv_heads"], c["keys"], c["head_dim"]

        def expand(t):  # the head expansion of GroupedQueryAttention.forward
            u = O.broadcastTo(O.reshape(t, [b, kv, 1, s, d]), [b, kv, h // kv, s, d],
                              [0, 1, 2, 3, 4])
            return O.reshape(u, [b, h, s, d])

        return [nn.scaledDotProductAttention(a[0], expand(a[1]), expand(a[2]),
                                             causal=c["causal"])]

    def decoder(a):
        H, nh, nkv, hd, _, _, theta = MODELS[c["model"]]
        x = O.reshape(nn.Embedding(a[1]).lookup(a[0]), [c["batch"], c["seq"], H])
        lin = [nn.Linear(a[2 + 2 * i], a[3 + 2 * i]) for i in range(7)]
        rope = nn.RotaryPositionEncoding(a[16], a[17], theta, hd, c["seq"])
        if c["norm"] == "rms":
            norms = [nn.RMSNorm(a[18], EPS), nn.RMSNorm(a[20], EPS)]
        else:
            norms = [nn.LayerNorm(a[18], a[19], [H], EPS), nn.LayerNorm(a[20], a[21], [H], EPS)]
        attn = nn.GroupedQueryAttention(*lin[:4], nh, nkv, hd, rope)
        layer = nn.LlamaDecoderLayer(attn, nn.GatedFeedForward(*lin[4:]), *norms)
        return [layer.forward(x, causal=True)]

    def moe(a):
        return [nn.moeFromParams(a[1:], c["shared"], c["routed"], c["top_k"]).forward(a[0])]

    return J.lazy(locals()[kind], "perf_" + kind)


def prepare(case, seed):
    E.installEagerBackend(E.mi355x(0))
    E.sync()
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    args = _inputs(case, _Maker(seed, False))
    torch.cuda.synchronize()
    return {"kind": case["kind"], "fn": _traced(key), "args": args}


def run(state):
    outs = state["fn"].call(state["args"])
    if state["kind"] == "classifier":
        return {"probabilities": _view(outs[0]), "ids": _view(O.argmax(outs[0], 1))}
    return [_view(t) for t in outs]


# ---- what a pass cannot do without -----------------------------------------------------

def _pairs(c):
    """(query, key) pairs the mask keeps: key j is visible to query i when j >= i."""
    q, k = c["queries"], c["keys"]
    return sum(max(0, k - i) for i in range(q)) if c["causal"] else q * k


def work(case):
    c, kind = case, case["kind"]
    size = 4 if c.get("dtype") == "float32" else 2
    if kind == "classifier":
        r, d, h, n = c["rows"], c["inputs"], c["hidden"], c["classes"]
        return {"bytes": 4 * (r * d + d * h + h * n + h + n + r * n + r),
                "flops": 2 * r * (d * h + h * n)}
    if kind == "rows":
        n = c["rows"] * c["cols"]
        return {"bytes": 4 * (4 * n + 3 * c["rows"] + c["cols"]), "flops": 15 * n}
    if kind == "linear":
        m, k, n = c["rows"], c["inputs"], c["outputs"]
        return {"bytes": size * (m * k + k * n + n + m * n), "flops": 2 * m * k * n}
    if kind == "ffn":
        t, h, i = c["tokens"], c["hidden"], c["inner"]
        return {"bytes": size * (2 * t * h + 3 * h * i + 2 * i + h), "flops": 6 * t * h * i}
    if kind == "attention":
        b, h, kv, d = c["batch"], c["heads"], c["kv_heads"], c["head_dim"]
        return {"bytes": size * b * d * (2 * h * c["queries"] + 2 * kv * c["keys"]),
                "flops": 4 * b * h * d * _pairs(c)}
    if kind == "decoder":
        H, nh, nkv, hd, I, V, _ = MODELS[c["model"]]
        t, s = c["batch"] * c["seq"], c["seq"]
        w = H * (nh + 2 * nkv) * hd + nh * hd * H + 3 * H * I
        return {"bytes": size * (2 * t * H + w) + 4 * (t + 2 * s * hd),
                "flops": 2 * t * w + 4 * c["batch"] * nh * hd * (s * (s + 1) // 2)}
    t, H, I, e, k = c["tokens"], c["hidden"], c["inner"], c["routed"], c["top_k"]
    hit = e * (1.0 - (1.0 - k / e) ** t)  # experts that some token is routed to
    return {"bytes": 2 * (2 * t * H + 3 * H * I * (hit + c["shared"])) + 4 * H * e,
            "flops": 2 * t * H * e + 6 * t * H * I * (k + c["shared"])}


def tolerance(case):
    """About four times the distance from `exact` that these layers show in float32
    (reductions 8e-8, products over up to 2816 terms 6e-7); in bfloat16 the largest
    distance of another order of the same sums, whose roundings travel on."""
    if case["kind"] == "classifier":
        return {"rel": 1.5e-6, "max": 6e-5, "differ": 0.01}
    if case["kind"] == "rows":
        return {"rel": 4e-7, "max": 1e-5}
    if case.get("dtype") == "float32":
        return {"rel": 2.5e-6, "max": 1e-4}
    if case["kind"] in ("decoder", "moe"):
        return {"rel": 1.5e-2, "max": 0.3}
    return {"rel": 1e-2, "max": 0.2}


# ---- the same in 64 bits -----------------------------------------------------------------

def exact(case, seed):
    c, kind = case, case["kind"]
    a = _inputs(c, _Maker(seed, True))
    f = lambda t: t.double()  # noqa: E731

    def lin(x, i):
        return x @ f(a[i]) + f(a[i + 1])

    def gated(x, i):
        return lin(torch.nn.functional.silu(lin(x, i)) * lin(x, i + 2), i + 4)

    def attend(q, k, v, causal):
        """[B, H, S, D] x [B, Hkv, Sk, D], one head after another."""
        out = torch.empty_like(q)
        group = q.shape[1] // k.shape[1]
        scale = 1.0 / math.sqrt(q.shape[-1])
        hidden = None
        if causal:
            hidden = torch.ones(q.shape[2], k.shape[2], dtype=torch.bool, device="cuda").tril(-1)
        for b in range(q.shape[0]):
            for h in range(q.shape[1]):
                s = (q[b, h] @ k[b, h // group].t().contiguous()) * scale
                if hidden is not None:
                    s -= 1e9 * hidden
                out[b, h] = torch.softmax(s, -1) @ v[b, h // group]
        return out

    if kind == "classifier":
        p = torch.softmax(lin(torch.relu(lin(f(a[0]), 1)), 3), 1)
        return {"probabilities": p, "ids": None}
    if kind == "rows":
        x, g = f(a[0]), f(a[1])
        y = torch.relu(x + x)
        return [y, y.sum(1), y.mean(1), y.max(1).values, torch.softmax(x, 1),
                g * (x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS))]
    if kind == "linear":
        return [lin(f(a[0]), 1)]
    if kind == "ffn":
        return [gated(f(a[0]), 1)]
    if kind == "attention":
        return [attend(f(a[0]), f(a[1]), f(a[2]), c["causal"])]
    if kind == "decoder":
        H, nh, nkv, hd, _, _, _ = MODELS[c["model"]]
        B, S = c["batch"], c["seq"]

        def norm(x, i):
            if c["norm"] == "rms":
                return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * f(a[i])
            d = x - x.mean(-1, keepdim=True)
            return d / torch.sqrt((d * d).mean(-1, keepdim=True) + EPS) * f(a[i]) + f(a[i + 1])

        def rotate(t):
            cos, sin = f(a[16])[:, ::2], f(a[17])[:, ::2]
            x0, x1 = t[..., ::2], t[..., 1::2]
            return torch.stack([cos * x0 - sin * x1, sin * x0 + cos * x1], -1).flatten(-2)

        def heads(t, n):
            return t.reshape(B, S, n, hd).transpose(1, 2).contiguous()

        x = f(a[1][a[0].long()])
        z = norm(x, 18)
        o = attend(rotate(heads(lin(z, 2), nh)), rotate(heads(lin(z, 4), nkv)),
                   heads(lin(z, 6), nkv), True)
        x = x + lin(o.transpose(1, 2).reshape(B * S, nh * hd), 8)
        return [(x + gated(norm(x, 20), 10)).reshape(B, S, H)]
    x = f(a[0])
    top, ids = torch.topk(torch.softmax(lin(x, 1), 1), c["top_k"], 1)
    top = top / top.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for e in range(c["shared"] + c["routed"]):
        if e < c["shared"]:
            out += gated(x, 3 + 6 * e)
            continue
        w = (top * (ids == e - c["shared"])).sum(1)
        at = w.nonzero()[:, 0]
        if at.numel():
            out[at] += gated(x[at], 3 + 6 * e) * w[at, None]
    return [out]
