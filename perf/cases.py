"""The work this framework is timed on: what a program written against it has it do, from single
small calls to a whole training step, over the range of sizes that such programs use.

Everything runs through the public entry points: the `Tensor` front-end and `nn` modules, `Backend`
methods where `Tensor` has no method (gradients, AdamW), `HIPBackend.batching` and `HIPBackend.capture`.
Inputs are generated on the GPU into the backend's own buffers.

  small        one token position's residual connection: add, LayerNorm. Latency of a few small calls.
  matmul       one product, from decoding a few rows through ragged sizes to the 4096^3 benchmark.
  attention    q k^T, scale, mask, softmax, x v over the heads of a batch, issued under batching.
  row_ops      the bandwidth-bound companions: bias add, GELU, and sum / max / argmax over rows.
  embedding    rows of an embedding table by token id, and the table's gradient.
  transformer  the forward pass of the decoder-only model in `nn`, recorded once and replayed.
  train_step   forward, backward and AdamW of a one-block language model, call by call.
  sampling     what picks the next token: softmax, sort by probability, running sum (nucleus).
"""
import math

import torch

from honeycrisp_amd import nn
from honeycrisp_amd.backend import Backend, HIPBackend
from honeycrisp_amd.descriptors import DType, ElemwiseOp, ReduceDims, product
from honeycrisp_amd.tensor import Tensor

_DTYPES = {"f16": DType.float16, "f32": DType.float32}
_TORCH = {DType.float16: torch.float16, DType.float32: torch.float32, DType.int64: torch.int64, DType.bool: torch.bool}
_TYPESTR = {DType.float16: "<f2", DType.float32: "<f4", DType.int64: "<i8", DType.bool: "|b1"}
_backend = None


def backend():
    """One context for the life of the program, installed as the default backend."""
    global _backend
    if _backend is None:
        _backend = HIPBackend()
        Backend.setDefault(_backend)
    return _backend


class _Buffer:
    """A tensor's device buffer as torch sees it (no copy; keeps the buffer alive)."""

    def __init__(self, data, shape, dtype):
        self.data = data
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": _TYPESTR[dtype], "data": (data.ptr, False),
                                         "version": 2}


def _view(t):
    return torch.as_tensor(_Buffer(t.data, t.shape, t.dtype), device="cuda")


def _upload(values):
    """The values of a torch tensor in a buffer of the backend."""
    dtype = next(d for d, kind in _TORCH.items() if kind == values.dtype)
    t = Tensor(dataHandle=backend().allocate(values.numel() * dtype.byteSize), shape=list(values.shape), dtype=dtype)
    _view(t).copy_(values)
    return t


class _Random:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        backend().sync()        # blocks of the pool may still be read by work in flight

    def normal(self, shape, dtype, scale=1.0):
        return _upload((torch.randn(shape, generator=self.g, device="cuda") * scale).to(_TORCH[dtype]))

    def positive(self, shape, dtype, scale=1.0):
        return _upload((torch.randn(shape, generator=self.g, device="cuda").square() * scale).to(_TORCH[dtype]))

    def ids(self, count, below):
        return _upload(torch.randint(below, (count,), generator=self.g, device="cuda"))


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # 16 rows of a d_model 512 model: what a decoding step does between two products
        {"name": "small_f16", "kind": "small", "dtype": "f16", "rows": 16, "cols": 512},
        # 16 sequences decoded together against a square weight
        {"name": "matmul_decode_f16", "kind": "matmul", "dtype": "f16", "m": 16, "k": 4096, "n": 4096, "ta": False, "tb": False},
        # the plain fp32 product of the reference's benchmark
        {"name": "matmul_f32_1024", "kind": "matmul", "dtype": "f32", "m": 1024, "k": 1024, "n": 1024, "ta": False, "tb": False},
        # ragged sizes, second operand stored transposed
        {"name": "matmul_ragged_f16", "kind": "matmul", "dtype": "f16", "m": 1000, "k": 4097, "n": 4097, "ta": False, "tb": True},
        # the benchmark's headline product
        {"name": "matmul_4096_f16", "kind": "matmul", "dtype": "f16", "m": 4096, "k": 4096, "n": 4096, "ta": False, "tb": False},
        # 8 sequences x 8 heads at a context of 1024
        {"name": "attention_f16", "kind": "attention", "dtype": "f16", "heads": 64, "t": 1024, "hd": 64},
        # activations of 8192 tokens, 4096 wide, in fp32
        {"name": "row_ops_f32", "kind": "row_ops", "dtype": "f32", "rows": 8192, "cols": 4096},
        # 65536 token ids into a table of 32000 rows
        {"name": "embedding_f32", "kind": "embedding", "dtype": "f32", "ids": 65536, "vocab": 32000, "width": 1024},
        # the benchmark's model: prefill of 8 sequences of 256 tokens, half precision
        {"name": "transformer_f16", "kind": "transformer", "dtype": "f16", "batch": 8, "t": 256, "layers": 6, "d": 512, "heads": 8, "vocab": 8192},
        # the same model in fp32 on a small batch with a sequence length that is no multiple of anything
        {"name": "transformer_f32", "kind": "transformer", "dtype": "f32", "batch": 3, "t": 201, "layers": 6, "d": 512, "heads": 8, "vocab": 8192},
        # one optimizer step over 2048 tokens, products in half precision, parameters in fp32
        {"name": "train_step_f16", "kind": "train_step", "dtype": "f16", "tokens": 2048, "d": 512, "mlp": 2048, "vocab": 8192},
        # the next token of 8 sequences over a vocabulary of 50257
        {"name": "sampling_f32", "kind": "sampling", "dtype": "f32", "rows": 8, "vocab": 50257},
    ]


def _size(rng, low, high, odd=0.25):
    """Log-uniform over [low, high], mostly multiples of 8 (as model sizes are), some of them not."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() >= odd:
        n = (n + 4) // 8 * 8
    return min(max(n, low), high)


def draw(rng):
    kind = rng.choice(["small", "matmul", "attention", "row_ops", "embedding", "transformer", "train_step", "sampling"])
    case = {"kind": kind, "dtype": rng.choice(["f16", "f32"])}
    if kind == "small":
        case.update(rows=_size(rng, 1, 256), cols=_size(rng, 64, 2048))
    elif kind == "matmul":
        m, k, n = _size(rng, 1, 4096), _size(rng, 64, 4352), _size(rng, 64, 4352)
        case.update(m=m, k=k, n=n, ta=rng.random() < 0.4, tb=rng.random() < 0.4)
    elif kind == "attention":
        t = _size(rng, 64, 2048)
        heads = min(_size(rng, 8, 128), max(8, (64 << 20) // (t * t)))
        case.update(heads=heads, t=t, hd=rng.choice([32, 64, 64, 128]))
    elif kind == "row_ops":
        rows = _size(rng, 64, 16384)
        case.update(rows=rows, cols=min(_size(rng, 64, 8192), (32 << 20) // rows))
    elif kind == "embedding":
        case.update(ids=_size(rng, 256, 65536), vocab=_size(rng, 1000, 32000), width=_size(rng, 64, 1024))
    elif kind == "transformer":
        t = _size(rng, 16, 256)
        d = rng.choice([256, 512])
        case.update(batch=rng.randint(1, max(1, min(16, 2048 // t))), t=t, layers=rng.randint(2, 6), d=d, heads=d // 64,
                    vocab=_size(rng, 1000, 8192))
    elif kind == "train_step":
        d = rng.choice([128, 256, 384, 512])
        case.update(tokens=_size(rng, 64, 2048), d=d, mlp=4 * d, vocab=_size(rng, 1000, 8192))
    else:
        case.update(rows=_size(rng, 1, 32), vocab=_size(rng, 1000, 50257))
    return case


# ---------------------------------------------------------------- what a program has in hand

_PARAMETERS = ("table", "gain", "shift", "w1", "b1", "w2", "b2", "wo")


def _parameter_shapes(c):
    d, mlp, vocab = c["d"], c["mlp"], c["vocab"]
    return {"table": [vocab, d], "gain": [d], "shift": [d], "w1": [d, mlp], "b1": [mlp], "w2": [mlp, d], "b2": [d], "wo": [d, vocab]}


def prepare(case, seed):
    c, b = dict(case), backend()
    dtype, r = _DTYPES[c["dtype"]], _Random(seed)
    s = {"case": c, "dtype": dtype}
    if c["kind"] == "small":
        shape = [c["rows"], c["cols"]]
        s.update(x=r.normal(shape, dtype), y=r.normal(shape, dtype), gain=r.normal([c["cols"]], dtype, 0.1),
                 bias=r.normal([c["cols"]], dtype, 0.1))
    elif c["kind"] == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        scale = 1 / math.sqrt(k)
        s.update(a=r.normal([k, m] if c["ta"] else [m, k], dtype, scale), b=r.normal([n, k] if c["tb"] else [k, n], dtype, scale))
    elif c["kind"] == "attention":
        shape, t = [c["heads"], c["t"], c["hd"]], c["t"]
        causal = torch.full((t, t), -1e4, device="cuda").triu(1)
        s.update(q=r.normal(shape, dtype), k=r.normal(shape, dtype), v=r.normal(shape, dtype), mask=_upload(causal.to(_TORCH[dtype])))
    elif c["kind"] == "row_ops":
        s.update(x=r.normal([c["rows"], c["cols"]], dtype), bias=r.normal([1, c["cols"]], dtype))
    elif c["kind"] == "embedding":
        s.update(table=r.normal([c["vocab"], c["width"]], dtype, 0.02), ids=r.ids(c["ids"], c["vocab"]),
                 grad=r.normal([c["ids"], c["width"]], dtype, 0.1))
    elif c["kind"] == "transformer":
        model = nn.Transformer(layers=c["layers"], d_model=c["d"], heads=c["heads"], mlp=4 * c["d"], vocab=c["vocab"],
                               seq=c["t"], seed=seed, dtype=dtype)
        ids = r.ids(c["batch"] * c["t"], c["vocab"]).reshape([c["batch"], c["t"]])
        model(ids)              # builds the mask, which a recording cannot upload
        with b.capture() as recording:
            logits = model(ids)
        s.update(model=model, ids=ids, recording=recording, logits=logits, out=_view(logits))
    elif c["kind"] == "train_step":
        p = {}
        for name, shape in _parameter_shapes(c).items():
            scale = 1 / math.sqrt(shape[0]) if name.startswith("w") else 0.02 if name == "table" else 0.1
            p[name] = {"value": r.normal(shape, DType.float32, scale), "m": r.normal(shape, DType.float32, 0.1),
                       "v": r.positive(shape, DType.float32, 0.01)}
        s.update(params=p, ids=r.ids(c["tokens"], c["vocab"]), targets=r.ids(c["tokens"], c["vocab"]))
    else:
        s.update(logits=r.normal([c["rows"], c["vocab"]], dtype, 3.0))
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass

def _train_step(s):
    """Embedding, LayerNorm, MLP with a residual, output projection; cross entropy summed over the
    tokens; gradients of everything; one AdamW update. Products run in the case's type."""
    c, b, half, f32 = s["case"], backend(), s["dtype"], DType.float32
    n, d, mlp, vocab = c["tokens"], c["d"], c["mlp"], c["vocab"]
    p = {name: v["value"] for name, v in s["params"].items()}
    ids, targets = s["ids"], s["targets"]
    mm, rows = Tensor.matmul, ReduceDims(n, d, 1)

    def wrap(data, shape, dtype=f32):
        return Tensor(dataHandle=data, shape=shape, dtype=dtype)

    w1, w2, wo = (p[k].cast(half) for k in ("w1", "w2", "wo"))
    x = p["table"].gather(0, ids)
    normed = x.normalize(axis=1, eps=1e-5)
    gain = p["gain"] + 1
    h = normed.mul(gain, thenAdd=p["shift"]).cast(half)
    f = mm(h, False, w1, False, False) + p["b1"].cast(half)
    g = f.gelu()
    y = (x.cast(half) + (mm(g, False, w2, False, False) + p["b2"].cast(half)))
    logits = mm(y, False, wo, False, False).cast(f32)
    logprobs = logits.logSoftmax()
    loss = -logprobs.gather(1, targets.reshape([n, 1])).sum()

    # d loss / d logprobs: -1 at each row's target
    seed_grad = Tensor.constant(-1, [n, 1]).scatter(1, vocab, targets.reshape([n, 1]), indicesAreUnique=False)
    dlogits = wrap(b.logSoftmaxGrad(logits.data, seed_grad.data, ReduceDims(n, vocab, 1), f32), [n, vocab]).cast(half)
    grads = {"wo": mm(y, True, dlogits, False, False).cast(f32)}
    dy = mm(dlogits, False, wo, True, False)
    grads["b2"] = dy.sum(axis=0).cast(f32)
    grads["w2"] = mm(g, True, dy, False, False).cast(f32)
    dg = mm(dy, False, w2, True, False)
    df = wrap(b.elemwise(f.data, ElemwiseOp.geluApproxGrad, dg.data, n * mlp, half), [n, mlp], half)
    grads["b1"] = df.sum(axis=0).cast(f32)
    grads["w1"] = mm(h, True, df, False, False).cast(f32)
    dh = mm(df, False, w1, True, False).cast(f32)
    grads["gain"] = (normed * dh).sum(axis=0)
    grads["shift"] = dh.sum(axis=0)
    dnormed = dh * gain
    dx = wrap(b.normalizeGrad(x.data, dnormed.data, rows, 1e-5, f32), [n, d]) + dy.cast(f32)
    grads["table"] = dx.scatter(0, vocab, ids)

    out = {"loss": _view(loss)}
    for name in _PARAMETERS:
        q = s["params"][name]
        shape = q["value"].shape
        new = b.adamW(q["value"].data, grads[name].data, q["m"].data, q["v"].data, 0.9, 0.999, 1e-8, 0.01, 1e-3, 10.0,
                      product(shape), f32)
        for key, data in zip(("value", "m", "v"), new):
            out[name + "." + key] = _view(wrap(data, shape))
    return out


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "small":
        x = s["x"] + s["y"]
        return [_view(x), _view(x.normalize(axis=1, eps=1e-5).mul(s["gain"] + 1, thenAdd=s["bias"]))]
    if kind == "matmul":
        return _view(Tensor.matmul(s["a"], c["ta"], s["b"], c["tb"], False))
    if kind == "attention":
        with backend().batching():
            scores = Tensor.batchedMatmul(s["q"], False, s["k"], True, False) * (1.0 / math.sqrt(c["hd"]))
            probs = (scores + s["mask"]).softmax()
            del scores
            out = Tensor.batchedMatmul(probs, False, s["v"], False, False)
            del probs
        return _view(out)
    if kind == "row_ops":
        h = (s["x"] + s["bias"]).gelu()
        return {"h": _view(h), "sum": _view(h.sum(axis=1)), "max": _view(h.max(axis=1)), "argmax": _view(h.argmax(axis=1))}
    if kind == "embedding":
        return [_view(s["table"].gather(0, s["ids"])), _view(s["grad"].scatter(0, c["vocab"], s["ids"]))]
    if kind == "transformer":
        s["recording"].graph.launch()
        return s["out"]
    if kind == "train_step":
        return _train_step(s)
    probs = s["logits"].softmax()
    order = s["logits"].argsort(1, descending=True)
    ranked = probs.gather(1, order)
    return {"order": _view(order), "ranked": _view(ranked), "cumulative": _view(ranked.cumulativeSum(1))}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c, z = case, _DTYPES[case["dtype"]].byteSize
    kind = c["kind"]
    if kind == "small":
        n = c["rows"] * c["cols"]
        return {"bytes": z * (4 * n + 2 * c["cols"]), "flops": 0}
    if kind == "matmul":
        m, k, n = c["m"], c["k"], c["n"]
        return {"bytes": z * (m * k + k * n + m * n), "flops": 2 * m * k * n}
    if kind == "attention":
        heads, t, hd = c["heads"], c["t"], c["hd"]
        return {"bytes": z * (4 * heads * t * hd + t * t), "flops": 4 * heads * t * t * hd}
    if kind == "row_ops":
        rows, cols = c["rows"], c["cols"]
        return {"bytes": z * (2 * rows * cols + cols + 2 * rows) + 8 * rows, "flops": 0}
    if kind == "embedding":
        ids, vocab, width = c["ids"], c["vocab"], c["width"]
        return {"bytes": 8 * ids + z * width * (min(ids, vocab) + 2 * ids + vocab), "flops": ids * width}
    if kind == "transformer":
        tokens, t, d, layers, vocab = c["batch"] * c["t"], c["t"], c["d"], c["layers"], c["vocab"]
        weights = layers * 12 * d * d + d * vocab
        return {"bytes": z * (weights + tokens * (d + vocab) + t * t + t * d) + 8 * tokens,
                "flops": 2 * tokens * weights + layers * 4 * tokens * t * d}
    if kind == "train_step":
        products = 2 * c["d"] * c["mlp"] + c["d"] * c["vocab"]
        params = sum(product(shape) for shape in _parameter_shapes(c).values())
        return {"bytes": 24 * params + 16 * c["tokens"], "flops": 6 * c["tokens"] * products}
    n = c["rows"] * c["vocab"]
    return {"bytes": n * (3 * z + 8), "flops": 0}


#: About four times the largest error seen over these ranges against the same calls with 64-bit arithmetic,
#: once with every stored value rounded to its type as the calls round it and once with none of them rounded
#: (what a correct implementation may keep in a wider type on the way).
_TOLERANCE = {
    "f32": {"train_step": {"rel": 6e-5, "max": 4.4e-3}, None: {"rel": 5e-6, "max": 4e-5}},
    "f16": {
        "small": {"rel": 2.4e-3, "max": 1e-2},
        "matmul": {"rel": 8e-4, "max": 4e-3},
        "attention": {"rel": 3.8e-3, "max": 7.5e-2},
        "row_ops": {"rel": 1.3e-3, "max": 4e-3, "differ": 7e-3},    # half values tie: argmax of the rounded ones
        "embedding": {"rel": 8e-4, "max": 2e-3},
        "transformer": {"rel": 4e-3, "max": 2.5e-2},
        "train_step": {"rel": 2e-2},                                 # gradients of a few ulps next to zero
        "sampling": {"rel": 2.4e-3, "max": 8e-3},
    },
}


def tolerance(case):
    by_kind = _TOLERANCE[case["dtype"]]
    return dict(by_kind.get(case["kind"], by_kind.get(None)))


# ---------------------------------------------------------------- the same in 64 bits

def _exact_norm(x):
    centered = x - x.mean(-1, keepdim=True)
    return centered / (centered.square().mean(-1, keepdim=True) + 1e-5).sqrt()


def _exact_gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _exact_attention(q, k, v, mask):
    scores = q @ k.transpose(-1, -2).contiguous() / math.sqrt(q.shape[-1]) + mask
    return scores.softmax(-1) @ v


def _exact_transformer(model, ids, heads):
    batch, t = ids.shape
    mask = torch.full((t, t), -1e4, device="cuda", dtype=torch.float64).triu(1)

    def value(tensor):
        return _view(tensor).double()

    def linear(layer, x):
        return x @ value(layer.weight) + value(layer.bias)

    def norm(layer, x):
        return _exact_norm(x) * (1 + value(layer.gain)) + value(layer.bias)

    def split(x):
        return x.reshape(batch, t, heads, -1).transpose(1, 2).contiguous()

    x = value(model.table)[ids] + value(model.pos)[:t]
    for block in model.blocks:
        h = norm(block.ln1, x)
        mixed = _exact_attention(split(linear(block.q, h)), split(linear(block.k, h)), split(linear(block.v, h)), mask)
        x = x + linear(block.o, mixed.transpose(1, 2).reshape(x.shape))
        x = x + linear(block.fc2, _exact_gelu(linear(block.fc1, norm(block.ln2, x))))
    return linear(model.unembed, norm(model.ln_f, x))


def _exact_train_step(s):
    ids, targets = _view(s["ids"]), _view(s["targets"])
    p = {name: _view(s["params"][name]["value"]).double().requires_grad_() for name in _PARAMETERS}
    x = p["table"][ids]
    f = (_exact_norm(x) * (1 + p["gain"]) + p["shift"]) @ p["w1"] + p["b1"]
    y = x + _exact_gelu(f) @ p["w2"] + p["b2"]
    loss = -(y @ p["wo"]).log_softmax(1).gather(1, targets[:, None]).sum()
    loss.backward()
    beta1, beta2, eps, decay, lr = torch.tensor([0.9, 0.999, 1e-8, 0.01, 1e-3], dtype=torch.float32).double().tolist()
    out = {"loss": loss.detach().reshape([])}
    for name in _PARAMETERS:
        g = p[name].grad
        m = beta1 * _view(s["params"][name]["m"]).double() + (1 - beta1) * g
        v = beta2 * _view(s["params"][name]["v"]).double() + (1 - beta2) * g * g
        moved = m / (1 - beta1 ** 10) / ((v / (1 - beta2 ** 10)).sqrt() + eps)
        out[name + ".value"] = p[name].detach() * (1 - lr * decay) - lr * moved
        out[name + ".m"], out[name + ".v"] = m, v
    return out


def exact(case, seed):
    """What `run` returns for these inputs, in plain torch with 64-bit numbers and nothing rounded on the way.
    None in the place of whole numbers that ties of rounded values decide."""
    c, s = case, prepare(case, seed)
    kind, half = c["kind"], c["dtype"] == "f16"
    if kind == "transformer":
        return _exact_transformer(s["model"], _view(s["ids"]), c["heads"])
    if kind == "train_step":
        return _exact_train_step(s)
    v = {name: _view(t) for name, t in s.items() if isinstance(t, Tensor)}
    v = {name: t if t.dtype == torch.int64 else t.double() for name, t in v.items()}
    if kind == "small":
        x = v["x"] + v["y"]
        return [x, _exact_norm(x) * (v["gain"] + 1) + v["bias"]]
    if kind == "matmul":
        return (v["a"].t() if c["ta"] else v["a"]) @ (v["b"].t() if c["tb"] else v["b"])
    if kind == "attention":
        return _exact_attention(v["q"], v["k"], v["v"], v["mask"])
    if kind == "row_ops":
        h = _exact_gelu(v["x"] + v["bias"])
        return {"h": h, "sum": h.sum(1), "max": h.max(1).values, "argmax": None if half else h.argmax(1)}
    if kind == "embedding":
        table = torch.zeros(c["vocab"], c["width"], dtype=torch.float64, device="cuda")
        return [v["table"][v["ids"]], table.index_add_(0, v["ids"], v["grad"])]
    ranked, order = v["logits"].sort(dim=1, descending=True, stable=True)
    ranked = ranked.softmax(1)
    return {"order": order, "ranked": ranked, "cumulative": ranked.cumsum(1)}
