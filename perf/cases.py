"""The work that a user of the 'hip' device has it do, at the sizes it is used at.

All of it is float32, the only floating type that the device computes in.
Every case goes through the public entry points (nn modules, functional ops,
the workload models, backward() and the optimizers).  `listed()` holds fixed
sizes, `draw()` others of the same ranges.

Inputs are made by torch on the GPU from the seed and copied into the
library's tensors; outputs are returned as torch views of the library's own
memory (no copy)."""
import math

import torch
import torch.nn.functional as TF

import __graft_entry__ as graft

hip = graft.load_package()
from torchjs_amd import workloads as W  # noqa: E402  (the package is loaded by the line above)

F = hip.functional

VOCAB, CTX, D, HEADS, LAYERS = 50257, 1024, 768, 12, 12  # GPT-2 small


def listed():
    return [
        # the smallest training program: a 784-256-10 classifier, one whole
        # step with Adam; launches and host work are most of it
        dict(name="mlp train 64", kind="mlp", batch=64, din=784, hidden=256, classes=10),
        # an elementwise chain with a broadcast bias and reductions, forward
        # and backward: what activation code outside the fused layers does
        dict(name="chain 4096x4096", kind="chain", rows=4096, cols=4096),
        # a small convolutional classifier, forward and backward
        dict(name="cnn 32x64x64", kind="cnn", batch=32, side=64),
        # one transformer block at GPT-2's training size, forward and backward
        dict(name="block 8x1024x768", kind="block", batch=8, seq=1024, heads=12, dim=768),
        # the same layer in a smaller model on an odd sequence length
        dict(name="block 3x509x384", kind="block", batch=3, seq=509, heads=6, dim=384),
        # bidirectional attention over an odd length with a head size that is
        # no power of two, forward and backward
        dict(name="attention 4x16x701x80", kind="attention", batch=4, heads=16, q=701, k=701,
             dim=80, causal=False),
        # one norm of an odd row count and a width outside GPT-2's
        dict(name="layernorm 4099x1000", kind="layernorm", rows=4099, cols=1000),
        # the language-model head and its loss on two sequences
        dict(name="head 2048x768x50257", kind="head", rows=2048, dim=768, vocab=VOCAB),
        # the optimizer over a large embedding and one block's parameters
        dict(name="adamw 46M", kind="adamw", dim=768, vocab=VOCAB, seq=1024),
        # the headline: one GPT-2 small training step
        dict(name="gpt2 train 8x1024", kind="gpt2_train", batch=8, seq=1024, dim=D, layers=LAYERS,
             vocab=VOCAB),
        # reading a prompt without gradients
        dict(name="gpt2 prompt 1x777", kind="gpt2_prompt", batch=1, seq=777, dim=D, layers=LAYERS,
             vocab=VOCAB),
        # one cached token for each of four sequences
        dict(name="gpt2 decode 4x700", kind="gpt2_decode", batch=4, seq=700, dim=D, layers=LAYERS,
             vocab=VOCAB),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "chain", "cnn", "block", "attention", "layernorm", "head", "adamw",
                       "gpt2_train", "gpt2_prompt", "gpt2_decode"])
    if kind == "mlp":
        return dict(kind=kind, batch=_log(rng, 1, 1024), din=_log(rng, 32, 2048),
                    hidden=_log(rng, 32, 1024), classes=_log(rng, 2, 1000))
    if kind == "chain":
        return dict(kind=kind, rows=_log(rng, 64, 4096), cols=_log(rng, 64, 4096))
    if kind == "cnn":
        return dict(kind=kind, batch=_log(rng, 1, 64), side=rng.randint(15, 96))
    if kind == "block":
        heads = rng.randint(2, 16)
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log(rng, 17, 1024), heads=heads,
                    dim=heads * rng.choice([32, 64, 64, 80]))
    if kind == "attention":
        causal = rng.random() < 0.5
        q = _log(rng, 16, 1024)
        return dict(kind=kind, batch=rng.randint(1, 8), heads=rng.randint(1, 16), q=q,
                    k=q if causal else _log(rng, 16, 1024), dim=rng.choice([32, 40, 64, 80, 96, 128]),
                    causal=causal)
    if kind == "layernorm":
        return dict(kind=kind, rows=_log(rng, 64, 16384), cols=_log(rng, 64, 3072))
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 64, 4096), dim=64 * rng.randint(2, 16),
                    vocab=_log(rng, 1000, 50257))
    if kind == "adamw":
        return dict(kind=kind, dim=64 * rng.randint(2, 12), vocab=_log(rng, 1000, 50257),
                    seq=rng.randint(64, 1024))
    dim = 64 * rng.randint(4, 12)
    if kind == "gpt2_train":
        return dict(kind=kind, batch=rng.randint(1, 8), seq=_log(rng, 64, 1024), dim=dim,
                    layers=rng.randint(1, 12), vocab=_log(rng, 5000, 50257))
    return dict(kind=kind, batch=rng.randint(1, 8), seq=_log(rng, 16, 1000), dim=dim,
                layers=rng.randint(1, 12), vocab=_log(rng, 5000, 50257))


# ------------------------------------------------- tensors to and from torch


class _Array:
    """A library tensor's memory for torch.as_tensor, which keeps this object
    (and with it the memory) as long as the torch tensor lives."""

    def __init__(self, t):
        self.tensor = t
        self.__cuda_array_interface__ = {
            "shape": t.shape, "strides": tuple(4 * s for s in t.stride()),
            "typestr": "<f4" if t.dtype == "float32" else "<i4", "data": (t.data_ptr(), False),
            "version": 2}


def _view(t):
    return torch.as_tensor(_Array(t.detach()), device="cuda")


def _to_hip(x, grad=False):
    """`x` in a tensor of the library."""
    hip.init(0)
    t = hip.empty(tuple(x.shape), dtype="int32" if x.dtype == torch.int32 else "float32")
    _view(t).copy_(x)
    torch.cuda.synchronize()
    t.requires_grad = grad
    return t


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda") * std + mean


def _ids(g, high, *shape):
    return torch.randint(0, high, shape, generator=g, device="cuda", dtype=torch.int32)


# --------------------------------------------------------------------- inputs


def _block_weights(g, d, pre=""):
    w = {}
    for ln in ("ln_1", "ln_2"):
        w[pre + ln + ".weight"] = _randn(g, d, std=0.1, mean=1.0)
        w[pre + ln + ".bias"] = _randn(g, d, std=0.1)
    for name, n, k in (("attn.c_attn", 3 * d, d), ("attn.c_proj", d, d), ("mlp.c_fc", 4 * d, d),
                       ("mlp.c_proj", d, 4 * d)):
        w[pre + name + ".weight"] = _randn(g, n, k, std=0.5 / math.sqrt(k))
        w[pre + name + ".bias"] = _randn(g, n, std=0.02)
    return w


def _gpt2_weights(g, c):
    d = c["dim"]
    w = {"wte.weight": _randn(g, c["vocab"], d, std=0.02), "wpe.weight": _randn(g, CTX, d, std=0.02)}
    for i in range(c["layers"]):
        w.update(_block_weights(g, d, "h.%d." % i))
    w["ln_f.weight"], w["ln_f.bias"] = _randn(g, d, std=0.1, mean=1.0), _randn(g, d, std=0.1)
    return w


def _inputs(c, seed):
    """(weights by name, other inputs by name) as torch tensors."""
    g, kind = _gen(seed), c["kind"]
    if kind == "mlp":
        a, h, n = c["din"], c["hidden"], c["classes"]
        w = {"0.weight": _randn(g, h, a, std=a ** -0.5), "0.bias": _randn(g, h, std=a ** -0.5),
             "2.weight": _randn(g, n, h, std=h ** -0.5), "2.bias": _randn(g, n, std=h ** -0.5)}
        return w, {"x": _randn(g, c["batch"], a), "t": _ids(g, n, c["batch"])}
    if kind == "chain":
        r, n = c["rows"], c["cols"]
        return {}, {"x": _randn(g, r, n), "bias": _randn(g, n),
                    "y": torch.rand((r, n), generator=g, device="cuda") * 2 - 1}
    if kind == "cnn":
        w = {"conv1.weight": _randn(g, 32, 3, 3, 3, std=0.2), "conv1.bias": _randn(g, 32, std=0.1),
             "conv2.weight": _randn(g, 64, 32, 3, 3, std=0.06), "conv2.bias": _randn(g, 64, std=0.1),
             "fc.weight": _randn(g, 10, 64, std=0.125), "fc.bias": _randn(g, 10, std=0.1)}
        b, s = c["batch"], c["side"]
        return w, {"x": _randn(g, b, 3, s, s), "t": _ids(g, 10, b)}
    if kind == "block":
        s = (c["batch"], c["seq"], c["dim"])
        return _block_weights(g, c["dim"]), {"x": _randn(g, *s), "g": _randn(g, *s, std=1e-3)}
    if kind == "attention":
        b, h, d = c["batch"], c["heads"], c["dim"]
        return {}, {"q": _randn(g, b, h, c["q"], d), "k": _randn(g, b, h, c["k"], d),
                    "v": _randn(g, b, h, c["k"], d), "g": _randn(g, b, h, c["q"], d, std=1e-3)}
    if kind == "layernorm":
        r, n = c["rows"], c["cols"]
        return ({"weight": _randn(g, n, std=0.1, mean=1.0), "bias": _randn(g, n, std=0.1)},
                {"x": _randn(g, r, n, std=2.0, mean=0.3), "g": _randn(g, r, n, std=1e-3)})
    if kind == "head":
        return ({"weight": _randn(g, c["vocab"], c["dim"], std=0.02)},
                {"x": _randn(g, c["rows"], c["dim"]), "t": _ids(g, c["vocab"], c["rows"])})
    if kind == "adamw":
        d = c["dim"]
        w = {"wte": _randn(g, c["vocab"], d, std=0.02), "wpe": _randn(g, c["seq"], d, std=0.02)}
        w.update(_block_weights(g, d))
        return w, {"g." + k: _randn(g, *v.shape, std=1e-3) for k, v in w.items()}
    w = _gpt2_weights(g, c)
    if kind == "gpt2_train":
        toks = _ids(g, c["vocab"], c["batch"], c["seq"] + 1)
        return w, {"ids": toks[:, :-1].contiguous(), "t": toks[:, 1:].contiguous()}
    if kind == "gpt2_prompt":
        return w, {"ids": _ids(g, c["vocab"], c["batch"], c["seq"])}
    # decode: one token each after `seq` earlier positions
    x = {"ids": _ids(g, c["vocab"], c["batch"], 1)}
    for i in range(c["layers"]):
        x["k%d" % i] = _randn(g, c["batch"], c["dim"] // 64, c["seq"], 64)
        x["v%d" % i] = _randn(g, c["batch"], c["dim"] // 64, c["seq"], 64)
    return w, x


def _load(module, w):
    """`w` in the module's parameters."""
    params = dict(module.named_parameters())
    for k, v in w.items():
        _view(params[k]).copy_(v)
    torch.cuda.synchronize()
    return module


def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    w, x = _inputs(case, seed)
    s = {"kind": kind}
    if kind in ("block", "attention", "layernorm", "head", "chain"):
        s.update({k: _to_hip(v, grad=k not in ("g", "t")) for k, v in x.items()})
        if kind == "block":
            s["model"] = _load(W.Block(case["dim"], case["heads"]), w)
        else:
            s.update({k: _to_hip(v, grad=True) for k, v in w.items()})
        s["causal"] = case.get("causal")
        return s
    if kind == "adamw":
        s["p"] = {k: _to_hip(v, grad=True) for k, v in w.items()}
        for k, p in s["p"].items():
            p.grad = _to_hip(x["g." + k])
        s["opt"] = hip.optim.AdamW(list(s["p"].values()), lr=6e-4, weight_decay=0.1)
        s["views"] = {k: _view(p) for k, p in s["p"].items()}
        return s
    s.update({k: _to_hip(v) for k, v in x.items() if k in ("x", "t", "ids")})
    if kind == "mlp":
        s["model"] = _load(hip.nn.Sequential(hip.nn.Linear(case["din"], case["hidden"]), hip.nn.ReLU(),
                                             hip.nn.Linear(case["hidden"], case["classes"])), w)
        s["opt"] = hip.optim.Adam(s["model"].parameters(), lr=1e-3)
    elif kind == "cnn":
        s["model"] = _load(W.CNN(), w)
    else:
        s["model"] = _load(W.GPT2(case["vocab"], CTX, case["dim"], case["dim"] // 64, case["layers"]), w)
    if kind == "gpt2_train":
        s["opt"] = hip.optim.AdamW(s["model"].parameters(), lr=6e-4, weight_decay=0.1)
        # the tables, the last norm and three blocks: whole gradients of each
        last = case["layers"] - 1
        keep = ("wte.", "wpe.", "ln_f.", "h.0.", "h.%d." % (last // 2), "h.%d." % last)
        s["keep"] = {k: p for k, p in s["model"].named_parameters() if k.startswith(keep)}
    elif kind == "gpt2_decode":
        s["pos"] = case["seq"]
        s["cache"], s["views"] = s["model"].new_cache(case["batch"]), {}
        for i in range(case["layers"]):
            for name, to in (("k%d" % i, s["cache"].k[i]), ("v%d" % i, s["cache"].v[i])):
                s["views"][name] = _view(to)
                s["views"][name][:, :, :case["seq"]].copy_(x[name])
        torch.cuda.synchronize()
    if kind == "mlp":
        s["views"] = {k: _view(p) for k, p in s["model"].named_parameters()}
    return s


# ----------------------------------------------------------------- one pass


def run(s):
    kind = s["kind"]
    if kind == "mlp":
        s["opt"].zero_grad()
        loss = F.cross_entropy(s["model"](s["x"]), s["t"])
        loss.backward()
        s["opt"].step()
        return dict(s["views"], loss=_view(loss))
    if kind == "chain":
        ts = {k: s[k] for k in ("x", "bias", "y")}
        for t in ts.values():
            t.grad = None
        loss = W.chain_loss(s["x"], s["bias"], s["y"])
        loss.backward()
        return dict({k: _view(t.grad) for k, t in ts.items()}, loss=_view(loss))
    if kind == "cnn":
        m = s["model"]
        m.zero_grad()
        logits = m(s["x"])
        F.cross_entropy(logits, s["t"]).backward()
        return dict({k: _view(p.grad) for k, p in m.named_parameters()}, logits=_view(logits))
    if kind == "block":
        m, x = s["model"], s["x"]
        m.zero_grad()
        x.grad = None
        y = m(x)
        y.backward(s["g"])
        return dict({k: _view(p.grad) for k, p in m.named_parameters()}, y=_view(y), x=_view(x.grad))
    if kind == "attention":
        ts = {k: s[k] for k in ("q", "k", "v")}
        for t in ts.values():
            t.grad = None
        y = F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=s["causal"])
        y.backward(s["g"])
        return dict({k: _view(t.grad) for k, t in ts.items()}, y=_view(y))
    if kind == "layernorm":
        ts = {k: s[k] for k in ("x", "weight", "bias")}
        for t in ts.values():
            t.grad = None
        y = F.layer_norm(s["x"], (s["x"].shape[1],), s["weight"], s["bias"])
        y.backward(s["g"])
        return dict({k: _view(t.grad) for k, t in ts.items()}, y=_view(y))
    if kind == "head":
        ts = {k: s[k] for k in ("x", "weight")}
        for t in ts.values():
            t.grad = None
        logits = F.linear(s["x"], s["weight"])
        loss = F.cross_entropy(logits, s["t"])
        loss.backward()
        return dict({k: _view(t.grad) for k, t in ts.items()}, logits=_view(logits), loss=_view(loss))
    if kind == "adamw":
        s["opt"].step()
        if "moments" not in s:  # the optimizer made them in its first step
            s["moments"] = {"%s.%s" % (m, k): _view(s["opt"].state[id(p)][m])
                            for k, p in s["p"].items() for m in ("exp_avg", "exp_avg_sq")}
        return dict(s["views"], **s["moments"])
    if kind == "gpt2_train":
        s["opt"].zero_grad()
        loss = s["model"].loss(s["ids"], s["t"])
        loss.backward()
        s["opt"].step()
        return dict({k: _view(p.grad) for k, p in s["keep"].items()}, loss=_view(loss))
    with hip.no_grad():
        if kind == "gpt2_prompt":
            return _view(s["model"](s["ids"]))
        logits = s["model"].forward_cached(s["ids"], s["cache"], s["pos"])
        return dict(s["views"], logits=_view(logits))


# ---------------------------------------------------------------- what it is


def _block_flops(b, t, d, past=0):
    """Products of one block, forward: the four linears and causal attention
    (each query with the keys up to its own)."""
    return b * t * 24 * d * d + 4 * b * d * (t * (t + 1) // 2 + t * past)


def work(c):
    kind = c["kind"]
    if kind == "mlp":
        n = c["din"] * c["hidden"] + c["hidden"] * c["classes"] + c["hidden"] + c["classes"]
        m = c["batch"]
        return {"bytes": 4 * (m * c["din"] + m + 6 * n),
                "flops": 2 * m * (2 * c["din"] * c["hidden"] + 3 * c["hidden"] * c["classes"])}
    if kind == "chain":
        n = c["rows"] * c["cols"]
        return {"bytes": 4 * (4 * n + 2 * c["cols"]), "flops": 40 * n}
    if kind == "cnn":
        b, s = c["batch"], c["side"]
        h = (s + 1) // 2
        conv1, conv2 = 2 * b * s * s * 32 * 27, 2 * b * h * h * 64 * 288
        n = 32 * 28 + 64 * 289 + 650
        return {"bytes": 4 * (b * 3 * s * s + 2 * n + 10 * b), "flops": 2 * conv1 + 3 * conv2}
    if kind == "block":
        n = c["batch"] * c["seq"] * c["dim"]
        p = 12 * c["dim"] ** 2 + 13 * c["dim"]
        return {"bytes": 4 * (4 * n + 2 * p), "flops": 3 * _block_flops(c["batch"], c["seq"], c["dim"])}
    if kind == "attention":
        b, h, d = c["batch"], c["heads"], c["dim"]
        pairs = c["q"] * (c["q"] + 1) // 2 if c["causal"] else c["q"] * c["k"]
        # forward two products of that size, backward five
        return {"bytes": 4 * b * h * d * (4 * c["q"] + 4 * c["k"]),
                "flops": 14 * b * h * pairs * d}
    if kind == "layernorm":
        n = c["rows"] * c["cols"]
        return {"bytes": 4 * (4 * n + 4 * c["cols"]), "flops": 20 * n}
    if kind == "head":
        r, d, v = c["rows"], c["dim"], c["vocab"]
        return {"bytes": 4 * (2 * r * d + 2 * v * d + r * v + r), "flops": 6 * r * d * v}
    if kind == "adamw":
        d = c["dim"]
        n = (c["vocab"] + c["seq"]) * d + 12 * d * d + 13 * d
        return {"bytes": 28 * n, "flops": 12 * n}
    d, v, b = c["dim"], c["vocab"], c["batch"]
    block = 12 * d * d + 13 * d
    n = (v + CTX) * d + c["layers"] * block + 2 * d
    if kind == "gpt2_train":
        r = b * c["seq"]
        # weights and moments read and written, gradients written
        return {"bytes": 4 * (7 * n + 2 * r),
                "flops": 3 * (c["layers"] * _block_flops(b, c["seq"], d) + 2 * r * d * v) + 12 * n}
    if kind == "gpt2_prompt":
        r = b * c["seq"]
        return {"bytes": 4 * (n - (CTX - c["seq"]) * d + r * v + r),
                "flops": c["layers"] * _block_flops(b, c["seq"], d) + 2 * r * d * v}
    kv = 2 * b * (c["seq"] + 1) * d
    return {"bytes": 4 * (n - CTX * d + c["layers"] * kv + b * v),
            "flops": c["layers"] * _block_flops(b, 1, d, c["seq"]) + 2 * b * d * v}


def tolerance(c):
    """About four times the difference between a float32 path and one in 64
    bits, as measured at the listed sizes."""
    return {"rel": {
        "adamw": 2e-7,      # 3e-8: a few roundings per element
        "layernorm": 6e-7,  # 1.3e-7
        "chain": 6e-7,      # 1.3e-7: erf and exp
        "mlp": 4e-6,        # 1e-6: weights after a step, g / (|g| + eps) of small gradients
        # 2.4e-7 where no ReLU input rounds across 0; one that does moves a
        # gradient of some 1e5 summed terms by one of them
        "cnn": 2e-5,
        # products summed over up to 50257 terms, and what follows from them:
        # 2e-6 in the gradients of a whole model or of attention
    }.get(c["kind"], 1e-5)}


# -------------------------------------------------------- the same in 64 bits


def _attend(q, k, v, causal):
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        t = q.shape[-2]
        s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.contiguous())


def _block(w, pre, x, heads, past=None, kv=None):
    """`past`: earlier keys and values; `kv` gets all of them."""
    b, t, d = x.shape
    h = TF.layer_norm(x, (d,), w[pre + "ln_1.weight"], w[pre + "ln_1.bias"])
    h = TF.linear(h, w[pre + "attn.c_attn.weight"], w[pre + "attn.c_attn.bias"])
    q, k, v = (a.reshape(b, t, heads, d // heads).transpose(1, 2) for a in h.split(d, 2))
    if past is not None:
        k, v = torch.cat([past[0], k], 2), torch.cat([past[1], v], 2)
        kv.append((k, v))
    h = _attend(q, k, v, past is None).transpose(1, 2).reshape(b, t, d)
    x = x + TF.linear(h, w[pre + "attn.c_proj.weight"], w[pre + "attn.c_proj.bias"])
    h = TF.layer_norm(x, (d,), w[pre + "ln_2.weight"], w[pre + "ln_2.bias"])
    h = TF.gelu(TF.linear(h, w[pre + "mlp.c_fc.weight"], w[pre + "mlp.c_fc.bias"]))
    return x + TF.linear(h, w[pre + "mlp.c_proj.weight"], w[pre + "mlp.c_proj.bias"])


def _gpt2(w, c, ids, pos=0, past=None, kv=None):
    d = c["dim"]
    x = w["wte.weight"][ids.long()] + w["wpe.weight"][pos:pos + ids.shape[1]]
    for i in range(c["layers"]):
        x = _block(w, "h.%d." % i, x, d // 64, None if past is None else past[i], kv)
    x = TF.layer_norm(x, (d,), w["ln_f.weight"], w["ln_f.bias"])
    return TF.linear(x, w["wte.weight"])


def _adam(p, g, lr, wd):
    """One first step of Adam with decoupled decay `wd`: (p, m, v)."""
    return (p * (1 - lr * wd) - lr * g / (g.abs() + 1e-8), 0.1 * g, 0.001 * g * g)


def exact(case, seed):
    kind = case["kind"]
    w, x = _inputs(case, seed)
    train = kind not in ("adamw", "gpt2_prompt", "gpt2_decode")
    w = {k: v.double().requires_grad_(train) for k, v in w.items()}
    x = {k: v.double().requires_grad_(train and k not in ("g", "t")) if v.is_floating_point() else v
         for k, v in x.items()}

    def grads():
        return {k: v.grad for k, v in list(w.items()) + list(x.items()) if k not in ("g", "t", "ids")}

    if kind == "mlp":
        h = torch.relu(TF.linear(x["x"], w["0.weight"], w["0.bias"]))
        loss = TF.cross_entropy(TF.linear(h, w["2.weight"], w["2.bias"]), x["t"].long())
        loss.backward()
        return dict({k: _adam(p.detach(), p.grad, 1e-3, 0.0)[0] for k, p in w.items()},
                    loss=loss.detach())
    if kind == "chain":
        loss = (TF.gelu(x["x"] + x["bias"]) * x["y"]).sum(0).mean()
        loss.backward()
        return dict(grads(), loss=loss.detach())
    if kind == "cnn":
        h = torch.relu(_conv(x["x"], w["conv1.weight"], w["conv1.bias"], 1))
        h = torch.relu(_conv(h, w["conv2.weight"], w["conv2.bias"], 2))
        logits = TF.linear(h.mean((2, 3)), w["fc.weight"], w["fc.bias"])
        TF.cross_entropy(logits, x["t"].long()).backward()
        return dict({k: p.grad for k, p in w.items()}, logits=logits.detach())
    if kind == "block":
        y = _block(w, "", x["x"], case["heads"])
        y.backward(x["g"])
        return dict(grads(), y=y.detach())
    if kind == "attention":
        y = _attend(x["q"], x["k"], x["v"], case["causal"])
        y.backward(x["g"])
        return dict(grads(), y=y.detach())
    if kind == "layernorm":
        y = TF.layer_norm(x["x"], (case["cols"],), w["weight"], w["bias"])
        y.backward(x["g"])
        return dict(grads(), y=y.detach())
    if kind == "head":
        logits = TF.linear(x["x"], w["weight"])
        loss = TF.cross_entropy(logits, x["t"].long())
        loss.backward()
        return dict(grads(), logits=logits.detach(), loss=loss.detach())
    if kind == "adamw":
        out = {}
        for k, p in w.items():
            out[k], out["exp_avg." + k], out["exp_avg_sq." + k] = _adam(p, x["g." + k], 6e-4, 0.1)
        return out
    if kind == "gpt2_train":
        logits = _gpt2(w, case, x["ids"])
        loss = TF.cross_entropy(logits.view(-1, case["vocab"]), x["t"].long().view(-1))
        loss.backward()
        last = case["layers"] - 1
        keep = ("wte.", "wpe.", "ln_f.", "h.0.", "h.%d." % (last // 2), "h.%d." % last)
        return dict({k: v.grad for k, v in w.items() if k.startswith(keep)}, loss=loss.detach())
    if kind == "gpt2_prompt":
        return _gpt2(w, case, x["ids"])
    past = [(x["k%d" % i], x["v%d" % i]) for i in range(case["layers"])]
    kv = []
    out = {"logits": _gpt2(w, case, x["ids"], case["seq"], past, kv)}
    for i, both in enumerate(kv):
        for name, a in zip("kv", both):
            out["%s%d" % (name, i)] = TF.pad(a, (0, 0, 0, CTX - a.shape[2]))
    return out


def _conv(x, w, b, stride):
    """A 3x3 convolution with padding 1 as a product over unfolded patches."""
    h = (x.shape[2] - 1) // stride + 1
    cols = TF.unfold(x, 3, padding=1, stride=stride)
    y = torch.matmul(w.reshape(w.shape[0], -1), cols)
    return y.reshape(x.shape[0], w.shape[0], h, -1) + b.view(1, -1, 1, 1)
