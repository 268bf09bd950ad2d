"""The work that a user of this backend has it do, as cases that can be timed and checked.

A case is one call (for a linear layer's backward and for a head, the two calls that belong
together) through the public entry points on arrays that are already on the device: `mf.sgemm`
with the descriptor that a program fills once per layer, `mf.sgemv`, `mf.attention_fused`,
`mf.softmax` and `mf.argmax`. Outputs are written into arrays that the program keeps, as it does
between steps.

Kinds of case and the ranges that `draw` takes them from:
* gemm        C = act(alpha op(A) op(B) + beta C0 + bias), 16 .. 4096 a side, all four layouts;
* backward    a linear layer's dX = dY W^T and dW = X^T dY;
* gemv        y = alpha op(A) x + beta y0, 64 .. 16384 a side, both forms;
* attention   prefill (causal or with padded keys) and decode (one query per head);
* head        softmax over a row of logits, and the row's argmax.
"""
import math

import torch

import mensurflow_amd as mf

_STREAM = None


def _stream():
    """The program's one stream on the device: kernels, workspace and released arrays go with it."""
    global _STREAM
    if _STREAM is None:
        _STREAM = mf.Stream(0)
    return _STREAM


def listed():
    return [
        # A small layer: launches and latency.
        dict(name="gemm_small", kind="gemm", m=256, n=256, k=256, ta=False, tb=False,
             alpha=1.0, beta=0.0, bias=False, gelu=False),
        # matmul at a middle size.
        dict(name="gemm_square", kind="gemm", m=1024, n=1024, k=1024, ta=False, tb=False,
             alpha=1.0, beta=0.0, bias=False, gelu=False),
        # The large square product, with B stored transposed, alpha and beta C0.
        dict(name="gemm_large", kind="gemm", m=4096, n=4096, k=4096, ta=False, tb=True,
             alpha=1.5, beta=0.5, bias=False, gelu=False),
        # A serving step's layer: a few rows against a large weight stored [out, in].
        dict(name="gemm_few_rows", kind="gemm", m=32, n=4096, k=4096, ta=False, tb=True,
             alpha=1.0, beta=0.0, bias=True, gelu=False),
        # An MLP layer with ragged sizes, bias and the tanh gelu.
        dict(name="mlp_gelu", kind="gemm", m=4093, n=4099, k=1023, ta=False, tb=False,
             alpha=1.0, beta=0.0, bias=True, gelu=True),
        # The two products of a linear layer's backward pass.
        dict(name="linear_backward", kind="backward", rows=2000, cin=1000, cout=1960),
        # The large gemv.
        dict(name="gemv_large", kind="gemv", rows=16384, cols=16384, trans=False,
             alpha=2.0, beta=0.5),
        # A^T x on an odd, smaller matrix.
        dict(name="gemv_t_ragged", kind="gemv", rows=4093, cols=1023, trans=True,
             alpha=1.0, beta=0.0),
        # Attention over a whole sequence, causal.
        dict(name="attention_prefill", kind="attention", batch=8, heads=16, lq=1024, lk=1024,
             d=64, causal=True, mask=False),
        # One new query per head against the keys so far.
        dict(name="attention_decode", kind="attention", batch=8, heads=16, lq=1, lk=4096,
             d=64, causal=False, mask=False),
        # Sequences of several lengths in one batch: padded keys masked out.
        dict(name="attention_padded", kind="attention", batch=4, heads=16, lq=1000, lk=1000,
             d=128, causal=False, mask=True),
        # Probabilities and greedy choice over a vocabulary, rows of odd length.
        dict(name="head", kind="head", rows=512, width=32003),
    ]


def _log(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "gemm", "backward", "gemv", "gemv", "attention",
                       "attention", "attention", "head"])
    if kind == "gemm":
        beta = rng.choice([0.0, 0.0, 0.5])
        bias = rng.random() < 0.5
        return dict(kind="gemm", m=_log(rng, 16, 4096), n=_log(rng, 64, 4096),
                    k=_log(rng, 64, 4096), ta=rng.random() < 0.25, tb=rng.random() < 0.5,
                    alpha=rng.choice([1.0, 1.5]), beta=beta, bias=bias,
                    gelu=bias and rng.random() < 0.5)
    if kind == "backward":
        return dict(kind="backward", rows=_log(rng, 64, 4096), cin=_log(rng, 64, 3000),
                    cout=_log(rng, 64, 3000))
    if kind == "gemv":
        return dict(kind="gemv", rows=_log(rng, 64, 16384), cols=_log(rng, 64, 16384),
                    trans=rng.random() < 0.5, alpha=rng.choice([1.0, 2.0]),
                    beta=rng.choice([0.0, 0.5]))
    if kind == "attention":
        form = rng.choice(["causal", "padded", "plain", "decode"])
        lk = _log(rng, 64, 4096 if form == "decode" else 1024)
        return dict(kind="attention", batch=rng.randint(1, 8), heads=rng.randint(1, 16),
                    lq=1 if form == "decode" else lk, lk=lk, d=rng.choice([32, 64, 96, 128]),
                    causal=form == "causal", mask=form == "padded")
    return dict(kind="head", rows=_log(rng, 1, 512), width=_log(rng, 1000, 32003))


def _values(case, seed):
    """The inputs, from the seed alone, as torch tensors on the device."""
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def uniform(shape, low=-1.0, high=1.0):
        return torch.rand(shape, generator=gen, device="cuda") * (high - low) + low

    def normal(shape, std=1.0):
        return torch.randn(shape, generator=gen, device="cuda") * std

    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        a_shape = (k, m) if case["ta"] else (m, k)
        b_shape = (n, k) if case["tb"] else (k, n)
        if case["bias"]:  # a layer: activations and weights
            v = {"a": normal(a_shape), "b": normal(b_shape, 1 / math.sqrt(k)),
                 "bias": uniform((n,), -0.1, 0.1)}
        else:
            v = {"a": uniform(a_shape), "b": uniform(b_shape)}
        if case["beta"]:
            v["c0"] = normal((m, n))
        return v
    if kind == "backward":
        rows, cin, cout = case["rows"], case["cin"], case["cout"]
        return {"x": normal((rows, cin)), "w": normal((cin, cout), 1 / math.sqrt(cin)),
                "dy": normal((rows, cout), 0.1)}
    if kind == "gemv":
        rows, cols = case["rows"], case["cols"]
        n_in, n_out = (rows, cols) if case["trans"] else (cols, rows)
        v = {"a": uniform((rows, cols)), "x": uniform((n_in,))}
        if case["beta"]:
            v["y0"] = normal((n_out,))
        return v
    if kind == "attention":
        lead = (case["batch"], case["heads"])
        v = {"q": normal(lead + (case["lq"], case["d"])), "k": normal(lead + (case["lk"], case["d"])),
             "v": normal(lead + (case["lk"], case["d"]))}
        if case["mask"]:
            lk = case["lk"]
            lengths = torch.randint((lk + 1) // 2, lk + 1, (case["batch"], 1), generator=gen,
                                    device="cuda")
            keep = torch.arange(lk, device="cuda")[None, :] < lengths
            v["mask"] = keep.to(torch.uint8).reshape(case["batch"], 1, 1, lk)
        return v
    return {"x": normal((case["rows"], case["width"]), 4.0)}


_NUMPY = {torch.float32: "float32", torch.uint8: "uint8", torch.int64: "int64"}


class _Exposed:
    """A contiguous device array as torch sees it."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {
            "shape": array.shape, "typestr": array.dtype.str, "data": (array.ptr, False),
            "version": 2}


def _tensor(array):
    return torch.as_tensor(_Exposed(array), device="cuda")


def _empty(shape, dtype="float32"):
    return mf.DeviceArray.empty(shape, _stream(), dtype)


def _array(tensor):
    out = _empty(tuple(tensor.shape), _NUMPY[tensor.dtype])
    _tensor(out).copy_(tensor)
    return out


def _desc(a, b, c, alpha=1.0, c0=None, beta=0.0, bias=None, act=mf.ACT_NONE):
    """C = act(alpha A B + beta C0 + bias) of two-dimensional arrays, B and A perhaps views."""
    d = mf.GemmDesc()
    d.m, d.k = a.shape
    d.n = b.shape[1]
    d.a, (d.a_rs, d.a_cs) = a.ptr, a.strides
    d.b, (d.b_rs, d.b_cs) = b.ptr, b.strides
    d.c, d.c_rs = c.ptr, c.strides[0]
    if c0 is not None:
        d.c0, d.c0_rs = c0.ptr, c0.strides[0]
    if bias is not None:
        d.bias = bias.ptr
    d.alpha, d.beta, d.act = alpha, beta, act
    return d


def prepare(case, seed):
    v = {name: _array(t) for name, t in _values(case, seed).items()}
    torch.cuda.synchronize()  # the copies above run on torch's stream
    state = {"case": case, "in": v}
    kind = case["kind"]
    if kind == "gemm":
        c = _empty((case["m"], case["n"]))
        state["calls"] = [_desc(v["a"].T if case["ta"] else v["a"], v["b"].T if case["tb"] else v["b"],
                                c, case["alpha"], v.get("c0"), case["beta"], v.get("bias"),
                                mf.ACT_GELU_TANH if case["gelu"] else mf.ACT_NONE)]
        outs = {"c": c}
    elif kind == "backward":
        dx, dw = _empty((case["rows"], case["cin"])), _empty((case["cin"], case["cout"]))
        state["calls"] = [_desc(v["dy"], v["w"].T, dx), _desc(v["x"].T, v["dy"], dw)]
        outs = {"dx": dx, "dw": dw}
    elif kind == "gemv":
        outs = {"y": _empty((case["cols"] if case["trans"] else case["rows"],))}
    elif kind == "attention":
        outs = {"out": _empty(v["q"].shape)}
    else:
        outs = {"p": _empty(v["x"].shape), "choice": _empty(v["x"].shape[:1], "int64")}
    state["out"] = outs
    state["tensors"] = {name: _tensor(a) for name, a in outs.items()}
    return state


def run(state):
    case, v, out = state["case"], state["in"], state["out"]
    kind = case["kind"]
    if kind in ("gemm", "backward"):
        for desc in state["calls"]:
            mf.sgemm(_STREAM, desc)
    elif kind == "gemv":
        mf.sgemv(v["a"], v["x"], alpha=case["alpha"], y0=v.get("y0"), beta=case["beta"],
                 trans=case["trans"], out=out["y"])
    elif kind == "attention":
        mf.attention_fused(v["q"], v["k"], v["v"], mask=v.get("mask"), causal=case["causal"],
                           out=out["out"])
    else:
        mf.softmax(v["x"], out=out["p"])
        mf.argmax(v["x"], out=out["choice"])
    return state["tensors"]


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * (m * k + k * n + (2 if case["beta"] else 1) * m * n
                              + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    if kind == "backward":
        r, i, o = case["rows"], case["cin"], case["cout"]
        return {"bytes": 4 * (r * o + i * o + r * i + r * i + i * o), "flops": 4 * r * i * o}
    if kind == "gemv":
        r, c = case["rows"], case["cols"]
        n_in, n_out = (r, c) if case["trans"] else (c, r)
        return {"bytes": 4 * (r * c + n_in + (2 if case["beta"] else 1) * n_out),
                "flops": 2 * r * c}
    if kind == "attention":
        heads = case["batch"] * case["heads"]
        lq, lk, d = case["lq"], case["lk"], case["d"]
        pairs = lq * (lq + 1) // 2 if case["causal"] else lq * lk
        return {"bytes": 4 * heads * d * (2 * lq + 2 * lk)
                + (case["batch"] * lk if case["mask"] else 0), "flops": 4 * heads * pairs * d}
    r, w = case["rows"], case["width"]
    return {"bytes": 8 * r * w + 8 * r, "flops": 5 * r * w}


def tolerance(case):
    # About four times the error against 64 bits at the ranges' ends: 32-bit products and sums
    # (1.1e-6 at a depth of 4096, 1.3e-6 over 4096 keys), gemv's 64-bit sums rounded once
    # (2.6e-8), softmax's 32-bit exponentials over a 64-bit sum (4.1e-8).
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1.5e-7}
    if kind == "head":
        return {"rel": 4e-7, "differ": 0.0}
    return {"rel": 5e-6}


def exact(case, seed):
    v = _values(case, seed)
    kind = case["kind"]
    if kind == "gemm":
        a = v["a"].double().T if case["ta"] else v["a"].double()
        b = v["b"].double().T if case["tb"] else v["b"].double()
        c = (a @ b) * case["alpha"]
        if case["beta"]:
            c += case["beta"] * v["c0"].double()
        if case["bias"]:
            c += v["bias"].double()
        if case["gelu"]:
            c = torch.nn.functional.gelu(c, approximate="tanh")
        return {"c": c}
    if kind == "backward":
        dy = v["dy"].double()
        return {"dx": dy @ v["w"].double().T, "dw": v["x"].double().T @ dy}
    if kind == "gemv":
        a = v["a"].double()
        y = ((a.T if case["trans"] else a) @ v["x"].double()) * case["alpha"]
        return {"y": y + case["beta"] * v["y0"].double() if case["beta"] else y}
    if kind == "attention":
        out = torch.empty(v["q"].shape, dtype=torch.float64, device="cuda")
        lq, lk = case["lq"], case["lk"]
        drop = torch.zeros((lq, lk), dtype=torch.bool, device="cuda")
        if case["causal"]:
            drop = torch.ones_like(drop).triu(1)
        for b in range(case["batch"]):
            gone = drop if v.get("mask") is None else drop | (v["mask"][b, 0] == 0)
            for h in range(case["heads"]):
                s = v["q"][b, h].double() @ v["k"][b, h].double().T.contiguous()
                s = (s / math.sqrt(case["d"])).masked_fill(gone, -math.inf)
                out[b, h] = torch.softmax(s, -1) @ v["v"][b, h].double()
        return {"out": out}
    return {"p": torch.softmax(v["x"].double(), -1), "choice": v["x"].argmax(-1)}
