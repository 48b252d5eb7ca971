"""What this library's callers ask of it, as cases that can be timed and checked.

Every case goes through the C ABI (include/linalg_hip.h) with its descriptors built once, the
way a compiled caller holds them, on buffers from lg_alloc and on the context's own stream.
Operands come from torch's generator on the GPU; outputs are zero-copy torch views of the
library's buffers.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "pipeline-parallelism-deep-learning-library_amd"))

import linalg_hip as L  # noqa: E402
from linalg_hip import backend as B  # noqa: E402
from linalg_hip import permutation as P  # noqa: E402

F = ctypes.c_float
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "u32": torch.int32}

_context = None


def context():
    """The one context that a program keeps for its GPU."""
    global _context
    if _context is None:
        _context = L.Context.new(0)
    return _context


# ------------------------------------------------------------------------------ the cases


def listed():
    return [
        # The smallest product of the reference's own list: launch and latency.
        {"name": "gemm-512", "kind": "gemm", "m": 512, "n": 512, "k": 512, "ta": False, "tb": False, "alpha": 1.0, "beta": 0.0},
        # The headline: a large square row-major product.
        {"name": "gemm-4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "ta": False, "tb": False, "alpha": 1.0, "beta": 0.0},
        # No extent a multiple of four, so no row is 16-byte aligned; accumulates into C.
        {"name": "gemm-odd", "kind": "gemm", "m": 3001, "n": 2011, "k": 1537, "ta": False, "tb": True, "alpha": 0.5, "beta": 1.0},
        # bik,bjk->bij: a batch of products whose B is a permuted view, read in place.
        {"name": "contract-batched", "kind": "batched", "batch": 32, "m": 1024, "n": 1024, "k": 1024, "tb": True},
        # Many small products at once (the reference's own batch of 32x32s).
        {"name": "contract-small", "kind": "batched", "batch": 4096, "m": 32, "n": 32, "k": 32, "tb": False},
        # A long contraction with a short output (split along K).
        {"name": "gemm-long-k", "kind": "gemm", "m": 256, "n": 256, "k": 65536, "ta": False, "tb": False, "alpha": 1.0, "beta": 0.0},
        # ijkl,klmn->ijmn: a rank-4 contraction over two axes.
        {"name": "contract-rank4", "kind": "rank4", "e": 48},
        # One linear layer of a pipeline stage, forward and backward, in f32: X.W, bias, GELU,
        # then GELU', db, dX and dW.
        {"name": "layer-step", "kind": "layer", "rows": 2048, "d_in": 2048, "d_out": 8192},
        # A 16-bit layer product on the backend surface (the CPU backend's bits).
        {"name": "gemm16-bf16", "kind": "gemm16", "dtype": "bf16", "m": 2048, "n": 4096, "k": 1024, "layout": "nn"},
        # The f16 contraction: every output is the exact sum rounded once.
        {"name": "gemm-f16", "kind": "gemmf16", "m": 2048, "n": 2048, "k": 2048, "ta": False, "tb": False},
        # A large rank-3 axis permutation (512 MiB read, 512 MiB written).
        {"name": "permute-3d", "kind": "permute", "shape": "512,1024,256", "perm": "2,0,1"},
        # A transpose whose rows are odd, so no row is 16-byte aligned.
        {"name": "permute-odd", "kind": "permute", "shape": "8191,4099", "perm": "1,0"},
    ]


def _spread(rng, lo, hi, step=1):
    """A size from lo to hi, even over its logarithm, in multiples of `step`."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, max(step, v // step * step)))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "batched", "longk", "rank4", "layer", "layer", "gemm16", "gemmf16", "permute", "permute"])
    # Half of the sizes are whole multiples of 64, as layers have them, half are anything.
    step = rng.choice([1, 64])
    if kind == "gemm":
        alpha, beta = rng.choice([(1.0, 0.0), (1.0, 1.0), (0.5, 1.0), (0.3, 0.0)])
        return {"kind": "gemm", "m": _spread(rng, 64, 5000, step), "n": _spread(rng, 64, 5000, step),
                "k": _spread(rng, 64, 5000, step), "ta": rng.random() < 0.3, "tb": rng.random() < 0.5,
                "alpha": alpha, "beta": beta}
    if kind == "batched":
        e = [_spread(rng, 16, 1024, 16 if step == 64 else 1) for _ in range(3)]
        b = _spread(rng, 2, max(3, min(4096, int(6e10 / (2 * e[0] * e[1] * e[2])), int(1e8 / max(e[0] * e[2], e[1] * e[2], e[0] * e[1])))))
        return {"kind": "batched", "batch": b, "m": e[0], "n": e[1], "k": e[2], "tb": rng.random() < 0.5}
    if kind == "longk":
        return {"kind": "gemm", "m": _spread(rng, 32, 512, 32 if step == 64 else 1), "n": _spread(rng, 32, 512, 32 if step == 64 else 1),
                "k": _spread(rng, 16384, 131072, step), "ta": False, "tb": rng.random() < 0.5, "alpha": 1.0, "beta": 0.0}
    if kind == "rank4":
        return {"kind": "rank4", "e": rng.randint(12, 56)}
    if kind == "layer":
        return {"kind": "layer", "rows": _spread(rng, 64, 4096, step), "d_in": _spread(rng, 64, 4096, step),
                "d_out": _spread(rng, 64, 4096, step)}
    if kind == "gemm16":
        return {"kind": "gemm16", "dtype": rng.choice(["bf16", "f16"]), "m": _spread(rng, 128, 2560, step),
                "n": _spread(rng, 128, 2560, step), "k": _spread(rng, 128, 2560, step), "layout": rng.choice(["nn", "nt", "tn"])}
    if kind == "gemmf16":
        return {"kind": "gemmf16", "m": _spread(rng, 128, 2560, step), "n": _spread(rng, 128, 2560, step),
                "k": _spread(rng, 128, 2560, step), "ta": rng.random() < 0.3, "tb": rng.random() < 0.5}
    rank = rng.choice([2, 3, 4])
    perm = list(range(rank))
    while perm == list(range(rank)):
        rng.shuffle(perm)
    total = math.exp(rng.uniform(math.log(1 << 18), math.log(1 << 27)))
    cuts = [rng.uniform(0.6, 1.4) for _ in range(rank)]
    shape = [max(2, int(total ** (c / sum(cuts)))) for c in cuts]
    if step == 64:
        shape = [max(4, s // 4 * 4) for s in shape]
    return {"kind": "permute", "shape": ",".join(map(str, shape)), "perm": ",".join(map(str, perm))}


# ------------------------------------------------------------------- buffers and descriptors


class Held:
    """A library buffer and a torch view of it; the buffer goes with the last reference."""

    def __init__(self, dtype, count):
        self.buffer = L.alloc_shared(context(), "u32", (count * TORCH[dtype].itemsize + 3) // 4)
        nbytes = count * TORCH[dtype].itemsize
        self.__cuda_array_interface__ = {"shape": (nbytes,), "typestr": "|u1", "data": (self.buffer.base, False), "version": 2}
        self.dtype = dtype

    def tensor(self, shape):
        return torch.as_tensor(self, device="cuda").view(TORCH[self.dtype]).view(*shape)

    def __del__(self):
        try:
            self.buffer.free()
        except Exception:  # the interpreter's own end
            pass


class Made:
    """Draws a case's operands in order, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, scale=1.0, dtype="f32"):
        return (torch.randn(shape, device="cuda", generator=self.g) * scale).to(TORCH[dtype])

    def words(self, shape):
        return torch.randint(-(2 ** 31), 2 ** 31, shape, device="cuda", generator=self.g, dtype=torch.int32)


def held(x):
    h = Held({v: k for k, v in TORCH.items()}[x.dtype], x.numel())
    t = h.tensor(x.shape)
    t.copy_(x)
    return h, t


def empty(dtype, shape):
    h = Held(dtype, math.prod(shape))
    return h, h.tensor(shape)


def view(h, shape, strides=None):
    dtype = "f32" if h.dtype == "u32" else h.dtype
    v = L.TensorView.row_major(h.buffer, 0, list(shape), dtype)
    return v if strides is None else L.TensorView(h.buffer, 0, list(shape), list(strides), dtype)


def tensor(h, shape, transposed=False):
    """A row-major backend tensor over `h`, or the transposed view of one (`shape` is then the stored one)."""
    dt = {"f32": B.DType.F32, "f16": B.DType.F16, "bf16": B.DType.BF16}[h.dtype]
    t = B.Tensor(B.Storage(h.buffer.base, h.buffer.nbytes, h.buffer), dt, list(shape), B.row_major_strides(shape))
    return (B.transpose_matrix(t) if transposed else t).to_c()


def call(name, *args):
    """One entry point with its arguments, ready to be called."""
    fn = getattr(L.lib(), name)
    refs = [ctypes.byref(a) if isinstance(a, ctypes.Structure) else a for a in args]

    def go():
        if fn(*refs) != 0:
            raise RuntimeError("%s: %s" % (name, L.lib().lg_last_error().decode()))
    go.keep = args
    return go


def on_stream(name, *args):
    ctx = context()
    return call(name, ctx.handle, ctx.queue.handle, *args)


# ------------------------------------------------------------------------------- operands


def _operands(case, seed):
    """The case's operands as torch tensors, in the order in which they are stored."""
    r, kind = Made(seed), case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s = 1.0 / math.sqrt(k)
        out = [r.normal((k, m) if case["ta"] else (m, k)), r.normal((n, k) if case["tb"] else (k, n), s)]
        return out + ([r.normal((m, n))] if case["beta"] else [])
    if kind == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return [r.normal((b, m, k)), r.normal((b, n, k) if case["tb"] else (b, k, n), 1.0 / math.sqrt(k))]
    if kind == "rank4":
        e = case["e"]
        return [r.normal((e, e, e, e)), r.normal((e, e, e, e), 1.0 / e)]
    if kind == "layer":
        m, k, n = case["rows"], case["d_in"], case["d_out"]
        return [r.normal((m, k)), r.normal((k, n), 1.0 / math.sqrt(k)), r.normal((n,), 0.1), r.normal((m, n), 1.0 / m)]
    if kind == "gemm16":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        return [r.normal((k, m) if case["layout"] == "tn" else (m, k), 1.0, dt),
                r.normal((n, k) if case["layout"] == "nt" else (k, n), 1.0 / math.sqrt(k), dt)]
    if kind == "gemmf16":
        m, n, k = case["m"], case["n"], case["k"]
        return [r.normal((k, m) if case["ta"] else (m, k), 1.0, "f16"),
                r.normal((n, k) if case["tb"] else (k, n), 1.0 / math.sqrt(k), "f16")]
    return [r.words(_ints(case["shape"]))]


def _ints(s):
    return [int(x) for x in s.split(",")]


def prepare(case, seed):
    kind = case["kind"]
    ops = [held(x) for x in _operands(case, seed)]
    keep = [h for h, _ in ops]
    if kind in ("gemm", "gemmf16"):
        m, n, k = case["m"], case["n"], case["k"]
        dt = "f32" if kind == "gemm" else "f16"
        a = view(keep[0], (m, k), (1, m) if case["ta"] else None)
        b = view(keep[1], (k, n), (1, k) if case["tb"] else None)
        alpha, beta = case.get("alpha", 1.0), case.get("beta", 0.0)
        h, out = ops[2] if beta else empty(dt, (m, n))
        calls = [on_stream("lg_encode_gemm_" + dt, F(alpha), a.to_c(), b.to_c(), F(beta), view(h, (m, n)).to_c())]
        outs = {"c": out}
    elif kind == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        h, out = empty("f32", (b, m, n))
        bv = view(keep[1], (b, n, k) if case["tb"] else (b, k, n))
        calls = [on_stream("lg_encode_contract_f32", F(1.0), view(keep[0], (b, m, k)).to_c(), b"bik", bv.to_c(),
                           b"bjk" if case["tb"] else b"bkj", F(0.0), view(h, (b, m, n)).to_c(), b"bij")]
        outs = {"c": out}
    elif kind == "rank4":
        e = (case["e"],) * 4
        h, out = empty("f32", e)
        calls = [on_stream("lg_encode_contract_f32", F(1.0), view(keep[0], e).to_c(), b"ijkl", view(keep[1], e).to_c(), b"klmn",
                           F(0.0), view(h, e).to_c(), b"ijmn")]
        outs = {"c": out}
    elif kind == "layer":
        m, k, n = case["rows"], case["d_in"], case["d_out"]
        x, w, bias, dy = keep
        (hpre, pre), (hy, y), (hg, g) = (empty("f32", (m, n)) for _ in range(3))
        (hdx, dx), (hdw, dw), (hdb, db) = empty("f32", (m, k)), empty("f32", (k, n)), empty("f32", (n,))
        keep += [hpre, hy, hg, hdx, hdw, hdb]
        h = hdb
        X, W, T = tensor(x, (m, k)), tensor(w, (k, n)), lambda q: tensor(q, (m, n))
        calls = [
            on_stream("lg_backend_gemm", X, W, T(hpre), F(1.0), F(0.0)),
            on_stream("lg_backend_add_bias", T(hpre), tensor(bias, (n,)), T(hpre)),
            on_stream("lg_backend_gelu", T(hpre), T(hy)),
            on_stream("lg_backend_gelu_backward", T(hpre), T(dy), T(hg)),
            on_stream("lg_backend_bias_grad", T(hg), tensor(hdb, (n,))),
            on_stream("lg_backend_gemm", T(hg), tensor(w, (k, n), True), tensor(hdx, (m, k)), F(1.0), F(0.0)),
            on_stream("lg_backend_gemm", tensor(x, (m, k), True), T(hg), tensor(hdw, (k, n)), F(1.0), F(0.0)),
        ]
        outs = {"y": y, "dx": dx, "db": db, "dw": dw}
    elif kind == "gemm16":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        h, out = empty(dt, (m, n))
        a = tensor(keep[0], (k, m), True) if case["layout"] == "tn" else tensor(keep[0], (m, k))
        b = tensor(keep[1], (n, k), True) if case["layout"] == "nt" else tensor(keep[1], (k, n))
        calls = [on_stream("lg_backend_gemm", a, b, tensor(h, (m, n)), F(1.0), F(0.0))]
        outs = {"c": out}
    else:
        shape, perm = _ints(case["shape"]), _ints(case["perm"])
        src = P.permute_view(view(keep[0], shape), perm)
        h, out = empty("u32", src.shape)
        calls = [on_stream("lg_encode_materialize", src.elem, src.to_c(), view(h, src.shape).to_c())]
        outs = {"y": out}
    keep.append(h)
    return {"calls": calls, "outs": outs, "keep": keep}


def run(state):
    for go in state["calls"]:
        go()
    return state["outs"]


# ------------------------------------------------------------------- work, tolerance, exact


def work(case):
    kind = case["kind"]
    if kind == "layer":
        m, k, n = case["rows"], case["d_in"], case["d_out"]
        # x, w, bias, dy read once; y, dx, db, dw written once.
        return {"bytes": 4 * (m * k + k * n + n + m * n + m * n + m * k + n + k * n), "flops": 6 * m * n * k}
    if kind == "permute":
        return {"bytes": 8 * math.prod(_ints(case["shape"])), "flops": 0}
    if kind == "rank4":
        e2 = case["e"] ** 2
        return {"bytes": 12 * e2 * e2, "flops": 2 * e2 ** 3}
    b, m, n, k = case.get("batch", 1), case["m"], case["n"], case["k"]
    size = 4 if kind in ("gemm", "batched") else 2
    c = 2 if case.get("beta") else 1
    return {"bytes": size * b * (m * k + k * n + c * m * n), "flops": 2 * b * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "permute" or kind == "gemm16":
        # Bits: words are moved, and the 16-bit backend product is the CPU backend's own f32 chain.
        return "exact"
    if kind == "gemmf16":
        # Correctly rounded outputs: two f64 sums of one dot product rarely round apart, and
        # then by one f16 step.
        return {"rel": 2e-5, "max": 4e-3}
    # f32 sums of K products in any order. One chain over K is measured to be 1.8e-8 * sqrt(K)
    # off the 64-bit sum (1.1e-6 at K = 4096), so two orders differ by about 3e-8 * sqrt(K); four
    # times that, from 1e-6 for the shortest to the 1e-5 of a chain over the longest.
    k = {"rank4": lambda: case["e"] ** 2, "layer": lambda: max(case["rows"], case["d_in"], case["d_out"])}.get(kind, lambda: case.get("k"))()
    return {"rel": min(1e-5, max(1e-6, 1.2e-7 * math.sqrt(k)))}


def exact(case, seed):
    kind = case["kind"]
    ops = [x.double() if x.is_floating_point() else x for x in _operands(case, seed)]
    if kind in ("gemm", "gemmf16"):
        a = ops[0].t() if case["ta"] else ops[0]
        b = ops[1].t() if case["tb"] else ops[1]
        alpha, beta = (float(torch.tensor(case.get(s, d), dtype=torch.float32)) for s, d in (("alpha", 1.0), ("beta", 0.0)))
        c = alpha * (a @ b)
        return {"c": c + beta * ops[2] if beta else c}
    if kind == "batched":
        b = ops[1].transpose(1, 2).contiguous() if case["tb"] else ops[1]
        return {"c": torch.stack([x @ y for x, y in zip(ops[0], b)])}
    if kind == "rank4":
        e = case["e"]
        return {"c": (ops[0].reshape(e * e, e * e) @ ops[1].reshape(e * e, e * e)).reshape(e, e, e, e)}
    if kind == "layer":
        x, w, bias, dy = ops
        pre = x @ w + bias
        phi = 0.5 * (1.0 + torch.erf(pre / math.sqrt(2.0)))
        g = dy * (phi + pre * torch.exp(-0.5 * pre * pre) / math.sqrt(2.0 * math.pi))
        return {"y": pre * phi, "dx": g @ w.t(), "db": g.sum(0), "dw": x.t() @ g}
    if kind == "gemm16":
        a = ops[0].t() if case["layout"] == "tn" else ops[0]
        b = ops[1].t() if case["layout"] == "nt" else ops[1]
        return {"c": a @ b}
    return {"y": ops[0].permute(_ints(case["perm"])).contiguous()}
