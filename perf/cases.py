"""Performance cases of the library: what its users run, over the sizes they run it at.

Each case goes through public entry points only: the Tensor API (`compute.Tensors`), or the C ABI
(include/csmi.h) on device memory that the caller owns, as a program that keeps compiled kernels
and buffers does. Imported with the repository's root as the working folder.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("compute.scala_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from compute import Tensors, workloads  # noqa: E402
from compute import _capi as capi  # noqa: E402

_VARIANTS = {"fp32": capi.GEMM_FP32, "bf16": capi.GEMM_BF16, "bf16x3": capi.GEMM_BF16X3, "fp8": capi.GEMM_FP8}
_back_end = None


def _tensors():
    """The process's back-end on GPU 0, as a program keeps one."""
    global _back_end
    if _back_end is None:
        _back_end = Tensors(0)
    return _back_end


def listed():
    return [
        # The smallest whole calls of the Tensor API: an expression with views and its sum, built
        # lazily, launched and read back. Latency, launches and host work are all of it.
        {"name": "api_small", "kind": "api", "b": 4, "h": 16, "w": 32},
        # The benchmark's view-heavy fused chain (permute, broadcast, translate, exp and tanh) with
        # its kernel compiled once, at the benchmark's size ...
        {"name": "chain", "kind": "chain", "b": 64, "h": 256, "w": 256},
        # ... and at sizes that divide by nothing, as data with a time or an image axis has.
        {"name": "chain_ragged", "kind": "chain", "b": 37, "h": 251, "w": 509},
        # The convolution of the reference's benchmark suite, one generated kernel.
        {"name": "conv", "kind": "conv", "batch": 128, "hw": 32, "depth": 8, "k": 3, "filters": 8},
        # Row sums, row maxima and the total of a large matrix in one pass (the benchmark's).
        {"name": "rows_wide", "kind": "rows", "rows": 16384, "cols": 4096},
        # The same statistics of many short records: a table with a few dozen columns.
        {"name": "rows_narrow", "kind": "rows", "rows": 120011, "cols": 77},
        # Column sums of such a table: one value per feature over all records.
        {"name": "cols", "kind": "cols", "rows": 20011, "cols": 1003},
        # matrixMultiply in FP32, the default data type, at the benchmark's size ...
        {"name": "gemm_fp32", "kind": "gemm", "variant": "fp32", "m": 4096, "n": 4096, "k": 4096},
        # ... and at the size of one layer over a small batch, where the chip is far from full.
        {"name": "gemm_small", "kind": "gemm", "variant": "fp32", "m": 300, "n": 200, "k": 1000},
        # matrixMultiply on rounded operands, for those who trade accuracy for speed.
        {"name": "gemm_bf16", "kind": "gemm", "variant": "bf16", "m": 4096, "n": 4096, "k": 4096},
        # One gradient of the cost model's network (forward and backward) at its training batch.
        {"name": "mlp", "kind": "mlp", "n": 512, "features": 23, "hidden": 64, "layers": 3},
        # Tensor.randomNormal of a large odd length: synthetic inputs and initial weights.
        {"name": "random_normal", "kind": "random", "n": 16777259, "normal": True},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], evenly spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["api", "chain", "chain", "conv", "rows", "rows", "cols", "gemm", "gemm", "gemm", "mlp", "random"])
    if kind == "api":
        return {"kind": kind, "b": rng.randint(1, 16), "h": _log(rng, 4, 64), "w": _log(rng, 4, 64)}
    if kind == "chain":
        total = _log(rng, 1 << 16, 1 << 22)
        w = _log(rng, 16, 2048)
        h = _log(rng, 1, max(1, min(1024, total // w)))
        return {"kind": kind, "b": max(1, total // (h * w)), "h": h, "w": w}
    if kind == "conv":
        return {"kind": kind, "batch": _log(rng, 4, 64), "hw": rng.randint(12, 48), "depth": rng.choice([1, 3, 4]),
                "k": rng.choice([1, 3]), "filters": rng.choice([2, 4, 6])}
    if kind == "rows" or kind == "cols":
        cols = _log(rng, 8, 16384)
        rows = max(1, min(1 << 19, _log(rng, 1 << 14, 1 << 24) // cols))
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "gemm":
        variant = rng.choice(["fp32", "fp32", "bf16", "bf16x3", "fp8"])
        return {"kind": kind, "variant": variant, "m": _log(rng, 16, 4096), "n": _log(rng, 16, 4096),
                "k": _log(rng, 16, 4096)}
    if kind == "mlp":
        return {"kind": kind, "n": _log(rng, 32, 512), "features": rng.randint(3, 32), "hidden": _log(rng, 16, 128),
                "layers": rng.randint(1, 3)}
    return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 23), "normal": rng.random() < 0.7}


# --------------------------------------------------------------------------------- inputs
def _seeded(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _uniform(g, *shape):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * 2 - 1


def _heavy_tailed(g, rows, cols):
    """N(0, 1) with one entry in a hundred 10^4 times as large, as the reduction benchmark has."""
    x = _normal(g, rows, cols)
    x[torch.rand(x.shape, generator=g, device="cuda") < 0.01] *= 1e4
    return x


def _chain_inputs(case, seed):
    g = _seeded(seed)
    return _normal(g, case["b"], case["h"], case["w"]), _uniform(g, case["h"]) / 2


def _conv_inputs(case, seed):
    g = _seeded(seed)
    k, d, f = case["k"], case["depth"], case["filters"]
    return (_uniform(g, case["batch"], case["hw"], case["hw"], d), _uniform(g, k, k, d, f), _uniform(g, f))


def _gemm_inputs(case, seed):
    g = _seeded(seed)
    return _uniform(g, case["m"], case["k"]), _uniform(g, case["k"], case["n"])


def _mlp_widths(case):
    return [case["features"]] + [case["hidden"]] * case["layers"] + [1]


def _mlp_inputs(case, seed):
    """Standardised features, targets and He-uniform parameters in the library's flat layout."""
    g = _seeded(seed)
    widths = _mlp_widths(case)
    x, t = _normal(g, case["n"], widths[0]), _normal(g, case["n"])
    parts = []
    for din, dout in zip(widths[:-1], widths[1:]):
        parts += [(_uniform(g, din, dout) * math.sqrt(6.0 / din)).reshape(-1), _uniform(g, dout) * 0.1]
    return x, t, torch.cat(parts)


# --------------------------------------------------------------------------------- states
class _State(object):
    pass


def _chain(T, x, b):
    p = x.permute([1, 0, 2])
    y = p + b.broadcast(p.shape) + p.translate([0, 0, 1])
    return T.Tensor.exp(-(y * y)) * T.Tensor.tanh(y)


def _compiled(T, closure, shape, data):
    """The kernel of `closure` and its leaf pointers. `data`: (leaf tensor, device tensor) pairs."""
    handle, leaves, _ = T.compile(closure, shape)
    by_id = {id(t): d.data_ptr() for t, d in data}
    return handle, (ctypes.c_void_p * len(leaves))(*[by_id[id(leaf.id)] for leaf in leaves])


class _Network(object):
    """A cs_mlp handle that goes with its state."""

    def __init__(self, T, widths, params):
        h = ctypes.c_void_p()
        capi.check(capi.lib.cs_mlp_create(T.device, (ctypes.c_int32 * len(widths))(*widths), len(widths), 1,
                                          ctypes.byref(h)))
        self.handle = h.value
        host = np.ascontiguousarray(params.cpu().numpy())
        capi.check(capi.lib.cs_mlp_set_params(T.stream, self.handle, host.ctypes.data_as(ctypes.c_void_p), host.size))

    def __del__(self):
        capi.lib.cs_mlp_release(self.handle)


def prepare(case, seed):
    T = _tensors()
    s = _State()
    s.kind, s.T, s.case = case["kind"], T, case
    new = lambda *shape: torch.empty(shape, device="cuda", dtype=torch.float32)  # noqa: E731
    if s.kind == "api":
        x, b = _chain_inputs(case, seed)
        s.x, s.b = (T.Tensor(v.cpu().numpy()).doCache() for v in (x, b))
    elif s.kind == "chain":
        s.x, s.b = _chain_inputs(case, seed)
        X, B = T.Tensor.fill(0.0, s.x.shape).nonInline, T.Tensor.fill(0.0, s.b.shape).nonInline
        e = _chain(T, X, B)
        s.out = new(*e.shape)
        s.fused, s.leaves = _compiled(T, e.closure, e.shape, [(X, s.x), (B, s.b)])
    elif s.kind == "conv":
        s.x, s.w, s.b = _conv_inputs(case, seed)
        leaves = [T.Tensor.fill(0.0, v.shape).nonInline for v in (s.x, s.w, s.b)]
        e = workloads.convolute(T, *leaves)
        (closure,), _ = e.closures()
        s.out = new(*e.shape)
        s.fused, s.leaves = _compiled(T, closure, e.shape[:-1], list(zip(leaves, (s.x, s.w, s.b))))
    elif s.kind == "rows":
        s.x = _heavy_tailed(_seeded(seed), case["rows"], case["cols"])
        s.sum, s.max, s.total = new(case["rows"]), new(case["rows"]), new(1)
        s.total64 = torch.empty(1, device="cuda", dtype=torch.float64)
    elif s.kind == "cols":
        s.x = _heavy_tailed(_seeded(seed), case["rows"], case["cols"])
        s.out = new(case["cols"])
    elif s.kind == "gemm":
        s.a, s.b = _gemm_inputs(case, seed)
        s.out = new(case["m"], case["n"])
        s.variant = _VARIANTS[case["variant"]]
    elif s.kind == "mlp":
        s.x, s.t, params = _mlp_inputs(case, seed)
        s.net = _Network(T, _mlp_widths(case), params)
        s.loss, s.grads = new(1), new(params.numel())
    else:
        s.n, s.seed = case["n"], int(seed) * 2654435761 % (1 << 32)
        s.out = new(s.n + (s.n & 1 if case["normal"] else 0))
    torch.cuda.synchronize()  # the library's stream is another than torch's
    return s


def run(s):
    T, lib, st, c = s.T, capi.lib, s.T.stream, s.case
    if s.kind == "api":
        e = _chain(T, s.x, s.b)
        return e.flatArray(), (e * e).sum().flatArray()
    if s.kind in ("chain", "conv"):
        capi.check(lib.cs_fused_launch(st, s.fused, s.leaves, len(s.leaves), s.out.data_ptr()))
        return s.out
    if s.kind == "rows":
        capi.check(lib.cs_reduce_rows(st, s.x.data_ptr(), c["rows"], c["cols"], s.sum.data_ptr(), s.max.data_ptr(),
                                      s.total.data_ptr(), s.total64.data_ptr()))
        return s.sum, s.max, s.total, s.total64
    if s.kind == "cols":
        capi.check(lib.cs_reduce_cols(st, s.x.data_ptr(), c["rows"], c["cols"], s.out.data_ptr()))
        return s.out
    if s.kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        capi.check(lib.cs_gemm(st, s.variant, m, n, k, s.a.data_ptr(), k, s.b.data_ptr(), n, s.out.data_ptr(), n))
        return s.out
    if s.kind == "mlp":
        capi.check(lib.cs_mlp_backward(st, s.net.handle, s.x.data_ptr(), s.t.data_ptr(), c["n"], s.loss.data_ptr(),
                                       s.grads.data_ptr()))
        return s.loss, s.grads
    if c["normal"]:
        capi.check(lib.cs_random_normal(st, s.out.data_ptr(), s.n, s.seed))
    else:
        capi.check(lib.cs_random(st, s.out.data_ptr(), s.n, s.seed))
    return s.out


def work(case):
    kind, c = case["kind"], case
    if kind in ("api", "chain"):
        n = c["b"] * c["h"] * c["w"]
        return {"bytes": 4 * (2 * n + c["h"]), "flops": 7 * n}
    if kind == "conv":
        px = c["batch"] * c["hw"] ** 2
        taps = c["k"] ** 2 * c["depth"]
        return {"bytes": 4 * (px * (c["depth"] + c["filters"]) + (taps + 1) * c["filters"]),
                "flops": 2 * px * taps * c["filters"]}
    if kind == "rows":
        return {"bytes": 4 * c["rows"] * (c["cols"] + 2) + 12, "flops": 2 * c["rows"] * c["cols"]}
    if kind == "cols":
        return {"bytes": 4 * (c["rows"] + 1) * c["cols"], "flops": c["rows"] * c["cols"]}
    if kind == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": 4 * (m * k + k * n + m * n), "flops": 2 * m * n * k}
    if kind == "mlp":
        w = _mlp_widths(c)
        weights = sum(i * o for i, o in zip(w[:-1], w[1:]))
        return {"bytes": 4 * (c["n"] * (w[0] + 1) + 2 * (weights + sum(w[1:])) + 1),
                "flops": c["n"] * (6 * weights - 2 * w[0] * w[1])}
    return {"bytes": 4 * (c["n"] + (c["n"] & 1 if c["normal"] else 0)), "flops": 8 * c["n"]}


# --------------------------------------------------------------------------------- 64-bit values
def _chain_exact(x, b):
    p = x.double().permute(1, 0, 2)
    y = p + b.double()[:, None, None] + torch.nn.functional.pad(p, (1, 0))[:, :, :-1]
    return torch.exp(-(y * y)) * torch.tanh(y)


def _wang(i, seed):
    with np.errstate(over="ignore"):
        v = i ^ np.uint32(seed)
        v = (v ^ np.uint32(61)) ^ (v >> np.uint32(16))
        v = v * np.uint32(9)
        v = v ^ (v << np.uint32(4))
        v = v * np.uint32(0x27D4EB2D)
        return v ^ (v >> np.uint32(15))


def _random_exact(case, seed):
    n, seed = case["n"], int(seed) * 2654435761 % (1 << 32)
    if not case["normal"]:
        return torch.from_numpy((_wang(np.arange(n, dtype=np.uint32), seed).astype(np.float32) / np.float32(2.0 ** 32))
                                .astype(np.float64))
    h = _wang(np.arange((n + 1) // 2, dtype=np.uint32), seed)
    t = h ^ (h << np.uint32(13))
    t = t ^ (t >> np.uint32(17))
    t = t ^ (t << np.uint32(5))
    # the two uniform draws are single-precision numbers by definition
    u1, u2 = ((v.astype(np.float32) / np.float32(2.0 ** 32)).astype(np.float64) for v in (h, t))
    with np.errstate(divide="ignore", invalid="ignore"):
        r = np.sqrt(-2.0 * np.log(u1))
        out = np.stack([r * np.cos(2 * np.pi * u2), r * np.sin(2 * np.pi * u2)], axis=1)
    return torch.from_numpy(out.reshape(-1))


def _mlp_exact(case, seed):
    x, t, params = _mlp_inputs(case, seed)
    widths = _mlp_widths(case)
    p = params.double().requires_grad_(True)
    y, at = x.double(), 0
    for layer, (din, dout) in enumerate(zip(widths[:-1], widths[1:])):
        w = p[at:at + din * dout].reshape(din, dout)
        y = y @ w + p[at + din * dout:at + (din + 1) * dout]
        at += (din + 1) * dout
        if layer < len(widths) - 2:
            y = torch.relu(y)
    loss = ((y[:, 0] - t.double()) ** 2).mean()
    loss.backward()
    return loss.detach().reshape(1), p.grad


def exact(case, seed):
    kind = case["kind"]
    if kind == "api":
        e = _chain_exact(*_chain_inputs(case, seed))
        return e.reshape(-1).cpu().numpy(), (e * e).sum().reshape(1).cpu().numpy()
    if kind == "chain":
        return _chain_exact(*_chain_inputs(case, seed))
    if kind == "conv":
        x, w, b = (v.double() for v in _conv_inputs(case, seed))
        k, d, f, hw = case["k"], case["depth"], case["filters"], case["hw"]
        # out[y, x] takes input[y - dy, x - dx] for dy, dx of [-(k // 2), k - k // 2)
        pad = torch.nn.functional.pad(x, (0, 0, k, k, k, k))
        out = b.expand(*x.shape[:3], f).clone()
        for i in range(k):
            for j in range(k):
                y0, x0 = k - (i - k // 2), k - (j - k // 2)
                out += (pad[:, y0:y0 + hw, x0:x0 + hw].reshape(-1, d) @ w[i, j]).reshape(out.shape)
        return out
    if kind == "rows":
        x = _heavy_tailed(_seeded(seed), case["rows"], case["cols"]).double()
        total = x.sum().reshape(1)
        return x.sum(1), x.amax(1), total, total
    if kind == "cols":
        return _heavy_tailed(_seeded(seed), case["rows"], case["cols"]).double().sum(0)
    if kind == "gemm":
        a, b = _gemm_inputs(case, seed)
        return a.double() @ b.double()
    if kind == "mlp":
        return _mlp_exact(case, seed)
    return _random_exact(case, seed)

