"""The work that programs have this library do, as cases that can be timed and compared.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw()` more of the same ranges,
`prepare()` what a program holds before the call (operands in limb planes on the GPU, plans, host arrays),
`run()` one pass through the public entry points, `work()` the bytes and word products that a pass cannot
do without.  Every result is a correctly rounded integer record (limbs, exponent, sign, status), so
outputs are 32-bit whole numbers.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from limbforge_amd import capi

TERNARY = ("fma", "fms")
UNARY = ("square", "sqrt")


def listed():
    return [
        # the headline workload: a resident batch multiplied by its factors 16 times, rounded every time
        {"name": "chain_1024b_65536x16", "kind": "chain", "bits": 1024, "count": 65536, "steps": 16},
        # one small element-wise call: launch latency and call overhead
        {"name": "mul_256b_1000", "kind": "elementwise", "op": "mul", "bits": 256, "count": 1000, "period": 0},
        # a large ragged batch of fused multiply-adds with a short coefficient table (Horner steps, stencils)
        {"name": "fma_512b_1000003_p64", "kind": "elementwise", "op": "fma", "bits": 512, "count": 1000003, "period": 64},
        # division of a large batch at the widest precision
        {"name": "div_1024b_1048576", "kind": "elementwise", "op": "div", "bits": 1024, "count": 1048576, "period": 0},
        # composed complex division at the usual precision
        {"name": "complex_div_256b_262147", "kind": "elementwise", "op": "complex_div", "bits": 256, "count": 262147, "period": 0},
        # a program whose values live in host arrays: one call in, one out
        {"name": "host_div_256b_65536", "kind": "host", "op": "div", "bits": 256, "count": 65536},
        # values of 31 precisions with multiplication / fma chains of uneven length, as one graph
        {"name": "mixed_1000000", "kind": "mixed", "count": 1000000},
        # the exact dense product of entries in three exponent bands
        {"name": "gemm_512b_512x512x512", "kind": "gemm", "bits": 512, "m": 512, "n": 512, "k": 512, "transpose": False, "exponents": "bands"},
        # a small ragged exact product, as called between other steps of an iteration
        {"name": "gemm_256b_96x75x130", "kind": "gemm", "bits": 256, "m": 96, "n": 75, "k": 130, "transpose": False, "exponents": "single"},
        # the normal equations of a least-squares step: S = A^T A
        {"name": "syrk_256b_2048x512", "kind": "syrk", "bits": 256, "rows": 2048, "cols": 512, "exponents": "single"},
        # their factorization
        {"name": "cholesky_256b_512", "kind": "cholesky", "bits": 256, "n": 512, "block": 32},
        # and the forward and backward solves with 64 right-hand sides
        {"name": "solve_256b_512_64rhs", "kind": "solve", "bits": 256, "n": 512, "nrhs": 64, "block": 32},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["chain", "elementwise", "elementwise", "elementwise", "host", "mixed", "gemm", "gemm", "gemm", "syrk", "syrk",
                       "cholesky", "cholesky", "solve", "solve"])
    bits = 32 * rng.randint(2, 32)
    if kind == "chain":
        return {"kind": kind, "bits": bits, "count": _log_int(rng, 256, 131072), "steps": rng.randint(4, 64)}
    if kind == "elementwise":
        op = rng.choice(["add", "sub", "mul", "square", "div", "sqrt", "fma", "fms", "complex_add", "complex_mul", "complex_div"])
        return {"kind": kind, "op": op, "bits": bits, "count": _log_int(rng, 500, 1048576),
                "period": rng.choice([0, rng.randint(1, 500)]) if op in TERNARY else 0}
    if kind == "host":
        return {"kind": kind, "op": rng.choice(["add", "mul", "div", "sqrt", "complex_div"]), "bits": bits, "count": _log_int(rng, 500, 131072)}
    if kind == "mixed":
        return {"kind": kind, "count": _log_int(rng, 2000, 1000000)}
    if kind == "gemm":
        bits = 32 * rng.randint(2, 24)
        m, n, k = (_log_int(rng, 8, 700) for _ in range(3))
        while m * n * k * bits > 512 ** 4:
            m, n, k = (_log_int(rng, 8, 700) for _ in range(3))
        return {"kind": kind, "bits": bits, "m": m, "n": n, "k": k, "transpose": rng.random() < 0.5,
                "exponents": rng.choice(["single", "bands", "qsc"])}
    if kind == "syrk":
        bits = 32 * rng.randint(2, 16)
        rows, cols = _log_int(rng, 32, 2048), _log_int(rng, 16, 640)
        while rows * cols * cols * bits > 2048 * 512 * 512 * 256:
            rows, cols = _log_int(rng, 32, 2048), _log_int(rng, 16, 640)
        return {"kind": kind, "bits": bits, "rows": rows, "cols": cols, "exponents": rng.choice(["single", "qsc"])}
    # the factorization and the solves: a column's cost grows with the precision, so wide values come smaller
    bits = 32 * rng.randint(2, 16)
    n = _log_int(rng, 40, min(500, 500 * 256 // bits))
    if kind == "cholesky":
        return {"kind": kind, "bits": bits, "n": n, "block": rng.choice([16, 24, 32, 32, 32])}
    return {"kind": kind, "bits": bits, "n": n, "nrhs": _log_int(rng, 1, 64), "block": rng.choice([16, 24, 32, 32, 32])}


# ------------------------------------------------------------------ operands on the GPU
class Planes:
    """A resident operand over a torch tensor: (n + 3) planes of `pitch` 32-bit words, the imaginary planes
    after the real ones.  It stands where the binding takes a Buffer."""

    def __init__(self, bits, count, complex_values=False, words=None):
        self.bits, self.count, self.complex = bits, count, complex_values
        self.pitch = int(capi.lib().lf_plane_pitch(count))
        rows = capi.record_words(bits, complex_values)
        self.words = torch.zeros((rows, self.pitch), dtype=torch.int32, device="cuda")
        if words is not None:
            self.words[:, :count] = words

    @property
    def operand(self):
        return capi.Operand(self.words.data_ptr(), self.pitch)

    def values(self):
        return self.words[:, :self.count]


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, lo, hi, count):
    return torch.randint(lo, hi + 1, (count,), generator=g, device="cuda", dtype=torch.int64)


def _normal(g, sigma, count):
    return torch.round(sigma * torch.randn(count, generator=g, device="cuda", dtype=torch.float64)).to(torch.int64)


def _numbers(g, bits, exponents, positive=False):
    """Planes of random values: uniform limbs with the top bit set, the given exponents, random signs."""
    n, count = bits // 32, exponents.numel()
    w = torch.zeros((n + 3, count), dtype=torch.int32, device="cuda")
    w[:n] = torch.randint(-(1 << 31), 1 << 31, (n, count), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    w[n - 1] |= -(1 << 31)
    w[n] = exponents.to(torch.int32)
    w[n + 1] = 1 if positive else (2 * _uniform(g, 0, 1, count) - 1).to(torch.int32)
    return w


def _real(g, bits, exponents, positive=False):
    return Planes(bits, exponents.numel(), False, _numbers(g, bits, exponents, positive))


def _operand(g, bits, count, complex_values, positive, span):
    parts = [_numbers(g, bits, _uniform(g, -span, span, count), positive) for _ in range(2 if complex_values else 1)]
    return Planes(bits, count, complex_values, torch.cat(parts))


def _matrix(g, bits, rows, cols, exponents):
    """A row-major rows x cols matrix: one exponent band per line, three bands (centres -200, 0 and 200), or the
    columns of a Jacobian of scaled, partly sparse quantities with a rare tiny entry."""
    count = rows * cols
    if exponents == "single":
        return _real(g, bits, _normal(g, 8, count))
    if exponents == "bands":
        return _real(g, bits, 200 * _uniform(g, -1, 1, count) + _normal(g, 8, count))
    scale = _uniform(g, -60, 60, cols)
    e = _uniform(g, -15, 15, count).view(rows, cols) + scale[None, :] - 10
    odd = torch.arange(5, cols, 17, device="cuda")
    at = _uniform(g, 0, rows - 1, odd.numel())
    e[at, odd] = scale[odd] - 150
    w = _numbers(g, bits, e.reshape(-1))
    w[:, _uniform(g, 0, 3, count) == 0] = 0
    return Planes(bits, count, False, w)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _normal_equations(g, bits, n):
    """S = A^T A + I of a (4n x n) matrix."""
    A = _matrix(g, bits, 4 * n, n, "single")
    S = Planes(bits, n * n)
    capi.syrk_resident(bits, A, 4 * n, n, S, lower_only=False, stream=_stream())
    one = torch.zeros((bits // 32 + 3, n), dtype=torch.int32, device="cuda")
    one[bits // 32 - 1] = -(1 << 31)
    one[bits // 32 + 1] = 1
    at = torch.arange(n, device="cuda") * (n + 1)
    d, e, f = Planes(bits, n, False, S.words[:, at]), Planes(bits, n, False, one), Planes(bits, n)
    capi.elementwise(bits, "add", d, e, None, f, stream=_stream())
    S.words[:, at] = f.values()
    return S


def _factor_library():
    lib = capi.lib()
    P, op = C.POINTER, C.POINTER(capi.Operand)
    lib.lf_cholesky.argtypes = [C.c_int, op, C.c_uint64, op, P(capi.FactorOptions), P(capi.LinalgOptions), P(capi.CholeskyInfo), C.c_void_p]
    lib.lf_solve.argtypes = [C.c_int, C.c_int, op, C.c_uint64, op, C.c_uint64, op, P(capi.FactorOptions), P(capi.LinalgOptions),
                             P(C.c_double), P(C.c_double), C.c_void_p]
    return lib


def _cholesky(lib, bits, S, n, L, options):
    info = capi.CholeskyInfo()
    s, l = S.operand, L.operand
    capi.check(lib.lf_cholesky(bits, C.byref(s), n, C.byref(l), C.byref(options), None, C.byref(info), _stream()))
    return int(info.pivot)


class Bucket:
    """The values of one precision of a mixed batch."""

    def __init__(self, g, bits, length, mask):
        self.bits, self.count = bits, length.numel()
        self.x, self.f, self.g = (_real(g, bits, _uniform(g, -64, 64, self.count)) for _ in range(3))
        self.out, self.length, self.mask = Planes(bits, self.count), length, mask

    def struct(self):
        return capi.ChainBucket(self.bits, self.x.operand, self.f.operand, self.g.operand, self.out.operand, self.length.data_ptr(),
                                self.mask.data_ptr(), self.count)


class Graph:
    def __init__(self, buckets):
        self.buckets, self.handle = buckets, capi.mixed_graph(buckets)

    def __del__(self):
        if getattr(self, "handle", None):
            torch.cuda.synchronize()
            capi.graph_destroy(self.handle)


def _mixed_counts(case):
    """Values of each of the 31 precisions: P(64 + 32 k bits) ~ 0.85^k, every precision present."""
    p = 0.85 ** np.arange(31)
    return np.maximum(1, np.floor(case["count"] * p / p.sum())).astype(np.int64)


# ------------------------------------------------------------------ one case
def prepare(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind == "host":
        rng, op = np.random.default_rng(seed), case["op"]
        n, parts = case["bits"] // 32, 2 if op.startswith("complex") else 1

        def records():
            r = np.zeros((case["count"] * parts, n + 3), dtype=np.uint32)
            r[:, :n] = rng.integers(0, 1 << 32, size=(r.shape[0], n), dtype=np.uint32)
            r[:, n - 1] |= np.uint32(0x80000000)
            r[:, n] = rng.integers(-512, 513, size=r.shape[0]).astype(np.int32).view(np.uint32)
            r[:, n + 1] = (1 if op == "sqrt" else 2 * rng.integers(0, 2, size=r.shape[0]) - 1)
            return r.reshape(case["count"], parts * (n + 3))

        return {"case": case, "a": records(), "b": None if op in UNARY else records()}
    if kind == "mixed":
        buckets = []
        for k, count in enumerate(_mixed_counts(case)):
            length = torch.sort(_uniform(g, 1, 64, int(count)), descending=True).values.to(torch.int32)
            mask = torch.randint(-(1 << 62), 1 << 62, (int(count),), generator=g, device="cuda", dtype=torch.int64) * 2 + _uniform(g, 0, 1, int(count))
            buckets.append(Bucket(g, 64 + 32 * k, length, mask))
        return {"case": case, "graph": Graph(buckets)}
    bits = case["bits"]
    if kind == "chain":
        x, f = (_real(g, bits, _uniform(g, -64, 64, case["count"])) for _ in range(2))
        return {"case": case, "x": x, "f": f, "out": Planes(bits, case["count"])}
    if kind == "elementwise":
        op, count = case["op"], case["count"]
        cpx = op.startswith("complex")
        a = _operand(g, bits, count, cpx, op == "sqrt", 512)
        b = None if op in UNARY else _operand(g, bits, case["period"] or count, cpx, False, 512)
        c = _operand(g, bits, count, cpx, False, 512) if op in TERNARY else None
        return {"case": case, "a": a, "b": b, "c": c, "out": Planes(bits, count, cpx), "index": (1, case["period"]) if case["period"] else None}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        a = _matrix(g, bits, k, m, case["exponents"]) if case["transpose"] else _matrix(g, bits, m, k, case["exponents"])
        return {"case": case, "a": a, "b": _matrix(g, bits, k, n, case["exponents"]), "c": Planes(bits, m * n)}
    if kind == "syrk":
        return {"case": case, "a": _matrix(g, bits, case["rows"], case["cols"], case["exponents"]), "c": Planes(bits, case["cols"] ** 2)}
    lib, n = _factor_library(), case["n"]
    options = capi.FactorOptions.default(block=case["block"])
    S, L = _normal_equations(g, bits, n), Planes(bits, n * n)
    if kind == "cholesky":
        return {"case": case, "lib": lib, "options": options, "s": S, "l": L}
    _cholesky(lib, bits, S, n, L, options)
    b = _real(g, bits, _uniform(g, -10, 10, n * case["nrhs"]))
    return {"case": case, "lib": lib, "options": options, "l": L, "b": b, "x": Planes(bits, n * case["nrhs"])}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "host":
        out, _, _ = capi.run_host(case["bits"], case["op"], state["a"], state["b"])
        return out.view(np.int32)
    if kind == "mixed":
        graph = state["graph"]
        capi.graph_launch(graph.handle, _stream())
        return [b.out.values() for b in graph.buckets]
    bits = case["bits"]
    if kind == "chain":
        capi.mul_chain(bits, state["x"], state["f"], state["out"], case["steps"], stream=_stream())
        return state["out"].values()
    if kind == "elementwise":
        capi.elementwise(bits, case["op"], state["a"], state["b"], state["c"], state["out"], b_index=state["index"], stream=_stream())
        return state["out"].values()
    if kind == "gemm":
        capi.gemm_resident(bits, case["transpose"], state["a"], state["b"], case["m"], case["n"], case["k"], state["c"], stream=_stream())
        return state["c"].values()
    if kind == "syrk":
        capi.syrk_resident(bits, state["a"], case["rows"], case["cols"], state["c"], lower_only=True, stream=_stream())
        return state["c"].values()
    if kind == "cholesky":
        pivot = _cholesky(state["lib"], bits, state["s"], case["n"], state["l"], state["options"])
        return [state["l"].values(), pivot]
    l, b, x = state["l"].operand, state["b"].operand, state["x"].operand
    capi.check(state["lib"].lf_solve(bits, 3, C.byref(l), case["n"], C.byref(b), case["nrhs"], C.byref(x), C.byref(state["options"]), None,
                                     None, None, _stream()))
    return state["x"].values()


def exact(case, seed):
    """Outputs are whole numbers (limbs, exponents, signs, statuses), equal or not: no 64-bit reference applies."""
    return None


def work(case):
    """Each operand record read once and each result record written once; 32 x 32-bit word products of the
    exact operation, a multiplication and an addition each."""
    kind = case["kind"]
    if kind == "mixed":
        counts = _mixed_counts(case)
        n = np.arange(31) + 2
        return {"bytes": float((counts * (16.0 * (n + 3) + 12)).sum()), "flops": float((2.0 * 32.5 * counts * n * n).sum())}
    n = case["bits"] // 32
    record = 4.0 * (n + 3)
    if kind == "chain":
        return {"bytes": 3 * record * case["count"], "flops": 2.0 * n * n * case["steps"] * case["count"]}
    if kind in ("elementwise", "host"):
        op, count = case["op"], case["count"]
        per = {"add": 0, "sub": 0, "complex_add": 0, "mul": n * n, "square": n * n, "fma": n * n, "fms": n * n, "div": n * (n + 1), "sqrt": n * n,
               "complex_mul": 4 * n * n, "complex_div": 6 * n * n + 2 * n * (n + 1)}[op]
        reads = count if op in UNARY else count + (case.get("period") or count) + (count if op in TERNARY else 0)
        return {"bytes": record * (2 if op.startswith("complex") else 1) * (reads + count), "flops": 2.0 * (per or n) * count}
    if kind == "gemm":
        m, k, o = case["m"], case["k"], case["n"]
        return {"bytes": record * (m * k + k * o + m * o), "flops": 2.0 * n * n * m * k * o}
    if kind == "syrk":
        r, c = case["rows"], case["cols"]
        return {"bytes": record * (r * c + c * (c + 1) / 2), "flops": 1.0 * n * n * r * c * (c + 1)}
    size = case["n"]
    if kind == "cholesky":
        return {"bytes": record * 1.5 * size * size, "flops": 2.0 * n * n * size ** 3 / 6}
    return {"bytes": record * (size * (size + 1) / 2 + 2 * size * case["nrhs"]), "flops": 2.0 * n * n * size * size * case["nrhs"]}
