"""The calls this library is used for, as cases that can be timed.

Every case is one call (or one training step) through the Python entry points
of jblas_amd on device-resident operands, which land on the same C entry
points that Julia `ccall`s.  The sizes are those of the repository's own
configurations, tests and benchmark, plus generic ragged ones.

kind      what a program does
fastmul   one small product D = A*X, the whole-matrix microkernel
jmul      D = A*X with the reference recurrence, Float64 or Float32
dgemm     C = alpha*op(A)*op(B) + beta*C on the FP64 matrix cores
emulated  the same through split-BF16 or split-INT8 slices
autograd  Y = A @ B and both gradients through the torch binding
grouped   many uneven products replayed from a plan
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.abspath("jblas.jl_amd"))
import jblas_amd as jb  # noqa: E402
from jblas_amd.grouped import GemmDesc, GroupedPlan  # noqa: E402
from jblas_amd.rrule import matmul  # noqa: E402

DTYPES = {"f64": torch.float64, "f32": torch.float32}
PRODUCTS = {"f32": 1, "f64": 1, "f32_bf16x3": 6}  # slice products per product of the method


def listed():
    return [
        # the reference's own benchmark, C(16x14) = A(16x32) B(32x14): one call's latency
        dict(name="fastmul_16x32x14_f64", kind="fastmul", dtype="f64", m=16, n=14, k=32),
        # the bit-parity configuration, 256^3 Float64: a small call that still needs many workgroups
        dict(name="jmul_256_f64", kind="jmul", dtype="f64", m=256, n=256, k=256),
        # Float32 jmul! at the largest shape the reference's test script exercises
        dict(name="jmul_800x900x840_f32", kind="jmul", dtype="f32", m=800, n=840, k=900),
        # native FP64 gemm! with alpha and beta, the smallest square of that configuration, one operand transposed
        dict(name="dgemm_1024_tn", kind="dgemm", ta="T", tb="N", m=1024, n=1024, k=1024, pad=0, alpha=1.5, beta=0.5),
        # a ragged product on views of larger matrices: no extent or leading dimension fits a tile or a vector
        dict(name="dgemm_ragged_nt", kind="dgemm", ta="N", tb="T", m=2999, n=1777, k=2111, pad=4, alpha=1.0, beta=0.0),
        # the largest native FP64 product of the configurations
        dict(name="dgemm_8192_nn", kind="dgemm", ta="N", tb="N", m=8192, n=8192, k=8192, pad=0, alpha=1.5, beta=0.5),
        # the headline: emulated FP64 on BF16 slices, wide-range entries
        dict(name="emulated_bf16_8192", kind="emulated", method="ozaki", slices=6, ta="N", tb="N", m=8192, n=8192, k=8192),
        # emulated FP64 on INT8 slices, the faster method, at a middling ragged size
        dict(name="emulated_int8_2500", kind="emulated", method="ozaki_int8", slices=7, ta="N", tb="T", m=2500, n=1900,
             k=3001),
        # differentiable product of the rrule configuration, 3xBF16: forward, dA and dB
        dict(name="autograd_4096_bf16x3", kind="autograd", method="f32_bf16x3", m=4096, n=4096, k=2048),
        # a small differentiable layer with the default Float32 method: launches and host work count
        dict(name="autograd_512_f32", kind="autograd", method="f32", m=512, n=384, k=256),
        # 1024 uneven problems, log-uniform in [16, 2048] in steps of 8, native FP64
        dict(name="grouped_1024_f64", kind="grouped", method="f64", count=1024, ta="N", tb="N", lo=16, hi=2048, mult=8,
             shapes=52),
        # the same set in Float32 through 3xBF16
        dict(name="grouped_1024_bf16x3", kind="grouped", method="f32_bf16x3", count=1024, ta="N", tb="N", lo=16, hi=2048,
             mult=8, shapes=52),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _sizes(rng, lo, hi):
    """Three extents, spread over their logarithm; every other draw rounds them to a multiple of 8."""
    v = [_log(rng, lo, hi) for _ in range(3)]
    if rng.random() < 0.5:
        v = [max(lo, x // 8 * 8) for x in v]
    return v


def draw(rng):
    kind = rng.choice(["fastmul", "jmul", "dgemm", "dgemm", "emulated", "autograd", "grouped"])
    op = lambda: rng.choice("NT")  # noqa: E731
    if kind == "fastmul":
        m, n, k = _sizes(rng, 4, 128)
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), m=m, n=n, k=k)
    if kind == "jmul":
        m, n, k = _sizes(rng, 64, 2048)
        return dict(kind=kind, dtype=rng.choice(["f64", "f32"]), m=m, n=n, k=k)
    if kind == "dgemm":
        m, n, k = _sizes(rng, 128, 8192)
        beta = rng.choice([0.0, 0.5])
        return dict(kind=kind, ta=op(), tb=op(), m=m, n=n, k=k, pad=rng.choice([0, 0, 1, 4]), alpha=1.5 if beta else 1.0,
                    beta=beta)
    if kind == "emulated":
        m, n, k = _sizes(rng, 512, 8192)
        method = rng.choice(["ozaki", "ozaki_int8"])
        return dict(kind=kind, method=method, slices=rng.choice([5, 6] if method == "ozaki" else [6, 7]), ta=op(), tb=op(),
                    m=m, n=n, k=k)
    if kind == "autograd":
        m, n, k = _sizes(rng, 64, 4096)
        return dict(kind=kind, method=rng.choice(["f32", "f32_bf16x3", "f64"]), m=m, n=n, k=k)
    return dict(kind=kind, method=rng.choice(["f64", "f32_bf16x3", "f32"]), count=_log(rng, 16, 1024), ta=op(), tb=op(),
                lo=16, hi=2048, mult=rng.choice([1, 8]), shapes=rng.randrange(1 << 30))


# ---- inputs -------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(g, n, dtype):
    return torch.rand(n, generator=g, device="cuda", dtype=dtype) * 2 - 1


def _wide(g, n):
    """u * 2^e with e a whole number in [-12, 12]: the dynamic range the emulated methods are for."""
    e = torch.randint(-12, 13, (n,), generator=g, device="cuda")
    return torch.ldexp(_uniform(g, n, torch.float64), e)


def _colmajor(flat, rows, cols, ld=None):
    """A rows x cols column-major matrix on `flat` (leading dimension ld)."""
    ld = ld or rows
    return flat[:ld * cols].view(cols, ld).T[:rows]


def _stored(t, a, b):
    return (a, b) if t == "N" else (b, a)


def _shapes(case):
    r = random.Random(case["shapes"])
    lo, hi, mult = case["lo"], case["hi"], case["mult"]
    return [tuple(min(hi, max(lo, mult * round(_log(r, lo, hi) / mult))) for _ in range(3)) for _ in range(case["count"])]


def _offsets(sizes):
    """Start of each matrix in one arena, 64-element aligned, and the arena's length."""
    at, out = 0, []
    for s in sizes:
        out.append(at)
        at += -(-s // 64) * 64
    return out, at


def _group(case, seed):
    """Operands and results of a group, each kind in one arena: [(A, B, C)], and the arena of the results."""
    dt = torch.float64 if case["method"] == "f64" else torch.float32
    g, sh = _gen(seed), _shapes(case)
    oa, na = _offsets([m * k for m, n, k in sh])
    ob, nb = _offsets([k * n for m, n, k in sh])
    oc, nc = _offsets([m * n for m, n, k in sh])
    fa, fb, fc = _uniform(g, na, dt), _uniform(g, nb, dt), torch.zeros(nc, device="cuda", dtype=dt)
    out = []
    for (m, n, k), pa, pb, pc in zip(sh, oa, ob, oc):
        out.append((_colmajor(fa[pa:], *_stored(case["ta"], m, k)), _colmajor(fb[pb:], *_stored(case["tb"], k, n)),
                    _colmajor(fc[pc:], m, n)))
    return out, fc


def _operands(case, seed):
    """Plain tensors of the case's inputs: what prepare() hands to the library and exact() to torch."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("fastmul", "jmul"):
        m, n, k, dt = case["m"], case["n"], case["k"], DTYPES[case["dtype"]]
        return dict(A=_colmajor(_uniform(g, m * k, dt), m, k), X=_colmajor(_uniform(g, k * n, dt), k, n))
    if kind == "dgemm":
        m, n, k, pad = case["m"], case["n"], case["k"], case["pad"]
        (ar, ac), (br, bc) = _stored(case["ta"], m, k), _stored(case["tb"], k, n)
        return dict(A=_colmajor(_uniform(g, (ar + pad) * ac, torch.float64), ar, ac, ar + pad),
                    B=_colmajor(_uniform(g, (br + pad) * bc, torch.float64), br, bc, br + pad),
                    C=_colmajor(_uniform(g, (m + pad) * n, torch.float64), m, n, m + pad))
    if kind == "emulated":
        m, n, k = case["m"], case["n"], case["k"]
        (ar, ac), (br, bc) = _stored(case["ta"], m, k), _stored(case["tb"], k, n)
        return dict(A=_colmajor(_wide(g, ar * ac), ar, ac), B=_colmajor(_wide(g, br * bc), br, bc))
    if kind == "autograd":
        # torch's own row-major tensors, entries N(0, 1) / sqrt(k), and the loss gradient W
        m, n, k = case["m"], case["n"], case["k"]
        dt = torch.float64 if case["method"] == "f64" else torch.float32
        rn = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dt)  # noqa: E731
        return dict(A=rn(m, k) / math.sqrt(k), B=rn(k, n) / math.sqrt(k), W=rn(m, n))
    raise ValueError(kind)


def prepare(case, seed):
    jb.init(0)
    kind = case["kind"]
    if kind == "grouped":
        probs, flat = _group(case, seed)
        plan = GroupedPlan(case["method"], [GemmDesc(case["ta"], case["tb"], 1.0, a, b, 0.0, c) for a, b, c in probs])
        return dict(case=case, plan=plan, out=flat)
    state = dict(case=case, **_operands(case, seed))
    if kind in ("fastmul", "jmul"):
        state["D"] = jb.device_matrix(case["m"], case["n"], DTYPES[case["dtype"]])
    elif kind == "emulated":
        state["C"] = jb.device_matrix(case["m"], case["n"], torch.float64)
    elif kind == "autograd":
        state["A"].requires_grad_()
        state["B"].requires_grad_()
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fastmul":
        return jb.fastmul_(state["D"], state["A"], state["X"])
    if kind == "jmul":
        return jb.jmul_(state["D"], state["A"], state["X"])
    if kind == "dgemm":
        return jb.gemm_(case["ta"], case["tb"], case["alpha"], state["A"], state["B"], case["beta"], state["C"])
    if kind == "emulated":
        return jb.gemm_(case["ta"], case["tb"], 1.0, state["A"], state["B"], 0.0, state["C"], method=case["method"],
                        nslices=case["slices"])
    if kind == "autograd":
        method = None if case["method"] in ("f32", "f64") else case["method"]  # None: the binding's default
        Y = matmul(state["A"], state["B"], method)
        dA, dB = torch.autograd.grad(Y, (state["A"], state["B"]), state["W"])
        return Y.detach(), dA, dB
    state["plan"].launch()
    return state["out"]


def work(case):
    """Operands read once, results written (and, with beta, read) once; the slice methods' products are part of what was asked for."""
    kind = case["kind"]
    if kind == "grouped":
        e = 8 if case["method"] == "f64" else 4
        sh = _shapes(case)
        return {"bytes": e * sum(m * k + k * n + m * n for m, n, k in sh),
                "flops": 2 * PRODUCTS[case["method"]] * sum(m * n * k for m, n, k in sh)}
    m, n, k = case["m"], case["n"], case["k"]
    mults = m * n * k
    if kind == "autograd":
        e = 8 if case["method"] == "f64" else 4
        return {"bytes": e * (2 * (m * k + k * n) + 2 * m * n), "flops": 6 * PRODUCTS[case["method"]] * mults}
    if kind in ("fastmul", "jmul"):
        return {"bytes": (8 if case["dtype"] == "f64" else 4) * (m * k + k * n + m * n), "flops": 2 * mults}
    if kind == "emulated":
        s = case["slices"]
        return {"bytes": 8 * (m * k + k * n + m * n), "flops": s * (s + 1) * mults}
    return {"bytes": 8 * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2 * mults}


def exact(case, seed):
    kind = case["kind"]
    if kind == "grouped":
        probs, flat = _group(case, seed)
        out = torch.zeros(flat.numel(), device="cuda", dtype=torch.float64)
        for a, b, c in probs:
            m, n = c.shape
            p = (c.data_ptr() - flat.data_ptr()) // flat.element_size()
            a, b = (a if case["ta"] == "N" else a.T).double(), (b if case["tb"] == "N" else b.T).double()
            _colmajor(out[p:], m, n).copy_(a @ b)
        return out
    s = {name: t.double() for name, t in _operands(case, seed).items()}
    if kind in ("fastmul", "jmul"):
        return s["A"] @ s["X"]
    if kind == "autograd":
        return s["A"] @ s["B"], s["W"] @ s["B"].T, s["A"].T @ s["W"]
    a, b = (s["A"] if case["ta"] == "N" else s["A"].T), (s["B"] if case["tb"] == "N" else s["B"].T)
    if kind == "emulated":
        return a @ b
    return case["alpha"] * (a @ b) + (case["beta"] * s["C"] if case["beta"] else 0.0)
