"""The adjoint entry points on the single-problem kernels: their split-K sums (edges
of chunks and tiles, repeated calls) and operands stored either way.

  * FP64 / FP32 native: bit for bit the split-K chains that a grouped launch of the same
    adjoints would run (chunk products by the oracle's jmul! recurrence, added in order).
  * 3xBF16: |C - C*| <= 2 K 2^-24 |A||B| componentwise against the FP64 oracle.
"""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from jblas_amd.grouped import GemmDesc, grouped_choices
from jblas_amd.rrule import matmul, pullback_
from oracle import oracle as O

from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu

# dA sums over n, dB over m: one to four chunks of at least 256, ragged last ones, tile edges
SHAPES = [(64, 64, 64), (33, 513, 31), (1030, 40, 129), (700, 600, 65), (257, 1200, 127), (1, 2049, 3), (2048, 130, 128)]
DTYPES = {"f64": np.float64, "f32": np.float32, "f32_bf16x3": np.float32}


def chunked(P, Q, kc):
    """P @ Q as fma chains over chunks of kc k, the chunks' results added in order."""
    s = None
    for k0 in range(0, P.shape[1], kc):
        p = O.jmul(np.asfortranarray(P[:, k0:k0 + kc]), np.asfortranarray(Q[k0:k0 + kc]))
        s = p if s is None else s + p
    return s


def check(method, got, P, Q, kc):
    if method == "f32_bf16x3":
        ref = P.astype(np.float64) @ Q.astype(np.float64)
        mag = np.abs(P).astype(np.float64) @ np.abs(Q).astype(np.float64)
        assert np.all(np.abs(got - ref) <= 2 * P.shape[1] * 2.0**-24 * mag)
    else:
        assert np.array_equal(got, chunked(P, Q, kc))


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("method", list(DTYPES))
def test_adjoints_split_k(gpu, method, m, n, k):
    dt = DTYPES[method]
    A, B, W = (G.matrix(7 + i, *s, dtype=dt) for i, s in enumerate([(m, k), (k, n), (m, n)]))
    dev = [to_dev(gpu, x) for x in (A, B, W)]
    dA, dB = jb.device_matrix(m, k, dev[0].dtype), jb.device_matrix(k, n, dev[0].dtype)
    kc = [c[2] for c in grouped_choices(method, [GemmDesc("N", "T", 1.0, dev[2], dev[1], 0.0, dA),
                                                 GemmDesc("T", "N", 1.0, dev[0], dev[2], 0.0, dB)])]
    for ta in "NT":
        for tb in "NT":
            a, b = (to_dev(gpu, x if t == "N" else x.T) for x, t in ((A, ta), (B, tb)))
            ga, gb = jb.device_matrix(*a.shape, a.dtype), jb.device_matrix(*b.shape, b.dtype)
            pullback_(ta, tb, 1.0, a, b, dev[2], ga, gb, method=method)
            check(method, to_host(ga if ta == "N" else ga.T), W, B.T, kc[0])
            check(method, to_host(gb if tb == "N" else gb.T), A.T, W, kc[1])


def layouts(torch, x):
    """The same matrix row-major, column-major, inside a wider row-major one, with a stride in both directions."""
    r = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    wide = torch.full((x.shape[0], x.shape[1] + 3), float("nan"), dtype=r.dtype, device="cuda")
    wide[:, 1:-2] = r
    both = torch.full((2 * x.shape[0], 2 * x.shape[1]), float("nan"), dtype=r.dtype, device="cuda")
    both[::2, ::2] = r
    return [r, to_dev(torch, x), wide[:, 1:-2], both[::2, ::2]]


@pytest.mark.parametrize("m,n,k", [(1, 5, 3), (70, 1, 9), (33, 600, 65), (129, 66, 1), (130, 127, 520)])
@pytest.mark.parametrize("method", list(DTYPES))
def test_matmul_storage_orders(gpu, method, m, n, k):
    dt = DTYPES[method]
    A, B, W = (G.matrix(17 + i, *s, dtype=dt) for i, s in enumerate([(m, k), (k, n), (m, n)]))
    la, lb, lw = (layouts(gpu, x) for x in (A, B, W))
    want = None
    for i in range(4):
        for j in range(4):
            a, b = la[i].detach().requires_grad_(), lb[j].detach().requires_grad_()
            Y = matmul(a, b, method)
            assert Y.stride() == jb.device_matrix(m, n, a.dtype).stride()
            got = [Y.detach(), *gpu.autograd.grad(Y, (a, b), lw[(i + j) % 4])]
            assert [g.stride() for g in got[1:]] == [jb.device_matrix(*s, a.dtype).stride() for s in ((m, k), (k, n))]
            got = [to_host(g) for g in got]
            want = want or got
            assert all(np.array_equal(g, w) for g, w in zip(got, want))
    check(method, want[0], A, B, k)
    for g, P, Q in ((want[1], W, B.T), (want[2], A.T, W)):
        if method == "f32_bf16x3" or P.shape[1] < 512:  # (one chunk)
            check(method, g, P, Q, P.shape[1])
    # a broadcast cotangent has no unit stride
    a, b = la[0].detach().requires_grad_(), lb[0].detach().requires_grad_()
    ga, _ = gpu.autograd.grad(matmul(a, b, method).sum(), (a, b))
    ref = np.ones((m, n)) @ B.T.astype(np.float64)
    assert np.all(np.abs(to_host(ga) - ref) <= 2 * n * 2.0**-24 * (np.ones((m, n)) @ np.abs(B.T)))
