"""Pullbacks of small products while a captured emulated product replays on another stream:
they are no emulated calls, so the replay need not be ordered against them, and share no
workspace with it."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from jblas_amd.rrule import pullback_

from conftest import to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["f64", "f32", "f32_bf16x3"])
def test_pullback_beside_a_replay(gpu, method):
    torch, n = gpu, 2560
    big = [jb.fill_uniform_(torch.empty(n, n, dtype=torch.float64, device="cuda"), 3 + i).T for i in range(2)]
    dt = np.float64 if method == "f64" else np.float32
    m, p, k = 257, 1200, 127  # two chunks of k in both adjoints' sums over p and one over m
    A, B, W = (to_dev(torch, G.matrix(7 + i, *s, dtype=dt)) for i, s in enumerate([(m, k), (k, p), (m, p)]))

    def grads():
        dA, dB = jb.device_matrix(m, k, A.dtype), jb.device_matrix(k, p, A.dtype)
        return pullback_("N", "N", 1.0, A, B, W, dA, dB, method=method)

    C = jb.device_matrix(n, n, torch.float64)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        jb.gemm_("N", "N", 1.0, *big, 0.0, C, method="ozaki")
    want = [to_host(x) for x in grads()]
    torch.cuda.synchronize()
    eager = C.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        jb.gemm_("N", "N", 1.0, *big, 0.0, C, method="ozaki")
    torch.cuda.synchronize()
    for _ in range(3):
        C.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            g.replay()
        got = [grads() for _ in range(10)]
        torch.cuda.synchronize()
        assert torch.equal(C, eager)
        assert all(np.array_equal(to_host(x), w) for pair in got for x, w in zip(pair, want))
    del g
