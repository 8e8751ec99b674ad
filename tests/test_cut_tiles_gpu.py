"""The slice-pair GEMM's last round of tiles, run as two blocks each: bit for bit the
result of the same columns computed in panels of few tiles (all of them cut), with tile
counts at and around the rule's bounds."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G

from conftest import to_dev

pytestmark = pytest.mark.gpu

# 128 x 64 tiles (3xBF16 128 x 128): 256 whole, 256 + 1 and 256 + 128 with a cut rest, 256 + 129 whole, 128 cut, 129 whole
TILES = [(16, 16), (1, 257), (24, 16), (35, 11), (8, 16), (3, 43)]


@pytest.mark.parametrize("method,width", [("ozaki", 64), ("ozaki_int8", 64), ("bf16x3", 128)])
@pytest.mark.parametrize("tm,tn", TILES)
def test_cut_tiles(gpu, method, width, tm, tn):
    m, n, k = 128 * tm - 5, width * tn - 3, 70
    dt = np.float32 if method == "bf16x3" else np.float64
    A, B = to_dev(gpu, G.matrix(1, m, k, dtype=dt)), to_dev(gpu, G.matrix(2, k, n, dtype=dt))
    C = jb.device_matrix(m, n, A.dtype)
    jb.gemm_("N", "N", 1.0, A, B, 0.0, C, method=method)
    step = width * max(1, 16 // tm)
    for j in range(0, n, step):
        P = jb.device_matrix(m, min(step, n - j), A.dtype)
        jb.gemm_("N", "N", 1.0, A, B[:, j:j + step], 0.0, P, method=method)
        assert gpu.equal(P, C[:, j:j + step])
