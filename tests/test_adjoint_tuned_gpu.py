"""Adjoints whose split along k comes from a tuning table, on more tiles than the runtime
keeps arrival counters for (65536): bit for bit the chunks' fma chains added in order."""
import numpy as np
import pytest

import jblas_amd as jb
from jblas_amd import generators as G
from jblas_amd.grouped import GemmDesc, grouped_choices
from jblas_amd.rrule import pullback_
from oracle import oracle as O

from conftest import to_dev
from test_grouped_gpu import write_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["f64", "f32"])
def test_tuned_split_of_many_tiles(gpu, method, tmp_path):
    dt = np.float64 if method == "f64" else np.float32
    m, n, k, rows = 32 * 65536 + 5, 33, 1, 1024
    W0, B = G.matrix(5, rows, n, dtype=dt), G.matrix(6, k, n, dtype=dt)
    ref = O.jmul(W0[:, :32], np.asfortranarray(B.T[:32])) + O.jmul(W0[:, 32:], np.asfortranarray(B.T[32:]))
    w = to_dev(gpu, W0).T.repeat(1, -(-m // rows))[:, :m].contiguous().T  # the rows of W0 over and over
    a, b = jb.device_matrix(m, k, w.dtype), to_dev(gpu, B)
    got = jb.device_matrix(m, k, w.dtype)
    jb.tune_reset()
    write_table(str(tmp_path / "t.json"), method, [(m, k, n)], 0, 2)
    try:
        assert grouped_choices(method, [GemmDesc("N", "T", 1.0, w, b, 0.0, got)])[0][1:] == (2, 32)
        for _ in range(2):
            got.fill_(float("nan"))
            pullback_("N", "N", 1.0, a, b, w, got, None, method=method)
            out = got.cpu().numpy()[:, 0]
            assert np.array_equal(out, np.resize(ref[:, 0], m))
    finally:
        jb.tune_reset()
