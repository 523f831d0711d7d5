"""Mat-muls of prompts and batches at the edges of their kernels' tiles, against the oracle."""
import numpy as np
import pytest

import harness as T
import llama_box_amd as L

pytestmark = pytest.mark.gpu


# (K, N, M): one column tile and its neighbours, a half-empty tile, K of fewer chunks than partial sums, rows that are no whole panel (no panel copy),
# and tile counts on both sides of the line between the two splits
@pytest.mark.parametrize("K,N,M", [(128, 32, 33), (256, 33, 64), (1024, 96, 65), (2048, 160, 97), (640, 70, 129), (1152, 64, 200), (256, 4096, 960), (384, 4096, 1024), (256, 4128, 1057), (128, 4100, 1030)])
def test_q8_0_batches_of_33_columns_and_up(backend, H, K, N, M):
    """mmq_q80.hip: k_mmq_q80_cols — the same bits for a column whatever batch it is in (one wave per tile or four), and the oracle's values."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(L.Q8_0, K, N, rng)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    b = rng.standard_normal((M, N)).astype(np.float32)

    def build(c0, c1):
        def f(g):
            r = H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, N], w), g.new(L.F32, [K, c1 - c0], x[c0:c1]))
            return H.ggml_add(g.ctx, r, g.new(L.F32, [N, c1 - c0], b[c0:c1]))
        return f

    s0 = backend.stat("skinny_launches")
    got = T.run_case(build(0, M), backend)[0].reshape(M, N)
    assert backend.stat("skinny_launches") == s0 + 1
    for c, e in {(0, 33), (max(0, M - 63), M), (M // 2, min(M, M // 2 + 40))}:
        if e - c < 33:
            continue  # (another kernel)
        part = T.run_case(build(c, e), backend)[0].reshape(e - c, N)
        assert np.array_equal(got[c:e].view(np.uint32), part.view(np.uint32)), (c, e)
    rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))  # (the oracle on the first and last rows)
    wr, br = np.ascontiguousarray(w[rows]), np.ascontiguousarray(b[:, rows])
    ref = T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, len(rows)], wr), g.new(L.F32, [K, M], x)), g.new(L.F32, [len(rows), M], br)), "oracle")[0].reshape(M, -1)
    assert T.nmse(got[:, rows], ref) <= 1e-10
