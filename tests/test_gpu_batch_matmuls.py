"""Mat-muls of prompts and batches at the edges of their kernels' tiles, against the oracle."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import harness as T
import nigozen_ref as R
import llama_box_amd as L

pytestmark = pytest.mark.gpu


# (K, N, M): one column tile and its neighbours, a half-empty tile, K of fewer chunks than partial sums, rows that are no whole panel (no panel copy), many rows and columns (128 x 128 tiles)
@pytest.mark.parametrize("K,N,M", [(128, 32, 33), (256, 33, 64), (1024, 96, 65), (2048, 160, 97), (640, 70, 129), (1152, 64, 200), (256, 4096, 960), (384, 4096, 1024), (256, 4128, 1057), (128, 4100, 1030)])
def test_q8_0_batches_of_33_columns_and_up(backend, H, K, N, M):
    """mmq_q80.hip: k_mmq_q80_cols / k_mmq_q80_tile — the same bits for a column in any batch of 33 columns and more, and the oracle's values."""
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
            continue  # (another kernel: eight partial sums, not four)
        part = T.run_case(build(c, e), backend)[0].reshape(e - c, N)
        assert np.array_equal(got[c:e].view(np.uint32), part.view(np.uint32)), (c, e)
    rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))  # (the oracle on the first and last rows)
    wr, br = np.ascontiguousarray(w[rows]), np.ascontiguousarray(b[:, rows])
    ref = T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, len(rows)], wr), g.new(L.F32, [K, M], x)), g.new(L.F32, [len(rows), M], br)), "oracle")[0].reshape(M, -1)
    assert T.nmse(got[:, rows], ref) <= 1e-10


def round16(a, wt):
    return R.bf16_round(a) if wt == L.BF16 else a.astype(np.float16).astype(np.float32)


def bits16(a, wt):
    return (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16) if wt == L.BF16 else a.astype(np.float16)


# one step of K and many, row tiles of 64 / 128 with a remainder, column tiles with one column too many or too few, and sizes on both sides of the tiles' dispatch
@pytest.mark.parametrize("wt", [L.BF16, L.F16])
@pytest.mark.parametrize("K,N,M", [(64, 30, 17), (128, 64, 63), (192, 65, 64), (1024, 200, 65), (320, 129, 127), (64, 4100, 330), (256, 12300, 200), (128, 18500, 257), (4096, 96, 40)])
def test_16_bit_matrices_with_batches(backend, H, wt, K, N, M):
    """mmf_tile.hip against float64 over the rounded operands.  f32 sums of K products of size ~1 / sqrt(K): off by at most K eps |x| |w| ~ K 6e-8, in practice its root."""
    rng = np.random.default_rng(K + N + M)
    w = round16((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), wt)
    x = rng.standard_normal((M, K)).astype(np.float32)

    def build(g):
        return H.ggml_mul_mat(g.ctx, g.new(wt, [K, N], bits16(w, wt)), g.new(L.F32, [K, M], x))

    got = T.run_case(build, backend)[0].reshape(M, N)
    ref = round16(x, wt).astype(np.float64) @ w.astype(np.float64).T
    assert np.abs(got - ref).max() <= 6e-8 * np.sqrt(K) * 8


# every form of mmf_tile.hip (stages of its ring, tile of columns x rows) with fewer steps of K than its ring has stages, as many, one and two more, and enough for the ring to go round several
# times, on both sides of the line for short rows; remainders on both sides of the tiles
@pytest.mark.parametrize("stages,tm,tn,N,M,steps", [(3, 256, 128, 14401, 500, (16, 17, 18, 31)), (4, 128, 128, 9000, 330, (16, 17, 18, 31)), (5, 128, 64, 4100, 330, (16, 17, 18, 31)), (5, 64, 128, 9000, 190, (16, 17, 18, 31)),
                                                    (4, 64, 64, 2000, 70, (3, 4, 5, 6, 15, 16, 17, 31)), (3, 64, 64, 4161, 520, (2, 3, 4, 5, 15)), (2, 128, 128, 12101, 500, (1, 2, 3, 4, 15))])
def test_16_bit_tiles_and_their_rings(backend, H, stages, tm, tn, N, M, steps):
    for n_steps in steps:
        one_ring(backend, H, stages, tm, tn, N, M, n_steps)


def one_ring(backend, H, stages, tm, tn, N, M, steps):
    rng = np.random.default_rng(N + M + steps)
    K = 64 * steps
    w = round16((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), L.BF16)
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = T.run_case(lambda g: H.ggml_mul_mat(g.ctx, g.new(L.BF16, [K, N], bits16(w, L.BF16)), g.new(L.F32, [K, M], x)), backend)[0].reshape(M, N)
    assert backend.stat("mm_tile") == stages * 1000000 + tm * 1000 + tn
    ref = round16(x, L.BF16).astype(np.float64) @ w.astype(np.float64).T
    assert np.abs(got - ref).max() <= 6e-8 * np.sqrt(K) * 8  # (as above)


@pytest.mark.parametrize("M", [2, 16, 17, 150])
def test_16_bit_siblings_have_the_bits_of_single_launches(backend, H, M):
    """three bf16 matrices over one input: one launch (and one rounding of the input), the results of three"""
    rng = np.random.default_rng(M)
    K, Ns = 1024, (300, 64, 70)
    ws = [round16((rng.standard_normal((n, K)) / np.sqrt(K)).astype(np.float32), L.BF16) for n in Ns]
    x = rng.standard_normal((M, K)).astype(np.float32)

    def build(g):
        cur = g.new(L.F32, [K, M], x)
        return [H.ggml_mul_mat(g.ctx, g.new(L.BF16, [K, n], bits16(w, L.BF16)), cur) for n, w in zip(Ns, ws)]

    k0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)
    merged = backend.stat("kernel_launches") - k0
    backend.set_option("fusion", 0)
    try:
        plain = T.run_case(build, backend)
    finally:
        backend.set_option("fusion", 1)
    assert merged == (1 if M < 17 else 2)
    for a, b, w in zip(got, plain, ws):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        ref = round16(x, L.BF16).astype(np.float64) @ w.astype(np.float64).T
        assert np.abs(a.reshape(M, -1) - ref).max() <= 6e-8 * np.sqrt(K) * 8


# rows of one, two and four pieces a thread, and rows longer than the norm holds (no copy from that one); reshaped and as they are
@pytest.mark.parametrize("wt", [L.F16, L.BF16])
@pytest.mark.parametrize("K,M", [(512, 17), (1088, 70), (4096, 40), (4160, 40)])
@pytest.mark.parametrize("what", ["norm", "norm_add", "norm_twice", "gate", "gate_rows", "gelu", "silu", "relu_sqr"])
def test_producers_leave_the_16_bit_copy_of_a_product(backend, H, wt, K, M, what):
    """the operand rounded by the kernel that makes it: no launch for it, and bit for bit what a launch of its own leaves"""
    rng = np.random.default_rng(K + M)
    N = 2048
    w = (rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    x, r = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((M, K)).astype(np.float32)
    g1, g2 = rng.standard_normal(K).astype(np.float32), rng.standard_normal(K).astype(np.float32)

    def build(g):
        cur, res = g.new(L.F32, [K, M], x), g.new(L.F32, [K, M], r)
        outs = []
        if what.startswith("norm"):
            cur = H.ggml_mul(g.ctx, H.ggml_norm(g.ctx, cur, 1e-5), g.new(L.F32, [K], g1))
            if what != "norm":
                cur = H.ggml_add(g.ctx, cur, res)
            if what == "norm_twice":
                cur = H.ggml_mul(g.ctx, H.ggml_norm(g.ctx, cur, 1e-5), g.new(L.F32, [K], g2))
        elif what.startswith("gate"):
            if what == "gate_rows":
                cur, res = g.new(L.F32, [8, K // 8, M], x), g.new(L.F32, [8, K // 8, M], r)
            cur = H.ggml_mul(g.ctx, cur, H.ggml_unary(g.ctx, res, 7))  # GGML_UNARY_OP_SIGMOID
            if what == "gate_rows":
                cur = H.ggml_reshape_2d(g.ctx, cur, K, M)
        else:
            cur = H.ggml_unary(g.ctx, cur, {"relu_sqr": 6, "gelu": 8, "silu": 10}[what])  # GGML_UNARY_OP_RELU, _GELU, _SILU
            if what == "relu_sqr":
                cur = H.ggml_sqr(g.ctx, cur)
        return [H.ggml_mul_mat(g.ctx, g.new(wt, [K, N], bits16(round16(w, wt), wt)), cur), cur]

    k0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)
    launches = backend.stat("kernel_launches") - k0
    backend.set_option("fusion", 0)
    try:
        plain = T.run_case(build, backend)
    finally:
        backend.set_option("fusion", 1)
    assert launches == (3 if what.startswith("norm") and K > 4096 else 2)
    for a, b in zip(got, plain):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    ref = round16(got[1].reshape(M, K), wt).astype(np.float64) @ round16(w, wt).astype(np.float64).T
    assert np.abs(got[0].reshape(M, N) - ref).max() <= 6e-8 * np.sqrt(K) * 8 * max(1.0, np.abs(got[1]).max() / 4)  # (the bound above is for operands of up to about 4)


# columns of an expert: none, fewer than a tile, several tiles (one expert draws most); both sides of the lines between the tiles (whose input is rounded by a launch of its own) and mmf.hip's form
@pytest.mark.parametrize("K,N,n_exp,top,T_,tiled", [
    (64, 40, 5, 2, 40, False), (128, 200, 8, 1, 300, False), (192, 130, 3, 3, 70, True), (256, 4160, 6, 2, 100, True), (192, 130, 3, 3, 47, False), (192, 64, 4, 2, 96, True), (256, 70, 4, 1, 92, False),
    (256, 70, 4, 1, 93, True), (384, 1000, 8, 2, 92, False), (384, 1024, 16, 1, 64, True), (448, 96, 8, 2, 93, True), (512, 64, 64, 4, 16, True), (512, 40, 8, 2, 124, False), (512, 40, 8, 2, 125, True),
    (768, 33, 32, 2, 32, True), (1024, 300, 8, 2, 70, True)])
def test_experts_with_batches(backend, H, K, N, n_exp, top, T_, tiled):
    rng = np.random.default_rng(K + N + T_)
    w = round16((rng.standard_normal((n_exp, N, K)) / np.sqrt(K)).astype(np.float32), L.BF16)
    x = rng.standard_normal((T_, 1, K)).astype(np.float32)
    ids = np.stack([rng.permutation(n_exp - 1 if n_exp > top else n_exp)[:top] for _ in range(T_)]).astype(np.int32)  # (the last expert draws nothing when it can be left out)
    ids[: T_ // 2, 0], swap = 0, ids[: T_ // 2, 0].copy()
    for t in range(T_ // 2):
        ids[t, 1:][ids[t, 1:] == 0] = swap[t]

    def build(g):
        return H.ggml_mul_mat_id(g.ctx, g.new(L.BF16, [K, N, n_exp], bits16(w, L.BF16)), g.new(L.F32, [K, 1, T_], x), g.new(L.I32, [top, T_], ids))

    k0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)[0].reshape(T_, top, N)
    assert backend.stat("kernel_launches") - k0 == (2 if tiled else 1)
    xr = round16(x, L.BF16).astype(np.float64)[:, 0]
    ref = np.stack([[w[ids[t, u]].astype(np.float64) @ xr[t] for u in range(top)] for t in range(T_)])
    assert np.abs(got - ref).max() <= 6e-8 * np.sqrt(K) * 8


# every form of the small-batch kernel (K over the waves, with and without a K split; four tiles a workgroup; a tile per wave) and both sides of its groups of eight columns
@pytest.mark.parametrize("qt,K,N", [(L.Q4_K, 2816, 96), (L.Q5_K, 2048, 64), (L.Q6_K, 4096, 160), (L.Q4_K, 1024, 24576), (L.Q6_K, 768, 49152), (L.Q6_K, 256, 70016)])
def test_k_quant_batches_by_groups_of_eight_columns(backend, H, qt, K, N):
    """mmq_skinny.hip: a column's bits do not depend on how many others there are (the integer sums are exact, the f32 sums in the same order), and match the oracle."""
    rng = np.random.default_rng(K + N)
    w = T.rand_weight(qt, K, N, rng)
    x = (rng.standard_normal((32, K)) * rng.uniform(0.2, 3.0, (32, 1))).astype(np.float32)

    def run(M, where, ww):
        return T.run_case(lambda g: H.ggml_mul_mat(g.ctx, g.new(qt, [K, ww.shape[0]], ww), g.new(L.F32, [K, M], x[:M])), where)[0].reshape(M, -1)

    rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))
    w = w.reshape(N, -1)
    ref = run(32, "oracle", np.ascontiguousarray(w[rows]))
    full = run(32 if N < 65536 else 16, backend, w)  # (65536 rows and up: 17 columns and more run on another kernel)
    for M in (2, 3, 7, 8, 9, 15, 16, 17, 24):
        if M > len(full) or (qt == L.Q5_K and M == 2):  # (two columns of Q5_K: the mat-vec)
            continue
        got = run(M, backend, w)
        assert np.array_equal(got.view(np.uint32), full[:M].view(np.uint32)), M
    assert T.nmse(full[:, rows], ref[: len(full)]) <= 1e-10


# one super-block and many, K slices of unequal lengths, two and three token tiles a workgroup with ragged ends, both sides of the lines between the kernels (f: k_mmq_wide_few,
# w: k_mmq_wide, t: the tiled GEMM; for Q4_K, Q5_K, Q6_K), row groups that are not whole eights with as many slices as those allow, Q6_K rows of an odd number of blocks
@pytest.mark.parametrize("qt", [L.Q4_K, L.Q5_K, L.Q6_K])
@pytest.mark.parametrize("K,N,M,kernels", [
    (256, 128, 33, "ttt"), (512, 256, 65, "ttt"), (4608, 128, 77, "fff"), (2560, 384, 96, "fff"), (1024, 4096, 97, "fff"), (768, 512, 129, "fft"), (2048, 1024, 190, "fff"),
    (512, 8192, 288, "fwf"), (1536, 640, 384, "fff"), (1536, 16384, 385, "wwt"), (8192, 128, 33, "ttt"), (8448, 256, 64, "ttt"), (8704, 128, 65, "fff"),
    (1024, 1024, 77, "tft"), (2560, 384, 97, "fff"), (768, 2048, 77, "tft"), (2048, 896, 256, "fff"), (2560, 896, 257, "fff"), (3584, 3072, 288, "fff"),
    (8192, 1024, 384, "fff"), (8192, 4608, 33, "fff"), (512, 16384, 33, "wwt"), (512, 4096, 512, "wwt"), (4096, 4608, 77, "fff"), (4096, 128, 384, "fft"),
    (1536, 20480, 65, "fwf"), (1024, 24576, 64, "wwf")])
def test_k_quant_batches_of_33_columns_and_up(backend, H, qt, K, N, M, kernels):
    """mmq_skinny.hip: k_mmq_wide_few / k_mmq_wide against the oracle and, the sums of the K slices apart, the tiled GEMM: exact integer block sums, f32 sums over K / 256 terms."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(qt, K, N, rng).reshape(N, -1)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    b = rng.standard_normal((M, N)).astype(np.float32)

    def run(where, ww, bb):
        return T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(qt, [K, ww.shape[0]], ww), g.new(L.F32, [K, M], x)), g.new(L.F32, [ww.shape[0], M], bb)), where)[0].reshape(M, -1)

    COUNTERS = ("skinny_launches", "wide_launches", "wide_few_launches", "tiled_launches")
    c0 = [backend.stat(k) for k in COUNTERS]
    got = run(backend, w, b)
    served = [backend.stat(k) - c for k, c in zip(COUNTERS, c0)]
    assert served == {"f": [0, 1, 1, 0], "w": [0, 1, 0, 0], "t": [0, 0, 0, 1]}[kernels[(L.Q4_K, L.Q5_K, L.Q6_K).index(qt)]], served
    c0 = backend.stat("tiled_launches")
    backend.set_option("mmq_skinny", 0)
    try:
        tiled = run(backend, w, b)
    finally:
        backend.set_option("mmq_skinny", 1)
    assert backend.stat("tiled_launches") == c0 + 1
    assert T.nmse(got, tiled) <= 1e-12
    rows = np.unique(np.concatenate([np.arange(min(N, 40)), np.arange(max(0, N - 40), N)]))
    assert T.nmse(got[:, rows], run("oracle", np.ascontiguousarray(w[rows]), np.ascontiguousarray(b[:, rows]))) <= 1e-10


# one column and more, both sides of the lines between the kernels; matrices that the graph makes: a cast, rows stored into a matrix
@pytest.mark.parametrize("wt,M", [(L.BF16, 1), (L.BF16, 2), (L.BF16, 17), (L.BF16, 60), (L.F16, 16), (L.F16, 17), (L.F16, 60), (L.Q8_0, 9), (L.Q8_0, 33), (L.Q8_0, 140)])
@pytest.mark.parametrize("made", ["cast", "rows", "input"])
def test_siblings_wait_for_what_they_read(backend, H, wt, M, made):
    """A sibling is run with the first product of its input only if its matrix and the input are then what they are at its own place: the bits of the same graph node by node."""
    rng = np.random.default_rng(M)
    K, N = 256, 96
    w = [(rng.standard_normal((N, K)) / 16).astype(np.float32) for _ in range(2)]
    x, x2 = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((M, K)).astype(np.float32)

    def run():
        g = T.G(backend)
        try:
            xt, first = g.new(L.F32, [K, M], x), []

            def matrix(q):
                f = g.new(L.F32, [K, N], w[q])
                if made != "rows":
                    return H.ggml_cast(g.ctx, f, wt)
                return H.ggml_set_rows(g.ctx, g.new(wt, [K, N]), f, g.new(L.I64, [N], np.arange(N, dtype=np.int64)))

            ms = [matrix(0), matrix(1)]
            outs = [H.ggml_mul_mat(g.ctx, ms[0], xt)]
            if made == "input":  # both matrices are there before the first product, the input's rows change behind it
                first = [*ms, outs[0], H.ggml_set_rows(g.ctx, xt, g.new(L.F32, [K, M], x2), g.new(L.I64, [M], np.arange(M, dtype=np.int64)))]
            outs.append(H.ggml_mul_mat(g.ctx, ms[1], xt))
            return g.compute(outs, expand_first=first)
        finally:
            g.free()

    got = run()
    backend.set_option("fusion", 0)
    try:
        plain = run()
    finally:
        backend.set_option("fusion", 1)
    for a, b, wq, xq in zip(got, plain, w, (x, x2 if made == "input" else x)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
        assert T.nmse(a.reshape(M, N), xq.astype(np.float64) @ wq.T) < 1e-3  # (8-bit codes of both operands: 1e-4)


@pytest.mark.parametrize("wt", [L.BF16, L.F16, L.Q8_0])
def test_sibling_in_the_block_of_the_first_matrix(backend, H, wt):
    """The first product is the last reader of its matrix, and the sibling's result got that block: the sibling runs behind it."""
    rng = np.random.default_rng(3)
    K, N, M = 1024, 4096, 150
    w = [(rng.standard_normal((N, K)) / 32).astype(np.float32) for _ in range(2)]
    x = rng.standard_normal((M, K)).astype(np.float32)

    def run(recycled):
        g = T.G(backend)
        try:
            xt = g.new(L.F32, [K, M], x)
            ms = [H.ggml_cast(g.ctx, g.new(L.F32, [K, N], v), wt) for v in w]
            outs = [H.ggml_mul_mat(g.ctx, m, xt) for m in ms]
            k0 = backend.stat("kernel_launches")
            r = g.compute(outs, expand_first=ms, same_block=[(outs[1], ms[0])] if recycled else [])
            return r, backend.stat("kernel_launches") - k0
        finally:
            g.free()

    (got, n_got), (plain, n_plain) = run(True), run(False)
    assert n_got == n_plain + 1, (n_got, n_plain)
    for a, b in zip(got, plain):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# two views of one address and one extent whose rows are not the same: fewer rows further apart, or half as many rows of twice the length
@pytest.mark.parametrize("wt", [L.BF16, L.F16, L.Q8_0, L.Q4_K])
@pytest.mark.parametrize("form", ["stride", "length"])
def test_inputs_of_one_address_and_extent(backend, H, wt, form):
    """A converted input is used again for a product over the same rows only: the bits each product has alone."""
    rng = np.random.default_rng(5)
    K, N = 256, 96
    K2 = K if form == "stride" else 2 * K
    M, M2 = (33, 17) if form == "stride" else (40, 20)
    ws = [bits16((rng.standard_normal((N, k)) / 16).astype(np.float32), wt) if wt in (L.BF16, L.F16) else T.rand_weight(wt, k, N, rng) for k in (K, K2)]
    x = rng.standard_normal(40 * 512).astype(np.float32)

    def build(which):
        def f(g):
            xt = g.new(L.F32, [x.size], x)
            v = [H.ggml_view_2d(g.ctx, xt, K, M, K * (8 if form == "stride" else 4), 0), H.ggml_view_2d(g.ctx, xt, K2, M2, K * (16 if form == "stride" else 8), 0)]
            assert H.ggml_nbytes(v[0]) == H.ggml_nbytes(v[1])
            return [H.ggml_mul_mat(g.ctx, g.new(wt, [k, N], w), u) for k, w, u, q in zip((K, K2), ws, v, (0, 1)) if q in which]
        return f

    got = T.run_case(build((0, 1)), backend)
    for q in (0, 1):
        assert np.array_equal(got[q].view(np.uint32), T.run_case(build((q,)), backend)[0].view(np.uint32)), q


@pytest.mark.parametrize("M", [20, 70])
def test_input_of_16_bit_and_quantised_matrices(backend, H, M):
    """An input that both kinds of matrices read in turn (adapters beside a quantised matrix) is converted once for each kind."""
    rng = np.random.default_rng(M)
    K, N = 512, 96
    ws = [(wt, T.rand_weight(wt, K, N, rng) if wt == L.Q8_0 else bits16((rng.standard_normal((N, K)) / 22).astype(np.float32), wt)) for wt in (L.Q8_0, L.F16) * 3]
    x = rng.standard_normal((M, K)).astype(np.float32)

    def run(which):
        k0 = backend.stat("kernel_launches")

        def build(g):
            cur = g.new(L.F32, [K, M], x)
            return [H.ggml_mul_mat(g.ctx, g.new(wt, [K, N], w), cur) for wt, w in (ws[q] for q in which)]

        r = T.run_case(build, backend)
        return r, backend.stat("kernel_launches") - k0

    backend.set_option("fusion", 0)  # (node by node)
    try:
        got, n = run(range(6))
        alone = [run([q]) for q in range(6)]
    finally:
        backend.set_option("fusion", 1)
    assert n == sum(k for _, k in alone) - 4  # (two conversions instead of six)
    for q in range(6):
        assert np.array_equal(got[q].view(np.uint32), alone[q][0][0].view(np.uint32)), q


# both sides of every line of the choice between the tiles and the kernels without them (mul_mat_tile_pays): two launches (rounding, tiles) or one (or two: K slices and their sum)
@pytest.mark.parametrize("wt", [L.BF16, L.F16])
@pytest.mark.parametrize("K,N,M,tiled", [
    (1024, 1024, 128, False), (1024, 1024, 129, True), (1536, 1024, 72, False), (1536, 1024, 73, True), (2048, 512, 256, False), (2048, 512, 257, True), (3072, 1024, 76, False), (3072, 1024, 77, True),
    (4352, 512, 128, False), (4352, 512, 129, True), (512, 32, 40, True), (448, 32, 40, False), (64, 4096, 300, False), (128, 256, 48, False), (128, 256, 49, True), (192, 70, 32, False), (192, 70, 33, True),
    (384, 40, 17, True)])
def test_16_bit_matrices_around_the_lines_of_the_choice(backend, H, wt, K, N, M, tiled):
    rng = np.random.default_rng(K + N + M)
    w = round16((rng.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32), wt)
    x = rng.standard_normal((M, K)).astype(np.float32)

    def run():
        k0 = backend.stat("kernel_launches")
        r = T.run_case(lambda g: H.ggml_mul_mat(g.ctx, g.new(wt, [K, N], bits16(w, wt)), g.new(L.F32, [K, M], x)), backend)[0].reshape(M, N)
        return r, backend.stat("kernel_launches") - k0

    got, n = run()
    assert n == (2 if tiled else 1)
    backend.set_option("fusion", 0)
    try:
        tiles, _ = run()
    finally:
        backend.set_option("fusion", 1)
    ref = round16(x, wt).astype(np.float64) @ w.astype(np.float64).T
    for r in (got, tiles):
        assert np.abs(r - ref).max() <= 6e-8 * np.sqrt(K) * 8
    if tiled:
        assert np.array_equal(got.view(np.uint32), tiles.view(np.uint32))


# 128 x 128 tiles (short rows and many outputs; without a panel copy at any length) and the column kernel in one and two groups of column tiles; rows and columns that end inside a tile
@pytest.mark.parametrize("panels", [False, True])
@pytest.mark.parametrize("K,N,M", [(128, 4128, 600), (256, 2080, 1025), (384, 96, 1030), (1152, 1088, 2500), (128, 64, 1100), (640, 3008, 1090), (512, 14336, 512)])
def test_q8_0_batches_with_and_without_the_panel_copy(backend, H, panels, K, N, M):
    """mmq_q80.hip from 33 columns: the bits of a column are those of 40 columns alone (always the column kernel), and its values the oracle's."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(L.Q8_0, K, N, rng)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    r = rng.standard_normal((M, N)).astype(np.float32)

    def run(c0, c1):
        g = T.G(backend)
        try:
            out = H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, N], w), g.new(L.F32, [K, c1 - c0], x[c0:c1])), g.new(L.F32, [N, c1 - c0], r[c0:c1]))
            got = g.compute([out])[0]
            if panels:  # the same graph again, over a weights buffer
                p0 = backend.stat("decode_copy_launches")
                H.ggml_backend_buffer_set_usage(g.buf, 1)
                assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
                assert backend.stat("decode_copy_launches") == p0 + 1
                got = g.read(out)
            return got.reshape(c1 - c0, N)
        finally:
            g.free()

    backend.set_option("graphs", 0)
    try:
        got = run(0, M)
        for c in (0, M // 2, M - 40):
            assert np.array_equal(got[c:c + 40].view(np.uint32), run(c, c + 40).view(np.uint32)), c
    finally:
        backend.set_option("graphs", 1)
    rows = np.unique(np.concatenate([np.arange(40), np.arange(N - 40, N)]))
    wr, rr = np.ascontiguousarray(w[rows]), np.ascontiguousarray(r[:, rows])
    ref = T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, len(rows)], wr), g.new(L.F32, [K, M], x)), g.new(L.F32, [len(rows), M], rr)), "oracle")[0].reshape(M, -1)
    assert T.nmse(got[:, rows], ref) <= 1e-10


# 16 rows a workgroup over panel copies: one panel, 128 and 129 of them, 257; K of fewer chunks than waves, of a whole ring of four chunks a wave and of one more, of a last ring in part
@pytest.mark.parametrize("M", [2, 3, 15, 16, 17, 32])
@pytest.mark.parametrize("K,N", [(640, 2560), (128, 32), (1152, 4096), (2048, 4128), (2048, 8224), (4096, 64), (4224, 512), (5632, 96)])
def test_q8_0_batches_of_few_columns(backend, H, K, N, M):
    """mmq_q80.hip up to 32 columns: the same bits from the blocks (32 rows a workgroup) and from the panel copy, and the oracle's values."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(L.Q8_0, K, N, rng)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    g = T.G(backend)
    try:
        out = H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, N], w), g.new(L.F32, [K, M], x)), g.new(L.F32, [N], b))
        s0 = backend.stat("skinny_launches")
        blocks = g.compute([out])[0].reshape(M, N)
        p0 = backend.stat("decode_copy_launches")
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
        assert backend.stat("decode_copy_launches") == p0 + 1 and backend.stat("skinny_launches") == s0 + 2
        panels = g.read(out).reshape(M, N)
    finally:
        g.free()
    assert np.array_equal(panels.view(np.uint32), blocks.view(np.uint32))
    rows = np.unique(np.concatenate([np.arange(32), np.arange(N - 32, N)]))
    ref = T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, len(rows)], np.ascontiguousarray(w[rows])), g.new(L.F32, [K, M], x)), g.new(L.F32, [len(rows)], b[rows])), "oracle")[0].reshape(M, -1)
    assert T.nmse(panels[:, rows], ref) <= 1e-10


def test_q8_0_batches_without_the_skinny_kernel(built):
    """GGML_MI355X_Q80_SKINNY=0 turns off the kernels of 2 .. 32 columns; 33 and more stay on the matrix cores."""
    code = """if 1:
        import numpy as np, harness as T, llama_box_amd as L
        be, H, rng = L.Backend(0), L.host(), np.random.default_rng(1)
        w, x = T.rand_weight(L.Q8_0, 256, 64, rng), rng.standard_normal((33, 256)).astype(np.float32)
        for M in (32, 33):
            f = lambda g: H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [256, 64], w), g.new(L.F32, [256, M], x[:M]))
            s = be.stat("skinny_launches")
            got = T.run_case(f, be)[0]
            print(be.stat("skinny_launches") - s, T.nmse(got, T.run_case(f, "oracle")[0]) <= 1e-10)
    """
    env = dict(os.environ, GGML_MI355X_Q80_SKINNY="0", PYTHONPATH=os.pathsep.join([T.REPO, os.path.join(T.REPO, "tests")]))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split() == ["0", "True", "1", "True"], (r.stdout, r.stderr[-1000:])


# K-quants over panel copies: 576 and 577 tiles of 16 rows, rounds of one to several tiles a wave, a wave without a unit (3 super-blocks), one and two matrices a launch, both sides of 16 columns
@pytest.mark.parametrize("M", [2, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("wt,K,Ns,widest,narrowest", [  # (the columns for which panels are used)
    (L.Q4_K, 4096, (4608, 4608), 16, 2), (L.Q4_K, 4352, (9232,), 16, 2), (L.Q4_K, 2048, (9216,), 16, 9), (L.Q4_K, 4096, (33792,), 16, 2), (L.Q4_K, 4096, (9200,), 0, 0), (L.Q5_K, 1024, (9232,), 16, 2),
    (L.Q5_K, 2560, (4624, 4608), 32, 2), (L.Q5_K, 4352, (12288,), 32, 2), (L.Q5_K, 4608, (12288,), 16, 2), (L.Q5_K, 2048, (38400,), 32, 2), (L.Q6_K, 1024, (9216,), 16, 2), (L.Q6_K, 1280, (32784,), 16, 2),
    (L.Q6_K, 2304, (16384, 16384), 32, 2), (L.Q6_K, 3584, (32768,), 32, 2), (L.Q6_K, 8704, (9216,), 16, 2)])
def test_k_quants_over_panels(backend, H, wt, K, Ns, widest, narrowest, M):
    """mmq_panel.hip: the values of the block layout's kernels and of the oracle, with an addend."""
    rng = np.random.default_rng(K + sum(Ns) + M)
    ws = [T.rand_weight(wt, K, N, rng) for N in Ns]
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    bs = [rng.standard_normal(N).astype(np.float32) for N in Ns]

    def outs(g, rows=None):
        cur = g.new(L.F32, [K, M], x)
        sel = [(w, b) if rows is None else (np.ascontiguousarray(w[r]), b[r]) for w, b, r in zip(ws, bs, rows or Ns)]
        return [H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(wt, [K, len(b)], w), cur), g.new(L.F32, [len(b)], b)) for w, b in sel]

    g = T.G(backend)
    try:
        os_ = outs(g)
        blocks = [r.copy() for r in g.compute(os_)]
        k0, p0 = backend.stat("kernel_launches"), backend.stat("decode_copy_launches")
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
        panels = [g.read(o) for o in os_]
        over = narrowest <= M <= widest
        assert backend.stat("decode_copy_launches") == p0 + over
        if over:
            assert backend.stat("kernel_launches") == k0 + 2  # (the quantiser and one launch)
    finally:
        g.free()
    rows = [np.unique(np.concatenate([np.arange(16), np.arange(N - 16, N)])) for N in Ns]
    ref = T.run_case(lambda g: outs(g, rows), "oracle")
    for q, N in enumerate(Ns):
        assert T.nmse(panels[q], blocks[q]) <= 1e-12
        assert T.nmse(panels[q].reshape(M, N)[:, rows[q]], ref[q].reshape(M, -1)) <= 1e-10


# Q6_K beyond 64 columns on the tiled GEMM: panels of 64 and 128 rows in 1, 2, 3, 4, 6 and 8 slices, slices of unequal lengths, fewer super-blocks than slices, ragged last panels and column
# tiles, rows that are no multiple of four (no slices); tiled: also where k_mmq_wide_few could run
@pytest.mark.parametrize("K,N,M,tiled", [
    (256, 300, 65, True), (768, 70, 129, True), (1280, 1000, 140, True), (2304, 999, 300, True), (4096, 4096, 385, True), (4096, 14336, 257, True), (8192, 2044, 257, True), (8448, 8192, 100, True),
    (14336, 4096, 300, True), (14336, 4096, 160, False), (18944, 3584, 140, True), (18944, 3584, 257, False), (18944, 3580, 300, True), (18944, 3584, 400, True), (13824, 5120, 200, True)])
def test_q6_k_panels_and_slices(backend, H, K, N, M, tiled):
    """mmq_i8.hip: what mmq_q6_tile picks gives the oracle's values (exact integer block sums, f32 sums over K / 256 terms in another order)."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(L.Q6_K, K, N, rng).reshape(N, -1)
    x = (rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32)
    b = rng.standard_normal((M, N)).astype(np.float32)

    def run(where, ww, bb):
        return T.run_case(lambda g: H.ggml_add(g.ctx, H.ggml_mul_mat(g.ctx, g.new(L.Q6_K, [K, ww.shape[0]], ww), g.new(L.F32, [K, M], x)), g.new(L.F32, [ww.shape[0], M], bb)), where)[0].reshape(M, -1)

    c0 = backend.stat("tiled_launches")
    got = run(backend, w, b)
    assert backend.stat("tiled_launches") == c0 + tiled
    rows = np.unique(np.concatenate([np.arange(min(N, 20)), np.arange(max(0, N - 20), N)]))
    assert T.nmse(got[:, rows], run("oracle", np.ascontiguousarray(w[rows]), np.ascontiguousarray(b[:, rows]))) <= 1e-10


@pytest.mark.parametrize("copies", [1, 0])
@pytest.mark.parametrize("types,M,served", [  # (launches of the matrix-core kernels with / without the copies)
    ((L.Q8_0,), 2, (1, 0)), ((L.Q8_0,), 3, (1, 1)), ((L.Q5_K,), 2, (1, 0)), ((L.Q5_K,), 3, (1, 1)), ((L.Q5_K, L.Q6_K), 2, (2, 0)), ((L.Q4_K, L.Q6_K), 2, (2, 2)), ((L.Q4_K,), 2, (1, 1))])
def test_two_columns_with_and_without_second_copies(backend, H, copies, types, M, served):
    """graph.cpp: q80_mm_ok, mmq_min_cols_for: two columns of a model's weights leave the mat-vec for the matrix cores only where second copies of the matrices may exist."""
    K, N = 1024, 96
    rng = np.random.default_rng(M + len(types))
    ws = [T.rand_weight(t, K, N, rng) for t in types]
    xs = [(rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32) for _ in types]
    outs = lambda g: [H.ggml_mul_mat(g.ctx, g.new(t, [K, N], w), g.new(L.F32, [K, M], x)) for t, w, x in zip(types, ws, xs)]  # noqa: E731
    ref = T.run_case(outs, "oracle")
    backend.set_option("decode_copy", copies)
    g = T.G(backend)
    try:
        os_ = outs(g)
        g.compute(os_)
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        s0 = backend.stat("skinny_launches")
        assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
        assert backend.stat("skinny_launches") - s0 == served[0 if copies else 1]
        got = [g.read(o) for o in os_]
    finally:
        g.free()
        backend.set_option("decode_copy", 1)
    for a, b in zip(got, ref):
        assert T.nmse(a, b) <= 1e-10


@pytest.mark.parametrize("wt", [L.Q4_K, L.Q5_K, L.Q6_K])
def test_panel_copies_follow_their_weight(backend, H, wt):
    """backend.cpp: k_panel_copy: eager and captured runs follow a weight that is written again in part; a second backend may use a copy that the first has just been asked to make; without
    room the blocks are read."""
    K, N, M = 4096, 9216, 5
    rng = np.random.default_rng(wt)
    w = [T.rand_weight(wt, K, N, rng).reshape(N, -1) for _ in range(2)]
    x = [(rng.standard_normal((M, K)) * rng.uniform(0.2, 3.0, (M, 1))).astype(np.float32) for _ in range(2)]
    w_mixed = np.concatenate([w[0][:N // 2], w[1][N // 2:]])
    rows = np.unique(np.concatenate([np.arange(16), np.arange(N // 2 - 16, N // 2 + 16), np.arange(N - 16, N)]))

    def ref(ww, xx):
        return T.run_case(lambda g: H.ggml_mul_mat(g.ctx, g.new(wt, [K, len(rows)], np.ascontiguousarray(ww[rows])), g.new(L.F32, [K, M], xx)), "oracle")[0].reshape(M, -1)

    H.ggml_backend_graph_compute_async.argtypes = [C.c_void_p, C.POINTER(L.CGraph)]
    other = L.Backend(0)
    g = T.G(backend)
    try:
        wt_t = g.new(wt, [K, N], w[0])
        outs, graphs = [], []
        for xx in x:  # (eight nodes: a repeated graph is captured)
            cur = g.new(L.F32, [K, M], xx)
            for _ in range(8):
                cur = H.ggml_scale(g.ctx, cur, -1.0)
            outs.append(H.ggml_mul_mat(g.ctx, wt_t, cur))
        g.compute(outs)
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        for o in outs:
            graphs.append(H.ggml_new_graph_custom(g.ctx, 64, False))
            H.ggml_build_forward_expand(graphs[-1], o)
        bes = [backend, other]

        def both():
            for be, gf in zip(bes, graphs):
                assert H.ggml_backend_graph_compute_async(be.backend, gf) == 0
            for be in bes:
                H.ggml_backend_synchronize(be.backend)
            return [g.read(o).reshape(M, N)[:, rows] for o in outs]

        for ww in (w[0], w_mixed, w[1]):
            if ww is w_mixed:
                part = np.ascontiguousarray(w[1][N // 2:])
                H.ggml_backend_tensor_set(wt_t, part.ctypes.data, w[0][:N // 2].nbytes, part.nbytes)
            elif ww is w[1]:
                H.ggml_backend_tensor_set(wt_t, w[1].ctypes.data, 0, w[1].nbytes)
            want = [ref(ww, xx) for xx in x]
            n0, l0 = backend.stat("decode_copy_launches"), backend.stat("graph_launches")
            for _ in range(4):
                for a, b in zip(both(), want):
                    assert T.nmse(a, b) <= 1e-10
            assert backend.stat("decode_copy_launches") > n0 and backend.stat("graph_launches") > l0
            bes.reverse()  # (the other backend makes the next copy)
    finally:
        g.free()
        other.close()
    backend.set_option("decode_copy_headroom_gib", 1 << 20)
    g = T.G(backend)
    try:
        o = H.ggml_mul_mat(g.ctx, g.new(wt, [K, N], w[0]), g.new(L.F32, [K, M], x[0]))
        blocks = g.compute([o])[0].copy()
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        n0 = backend.stat("decode_copy_launches")
        assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
        assert backend.stat("decode_copy_launches") == n0
        assert np.array_equal(g.read(o).view(np.uint32), blocks.view(np.uint32))
        assert T.nmse(blocks.reshape(M, N)[:, rows], ref(w[0], x[0])) <= 1e-10
    finally:
        g.free()
        backend.set_option("decode_copy_headroom_gib", 2)


@pytest.mark.parametrize("wt,K,N,M", [(L.Q5_K, 2048, 18432, 4), (L.Q4_K, 2048, 512, 1), (L.Q8_0, 2048, 512, 4)])
def test_two_tensors_over_the_same_bytes(backend, H, wt, K, N, M):
    """backend.cpp: a second copy belongs to a matrix of one row length; another matrix over the same bytes (rows twice as long) does not read it."""
    rng = np.random.default_rng(K + N + M)
    w = T.rand_weight(wt, K, N, rng)
    xs = [rng.standard_normal((M, k)).astype(np.float32) for k in (K, 2 * K)]
    shapes = [(K, N), (2 * K, N // 2)]
    ref = [T.run_case(lambda g: H.ggml_mul_mat(g.ctx, g.new(wt, [k, 64], np.ascontiguousarray(w.reshape(n, -1)[:64])), g.new(L.F32, [k, M], x)), "oracle")[0].reshape(M, -1) for (k, n), x in zip(shapes, xs)]
    g = T.G(backend)
    try:
        ws = [g.new(wt, [k, n], w) for k, n in shapes]
        outs = [H.ggml_mul_mat(g.ctx, t, g.new(L.F32, [k, M], x)) for t, (k, n), x in zip(ws, shapes, xs)]
        g.compute(outs, same_block=[(ws[1], ws[0])])
        H.ggml_backend_buffer_set_usage(g.buf, 1)
        n0 = backend.stat("decode_copy_launches")
        for _ in range(2):
            assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
            for o, (k, n), r in zip(outs, shapes, ref):
                assert T.nmse(g.read(o).reshape(M, n)[:, :64], r) <= 1e-10
        assert backend.stat("decode_copy_launches") - n0 == 2
    finally:
        g.free()
