"""Attention of prompt portions over a bf16 cache at the edges of its kernel's blocks, against float64."""
import numpy as np
import pytest

import harness as T
import llama_box_amd as L
from test_gpu_nigozen import attention_case

pytestmark = pytest.mark.gpu


# cells: one block, a block and one cell, whole groups of four blocks and one more, many; queries: one wave, one more than two; long runs of hidden blocks in front (chunks)
@pytest.mark.parametrize("n_q,n_kv,heads,kv_heads,dk,dv,chunk,sink", [
    (32, 32, 2, 1, 128, 128, 0, True), (33, 33, 2, 2, 128, 128, 0, False), (65, 128, 4, 1, 128, 128, 64, True), (64, 161, 2, 1, 64, 64, 33, True),
    (130, 2100, 4, 2, 128, 128, 160, True), (40, 1500, 2, 1, 96, 96, 70, False), (100, 700, 2, 1, 128, 64, 0, True), (36, 260, 2, 1, 120, 96, 50, True), (300, 1030, 2, 1, 32, 32, 0, True)])
def test_prompt_attention_at_block_edges(backend, H, n_q, n_kv, heads, kv_heads, dk, dv, chunk, sink):
    """f32 sums of weights split into two bf16 terms (to 2^-17 of each): 2e-5 of the largest value"""
    rng = np.random.default_rng(n_q + 7 * n_kv)
    q = rng.standard_normal((n_q, heads, dk)).astype(np.float32)
    k = rng.standard_normal((n_kv, kv_heads, dk)).astype(np.float32)
    v = rng.standard_normal((n_kv, kv_heads, dv)).astype(np.float32)
    got, ref = attention_case(backend, H, L.BF16, n_q, n_kv, heads, kv_heads, dk, dv, chunk, sink, q, k, v, np.arange(n_kv - n_q, n_kv))
    assert np.abs(got - ref).max() <= 2e-5 * max(1.0, np.abs(ref).max())


# two tokens (eight slices of a head's dimensions) to more workgroups than CUs; lists of one cell, ragged, a full eight-wave trip and more than fit the chip's memory
@pytest.mark.parametrize("T_,NKV,G,per", [(2, 2, 4, 1), (3, 8, 4, 700), (5, 2, 7, 513), (2, 8, 8, 1024), (3, 4, 1, 1100), (16, 8, 2, 70), (17, 8, 4, 100)])
def test_few_tokens_over_listed_cells(backend, H, T_, NKV, G, per):
    """K.q -> SOFT_MAX -> V^T.p of a few tokens over scattered cells (attn_nf.hip), against float64 with the chain's two f16 roundings (queries, probabilities):
    sums of at most 1100 products in f32, and a probability next to a rounding boundary may round the other way: 2^-11 of it."""
    rng = np.random.default_rng(T_ + 31 * per + G)
    HD, NH = 128, NKV * G
    n_kv = min(max(256, (T_ * per + 255) // 256 * 256), 1024 * T_)  # (more cells a token: another route)
    k = rng.standard_normal((n_kv, NKV, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, HD, n_kv)).astype(np.float16)
    q = rng.standard_normal((T_, NH, HD)).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    for t in range(T_):
        mask[t, rng.choice(n_kv, per - t % min(per, 3), replace=False)] = 0

    def build(g):
        kc, vc = g.new(L.F16, [NKV * HD, n_kv], k.reshape(n_kv, -1)), g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        return H.ggml_mul_mat(g.ctx, vv, p)

    s0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)[0].reshape(NH, T_, HD)
    launches = backend.stat("kernel_launches") - s0
    assert launches <= 2, launches  # (the lists and the chain)
    qh = q.astype(np.float16).astype(np.float64)
    for h in range(NH):
        s = qh[:, h] @ k[:, h // G].astype(np.float64).T * HD ** -0.5 + mask
        p = np.exp(s - s.max(1, keepdims=True))
        p = (p / p.sum(1, keepdims=True)).astype(np.float16).astype(np.float64)
        ref = p @ v[h // G].astype(np.float64).T
        assert np.abs(got[h] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, h


# slices of the head dimensions (dq > 1: few tokens) and whole rows, an even and an odd number of heads on a key head
@pytest.mark.parametrize("recycled", [False, True])
@pytest.mark.parametrize("T_,NKV,G,per,dq", [(2, 2, 1, 9, 8), (3, 8, 4, 300, 8), (17, 2, 3, 40, 8), (20, 8, 2, 12, 2), (32, 8, 4, 30, 1), (32, 8, 3, 30, 1)])
def test_few_tokens_feed_a_quantised_matrix(backend, H, T_, NKV, G, per, dq, recycled):
    """... -> CONT(PERMUTE) -> MUL_MAT with a K-quant, the copy in a block of its own or in q's (where the graph allocator puts it).  No launch copies: the attention kernel writes the
    copy or, from whole rows of head pairs, its Q8_K blocks; where it may not write to q's block because other slices still read it, the quantiser takes the heads from the
    product.  Against the same graph node by node: only a Q8_K code next to a rounding boundary may differ (1e-5 of the product's size)."""
    rng = np.random.default_rng(T_ + 31 * per + G)
    HD, NH, n_kv, N = 128, NKV * G, max(256, (T_ * per + 255) // 256 * 256), 96
    k = rng.standard_normal((n_kv, NKV * HD)).astype(np.float16)
    v = rng.standard_normal((NKV * HD, n_kv)).astype(np.float16)
    wq, x = T.rand_weight(L.Q4_K, 256, NH * HD, rng), rng.standard_normal((T_, 256)).astype(np.float32)
    wo = T.rand_weight(L.Q4_K, NH * HD, N, rng)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    for t in range(T_):
        mask[t, rng.choice(n_kv, per, replace=False)] = 0

    def run(whole):  # the launches up to wo's product, or the product
        g = T.G(backend)
        try:
            q = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [256, NH * HD], wq), g.new(L.F32, [256, T_], x))
            qp = H.ggml_permute(g.ctx, H.ggml_reshape_3d(g.ctx, q, HD, NH, T_), 0, 2, 1, 3)
            kv = H.ggml_view_3d(g.ctx, g.new(L.F16, [NKV * HD, n_kv], k), HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
            vv = H.ggml_view_3d(g.ctx, g.new(L.F16, [n_kv, NKV * HD], v), n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
            p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
            o = H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, H.ggml_mul_mat(g.ctx, vv, p), 0, 2, 1, 3), NH * HD, T_)
            r = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [NH * HD, N], wo), o) if whole else H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [256, NH * HD], wq), g.new(L.F32, [256, T_], x))
            k0 = backend.stat("kernel_launches")
            out = g.compute([r], same_block=[(o, q)] if recycled else [])[0]
            return out, backend.stat("kernel_launches") - k0
        finally:
            g.free()

    got, launches = run(True)
    product = 1 + (NH * HD // 256 >= 8)  # wo: K slices and their sum from eight super-blocks on
    quantised = 0 if dq == 1 and G % 2 == 0 else 1
    assert launches == run(False)[1] + 2 + quantised + product, launches  # (q; the lists, the chain)
    backend.set_option("fusion", 0)
    try:
        plain, _ = run(True)
    finally:
        backend.set_option("fusion", 1)
    assert T.nmse(got, plain) <= 1e-5


@pytest.mark.parametrize("T_,n_kv", [(32, 32768), (512, 16384)])
def test_one_head_over_one_key_head(H, T_, n_kv):
    """K.q -> SOFT_MAX -> V^T.p with one query head on one key head: plain 2-D products by their shapes, and the chain's scratch is there for them too (more of it than a new
    backend's first allocation leaves over).  Against float64 with the chain's two f16 roundings: 2^-11 of a probability next to a rounding boundary."""
    rng = np.random.default_rng(T_)
    HD, backend = 128, L.Backend(0)
    k, v = rng.standard_normal((n_kv, HD)).astype(np.float16), rng.standard_normal((HD, n_kv)).astype(np.float16)
    q = rng.standard_normal((T_, 1, HD)).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    for t in range(T_):
        mask[t, rng.choice(n_kv, 40, replace=False)] = 0

    def build(g):
        kc, vc = g.new(L.F16, [HD, n_kv], k), g.new(L.F16, [n_kv, HD], v)
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, 1, T_], q), 0, 2, 1, 3)
        kv, vv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, 1, HD * 2, HD * 2, 0), H.ggml_view_3d(g.ctx, vc, n_kv, HD, 1, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        return H.ggml_mul_mat(g.ctx, vv, p)

    try:
        f0 = backend.stat("fused_nodes")
        got = T.run_case(build, backend)[0].reshape(T_, HD)
        assert backend.stat("fused_nodes") == f0 + 2  # (the soft-max and the second product)
    finally:
        backend.close()
    s = q[:, 0].astype(np.float16).astype(np.float64) @ k.astype(np.float64).T * HD ** -0.5 + mask
    p = np.exp(s - s.max(1, keepdims=True))
    ref = (p / p.sum(1, keepdims=True)).astype(np.float16).astype(np.float64) @ v.astype(np.float64).T
    assert np.abs(got - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5


# k_attn_mma_bf16 (attn_f32.hip): blocks of 32 cells, every fourth one a wave's.  Fewer blocks than waves, a last block of 1 and of 31 cells, masks that leave a wave nothing, holes between requests,
# biases, a row that sees nothing, rows of the f32's lowest value; heads in eights (the launch's other order) and not; head sizes of whole tiles and not
@pytest.mark.parametrize("n_q,n_kv,heads,kv_heads,dk,dv", [(32, 32, 8, 2, 128, 128), (33, 97, 3, 1, 64, 64), (70, 287, 16, 4, 32, 128), (64, 1000, 8, 8, 96, 96), (100, 130, 5, 5, 72, 40), (257, 700, 8, 1, 128, 64),
                                                           (40, 33, 6, 3, 24, 32)])
@pytest.mark.parametrize("kind", ["causal", "holes", "bias", "lowest"])
def test_prompts_over_a_bf16_cache(backend, H, n_q, n_kv, heads, kv_heads, dk, dv, kind):
    rng = np.random.default_rng(n_q + n_kv + dk)
    r16 = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32)
    bits = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    q, k, v = (r16(rng.standard_normal(s) * f) for s, f in (((n_q, heads, dk), 2.0), ((n_kv, kv_heads, dk), 1.0), ((n_kv, kv_heads, dv), 1.0)))
    low = np.finfo(np.float32).min if kind == "lowest" else -np.inf
    t, j = np.arange(n_q)[:, None], np.arange(n_kv)[None, :]
    ok = j <= t + max(0, n_kv - n_q)
    if kind == "holes":
        ok = ok & ((j // 40) % 3 == t % 3)
    m = np.full((n_q, n_kv), low, np.float32)
    m[ok] = 0.0
    if kind == "bias":
        m = np.where(ok, -0.01 * np.abs(t - j), -np.inf).astype(np.float32)
        m[5] = -np.inf  # (a row that sees nothing: zeros)
    mask = np.full((64 * ((n_q + 63) // 64), n_kv), -np.inf, np.float32)
    mask[:n_q] = m
    scale = 1.0 / np.sqrt(dk)

    def build(g):
        tk, tv = (g.new(L.BF16, [d * kv_heads, n_kv], bits(x)) for d, x in ((dk, k), (dv, v)))
        kk = H.ggml_view_3d(g.ctx, tk, dk, n_kv, kv_heads, dk * kv_heads * 2, dk * 2, 0)
        vv = H.ggml_view_3d(g.ctx, tv, dv, n_kv, kv_heads, dv * kv_heads * 2, dv * 2, 0)
        r = H.ggml_flash_attn_ext(g.ctx, H.ggml_permute(g.ctx, g.new(L.F32, [dk, heads, n_q], q), 0, 2, 1, 3), kk, vv, g.new(L.F32, [n_kv, mask.shape[0]], mask), scale, 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(r, 10)
        return r

    got = T.run_case(build, backend)[0].reshape(n_q, heads, dv)
    for h in range(heads):
        z = scale * (q[:, h].astype(np.float64) @ k[:, h // (heads // kv_heads)].astype(np.float64).T) + m
        top = z.max(axis=1, keepdims=True)
        w = np.where(np.isfinite(z), np.exp(z - np.where(np.isfinite(top), top, 0.0)), 0.0)
        den = w.sum(axis=1, keepdims=True)
        ref = np.where(den > 0, w, 0.0) / np.where(den > 0, den, 1.0) @ v[:, h // (heads // kv_heads)].astype(np.float64)
        # (a weight as two bf16 terms is off by 2^-17, a score of up to 40 in f32 sums by a few 2^-20)
        assert np.abs(got[:, h] - ref).max() <= 2.0 ** -15 * np.abs(v).max()


# up to three visible blocks of 32 cells, near the start and the end of a cache of one block, of up to 64 and of more (a wave alone, or four that meet), rows that are no whole fours, with and without sinks
@pytest.mark.parametrize("n_kv", [3, 31, 32, 35, 256, 1026, 2048, 2080])
@pytest.mark.parametrize("blocks", [0, 1, 2, 3])
@pytest.mark.parametrize("sinks", [False, True])
def test_prompts_that_see_few_blocks_of_a_bf16_cache(backend, H, n_kv, blocks, sinks):
    n_q, heads, kv_heads, d = 37, 8, 2, 64
    rng = np.random.default_rng(n_kv + blocks)
    r16 = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32)
    bits = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    q, k, v = (r16(rng.standard_normal(s) * f) for s, f in (((n_q, heads, d), 2.0), ((n_kv, kv_heads, d), 1.0), ((n_kv, kv_heads, d), 1.0)))
    sk = rng.standard_normal(heads).astype(np.float32)
    m = np.full((64, n_kv), -np.inf, np.float32)
    for b in [b for b in (1, (n_kv - 1) // 32, 4)[:blocks] if 32 * b < n_kv]:
        m[:n_q, 32 * b : 32 * b + 32] = np.where(rng.random((n_q, min(32, n_kv - 32 * b))) < 0.5, 0.0, -np.inf)

    def build(g):
        tk, tv = (g.new(L.BF16, [d * kv_heads, n_kv], bits(x)) for x in (k, v))
        kk, vv = (H.ggml_view_3d(g.ctx, t, d, n_kv, kv_heads, d * kv_heads * 2, d * 2, 0) for t in (tk, tv))
        r = H.ggml_flash_attn_ext(g.ctx, H.ggml_permute(g.ctx, g.new(L.F32, [d, heads, n_q], q), 0, 2, 1, 3), kk, vv, g.new(L.F32, [n_kv, 64], m), 0.125, 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(r, 10)
        if sinks:
            H.ggml_flash_attn_ext_add_sinks(r, g.new(L.F32, [heads], sk))
        return r

    got = T.run_case(build, backend)[0].reshape(n_q, heads, d)
    for h in range(heads):
        z = 0.125 * (q[:, h].astype(np.float64) @ k[:, h // 4].astype(np.float64).T) + m[:n_q]
        top = np.maximum(z.max(axis=1, keepdims=True), sk[h] if sinks else -1e300)
        w = np.exp(z - top)
        den = w.sum(axis=1, keepdims=True) + (np.exp(sk[h] - top) if sinks else 0.0)
        ref = np.where(den > 0, w, 0.0) / np.where(den > 0, den, 1.0) @ v[:, h // 4].astype(np.float64)
        assert np.abs(got[:, h] - ref).max() <= 2.0 ** -15 * np.abs(v).max()  # (as above)


# heads of 64 whose only reader is a Q8_0 product on the matrix cores: the combine pass leaves the product's quantised blocks — tokens on lists (9 .. 32) and prompts, 2 .. 8 records a row
@pytest.mark.parametrize("T_,n_kv,NH,NKV,splits", [(9, 640, 8, 2, 0), (16, 2560, 32, 4, 0), (32, 512, 8, 8, 8), (40, 512, 16, 4, 0), (130, 700, 8, 4, 5), (512, 1024, 16, 2, 0)])
def test_heads_of_64_leave_quantised_rows(backend, H, T_, n_kv, NH, NKV, splits):
    rng = np.random.default_rng(T_ + n_kv)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((NH, T_, 64), (NKV, n_kv, 64), (NKV, n_kv, 64)))
    w = T.rand_weight(L.Q8_0, NH * 64, 256, rng)
    mask = np.full(((T_ + 63) // 64 * 64, n_kv), -np.inf, np.float16)
    for t in range(T_):
        mask[t, : n_kv - T_ + t + 1] = 0

    def build(also):
        def f(g):
            tq, tk, tv = g.new(L.F32, [64, T_, NH], q), g.new(L.F16, [64, n_kv, NKV], k.astype(np.float16)), g.new(L.F16, [64, n_kv, NKV], v.astype(np.float16))
            a = H.ggml_flash_attn_ext(g.ctx, tq, tk, tv, g.new(L.F16, [n_kv, mask.shape[0]], mask), 0.125, 0.0, 0.0)
            H.ggml_flash_attn_ext_set_prec(a, 10)
            r = H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [NH * 64, 256], w), H.ggml_reshape_2d(g.ctx, a, NH * 64, T_))
            return [r, a] if also else [r]
        return f

    backend.set_option("fa_splits", splits)
    try:
        n = []
        out = []
        for also in (False, True):  # (an attention result that is an output itself exists in f32, with a quantiser behind it)
            k0 = backend.stat("kernel_launches")
            out.append(np.asarray(T.run_case(build(also), backend)[0], np.float32))
            n.append(backend.stat("kernel_launches") - k0)
    finally:
        backend.set_option("fa_splits", 0)
    assert n[0] == n[1] - 1, n
    # (the two combine passes sum the records' weights in another order: a value next to a rounding boundary moves by 1 / 127 of its block's largest, few of them)
    assert T.nmse(out[0], out[1]) <= 1e-6


# the option that widens the mat-vec fusions beyond 8 columns: products that take them quantise their f32 input themselves, so its producer (attention, norm, SwiGLU) may not leave panel blocks alone
@pytest.mark.parametrize("what", ["attention", "norm", "swiglu"])
@pytest.mark.parametrize("widest", [11, 12, 16])
def test_mat_vec_fusions_of_many_columns_find_their_input(backend, H, what, widest):
    T_, n_kv, NH, NKV, N = 12, 640, 8, 2, 256
    rng = np.random.default_rng(widest)
    K = NH * 64
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((NH, T_, 64), (NKV, n_kv, 64), (NKV, n_kv, 64)))
    x, w0, r1, r2 = (rng.standard_normal(s).astype(np.float32) for s in ((T_, K), (K,), (T_, N), (T_, N)))
    ws = [T.rand_weight(L.Q8_0, K, n, rng) for n in (N, N, K, K)]
    mask = np.full((64, n_kv), -np.inf, np.float16)
    for t in range(T_):
        mask[t, : n_kv - T_ + t + 1] = 0

    def build(g):
        def mm(i, y, n):
            return H.ggml_mul_mat(g.ctx, g.new(L.Q8_0, [K, n], ws[i]), y)

        if what == "attention":
            y = H.ggml_flash_attn_ext(g.ctx, g.new(L.F32, [64, T_, NH], q), g.new(L.F16, [64, n_kv, NKV], k.astype(np.float16)), g.new(L.F16, [64, n_kv, NKV], v.astype(np.float16)),
                                      g.new(L.F16, [n_kv, 64], mask), 0.125, 0.0, 0.0)
            H.ggml_flash_attn_ext_set_prec(y, 10)
            y = H.ggml_reshape_2d(g.ctx, y, K, T_)
        else:
            y = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, g.new(L.F32, [K, T_], x), 1e-5), g.new(L.F32, [K], w0))
            if what == "norm":
                return [H.ggml_swiglu_split(g.ctx, mm(0, y, N), mm(1, y, N))]
            y = H.ggml_swiglu_split(g.ctx, mm(2, y, K), mm(3, y, K))
        return [H.ggml_add(g.ctx, H.ggml_add(g.ctx, mm(0, y, N), g.new(L.F32, [N, T_], r1)), g.new(L.F32, [N, T_], r2))]

    backend.set_option("fa_splits", 4)  # (attention ends in the combine pass that can leave blocks)
    try:
        ref = T.run_case(build, backend)[0]
        backend.set_option("mmvq_max_cols", widest)
        got = T.run_case(build, backend)[0]
    finally:
        backend.set_option("mmvq_max_cols", 2)
        backend.set_option("fa_splits", 0)
    # (other kernels in front of the quantiser: a value next to a rounding boundary moves by 1 / 127 of its block's largest, few of them)
    assert T.nmse(got, ref) <= 1e-6


# tokens of one sequence, which see all cells, and tokens with a few cells each, for which most of a row's splits have none; heads of 128 and 64; a number of cells that no split divides
@pytest.mark.parametrize("T_,n_kv,NH,NKV,HD,seen", [
    (9, 1532, 8, 2, 128, 0), (9, 1532, 8, 2, 128, 3), (2, 260, 4, 4, 128, 1), (5, 6000, 16, 2, 128, 0), (20, 1600, 32, 8, 128, 77), (9, 1000, 16, 4, 64, 0), (16, 2432, 32, 4, 64, 2), (31, 4096, 16, 8, 64, 130)])
def test_splits_of_few_tokens(backend, H, T_, n_kv, NH, NKV, HD, seen):
    """position lists in more splits than a token may have cells for, against float64 on the f16 query: sums of at most 6000 products in f32"""
    rng = np.random.default_rng(T_ + n_kv)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((NH, T_, HD), (NKV, n_kv, HD), (NKV, n_kv, HD)))
    k, v = k.astype(np.float16), v.astype(np.float16)
    mask = np.full(((T_ + 63) // 64 * 64, n_kv), -np.inf, np.float16)
    for t in range(T_):
        if seen:
            mask[t, rng.choice(n_kv, seen, replace=False)] = 0
        else:
            mask[t, : n_kv - T_ + t + 1] = 0

    def build(g):
        a = H.ggml_flash_attn_ext(g.ctx, g.new(L.F32, [HD, T_, NH], q), g.new(L.F16, [HD, n_kv, NKV], k), g.new(L.F16, [HD, n_kv, NKV], v), g.new(L.F16, [n_kv, mask.shape[0]], mask), HD ** -0.5, 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(a, 10)
        return a

    s0 = backend.stat("fa_list_launches")
    got = T.run_case(build, backend)[0].reshape(T_, NH, HD)
    assert backend.stat("fa_list_launches") == s0 + 1
    for h in range(NH):
        z = q[h].astype(np.float16).astype(np.float64) @ k[h // (NH // NKV)].astype(np.float64).T * HD ** -0.5 + mask[:T_].astype(np.float64)
        p = np.exp(z - z.max(1, keepdims=True))
        ref = (p / p.sum(1, keepdims=True)) @ v[h // (NH // NKV)].astype(np.float64)
        # (scores are f32 sums over packed f16 products, the probabilities packed f16: 2^-10 of a weight, as the few-token tests above)
        assert np.abs(got[:, h] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, h


# one pass over all cells, two heads of a key head a workgroup, at the lines between it and the splits; group sizes that leave a last pair in part, Q8_0 rows, sinks, tokens on lists
@pytest.mark.parametrize("T_,n_kv,NH,NKV,HD,seen,q8,sinks,launches", [
    (1, 1, 7, 1, 128, 0, False, False, 1), (1, 255, 14, 2, 128, 0, False, True, 1), (1, 768, 14, 2, 128, 0, False, False, 1), (1, 772, 14, 2, 128, 0, False, False, 2), (1, 512, 8, 2, 128, 0, False, False, 1),
    (1, 513, 8, 2, 128, 0, False, False, 2), (1, 1, 4, 1, 128, 0, False, False, 1), (1, 256, 32, 8, 128, 0, False, True, 1), (1, 200, 6, 2, 128, 0, False, False, 1), (1, 257, 5, 1, 128, 0, True, False, 2), (1, 256, 6, 2, 128, 0, True, True, 1), (1, 70, 3, 3, 64, 0, False, False, 1), (1, 1024, 32, 4, 64, 0, False, True, 1),
    (1, 1025, 10, 2, 64, 0, False, False, 2), (2, 900, 8, 2, 128, 384, False, True, 2), (3, 900, 8, 2, 128, 385, False, False, 3), (17, 640, 16, 8, 128, 130, False, False, 2), (6, 500, 8, 2, 128, 256, True, False, 2),
    (6, 500, 12, 2, 128, 257, True, False, 3), (4, 4096, 7, 1, 64, 1000, False, True, 2), (4, 4096, 8, 1, 64, 200, False, False, 2), (32, 640, 24, 8, 64, 256, False, False, 2), (32, 644, 24, 8, 64, 257, False, False, 2)])
def test_one_pass_of_head_pairs(backend, H, T_, n_kv, NH, NKV, HD, seen, q8, sinks, launches):
    """against float64 on the rows and queries as the kernel reads them (f16; Q8_0 rows: 8-bit queries); `launches`: the attention's own and the list scan's"""
    rng = np.random.default_rng(T_ + n_kv + NH)
    q = rng.standard_normal((NH, T_, HD)).astype(np.float32)
    k, v = (rng.standard_normal((NKV, n_kv, HD)).astype(np.float32) for _ in range(2))
    sk = rng.standard_normal(NH).astype(np.float32)
    mask = np.full(((T_ + 63) // 64 * 64, n_kv), -np.inf, np.float16)
    for t in range(T_):
        if seen:
            mask[t, rng.choice(n_kv, seen, replace=False)] = 0
        else:
            mask[t, : n_kv - T_ + t + 1] = 0
    if q8:
        def blocks(x):  # (bytes, values) of Q8_0 blocks
            b = x.reshape(-1, 32)
            d = (np.abs(b).max(1, keepdims=True) / 127).astype(np.float32)
            i = np.rint(b / d).astype(np.int8)
            return np.concatenate([d.astype(np.float16).view(np.uint8), i.view(np.uint8)], 1), (d.astype(np.float16).astype(np.float32) * i).reshape(x.shape)

        (kr, k), (vr, v), (_, qx) = blocks(k), blocks(v), blocks(q)
    else:
        kr, vr = (x.astype(np.float16) for x in (k, v))
        k, v, qx = kr, vr, q.astype(np.float16)

    def build(g):
        kt = L.Q8_0 if q8 else L.F16
        a = H.ggml_flash_attn_ext(g.ctx, g.new(L.F32, [HD, T_, NH], q), g.new(kt, [HD, n_kv, NKV], kr), g.new(kt, [HD, n_kv, NKV], vr),
                                  H.ggml_cast(g.ctx, g.new(L.F32, [n_kv, mask.shape[0]], mask.astype(np.float32), "KQ_mask"), L.F16), HD ** -0.5, 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(a, 10)
        if sinks:
            H.ggml_flash_attn_ext_add_sinks(a, g.new(L.F32, [NH], sk))
        return a

    n0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)[0].reshape(T_, NH, HD)
    assert backend.stat("kernel_launches") - n0 == launches + 1  # (the mask's conversion)
    for h in range(NH):
        z = qx[h].astype(np.float64) @ k[h // (NH // NKV)].astype(np.float64).T * HD ** -0.5 + mask[:T_].astype(np.float64)
        m = np.maximum(z.max(1, keepdims=True), sk[h] if sinks else -np.inf)
        p = np.exp(z - m)
        ref = (p / (p.sum(1, keepdims=True) + (np.exp(sk[h] - m) if sinks else 0.0))) @ v[h // (NH // NKV)].astype(np.float64)
        # (f32 sums and probabilities: 2^-11 of headroom over the query's own rounding, whose f16 scale a Q8_0 block holds)
        assert np.abs(got[:, h] - ref).max() <= 1e-3 * np.abs(ref).max() + 1e-5, h


# one token of a batch on lists sees nothing: with sinks its result is zero (all weight is the sink's), without them NaN, of which quantisers make Q8_K blocks of zeros and Q8_0 scales of NaN; f32 rows and
# such blocks (whose scratch holds another step's before), pairs of heads and whole groups
@pytest.mark.parametrize("T_,n_kv,NH,NKV,HD,seen,kq,sinks,reader", [
    (3, 900, 8, 2, 128, 300, False, True, None), (3, 900, 8, 2, 128, 300, False, False, None), (5, 500, 8, 2, 128, 200, True, True, None), (4, 1024, 7, 1, 64, 200, False, True, None), (4, 1024, 8, 2, 64, 900, False, False, None),
    (24, 640, 32, 8, 128, 100, False, True, None), (3, 900, 8, 2, 128, 300, False, True, "Q4_K"), (3, 900, 8, 2, 128, 300, False, False, "Q4_K"), (24, 640, 32, 8, 128, 100, False, False, "Q4_K"),
    (24, 640, 16, 8, 128, 100, True, True, "Q6_K"), (4, 1024, 8, 2, 64, 200, False, False, "Q8_0"), (4, 1024, 8, 2, 64, 900, False, False, "Q8_0"), (4, 1024, 8, 2, 64, 200, False, True, "Q8_0"), (1, 256, 8, 2, 128, 100, False, True, None),
    (1, 256, 8, 2, 128, 100, False, False, None), (1, 300, 14, 2, 128, 100, False, True, "Q4_K"), (1, 200, 8, 2, 128, 100, True, True, None), (1, 700, 8, 1, 64, 100, False, True, None), (1, 700, 8, 1, 64, 100, False, False, None)])
def test_token_without_cells(backend, H, T_, n_kv, NH, NKV, HD, seen, kq, sinks, reader):
    """one pass against splits and their merge (option fa_splits), where the merge speaks for such a token"""
    rng = np.random.default_rng(T_ + n_kv + NH)
    q = rng.standard_normal((NH, T_, HD)).astype(np.float32)
    k, v = (T.rand_weight(L.Q8_0, HD, n_kv * NKV, rng) if kq else rng.standard_normal((NKV, n_kv, HD)).astype(np.float16) for _ in range(2))
    sk = rng.standard_normal(NH).astype(np.float32)
    w = T.rand_weight(getattr(L, reader), NH * HD, 96, rng) if reader else None
    full = np.full((64, n_kv), -np.inf, np.float32)
    for t in range(T_):
        full[t, rng.choice(n_kv, seen, replace=False)] = 0
    blind = full.copy()
    blind[T_ // 2] = -np.inf

    def build(mask):
        def f(g):
            kt = L.Q8_0 if kq else L.F16
            a = H.ggml_flash_attn_ext(g.ctx, g.new(L.F32, [HD, T_, NH], q), g.new(kt, [HD, n_kv, NKV], k), g.new(kt, [HD, n_kv, NKV], v), H.ggml_cast(g.ctx, g.new(L.F32, [n_kv, 64], mask, "KQ_mask"), L.F16),
                                      HD ** -0.5, 0.0, 0.0)
            H.ggml_flash_attn_ext_set_prec(a, 10)
            if sinks:
                H.ggml_flash_attn_ext_add_sinks(a, g.new(L.F32, [NH], sk))
            return H.ggml_mul_mat(g.ctx, g.new(getattr(L, reader), [NH * HD, 96], w), H.ggml_reshape_2d(g.ctx, a, NH * HD, T_)) if reader else a
        return f

    def run(mask):
        k0 = backend.stat("kernel_launches")
        return T.run_case(build(mask), backend)[0].reshape(T_, -1), backend.stat("kernel_launches") - k0

    run(full)
    got, n_got = run(blind)
    backend.set_option("fa_splits", 3)
    try:
        ref, n_ref = run(blind)
    finally:
        backend.set_option("fa_splits", 0)
    assert n_got < n_ref or (sinks and reader == "Q8_0")
    t = T_ // 2
    assert np.array_equal(got[t], ref[t], equal_nan=True) and (np.isnan(ref[t]).all() if not sinks and reader in (None, "Q8_0") else (ref[t] == 0).all())
    # (f32 sums in another order; an 8-bit value next to a rounding boundary moves by 1 / 127 of its block's largest, few of them)
    assert T.nmse(np.delete(got, t, 0), np.delete(ref, t, 0)) <= 1e-6


# trips of 512 cells with eight waves (16, 32 and 64 rows of V^T a workgroup) and of 256 with four, the last tile and the last trip in part, waves without a tile; whole rows from 80 pairs of
# a token and a key head and 64 cells a token on (their 256- and 512-cell limits on both sides)
@pytest.mark.parametrize("T_,NKV,G,per", [
    (2, 8, 4, 17), (3, 8, 5, 513), (4, 8, 4, 1024), (6, 8, 3, 129), (6, 8, 8, 1000), (12, 8, 1, 1023), (14, 8, 6, 257), (10, 8, 4, 64), (10, 8, 7, 250), (10, 8, 4, 260), (20, 8, 4, 500), (20, 8, 5, 520), (9, 8, 4, 100)])
def test_few_tokens_on_matrix_cores(backend, H, T_, NKV, G, per):
    """attn_nf.hip; infinities and NaN in cells that a token does not see stay out of its result"""
    rng = np.random.default_rng(T_ + 31 * per + G)
    HD, NH = 128, NKV * G
    n_kv = max(256, (T_ * per + 255) // 256 * 256)
    k = rng.standard_normal((n_kv, NKV, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, HD, n_kv)).astype(np.float16)
    q = (3 * rng.standard_normal((T_, NH, HD))).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    cells = rng.permutation(n_kv)[:T_ * per - 4]
    for t in range(T_):
        own = cells[t::T_]
        mask[t, own] = np.where(np.arange(len(own)) % 3, 0, -0.5)
    hidden = np.setdiff1d(np.arange(n_kv), cells)
    k[hidden], v[:, :, hidden] = np.inf, np.nan

    def build(g):
        kc, vc = g.new(L.F16, [NKV * HD, n_kv], k.reshape(n_kv, -1)), g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        return H.ggml_mul_mat(g.ctx, vv, p)

    s0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)[0].reshape(NH, T_, HD)
    assert backend.stat("kernel_launches") - s0 <= 2
    qh = q.astype(np.float16).astype(np.float64)
    for t in range(T_):
        see = np.flatnonzero(mask[t] > -1)
        kt, vt = k[see].astype(np.float64), v[:, :, see].astype(np.float64)
        for h in range(NH):
            s = kt[:, h // G] @ qh[t, h] * HD ** -0.5 + mask[t, see]
            p = np.exp(s - s.max())
            p = (p / p.sum()).astype(np.float16).astype(np.float64)
            ref = vt[h // G] @ p
            # f32 sums; a probability next to a rounding boundary may round the other way: 2^-11 of it
            assert np.abs(got[h, t] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, (t, h)


def test_few_tokens_over_a_cache_beyond_32_bit_offsets(backend, H):
    """attn_nf.hip: cells 4 MiB apart, the last ones more than 2 GiB behind the first: one list and one launch, as of a dense cache."""
    rng = np.random.default_rng(5)
    HD, NKV, G, T_, n_kv, far = 128, 2, 4, 2, 768, 4 << 20
    NH = NKV * G
    k = rng.standard_normal((n_kv, NKV, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, HD, n_kv)).astype(np.float16)
    q = (3 * rng.standard_normal((T_, NH, HD))).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    mask[0, ::2] = mask[1, 1::2] = 0
    g = T.G(backend)
    try:
        base = g.new(L.F16, [far // 2, n_kv])
        vc = g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, base, HD, n_kv, NKV, far, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        out = H.ggml_mul_mat(g.ctx, vv, p)
        g.compute([out])
        for i in range(n_kv):
            row = np.ascontiguousarray(k[i])
            H.ggml_backend_tensor_set(base, row.ctypes.data, i * far, row.nbytes)
        s0 = backend.stat("kernel_launches")
        assert H.ggml_backend_graph_compute(backend.backend, g.gf) == 0
        assert backend.stat("kernel_launches") - s0 <= 2
        got = g.read(out).reshape(NH, T_, HD)
    finally:
        g.free()
    qh = q.astype(np.float16).astype(np.float64)
    for t in range(T_):
        see = np.flatnonzero(mask[t] == 0)
        for h in range(NH):
            s = k[see, h // G].astype(np.float64) @ qh[t, h] * HD ** -0.5
            p = np.exp(s - s.max())
            p = (p / p.sum()).astype(np.float16).astype(np.float64)
            ref = v[h // G][:, see].astype(np.float64) @ p
            # (as test_few_tokens_on_matrix_cores)
            assert np.abs(got[h, t] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, (t, h)


@pytest.mark.parametrize("T_,NKV,G,per,first", [(10, 8, 4, 71, 1), (16, 8, 5, 69, 0), (10, 8, 7, 75, 17), (12, 8, 8, 170, 7), (24, 8, 6, 33, 231)])
def test_few_tokens_over_runs_of_cells(backend, H, T_, NKV, G, per, first):
    """attn_nf.hip, whole rows: eight consecutive cells are one load wherever they begin, up to the last cell of the cache; a cell out of the row ends a run."""
    rng = np.random.default_rng(T_ + per + G)
    HD, NH = 128, NKV * G
    n_kv = (first + T_ * per + 255) // 256 * 256
    k = rng.standard_normal((n_kv, NKV, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, HD, n_kv)).astype(np.float16)
    q = (3 * rng.standard_normal((T_, NH, HD))).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    for t in range(T_):
        mask[t, first + t * per:first + (t + 1) * per] = 0
        mask[t, (7 * t) % n_kv] = 0
    mask[T_ - 1, n_kv - 9:] = 0

    def build(g):
        kc, vc = g.new(L.F16, [NKV * HD, n_kv], k.reshape(n_kv, -1)), g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        return H.ggml_mul_mat(g.ctx, vv, p)

    s0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)[0].reshape(NH, T_, HD)
    assert backend.stat("kernel_launches") - s0 <= 2
    qh = q.astype(np.float16).astype(np.float64)
    for t in range(T_):
        see = np.flatnonzero(mask[t] == 0)
        for h in range(NH):
            s = k[see, h // G].astype(np.float64) @ qh[t, h] * HD ** -0.5
            p = np.exp(s - s.max())
            p = (p / p.sum()).astype(np.float16).astype(np.float64)
            ref = v[h // G][:, see].astype(np.float64) @ p
            # (as test_few_tokens_on_matrix_cores)
            assert np.abs(got[h, t] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, (t, h)


# one launch over a short cache (attn_nf_once: 16 and 32 columns a workgroup, pairs and single heads, one, two and four blocks a wave) and two passes behind it; ragged batches, a last block in part
@pytest.mark.parametrize("HD,NH,NKV,T_,n_kv", [
    (128, 8, 2, 33, 40), (128, 8, 2, 77, 256), (128, 7, 1, 45, 264), (128, 4, 4, 129, 512), (128, 8, 2, 250, 520), (128, 14, 2, 130, 1024), (128, 4, 2, 257, 768),
    (64, 8, 1, 33, 48), (64, 8, 2, 128, 512), (64, 6, 2, 140, 1000), (64, 3, 1, 65, 256), (64, 8, 2, 70, 1032), (64, 4, 1, 300, 1024)])
@pytest.mark.parametrize("mask_kind", ["causal", "scattered"])
def test_prompt_over_a_short_cache(backend, H, HD, NH, NKV, T_, n_kv, mask_kind):
    """K.q -> SOFT_MAX -> V^T.p -> CONT of a prompt's batch; cells that no query sees hold infinities and NaN (whole blocks of 64 of them: such blocks are not multiplied), one query sees nothing: NaN.
    Against float64 with the chain's two f16 roundings, as test_few_tokens_on_matrix_cores."""
    rng = np.random.default_rng(HD + NH + T_ + n_kv)
    G = NH // NKV
    k = rng.standard_normal((n_kv, NKV, HD)).astype(np.float16)
    v = rng.standard_normal((NKV, HD, n_kv)).astype(np.float16)
    q = (2 * rng.standard_normal((T_, NH, HD))).astype(np.float32)
    mask = np.full((T_, n_kv), -np.inf, np.float32)
    for t in range(T_):
        if mask_kind == "causal":
            mask[t, :max(1, n_kv - T_ + t + 1 - 8)] = 0
        else:
            mask[t, rng.random(n_kv) < 0.2] = -0.5 * (t % 3)
            mask[t, t % 8] = 0
            if n_kv > 200:
                mask[t, 64:128] = -np.inf
    mask[T_ // 2] = -np.inf
    if mask_kind == "scattered" and n_kv > 200:
        k[64:128], v[:, :, 64:128] = np.inf, np.nan

    def build(g):
        kc, vc = g.new(L.F16, [NKV * HD, n_kv], k.reshape(n_kv, -1)), g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
        return H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, H.ggml_mul_mat(g.ctx, vv, p), 0, 2, 1, 3), HD * NH, T_)

    k0, c0 = backend.stat("kernel_launches"), backend.stat("nf_mma_chains")
    got = T.run_case(build, backend)[0].reshape(T_, NH, HD)
    launches = backend.stat("kernel_launches") - k0
    once = n_kv <= (1024 if HD == 64 or T_ <= 256 else 512)
    assert backend.stat("nf_mma_chains") - c0 == 1 and (launches == 1 if once else launches in (3, 4)), launches
    qh = q.astype(np.float16).astype(np.float64)
    for t in range(T_):
        see = np.flatnonzero(mask[t] > -1e30)
        if len(see) == 0:
            assert np.isnan(got[t]).all()
            continue
        kt, vt = k[see].astype(np.float64), v[:, :, see].astype(np.float64)
        for h in range(NH):
            s = kt[:, h // G] @ qh[t, h] * HD ** -0.5 + mask[t, see]
            p = np.exp(s - s.max())
            p = (p / p.sum()).astype(np.float16).astype(np.float64)
            ref = vt[h // G] @ p
            assert np.abs(got[t, h] - ref).max() <= 2e-3 * np.abs(ref).max() + 1e-5, (t, h)


# heads of 64: the sum of a row's weights is made in 64 bits, as SOFT_MAX makes it.  One weight of 1 and 31 of 2^-24.1 in the cells that one lane adds up (in 32 bits each of them is lost behind the 1), another
# cell's weight chosen so that the large probability lies 8e-7 of itself below a rounding boundary of f16: without the small ones it would round up
@pytest.mark.parametrize("NH,NKV,T_,n_kv", [(8, 2, 33, 1024), (3, 1, 40, 1024), (8, 2, 200, 1024), (6, 2, 130, 1000), (8, 2, 40, 2048), (8, 2, 300, 1032), (8, 1, 130, 4096)])
def test_sums_of_prompt_probabilities(backend, H, NH, NKV, T_, n_kv):
    HD = 64
    small = [1, 2, 3] + [8 * i + j for i in range(1, 8) for j in range(4)] if n_kv > 1024 else list(range(1, 8)) + [256 * i + j for i in range(1, 4) for j in range(8)]
    row = np.full(n_kv, -np.inf, np.float32)
    row[0], row[small] = 0, -16.7
    edge = 0.75 + 2.0 ** -12
    row[63] = np.log((1 + 8e-7) / edge - 1 - np.exp(row[small].astype(np.float64)).sum())
    p = 1 / np.exp(row.astype(np.float64)).sum()
    assert len(small) == 31 and 7e-7 < 1 - p / edge < 9e-7 and 3e-7 < p * (1 + 31 * p * np.exp(-16.7)) / edge - 1
    v = np.zeros((NKV, HD, n_kv), np.float16)
    v[:, :, 0] = 1 + np.arange(HD) % 2

    def build(g):
        kc, vc = g.new(L.F16, [NKV * HD, n_kv], np.ones((n_kv, NKV * HD), np.float16)), g.new(L.F16, [n_kv, NKV * HD], v.reshape(-1, n_kv))
        qp = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], np.zeros((T_, NH, HD), np.float32)), 0, 2, 1, 3)
        kv = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
        vv = H.ggml_view_3d(g.ctx, vc, n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], np.tile(row, (T_, 1))), HD ** -0.5, 0.0)
        return H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, H.ggml_mul_mat(g.ctx, vv, p), 0, 2, 1, 3), HD * NH, T_)

    c0 = backend.stat("nf_mma_chains")
    got = T.run_case(build, backend)[0].reshape(T_, NH, HD)
    assert backend.stat("nf_mma_chains") == c0 + 1
    assert np.array_equal(got, np.broadcast_to(np.float16(p).astype(np.float32) * v[0, :, 0].astype(np.float32), got.shape))


@pytest.mark.parametrize("recycled", [False, True])
@pytest.mark.parametrize("NH,NKV,T_", [(8, 2, 41), (8, 2, 160), (6, 2, 50)])
def test_prompt_over_a_short_cache_feeds_a_quantised_matrix(backend, H, NH, NKV, T_, recycled):
    """the same into a K-quant product: head pairs of a group leave as Q8_K blocks, an odd group's rows as the copy; only a Q8_K code next to a rounding boundary may differ from the graph run node by node"""
    rng = np.random.default_rng(NH + T_)
    HD, n_kv, N = 128, 256, 96
    k, v = rng.standard_normal((n_kv, NKV * HD)).astype(np.float16), rng.standard_normal((NKV * HD, n_kv)).astype(np.float16)
    wq, x = T.rand_weight(L.Q4_K, 256, NH * HD, rng), rng.standard_normal((T_, 256)).astype(np.float32)
    wo = T.rand_weight(L.Q4_K, NH * HD, N, rng)
    mask = np.where(np.arange(n_kv)[None, :] <= 30 + np.arange(T_)[:, None], 0, -np.inf).astype(np.float32)

    def run():
        g = T.G(backend)
        try:
            q = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [256, NH * HD], wq), g.new(L.F32, [256, T_], x))
            qp = H.ggml_permute(g.ctx, H.ggml_reshape_3d(g.ctx, q, HD, NH, T_), 0, 2, 1, 3)
            kv = H.ggml_view_3d(g.ctx, g.new(L.F16, [NKV * HD, n_kv], k), HD, n_kv, NKV, NKV * HD * 2, HD * 2, 0)
            vv = H.ggml_view_3d(g.ctx, g.new(L.F16, [n_kv, NKV * HD], v), n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
            p = H.ggml_soft_max_ext(g.ctx, H.ggml_mul_mat(g.ctx, kv, qp), g.new(L.F32, [n_kv, T_], mask), HD ** -0.5, 0.0)
            o = H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, H.ggml_mul_mat(g.ctx, vv, p), 0, 2, 1, 3), NH * HD, T_)
            r = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [NH * HD, N], wo), o)
            c0 = backend.stat("nf_mma_chains")
            out = g.compute([r], same_block=[(o, q)] if recycled else [])[0]
            return out, backend.stat("nf_mma_chains") - c0
        finally:
            g.free()

    got, chains = run()
    backend.set_option("fusion", 0)
    try:
        plain, plain_chains = run()
    finally:
        backend.set_option("fusion", 1)
    assert chains == 1 and plain_chains == 0
    assert T.nmse(got, plain) <= 1e-5
