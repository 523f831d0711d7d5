"""GPU parity at the shapes BASELINE.json names (Llama-3-8B Q4_K_M, TinyLlama-1.1B Q8_0, Qwen2-7B Q5_K/Q6_K, Llama-3-70B
Q4_K_M), all through the C-ABI against the CPU oracle.

Why this file exists: the op tests use small matrices, so the code the bench actually times —
k_mmvq_stream's multi-pass walk with its balanced tail (N > 4096, N % 4096 != 0: ffn gate/up N = 14336, output N = 128256,
Qwen2's 18944 / 152064), the 56- / 74- / 112-super-block rows of ffn_down, head_dim-128 attention over 8192 cells — never
ran in a test.  Here they do, and in the forms the decode graph uses them (norm prologue, SwiGLU pair, residual epilogue,
fused Q/K/V + rope + cache store).

Teacher forcing (test_layer_teacher_forced): a layer is evaluated node group by node group; every group — exactly the
launches of the decode path — is fed the ORACLE's values for its inputs, so no deviation can cascade from one group into the
next and the per-op gates apply to the real graph at the real shapes:
    quantised mat-vec chains (integer block sums exact, f32 accumulate order differs) ....... NMSE <= 1e-10
    f16 cache rows written by the fused Q/K/V launch .......................................... <= one f16 rounding (1e-6)
    FLASH_ATTN_EXT (the CPU accumulates V in f16, the kernel in f32) .......................... NMSE <= 1e-4, and closer to
                                                                                               float64 attention than the CPU is
"""
import os
import zlib

import numpy as np
import pytest

import harness as T
import llama_box_amd as L

pytestmark = pytest.mark.gpu

QNAME = {L.Q4_K: "q4_K", L.Q5_K: "q5_K", L.Q6_K: "q6_K", L.Q8_0: "q8_0"}
NT = T.host_threads()


def _seed(*key):
    return zlib.crc32(repr(key).encode())  # (hash() of a str is salted per process)


def _log(plog, msg):
    plog("[baseline-shapes] " + msg)


# ------------------------------------------------------------------------------------------------ (a) mat-vec at real shapes
# (tag, weight type, K, N, forms).  forms: plain = MUL_MAT; res = MUL_MAT + residual ADD; norm = RMS_NORM*w -> MUL_MAT (deferred
# into the mat-vec prologue); glu = RMS_NORM*w -> {gate, up} -> SwiGLU (one launch)
REAL_MV = [
    ("llama3-8b wo", L.Q4_K, 4096, 4096, ("plain", "res")),
    ("llama3-8b ffn_gate/up", L.Q4_K, 4096, 14336, ("plain", "norm", "glu")),
    ("llama3-8b ffn_down", L.Q4_K, 14336, 4096, ("plain", "res")),
    ("llama3-8b ffn_down (more-bits layer)", L.Q6_K, 14336, 4096, ("plain", "res")),
    ("llama3-8b output", L.Q6_K, 4096, 128256, ("norm",)),
    ("tinyllama ffn_gate/up", L.Q8_0, 2048, 5632, ("plain", "norm", "glu")),
    ("tinyllama ffn_down", L.Q8_0, 5632, 2048, ("plain", "res")),
    ("tinyllama output", L.Q8_0, 2048, 32000, ("norm",)),
    ("qwen2-7b ffn_gate/up", L.Q5_K, 3584, 18944, ("plain", "norm", "glu")),
    ("qwen2-7b ffn_down", L.Q6_K, 18944, 3584, ("plain", "res")),
    ("qwen2-7b wo", L.Q5_K, 3584, 3584, ("res",)),
    ("qwen2-7b output", L.Q6_K, 3584, 152064, ("norm",)),
    ("llama3-70b wo", L.Q4_K, 8192, 8192, ("res",)),
    ("llama3-70b ffn_gate/up", L.Q4_K, 8192, 28672, ("norm", "glu")),
    ("llama3-70b ffn_down", L.Q4_K, 28672, 8192, ("res",)),
    ("llama3-70b ffn_down (more-bits layer)", L.Q6_K, 28672, 8192, ("plain", "res")),
    ("llama3-70b attn_v", L.Q5_K, 8192, 1024, ("plain",)),
]
_MV_CASES = [(tag, qt, K, N, f) for tag, qt, K, N, forms in REAL_MV for f in forms]


@pytest.mark.parametrize("tag,qt,K,N,form", _MV_CASES, ids=[f"{t.replace(' ', '_')}-{QNAME[q]}-{f}" for t, q, _, _, f in _MV_CASES])
def test_mat_vec_real_shapes(backend, H, plog, tag, qt, K, N, form):
    rng = np.random.default_rng(_seed(K, N, qt, form))
    w = T.rand_weight(qt, K, N, rng)
    w2 = T.rand_weight(qt, K, N, rng) if form == "glu" else None
    x = (rng.standard_normal((1, K)) * rng.uniform(0.5, 2.0)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, K).astype(np.float32)
    r = rng.standard_normal((1, N)).astype(np.float32)

    def build(g):
        cur = g.new(L.F32, [K, 1], x)
        if form in ("norm", "glu"):
            cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, cur, 1e-5), g.new(L.F32, [K], nw))
        y = H.ggml_mul_mat(g.ctx, g.new(qt, [K, N], w), cur)
        if form == "glu":
            y = H.ggml_swiglu_split(g.ctx, y, H.ggml_mul_mat(g.ctx, g.new(qt, [K, N], w2), cur))
        if form == "res":
            y = H.ggml_add(g.ctx, y, g.new(L.F32, [N, 1], r))
        return y

    ref = T.run_case(build, "oracle", NT)
    k0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)
    launches = backend.stat("kernel_launches") - k0
    _log(plog, f"{tag} {QNAME[qt]} K={K} N={N} form={form}: {launches} launch(es)")
    assert launches == 1, f"{tag} {form}: expected the one fused launch of the decode path, got {launches}"
    T.compare(f"mat-vec {tag} {QNAME[qt]} K={K} N={N} {form}", got[0], ref[0], max_nmse=1e-10, log=plog)


# ------------------------------------------------------------------------------------------------ (b) one real layer, teacher-forced
class Spec:
    def __init__(self, name, E, FF, NH, NKV, HD, t_qk, t_v, t_o, t_gu, t_d, bias, neox, base, eps, n_past, n_ctx_train):
        self.__dict__.update(locals())


LAYERS = [
    # Llama-3-8B Q4_K_M: the plain layers (everything Q4_K) and the "more bits" layers (attn_v, ffn_down in Q6_K)
    Spec("llama3-8b q4_k_m layer (plain)", 4096, 14336, 32, 8, 128, L.Q4_K, L.Q4_K, L.Q4_K, L.Q4_K, L.Q4_K, False, False, 500000.0, 1e-5, 2063, 8192),
    Spec("llama3-8b q4_k_m layer (more bits)", 4096, 14336, 32, 8, 128, L.Q4_K, L.Q6_K, L.Q4_K, L.Q4_K, L.Q6_K, False, False, 500000.0, 1e-5, 2063, 8192),
    # Qwen2-7B, Q5_K / Q6_K mix, 8192 cells of context: NeoX rope, Q/K/V bias, 28/4 heads (7 per KV head)
    Spec("qwen2-7b q5_k/q6_k layer @8192", 3584, 18944, 28, 4, 128, L.Q5_K, L.Q6_K, L.Q5_K, L.Q5_K, L.Q6_K, True, True, 1000000.0, 1e-6, 8191, 32768),
    # Llama-3-70B Q4_K_M (config 4's model): attn_v in Q5_K in its plain layers
    Spec("llama3-70b q4_k_m layer", 8192, 28672, 64, 8, 128, L.Q4_K, L.Q5_K, L.Q4_K, L.Q4_K, L.Q6_K, False, False, 500000.0, 1e-5, 1030, 8192),
    # TinyLlama-1.1B Q8_0 (config 1's model): head_dim 64
    Spec("tinyllama-1.1b q8_0 layer", 2048, 5632, 32, 4, 64, L.Q8_0, L.Q8_0, L.Q8_0, L.Q8_0, L.Q8_0, False, False, 10000.0, 1e-5, 143, 2048),
    # ONE RANK of Llama-3-70B under --tensor-split 1,1,1,1,1,1,1,1 (engine_param.hpp:821-842, :902-916):
    # 8 Q heads on 1 KV head, wq 1024 x 8192, wk / wv 128 x 8192, wo's K slice 8192 x 1024, gate / up 3584 x 8192, ffn_down's K slice
    # 8192 x 3584 (14 super-blocks per row).  A rank's partial products carry the residual here, as the single-rank graph does; the
    # sum over ranks is tests/test_tp_* 's business.  Plain layers keep attn_v in Q5_K, the "more bits" layers have attn_v / ffn_down in Q6_K.
    Spec("llama3-70b q4_k_m TP8 rank shard (plain)", 8192, 3584, 8, 1, 128, L.Q4_K, L.Q5_K, L.Q4_K, L.Q4_K, L.Q4_K, False, False, 500000.0, 1e-5, 2063, 8192),
    Spec("llama3-70b q4_k_m TP8 rank shard (more bits)", 8192, 3584, 8, 1, 128, L.Q4_K, L.Q6_K, L.Q4_K, L.Q4_K, L.Q6_K, False, False, 500000.0, 1e-5, 2063, 8192),
]


def _attention_f64(q, kc, vc, n_kv, NH, NKV, HD):
    """Exact attention over cells [0, n_kv) in float64: q [NH, HD] f32 (already rotated; rounded to f16 first, as ggml-cpu's
    q_to_vec_dot and the kernel both do), caches [n_ctx, NKV*HD] f16."""
    q = q.astype(np.float16).astype(np.float64).reshape(NH, HD)
    k = kc[:n_kv].astype(np.float64).reshape(n_kv, NKV, HD)
    v = vc[:n_kv].astype(np.float64).reshape(n_kv, NKV, HD)
    g = NH // NKV
    out = np.empty((NH, HD))
    for h in range(NH):
        s = k[:, h // g, :] @ q[h] / np.sqrt(HD)
        p = np.exp(s - s.max())
        out[h] = (p / p.sum()) @ v[:, h // g, :]
    return out


@pytest.mark.parametrize("sp", LAYERS, ids=[s.name.replace(" ", "_") for s in LAYERS])
def test_layer_teacher_forced(backend, H, plog, sp):
    rng = np.random.default_rng(_seed(sp.name))
    E, FF, NH, NKV, HD = sp.E, sp.FF, sp.NH, sp.NKV, sp.HD
    EK = NKV * HD
    n_kv = (sp.n_past + 1 + 255) // 256 * 256  # cells the graph covers (llama_lite: used cells rounded up to 256)
    n_ctx = n_kv
    pos, slot = sp.n_past, sp.n_past
    mode = L.ROPE_NEOX if sp.neox else 0
    W = dict(wq=T.rand_weight(sp.t_qk, E, NH * HD, rng), wk=T.rand_weight(sp.t_qk, E, EK, rng), wv=T.rand_weight(sp.t_v, E, EK, rng),
             wo=T.rand_weight(sp.t_o, NH * HD, E, rng), wg=T.rand_weight(sp.t_gu, E, FF, rng), wu=T.rand_weight(sp.t_gu, E, FF, rng),
             wd=T.rand_weight(sp.t_d, FF, E, rng))
    nw1, nw2 = rng.uniform(0.5, 1.5, E).astype(np.float32), rng.uniform(0.5, 1.5, E).astype(np.float32)
    bq, bk, bv = (rng.standard_normal(n).astype(np.float32) * 0.1 for n in (NH * HD, EK, EK))
    x0 = rng.standard_normal((1, E)).astype(np.float32)
    kc0 = (rng.standard_normal((n_ctx, EK)) * 0.5).astype(np.float16)
    vc0 = (rng.standard_normal((n_ctx, EK)) * 0.5).astype(np.float16)
    mask = np.full((64, n_kv), -np.inf, np.float16)  # [n_kv, GGML_KQ_MASK_PAD] in ggml order
    mask[0, : sp.n_past + 1] = 0

    def rope(g, t, nh, tp):
        return H.ggml_rope_ext(g.ctx, H.ggml_reshape_3d(g.ctx, t, HD, nh, 1), tp, None, HD, mode, sp.n_ctx_train, sp.base, 1.0, 0.0, 1.0, 32.0, 1.0)

    # ---- the five node groups of a decode layer (= the launches of the decode path); `inp` holds the values a group reads
    def seg_qkv(g, inp):
        x = g.new(L.F32, [E, 1], inp["x"])
        cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, x, sp.eps), g.new(L.F32, [E], nw1))
        q = H.ggml_mul_mat(g.ctx, g.new(sp.t_qk, [E, NH * HD], W["wq"]), cur)
        k = H.ggml_mul_mat(g.ctx, g.new(sp.t_qk, [E, EK], W["wk"]), cur)
        v = H.ggml_mul_mat(g.ctx, g.new(sp.t_v, [E, EK], W["wv"]), cur)
        if sp.bias:
            q = H.ggml_add(g.ctx, q, g.new(L.F32, [NH * HD], bq))
            k = H.ggml_add(g.ctx, k, g.new(L.F32, [EK], bk))
            v = H.ggml_add(g.ctx, v, g.new(L.F32, [EK], bv))
        tp = g.new(L.I32, [1], np.array([pos], np.int32))
        idx = g.new(L.I64, [1], np.array([slot], np.int64))
        qr, kr = rope(g, q, NH, tp), rope(g, k, NKV, tp)
        v3 = H.ggml_reshape_3d(g.ctx, v, HD, NKV, 1)
        ks = H.ggml_set_rows(g.ctx, g.new(L.F16, [EK, n_ctx], inp["kc"]), H.ggml_reshape_2d(g.ctx, kr, EK, 1), idx)
        vs = H.ggml_set_rows(g.ctx, g.new(L.F16, [EK, n_ctx], inp["vc"]), H.ggml_reshape_2d(g.ctx, v3, EK, 1), idx)
        return dict(outs=[qr, ks, vs], first=[qr, kr, v3])

    def seg_attn(g, inp):
        qr = g.new(L.F32, [HD, NH, 1], inp["q_rope"])
        kc = g.new(L.F16, [EK, n_ctx], inp["kc"])
        vc = g.new(L.F16, [EK, n_ctx], inp["vc"])
        q = H.ggml_permute(g.ctx, qr, 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, EK * 2, HD * 2, 0)
        v = H.ggml_view_3d(g.ctx, vc, HD, n_kv, NKV, EK * 2, HD * 2, 0)
        fa = H.ggml_flash_attn_ext(g.ctx, q, k, v, g.new(L.F16, [n_kv, 64], mask), 1.0 / np.sqrt(HD), 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(fa, 10)
        return dict(outs=[fa], first=[])

    def seg_wo(g, inp):
        a = g.new(L.F32, [NH * HD, 1], inp["attn"])
        y = H.ggml_mul_mat(g.ctx, g.new(sp.t_o, [NH * HD, E], W["wo"]), a)
        return dict(outs=[H.ggml_add(g.ctx, y, g.new(L.F32, [E, 1], inp["x"]))], first=[])

    def seg_ffn(g, inp):
        f = g.new(L.F32, [E, 1], inp["ffn_inp"])
        cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, f, sp.eps), g.new(L.F32, [E], nw2))
        gate = H.ggml_mul_mat(g.ctx, g.new(sp.t_gu, [E, FF], W["wg"]), cur)
        up = H.ggml_mul_mat(g.ctx, g.new(sp.t_gu, [E, FF], W["wu"]), cur)
        return dict(outs=[H.ggml_swiglu_split(g.ctx, gate, up)], first=[])

    def seg_down(g, inp):
        a = g.new(L.F32, [FF, 1], inp["act"])
        y = H.ggml_mul_mat(g.ctx, g.new(sp.t_d, [FF, E], W["wd"]), a)
        return dict(outs=[H.ggml_add(g.ctx, y, g.new(L.F32, [E, 1], inp["ffn_inp"]))], first=[])

    def run(seg, target, inp):
        g = T.G(target)
        try:
            b = seg(g, inp)
            k0 = backend.stat("kernel_launches") if target != "oracle" else 0
            r = g.compute(b["outs"], NT, expand_first=b["first"])
            return r, (backend.stat("kernel_launches") - k0 if target != "oracle" else 0)
        finally:
            g.free()

    # ---- the oracle runs the layer end to end (its own outputs feed its next group), the GPU gets the oracle's values
    vals = {"x": x0, "kc": kc0, "vc": vc0}
    report = []
    (q_o, kc_o, vc_o), _ = run(seg_qkv, "oracle", vals)
    (q_g, kc_g, vc_g), n1 = run(seg_qkv, backend, vals)
    T.compare(f"{sp.name}: q_rope", q_g, q_o, max_nmse=1e-10, log=plog)
    for nm, a, b, c0 in (("k_cache", kc_g, kc_o, kc0), ("v_cache", vc_g, vc_o, vc0)):
        a32, b32 = np.asarray(a).astype(np.float32).reshape(n_ctx, EK), np.asarray(b).astype(np.float32).reshape(n_ctx, EK)
        T.compare(f"{sp.name}: {nm} new row", a32[slot], b32[slot], max_nmse=1e-6, log=plog)
        other = np.ones(n_ctx, bool)
        other[slot] = False
        assert np.array_equal(np.asarray(a).reshape(n_ctx, EK)[other], c0[other]), f"{nm}: rows other than the new one were touched"
    report.append(("qkv+rope+store", n1))

    vals.update(q_rope=q_o, kc=np.asarray(kc_o).reshape(n_ctx, EK), vc=np.asarray(vc_o).reshape(n_ctx, EK))
    (fa_o,), _ = run(seg_attn, "oracle", vals)
    (fa_g,), n2 = run(seg_attn, backend, vals)
    exact = _attention_f64(np.asarray(q_o), vals["kc"], vals["vc"], sp.n_past + 1, NH, NKV, HD)
    e_gpu, e_cpu = T.nmse(np.asarray(fa_g).reshape(NH, HD), exact), T.nmse(np.asarray(fa_o).reshape(NH, HD), exact)
    _log(plog, f"{sp.name}: attention vs float64: gpu nmse={e_gpu:.3e}, cpu oracle (f16 V accumulation) nmse={e_cpu:.3e}")
    # the CPU's f16 V accumulator loses precision with every cell (its distance from exact attention grows with n_kv: ~1e-5 at 2 k
    # cells, ~2e-4 at 8 k); the kernel must be (much) closer to exact attention than the CPU is, and no further from the CPU than
    # the CPU is from exact
    assert e_gpu <= 1e-9 and e_gpu <= e_cpu * 1.01 + 1e-12
    T.compare(f"{sp.name}: flash_attn n_kv={sp.n_past + 1} heads={NH}/{NKV} d={HD}", fa_g, fa_o, max_nmse=max(1e-4, 1.5 * e_cpu), log=plog)
    report.append(("flash_attn", n2))

    vals.update(attn=np.asarray(fa_o).reshape(1, NH * HD))
    (fi_o,), _ = run(seg_wo, "oracle", vals)
    (fi_g,), n3 = run(seg_wo, backend, vals)
    T.compare(f"{sp.name}: wo + residual (ffn_inp)", fi_g, fi_o, max_nmse=1e-10, log=plog)
    report.append(("wo+res", n3))

    vals.update(ffn_inp=np.asarray(fi_o).reshape(1, E))
    (act_o,), _ = run(seg_ffn, "oracle", vals)
    (act_g,), n4 = run(seg_ffn, backend, vals)
    T.compare(f"{sp.name}: norm -> gate/up -> swiglu", act_g, act_o, max_nmse=1e-10, log=plog)
    report.append(("gate/up/swiglu", n4))

    vals.update(act=np.asarray(act_o).reshape(1, FF))
    (lo_o,), _ = run(seg_down, "oracle", vals)
    (lo_g,), n5 = run(seg_down, backend, vals)
    T.compare(f"{sp.name}: ffn_down + residual (l_out)", lo_g, lo_o, max_nmse=1e-10, log=plog)
    report.append(("down+res", n5))
    _log(plog, f"{sp.name}: launches per group {report}")
    # the groups must be the fused launches the decode path (and the bench) runs, not node-by-node fallbacks
    # (qkv group: + the token's (cos, sin) table, which a whole-model graph launches once for all its layers)
    assert n1 == 2 and n3 == 1 and n4 == 1 and n5 == 1 and n2 <= 2, report


# ------------------------------------------------------------------------------------------------ (c) attention at 8192 cells
@pytest.mark.parametrize("NH,NKV,n_kv,n_vis", [(28, 4, 8192, 8192), (28, 4, 8192, 7000), (32, 8, 8192, 8192), (64, 8, 8192, 8100)])
def test_flash_attn_head_dim_128_at_8192(backend, H, plog, NH, NKV, n_kv, n_vis):
    rng = np.random.default_rng(NH * 31 + n_vis)
    HD, EK = 128, NKV * 128
    q = rng.standard_normal((1, NH, HD)).astype(np.float32)
    kc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    vc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    mask = np.full((64, n_kv), -np.inf, np.float16)
    mask[0, :n_vis] = 0

    def build(g):
        qq = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, 1], q), 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], kc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        v = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], vc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        fa = H.ggml_flash_attn_ext(g.ctx, qq, k, v, g.new(L.F16, [n_kv, 64], mask), 1.0 / np.sqrt(HD), 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(fa, 10)
        return fa

    ref = T.run_case(build, "oracle", NT)
    got = T.run_case(build, backend)
    exact = _attention_f64(q[0], kc, vc, n_vis, NH, NKV, HD)
    e, e_cpu = T.nmse(np.asarray(got[0]).reshape(NH, HD), exact), T.nmse(np.asarray(ref[0]).reshape(NH, HD), exact)
    _log(plog, f"flash_attn d=128 heads={NH}/{NKV} n_kv={n_kv} visible={n_vis}: vs float64 gpu nmse={e:.3e}, cpu oracle (f16 V accumulation) nmse={e_cpu:.3e}")
    assert e <= 1e-9 and e <= e_cpu
    # (at 8 k cells the CPU's own f16 accumulation error is ~2e-4: the gate against the CPU follows it)
    T.compare(f"flash_attn d=128 heads={NH}/{NKV} n_kv={n_kv} visible={n_vis}", got[0], ref[0], max_nmse=max(1e-4, 1.5 * e_cpu), log=plog)


# ------------------------------------------------------------------------------------------------ the non-flash attention chain at real shapes
# llama-box runs with -fa off unless asked (engine_param.hpp:772-779): K view . q -> SOFT_MAX(mask, scale) -> V^T view . p -> CONT, exactly as
# llama_lite / llm_build_llama build it.  Decode: two launches (grouped-head K.q, SOFT_MAX folded into V^T.p); a prompt chunk: the f16
# matrix-core kernels and the register-resident soft-max.  Gates are the per-op ones (the products are exact in f32, sums differ in order).
@pytest.mark.parametrize("NH,NKV,n_kv,n_vis,T_", [(32, 8, 2304, 2100, 1), (28, 4, 8192, 8000, 1), (64, 8, 4096, 4096, 1), (32, 8, 2304, 2304, 512), (28, 4, 1096, 1000, 300), (32, 8, 2304, 2000, 130), (32, 8, 7296, 7296, 32),
                                                  # small batches: one launch over the tokens' visible-cell lists (attn_nf.hip); 8 / 2 tokens take slices of the head dimensions
                                                  (28, 4, 2048, 2048, 8), (8, 8, 1024, 1024, 2), (32, 8, 512, 512, 16)])
def test_non_flash_attention_chain(backend, H, plog, NH, NKV, n_kv, n_vis, T_):
    rng = np.random.default_rng(NH * 17 + n_kv + T_)
    HD, EK = 128, NKV * 128
    q = rng.standard_normal((T_, NH, HD)).astype(np.float32)
    kc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    vt = (rng.standard_normal((EK, n_kv)) * 0.5).astype(np.float16)  # transposed V cache: [n_embd_v][n_ctx]
    TP = (T_ + 63) // 64 * 64
    mask = np.full((TP, n_kv), -np.inf, np.float16)
    if T_ == 1:
        mask[0, :n_vis] = 0
    elif T_ in (32, 8, 2):  # a -np batch: token t sees the cells of its own sequence (a prompt's run, then every T_-th cell)
        run = (n_kv // 2) // T_ // 4 * 4
        for t in range(T_):
            mask[t, t * run:(t + 1) * run] = 0
            mask[t, T_ * run + t::T_] = 0
    else:  # a prompt chunk at the end of the context (of the n_vis cells in use): causal
        for t in range(T_):
            mask[t, :n_vis - T_ + t + 1] = 0

    def build(g):
        qq = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], kc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        v = H.ggml_view_3d(g.ctx, g.new(L.F16, [n_kv, EK], vt), n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        kq = H.ggml_mul_mat(g.ctx, k, qq)
        mt = L.F32 if T_ in (8, 16, 512, 300, 130) else L.F16  # (llama.cpp's mask is f32 when flash attention is off; both are served)
        p = H.ggml_soft_max_ext(g.ctx, kq, g.new(mt, [n_kv, TP], mask.astype(np.float32) if mt == L.F32 else mask), 1.0 / np.sqrt(HD), 0.0)
        kqv = H.ggml_mul_mat(g.ctx, v, p)
        return H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, kqv, 0, 2, 1, 3), HD * NH, T_)

    ref = T.run_case(build, "oracle", NT)
    k0, c0 = backend.stat("kernel_launches"), backend.stat("nf_mma_chains")
    got = T.run_case(build, backend)
    launches = backend.stat("kernel_launches") - k0
    _log(plog, f"non-flash attention heads={NH}/{NKV} n_kv={n_kv} tokens={T_}: {launches} launches")
    # a prompt chunk with llama.cpp's f32 mask: the two-pass matrix-core form (tile states, row statistics, p.V, sum of the KV splits), not three dense launches
    assert backend.stat("nf_mma_chains") - c0 == (1 if T_ >= 33 else 0)
    # (the chain amplifies one effect: where a K.q sum differs from the CPU's double-accumulated one in its last bit, a probability can
    # round to the neighbouring f16 — 2^-11 of one weight; with a few hundred cells per row a single flip is ~3e-10 of the output)
    T.compare(f"non-flash attention heads={NH}/{NKV} n_kv={n_kv} tokens={T_}", got[0], ref[0], max_nmse=1e-9, log=plog)
    if T_ == 1:
        assert launches <= 3, launches  # K.q, SOFT_MAX + V^T.p, (CONT: a no-op copy for one token unless the allocator moved it)
    elif T_ <= 32:
        assert launches <= 3, launches  # list scan, the fused chain, CONT


def test_non_flash_list_chain_gate_follows_the_longest_row(backend, H, plog):
    """the fused K.q -> SOFT_MAX -> V^T.p launch keeps a token's first 1024 visible cells on chip and pushes longer
    rows through scratch memory (~100 us per layer).  The host used to know only the AVERAGE row (cache cells / tokens); since round 4 the
    backend notes every mask's longest row while the engine uploads it (set_tensor, tensor named as llama.cpp names it) — one 3000-cell
    sequence among three short ones now stays on the dense kernels although the average (825 cells) would have passed.  Same numbers either way."""
    NH, NKV, HD, n_kv, T_ = 32, 8, 128, 3300, 4
    n_kv = (n_kv + 255) // 256 * 256
    EK = NKV * HD
    rng = np.random.default_rng(77)
    q = rng.standard_normal((T_, NH, HD)).astype(np.float32)
    kc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    vt = (rng.standard_normal((EK, n_kv)) * 0.5).astype(np.float16)
    mask = np.full((64, n_kv), -np.inf, np.float32)
    mask[0, :3000] = 0
    for t in range(1, T_):
        mask[t, 3000 + 100 * (t - 1): 3000 + 100 * t] = 0

    def build(name):
        def b(g):
            qq = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
            k = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], kc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
            v = H.ggml_view_3d(g.ctx, g.new(L.F16, [n_kv, EK], vt), n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
            kq = H.ggml_mul_mat(g.ctx, k, qq)
            p = H.ggml_soft_max_ext(g.ctx, kq, g.new(L.F32, [n_kv, 64], mask, name=name), 1.0 / np.sqrt(HD), 0.0)
            kqv = H.ggml_mul_mat(g.ctx, v, p)
            return H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, kqv, 0, 2, 1, 3), HD * NH, T_)
        return b

    ref = T.run_case(build("KQ_mask"), "oracle", NT)
    res = {}
    for name in ("inp_anon", "KQ_mask"):  # (anonymous first: a mask the backend has no statistics for is judged by the average, as before)
        k0 = backend.stat("kernel_launches")
        got = T.run_case(build(name), backend)
        res[name] = (got[0], backend.stat("kernel_launches") - k0)
        T.compare(f"non-flash chain, one long row among short ones, mask named {name}", got[0], ref[0], max_nmse=1e-9, log=plog)
    _log(plog, f"non-flash list gate: launches with an anonymous mask {res['inp_anon'][1]} (fused over lists, long row through scratch), with llama.cpp's mask name {res['KQ_mask'][1]} (dense kernels)")
    assert res["inp_anon"][1] <= 2 and res["KQ_mask"][1] >= 3, (res["inp_anon"][1], res["KQ_mask"][1])


@pytest.mark.parametrize("NH,NKV,n_kv,T_,wt", [(32, 8, 7296, 32, L.Q4_K), (32, 8, 512, 16, L.Q6_K), (32, 8, 1024, 24, L.Q6_K), (28, 4, 2048, 32, L.Q5_K)])
def test_non_flash_attention_chain_into_wo(backend, H, plog, NH, NKV, n_kv, T_, wt):
    """The -np decode step of llama-box's default (non-flash) path up to the attention output projection: K.q -> SOFT_MAX -> V^T.p -> CONT ->
    wo.  When the copy is read only by quantised mat-muls, the list kernel leaves the rows as Q8_K blocks (two heads per block) in the
    activation scratch: no f32 rows, no quantiser launch.  Equal to the oracle within the mat-mul gate, and to the execution with the
    f32 rows + quantiser launch (prologue = 0) bit for bit — same sums, same quantiser arithmetic."""
    rng = np.random.default_rng(NH * 19 + n_kv + T_ + wt)
    HD, EK, E = 128, NKV * 128, NH * 128
    q = rng.standard_normal((T_, NH, HD)).astype(np.float32)
    kc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    vt = (rng.standard_normal((EK, n_kv)) * 0.5).astype(np.float16)
    wo = T.rand_weight(wt, E, 512, rng)
    TP = (T_ + 63) // 64 * 64
    mask = np.full((TP, n_kv), -np.inf, np.float32)
    run_ = (n_kv // 2) // T_ // 4 * 4
    for t in range(T_):
        mask[t, t * run_:(t + 1) * run_] = 0
        mask[t, T_ * run_ + t::T_] = 0

    def build(g):
        qq = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, T_], q), 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], kc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        v = H.ggml_view_3d(g.ctx, g.new(L.F16, [n_kv, EK], vt), n_kv, HD, NKV, n_kv * 2, n_kv * 2 * HD, 0)
        kq = H.ggml_mul_mat(g.ctx, k, qq)
        p = H.ggml_soft_max_ext(g.ctx, kq, g.new(L.F32, [n_kv, TP], mask), 1.0 / np.sqrt(HD), 0.0)
        kqv = H.ggml_mul_mat(g.ctx, v, p)
        cur = H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, kqv, 0, 2, 1, 3), HD * NH, T_)
        return H.ggml_mul_mat(g.ctx, g.new(wt, [E, 512], wo), cur)

    ref = T.run_case(build, "oracle", NT)
    k0 = backend.stat("kernel_launches")
    got = T.run_case(build, backend)
    launches = backend.stat("kernel_launches") - k0
    backend.set_option("prologue", 0)
    try:
        k1 = backend.stat("kernel_launches")
        plain = T.run_case(build, backend)
        launches_plain = backend.stat("kernel_launches") - k1
    finally:
        backend.set_option("prologue", 1)
    _log(plog, f"non-flash attention -> wo heads={NH}/{NKV} n_kv={n_kv} tokens={T_} wo={QNAME[wt]}: {launches} launches, {launches_plain} with the f32 rows + quantiser")
    G = NH // NKV
    # (Q8_K blocks are head pairs of whole rows: an even group size, and one workgroup per (token, KV head) — with fewer than 192 of those
    # the kernel slices the head dimensions to fill the chip and the rows leave as f32)
    handed_over = G % 2 == 0 and T_ * NKV >= 192
    assert launches == launches_plain - (1 if handed_over else 0), (launches, launches_plain)
    # (the attention's own rounding flips — see test_non_flash_attention_chain — pass through the 8-bit activation quantiser: ~1e-6 of the output)
    T.compare(f"non-flash attention -> wo heads={NH}/{NKV} n_kv={n_kv} tokens={T_} wo={QNAME[wt]}", got[0], ref[0], max_nmse=5e-6, log=plog)
    assert np.array_equal(np.asarray(got[0]), np.asarray(plain[0])), "Q8_K hand-off and f32 rows + quantiser differ"


# ------------------------------------------------------------------------------------------------ split graphs
def test_split_graph_keeps_tensors_read_by_another_split(backend, H, plog):
    """ggml_backend_sched hands a backend ONE split (a ggml_graph_view).  A tensor whose other reader sits in the next split
    must be written even if every reader inside this split could have absorbed it: RMS_NORM*w feeding wq here and wk in the
    next split; gate/up results that a later split reads next to the SwiGLU; a projection read behind its residual ADD."""
    rng = np.random.default_rng(77)
    E, N = 1024, 512
    x = rng.standard_normal((1, E)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, E).astype(np.float32)
    w1, w2, w3 = (T.rand_weight(L.Q4_K, E, N, rng) for _ in range(3))
    r = rng.standard_normal((1, N)).astype(np.float32)

    def build(g):
        cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, g.new(L.F32, [E, 1], x), 1e-5), g.new(L.F32, [E], nw))
        a = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [E, N], w1), cur)          # split 1: norm, mul, mm(w1), add
        a_res = H.ggml_add(g.ctx, a, g.new(L.F32, [N, 1], r))
        b = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [E, N], w2), cur)          # split 2: reads `cur` and `a` again
        c = H.ggml_mul_mat(g.ctx, g.new(L.Q4_K, [E, N], w3), cur)
        glu = H.ggml_swiglu_split(g.ctx, b, c)
        both = H.ggml_add(g.ctx, glu, a)
        return g, [a_res, both]

    def run(target, cuts):
        g = T.G(target)
        try:
            _, outs = build(g)
            return g.compute(outs, 4, cuts=cuts)
        finally:
            g.free()

    ref = run("oracle", None)
    whole = run(backend, None)
    for cuts in ([4], [3], [2], [4, 6], [3, 5, 7]):
        got = run(backend, cuts)
        for nm, a, b, c in zip(("mm+residual", "swiglu + earlier projection"), got, ref, whole):
            T.compare(f"split graph cuts={cuts}: {nm}", a, b, max_nmse=1e-10, log=plog)
            T.compare(f"split graph cuts={cuts}: {nm} vs unsplit", a, c, max_nmse=1e-12, log=plog)


def test_deferred_norm_result_is_still_written(backend, H, plog):
    """result_norm / t_embd: llama.cpp reads the final RMS_NORM*w from the host although only the lm_head consumes it in the
    graph and the tensor is not flagged as an output.  The norm is folded into the mat-vec prologue — and written anyway."""
    rng = np.random.default_rng(5)
    E, N = 2048, 1000
    x = rng.standard_normal((1, E)).astype(np.float32)
    nw = rng.uniform(0.5, 1.5, E).astype(np.float32)
    w = T.rand_weight(L.Q6_K, E, N, rng)
    res = {}
    for target in ("oracle", backend):
        g = T.G(target)
        try:
            m = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, g.new(L.F32, [E, 1], x), 1e-5), g.new(L.F32, [E], nw))
            y = H.ggml_mul_mat(g.ctx, g.new(L.Q6_K, [E, N], w), m)
            k0 = backend.stat("kernel_launches")
            out = g.compute([y], 4)
            launches = backend.stat("kernel_launches") - k0
            res[target == "oracle"] = (out[0], g.read(m), launches)  # m is NOT an output of the graph
        finally:
            g.free()
    assert res[False][2] == 1, "norm was not folded into the mat-vec launch"
    T.compare("lm_head over deferred norm", res[False][0], res[True][0], max_nmse=1e-10, log=plog)
    T.compare("result_norm read behind the fused launch", res[False][1], res[True][1], max_nmse=1e-12, log=plog)


# ------------------------------------------------------------------------------------------------ attention merged in wo's prologue
@pytest.mark.parametrize("NH,NKV,n_kv,n_vis,wt", [(32, 8, 2304, 2100, L.Q4_K), (32, 8, 2304, 2304, L.Q6_K), (28, 4, 8192, 8000, L.Q5_K), (64, 8, 1280, 1031, L.Q4_K),
                                                   (32, 8, 256, 17, L.Q4_K), (8, 4, 4352, 4300, L.Q8_0), (32, 8, 33 * 256, 8400, L.Q4_K)])
def test_decode_attention_merged_in_wo_prologue(backend, H, plog, NH, NKV, n_kv, n_vis, wt):
    """One decode token: FLASH_ATTN_EXT -> reshape -> wo MUL_MAT -> + residual, with option fa_wo = 1: the attention runs as a few
    fat splits (8-wave workgroups) and the merge of their partial records is the prologue of the wo mat-vec: two launches, no
    combine pass.  Gates: the
    attention tensor itself (still written, for any other reader) like every FLASH_ATTN_EXT; the mat-vec result against the
    oracle fed the ORACLE's attention within the f16-accumulation band of the CPU's attention, and against the unfused GPU path."""
    rng = np.random.default_rng(_seed(NH, NKV, n_kv, wt))
    HD, EK, E = 128, NKV * 128, NH * 128
    q = rng.standard_normal((1, NH, HD)).astype(np.float32)
    kc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    vc = (rng.standard_normal((n_kv, EK)) * 0.5).astype(np.float16)
    mask = np.full((64, n_kv), -np.inf, np.float16)
    mask[0, :n_vis] = 0
    wo = T.rand_weight(wt, E, E, rng)
    res = rng.standard_normal((1, E)).astype(np.float32)

    def build(g):
        qq = H.ggml_permute(g.ctx, g.new(L.F32, [HD, NH, 1], q), 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], kc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        v = H.ggml_view_3d(g.ctx, g.new(L.F16, [EK, n_kv], vc), HD, n_kv, NKV, EK * 2, HD * 2, 0)
        fa = H.ggml_flash_attn_ext(g.ctx, qq, k, v, g.new(L.F16, [n_kv, 64], mask), 1.0 / np.sqrt(HD), 0.0, 0.0)
        H.ggml_flash_attn_ext_set_prec(fa, 10)
        y = H.ggml_mul_mat(g.ctx, g.new(wt, [E, E], wo), H.ggml_reshape_2d(g.ctx, fa, E, 1))
        return fa, H.ggml_add(g.ctx, y, g.new(L.F32, [E, 1], res))

    def run(target):
        g = T.G(target)
        try:
            fa, out = build(g)
            k0 = backend.stat("kernel_launches")
            r = g.compute([out], NT)
            return r[0], g.read(fa), backend.stat("kernel_launches") - k0
        finally:
            g.free()

    y_o, fa_o, _ = run("oracle")
    backend.set_option("fa_splits", 4 if n_kv <= 512 else 0)  # (few cells are attended in one pass otherwise: nothing to merge)
    try:
        y_u, fa_u, launches_u = run(backend)
    finally:
        backend.set_option("fa_splits", 0)
    backend.set_option("fa_wo", 1)  # (off by default: measured slower than thin splits + combine — DESIGN.md §4)
    try:
        y_g, fa_g, launches = run(backend)
    finally:
        backend.set_option("fa_wo", 0)
    _log(plog, f"attention->wo heads={NH}/{NKV} n_kv={n_kv} visible={n_vis} wo={QNAME[wt]}: {launches} launches merged, {launches_u} unmerged")
    assert launches == 2 and launches_u == 3
    exact = _attention_f64(q[0], kc, vc, n_vis, NH, NKV, HD)
    e_gpu, e_cpu = T.nmse(np.asarray(fa_g).reshape(NH, HD), exact), T.nmse(np.asarray(fa_o).reshape(NH, HD), exact)
    assert e_gpu <= 1e-9 and e_gpu <= e_cpu  # the attention tensor left behind by the merged path
    T.compare(f"attention->wo merged: attention tensor heads={NH}/{NKV} n_kv={n_kv}", fa_g, fa_u, max_nmse=1e-11, log=plog)
    # mat-vec result: the merged and the unmerged GPU paths see attention values that differ by f32 summation order only
    T.compare(f"attention->wo merged vs unmerged heads={NH}/{NKV} n_kv={n_kv} wo={QNAME[wt]}", y_g, y_u, max_nmse=1e-6, log=plog)
    T.compare(f"attention->wo merged vs oracle heads={NH}/{NKV} n_kv={n_kv} wo={QNAME[wt]}", y_g, y_o, max_nmse=max(2e-4, 3.0 * e_cpu), log=plog)


# ------------------------------------------------------------------------------------------------ (d) one real layer on a BATCH, teacher-forced
# the kernels the -np 32 and prefill bench lines time (k_mmq_skinny[_tp], k_mmq_wide, k_mmq_i8,
# k_rope_qk_store / the rope epilogue, k_swiglu_q8_K, list attention, k_fattn_mma) ran in tests only at small shapes.  Here every node
# group of a REAL layer is evaluated on a batch — 32 sequences of a continuous-batching decode step over a unified cache (config 3;
# reference call site httpserver.hpp:3539-3623: one llama_decode over every slot's next token), and a 512-token prompt micro-batch
# (config 2, -b/-ub: engine_param.hpp:1181,:1190) — each group fed the ORACLE's inputs, same gates as the one-token test above, and
# which kernel served each mat-mul is asserted from the backend's counters.
def _np32_layout(M, R, D):
    """Unified cache of a -np step: sequence s owns prompt cells [s*R, (s+1)*R) and the decode cells M*R + d*M + s (d < D); the token
    of this step goes into its d = D-1 cell.  Returns (n_kv, slot[M], pos[M], visible[M, n_kv])."""
    n_kv = M * R + D * M
    slot = np.array([M * R + (D - 1) * M + s for s in range(M)], np.int64)
    pos = np.full(M, R + D - 1, np.int32)
    vis = np.zeros((M, n_kv), bool)
    for s in range(M):
        vis[s, s * R:(s + 1) * R] = True
        vis[s, M * R + s::M] = True
    return n_kv, slot, pos, vis


def _prefill_layout(M, n_past):
    n_kv = n_past + M
    slot = np.arange(n_past, n_past + M, dtype=np.int64)
    pos = np.arange(n_past, n_past + M, dtype=np.int32)
    vis = np.tril(np.ones((M, n_kv), bool), n_past)
    return n_kv, slot, pos, vis


def _draft_layout(S, R, D, n_draft):
    """A step that verifies drafts (llama-box speculative decoding: httpserver.hpp:4042-4069 batches every slot's sampled token plus its
    n_draft draft tokens, :4696-4768 verifies them): S sequences, each with R prompt cells and D - 1 earlier decode cells (interleaved as
    continuous batching leaves them), and 1 + n_draft NEW consecutive tokens per sequence in this batch; token j of a sequence sees the
    sequence's older cells and the batch's tokens 0..j of the same sequence.  Returns (n_kv, slot[M], pos[M], visible[M, n_kv])."""
    T1 = 1 + n_draft
    M = S * T1
    base = S * R + (D - 1) * S
    n_kv = (base + M + 255) // 256 * 256
    slot = np.array([base + s * T1 + j for s in range(S) for j in range(T1)], np.int64)
    pos = np.array([R + D - 1 + j for s in range(S) for j in range(T1)], np.int32)
    vis = np.zeros((M, n_kv), bool)
    for s in range(S):
        for j in range(T1):
            t = s * T1 + j
            vis[t, s * R:(s + 1) * R] = True
            vis[t, S * R + s:base:S] = True
            vis[t, base + s * T1:base + s * T1 + j + 1] = True
    return n_kv, slot, pos, vis


# mode -> (M, layout): "np32" / "pf512" are BASELINE configs 3 / 2; the rest are the speculative-decoding shapes of SURVEY §8 f4
# a -np 32 step with 1 / 4 drafts per slot (M = 64 / 160 — between the skinny kernels' 32 columns and the 512 the
# wide form was tuned on) and ONE sequence verifying 8 / 16 drafts (M = 9 / 17)
BATCH_MODES = {
    "np32": lambda: (32,) + _np32_layout(32, 64, 8),            # 2304 cells
    "pf512": lambda: (512,) + _prefill_layout(512, 1792),       # 2304 cells, the last micro-batch of a 2304-token context
    "np32d1": lambda: (64,) + _draft_layout(32, 64, 7, 1),      # 2304 cells
    "np32d4": lambda: (160,) + _draft_layout(32, 64, 4, 4),     # 2304 cells
    "sd8": lambda: (9,) + _draft_layout(1, 2288, 8, 8),         # 2304 cells
    "sd16": lambda: (17,) + _draft_layout(1, 2280, 8, 16),      # 2304 cells
}
BATCH_CASES = [
    # (layer spec index, mode, flash attention)
    (0, "np32", 1), (0, "np32", 0), (1, "np32", 1), (2, "np32", 1), (2, "np32", 0),
    (0, "pf512", 1), (0, "pf512", 0), (1, "pf512", 1), (2, "pf512", 1),
    # config 4: one TP8 rank of Llama-3-70B at M = 32 and M = 512 (M = 1 is test_layer_teacher_forced)
    (5, "np32", 1), (6, "np32", 1), (5, "pf512", 1), (6, "pf512", 1), (6, "np32", 0),
    # speculative-decoding shapes: Llama-3-8B plain / more-bits layers, flash and non-flash, and a TP8 rank
    (0, "np32d1", 1), (1, "np32d4", 1), (0, "np32d4", 0), (0, "sd8", 1), (1, "sd16", 1), (1, "sd8", 0), (6, "np32d4", 1), (5, "sd16", 1),
]


@pytest.mark.parametrize("li,mode,fa", BATCH_CASES, ids=[f"{LAYERS[li].name.replace(' ', '_')}-{m}-fa{f}" for li, m, f in BATCH_CASES])
def test_layer_teacher_forced_batch(backend, H, plog, li, mode, fa):
    sp = LAYERS[li]
    rng = np.random.default_rng(_seed(sp.name, mode, fa))
    E, FF, NH, NKV, HD = sp.E, sp.FF, sp.NH, sp.NKV, sp.HD
    EK = NKV * HD
    M, n_kv, slot, pos, vis = BATCH_MODES[mode]()
    assert n_kv % 256 == 0
    n_ctx = n_kv
    MP = (M + 63) // 64 * 64
    rope_mode = L.ROPE_NEOX if sp.neox else 0
    W = dict(wq=T.rand_weight(sp.t_qk, E, NH * HD, rng), wk=T.rand_weight(sp.t_qk, E, EK, rng), wv=T.rand_weight(sp.t_v, E, EK, rng),
             wo=T.rand_weight(sp.t_o, NH * HD, E, rng), wg=T.rand_weight(sp.t_gu, E, FF, rng), wu=T.rand_weight(sp.t_gu, E, FF, rng),
             wd=T.rand_weight(sp.t_d, FF, E, rng))
    nw1, nw2 = rng.uniform(0.5, 1.5, E).astype(np.float32), rng.uniform(0.5, 1.5, E).astype(np.float32)
    bq, bk, bv = (rng.standard_normal(n).astype(np.float32) * 0.1 for n in (NH * HD, EK, EK))
    x0 = (rng.standard_normal((M, E)) * rng.uniform(0.5, 2.0, (M, 1))).astype(np.float32)
    kc0 = (rng.standard_normal((n_ctx, EK)) * 0.5).astype(np.float16)
    vc0 = (rng.standard_normal((n_ctx, EK)) * 0.5).astype(np.float16)  # row-major [cell][EK]; the non-flash graph holds its transpose
    mask16 = np.full((MP, n_kv), -np.inf, np.float16)
    mask16[:M][vis] = 0
    v_idx = (np.arange(EK, dtype=np.int64)[None, :] * n_ctx + slot[:, None]).reshape(-1)  # llama.cpp's v_idxs: element j of token t -> j * n_ctx + cell

    def rope(g, t, nh, tp):
        return H.ggml_rope_ext(g.ctx, H.ggml_reshape_3d(g.ctx, t, HD, nh, M), tp, None, HD, rope_mode, sp.n_ctx_train, sp.base, 1.0, 0.0, 1.0, 32.0, 1.0)

    def v_cache_tensor(g, vc):  # [n_ctx, EK] values -> the graph's cache tensor
        if fa:
            return g.new(L.F16, [EK, n_ctx], vc)
        return g.new(L.F16, [n_ctx, EK], np.ascontiguousarray(vc.T))

    def seg_qkv(g, inp):
        x = g.new(L.F32, [E, M], inp["x"])
        cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, x, sp.eps), g.new(L.F32, [E], nw1))
        q = H.ggml_mul_mat(g.ctx, g.new(sp.t_qk, [E, NH * HD], W["wq"]), cur)
        if sp.bias:
            q = H.ggml_add(g.ctx, q, g.new(L.F32, [NH * HD], bq))
        k = H.ggml_mul_mat(g.ctx, g.new(sp.t_qk, [E, EK], W["wk"]), cur)
        if sp.bias:
            k = H.ggml_add(g.ctx, k, g.new(L.F32, [EK], bk))
        v = H.ggml_mul_mat(g.ctx, g.new(sp.t_v, [E, EK], W["wv"]), cur)
        if sp.bias:
            v = H.ggml_add(g.ctx, v, g.new(L.F32, [EK], bv))
        tp = g.new(L.I32, [M], pos)
        idx = g.new(L.I64, [M], slot)
        qr, kr = rope(g, q, NH, tp), rope(g, k, NKV, tp)
        v3 = H.ggml_reshape_3d(g.ctx, v, HD, NKV, M)
        ks = H.ggml_set_rows(g.ctx, g.new(L.F16, [EK, n_ctx], inp["kc"]), H.ggml_reshape_2d(g.ctx, kr, EK, M), idx)
        vct = v_cache_tensor(g, inp["vc"])
        if fa:
            vs = H.ggml_set_rows(g.ctx, vct, H.ggml_reshape_2d(g.ctx, v3, EK, M), idx)
        else:
            vs = H.ggml_set_rows(g.ctx, H.ggml_reshape_2d(g.ctx, vct, 1, n_ctx * EK), H.ggml_reshape_2d(g.ctx, v3, 1, M * EK), g.new(L.I64, [M * EK], v_idx))
        return dict(outs=[qr, ks, vs], first=[qr, kr, v3])

    def seg_attn(g, inp):
        qr = g.new(L.F32, [HD, NH, M], inp["q_rope"])
        kc = g.new(L.F16, [EK, n_ctx], inp["kc"])
        vct = v_cache_tensor(g, inp["vc"])
        q = H.ggml_permute(g.ctx, qr, 0, 2, 1, 3)
        k = H.ggml_view_3d(g.ctx, kc, HD, n_kv, NKV, EK * 2, HD * 2, 0)
        if fa:
            v = H.ggml_view_3d(g.ctx, vct, HD, n_kv, NKV, EK * 2, HD * 2, 0)
            out = H.ggml_flash_attn_ext(g.ctx, q, k, v, g.new(L.F16, [n_kv, MP], mask16, name="KQ_mask"), 1.0 / np.sqrt(HD), 0.0, 0.0)  # (llama.cpp's name for it)
            H.ggml_flash_attn_ext_set_prec(out, 10)
            out = H.ggml_reshape_2d(g.ctx, out, HD * NH, M)
        else:
            v = H.ggml_view_3d(g.ctx, vct, n_kv, HD, NKV, n_ctx * 2, n_ctx * 2 * HD, 0)
            kq = H.ggml_mul_mat(g.ctx, k, q)
            p = H.ggml_soft_max_ext(g.ctx, kq, g.new(L.F32, [n_kv, MP], mask16.astype(np.float32), name="KQ_mask"), 1.0 / np.sqrt(HD), 0.0)
            kqv = H.ggml_mul_mat(g.ctx, v, p)
            out = H.ggml_cont_2d(g.ctx, H.ggml_permute(g.ctx, kqv, 0, 2, 1, 3), HD * NH, M)
        return dict(outs=[out], first=[])

    def seg_wo(g, inp):
        a = g.new(L.F32, [NH * HD, M], inp["attn"])
        y = H.ggml_mul_mat(g.ctx, g.new(sp.t_o, [NH * HD, E], W["wo"]), a)
        return dict(outs=[H.ggml_add(g.ctx, y, g.new(L.F32, [E, M], inp["x"]))], first=[])

    def seg_ffn(g, inp):
        f = g.new(L.F32, [E, M], inp["ffn_inp"])
        cur = H.ggml_mul(g.ctx, H.ggml_rms_norm(g.ctx, f, sp.eps), g.new(L.F32, [E], nw2))
        gate = H.ggml_mul_mat(g.ctx, g.new(sp.t_gu, [E, FF], W["wg"]), cur)
        up = H.ggml_mul_mat(g.ctx, g.new(sp.t_gu, [E, FF], W["wu"]), cur)
        return dict(outs=[H.ggml_swiglu_split(g.ctx, gate, up)], first=[])

    def seg_down(g, inp):
        a = g.new(L.F32, [FF, M], inp["act"])
        y = H.ggml_mul_mat(g.ctx, g.new(sp.t_d, [FF, E], W["wd"]), a)
        return dict(outs=[H.ggml_add(g.ctx, y, g.new(L.F32, [E, M], inp["ffn_inp"]))], first=[])

    COUNTERS = ("kernel_launches", "skinny_launches", "wide_launches", "wide_few_launches", "tiled_launches", "rope_epilogues", "fa_list_launches")

    def run(seg, target, inp):
        g = T.G(target)
        try:
            b = seg(g, inp)
            c0 = {k: backend.stat(k) for k in COUNTERS} if target != "oracle" else None
            r = g.compute(b["outs"], NT, expand_first=b["first"])
            return r, ({k: backend.stat(k) - c0[k] for k in COUNTERS} if c0 else None)
        finally:
            g.free()

    def served(cnt, wtypes, group):
        """which kernel ran the group's quantised mat-muls: asserted, so that a silent fall-back to a slower (or untested) kernel fails here"""
        _log(plog, f"{sp.name} {mode} fa={fa}: {group}: {cnt}")
        if cnt is None:  # (the oracle target has no counters)
            return
        if M <= 32:
            assert cnt["skinny_launches"] >= 1 and cnt["wide_launches"] == 0 and cnt["tiled_launches"] == 0, (group, cnt)
        elif mode == "pf512" and li < 5:
            kq = [t for t in wtypes if t in (L.Q4_K, L.Q5_K)]
            if kq:
                assert cnt["wide_launches"] >= 1, (group, cnt)
            if L.Q6_K in wtypes:
                assert cnt["tiled_launches"] >= 1, (group, cnt)
            assert cnt["skinny_launches"] == 0, (group, cnt)
        else:
            # 33 .. 160 columns, or a rank's narrow shards: a wide form where it applies, the tiled int8 GEMM otherwise — never the 32-column skinny kernel, never a column-by-column mat-vec fall-back (one launch per matrix group at most,
            # + split-K reduce / quantiser launches)
            assert cnt["skinny_launches"] == 0 and cnt["wide_launches"] + cnt["tiled_launches"] >= 1, (group, cnt)
            if L.Q6_K in wtypes:  # (up to 384 columns: the wide form with K slices, but for 8192 x 3584 x 160, which would be a second round of it for a few items)
                tiled = M > 384 or (group.startswith("ffn_down") and (FF, E, M) == (3584, 8192, 160))
                assert cnt["tiled_launches" if tiled else "wide_few_launches"] >= 1, (group, cnt)
            assert cnt["kernel_launches"] <= 12, (group, cnt)

    tag = f"{sp.name} [{mode}, {M} tokens, n_kv {n_kv}, fa={fa}]"
    vals = {"x": x0, "kc": kc0, "vc": vc0}
    (q_o, kc_o, vc_o), _ = run(seg_qkv, "oracle", vals)
    (q_g, kc_g, vc_g), c1 = run(seg_qkv, backend, vals)
    served(c1, (sp.t_qk, sp.t_v), "qkv + rope + stores")
    T.compare(f"{tag}: q_rope", q_g, q_o, max_nmse=1e-10, log=plog)

    def cache_rows(a, transposed):  # -> float32 [n_ctx, EK]
        a = np.asarray(a)
        return (a.reshape(EK, n_ctx).T if transposed else a.reshape(n_ctx, EK)).astype(np.float32)

    other = np.ones(n_ctx, bool)
    other[slot] = False
    for nm, a, b, c0_, tr in (("k_cache", kc_g, kc_o, kc0, False), ("v_cache", vc_g, vc_o, vc0, not fa)):
        a32, b32 = cache_rows(a, tr), cache_rows(b, tr)
        T.compare(f"{tag}: {nm} new rows", a32[slot], b32[slot], max_nmse=1e-6, log=plog)
        assert np.array_equal(a32[other], c0_.astype(np.float32)[other]), f"{nm}: cells other than the batch's were touched"

    kc_n = cache_rows(kc_o, False).astype(np.float16)
    vc_n = cache_rows(vc_o, not fa).astype(np.float16)
    vals.update(q_rope=q_o, kc=kc_n, vc=vc_n)
    (at_o,), _ = run(seg_attn, "oracle", vals)
    (at_g,), c2 = run(seg_attn, backend, vals)
    _log(plog, f"{tag}: attention: {c2}")
    if fa:
        # which attention kernel: per-token position lists for up to 32 tokens and — the mask having passed through set_tensor under llama.cpp's
        # name, so that the backend knows how little of the cache a token sees — for the draft-verification batches of 64 / 160 tokens
        # (3 % visible here); the 512-token prompt chunk runs on the matrix-core kernel
        assert c2["fa_list_launches"] == (1 if M <= 256 else 0), (tag, c2)
    # exact attention in float64 over each token's visible cells (q rounded to f16 as both implementations do)
    qf = np.asarray(q_o).reshape(M, NH, HD).astype(np.float16).astype(np.float64)
    kf, vf = kc_n.astype(np.float64).reshape(n_ctx, NKV, HD), vc_n.astype(np.float64).reshape(n_ctx, NKV, HD)
    grp = NH // NKV
    exact = np.empty((M, NH, HD))
    for t in range(M):
        cells = np.nonzero(vis[t])[0]
        for h in range(NH):
            s_ = kf[cells, h // grp, :] @ qf[t, h] / np.sqrt(HD)
            p_ = np.exp(s_ - s_.max())
            exact[t, h] = (p_ / p_.sum()) @ vf[cells, h // grp, :]
    e_gpu, e_cpu = T.nmse(np.asarray(at_g).reshape(M, NH, HD), exact), T.nmse(np.asarray(at_o).reshape(M, NH, HD), exact)
    _log(plog, f"{tag}: attention vs float64: gpu nmse={e_gpu:.3e}, cpu oracle nmse={e_cpu:.3e}")
    if fa:
        # (prompt chunks run on the f16 matrix cores: the probabilities are rounded to f16 for the P.V product, ~1e-9 of the result; the
        # lane-parallel decode kernel keeps them in f32.  Either way the kernel must be closer to exact attention than the CPU's f16 V sum.)
        assert e_gpu <= (1e-9 if M <= 32 else 1e-8) and e_gpu <= e_cpu * 1.01 + 1e-12
        T.compare(f"{tag}: flash_attn", at_g, at_o, max_nmse=max(1e-4, 1.5 * e_cpu), log=plog)
    else:
        T.compare(f"{tag}: K.q -> soft_max -> V^T.p -> cont", at_g, at_o, max_nmse=1e-9, log=plog)

    vals.update(attn=np.asarray(at_o).reshape(M, NH * HD))
    (fi_o,), _ = run(seg_wo, "oracle", vals)
    (fi_g,), c3 = run(seg_wo, backend, vals)
    served(c3, (sp.t_o,), "wo + residual")
    T.compare(f"{tag}: wo + residual (ffn_inp)", fi_g, fi_o, max_nmse=1e-10, log=plog)

    vals.update(ffn_inp=np.asarray(fi_o).reshape(M, E))
    (act_o,), _ = run(seg_ffn, "oracle", vals)
    (act_g,), c4 = run(seg_ffn, backend, vals)
    served(c4, (sp.t_gu,), "norm -> gate/up -> swiglu")
    T.compare(f"{tag}: norm -> gate/up -> swiglu", act_g, act_o, max_nmse=1e-10, log=plog)

    vals.update(act=np.asarray(act_o).reshape(M, FF))
    (lo_o,), _ = run(seg_down, "oracle", vals)
    (lo_g,), c5 = run(seg_down, backend, vals)
    served(c5, (sp.t_d,), "ffn_down + residual")
    T.compare(f"{tag}: ffn_down + residual (l_out)", lo_g, lo_o, max_nmse=1e-10, log=plog)


# ------------------------------------------------------------------------------------------------ (e) config 2's prefill, end to end
def test_prefill_2048_in_four_micro_batches(backend, H, plog):
    """BASELINE config 2's prefill as llama-box drives it (-b 2048 -ub 512: four micro-batches of 512 tokens through one llama_decode), on a
    model with Llama-3-8B's layer shapes and Q4_K_M type map cut to four layers (two plain, two "more bits"), flash attention on:
    last-token logits against the oracle, judged beside the oracle's own order sensitivity (its block dots summed in reverse)."""
    from model_util import Context, Model, preset
    hp = preset("llama3-8b-q4_k_m", n_layer=4)
    rng = np.random.default_rng(2048)
    prompt = rng.integers(3, hp.n_vocab, 2048).tolist()
    want = [0] * 2047 + [1]
    mc = Model(hp, 7, H.ggml_backend_cpu_buffer_type())
    mg = Model(hp, 7, backend.buft)
    ctxs = []
    try:
        def last_logits(model, **kw):
            c = Context(model, n_ctx=2304, n_ubatch=512, flash_attn=1, **kw)
            ctxs.append(c)
            rc, lg = c.decode(prompt, range(2048), want=want)
            assert rc == 0
            return lg[-1].copy()

        ref = last_logits(mc, compute=T.oracle_compute_fn(NT))
        T.oracle().oracle_set_variant(1)
        try:
            var = last_logits(mc, compute=T.oracle_compute_fn(NT))
        finally:
            T.oracle().oracle_set_variant(0)
        c0 = {k: backend.stat(k) for k in ("wide_launches", "tiled_launches", "skinny_launches", "kernel_launches")}
        got = last_logits(mg, backend=backend)
        cnt = {k: backend.stat(k) - v for k, v in c0.items()}
        e, e_var = T.nmse(got, ref), T.nmse(var, ref)
        top2 = np.sort(ref)
        _log(plog, f"prefill 2048 tokens in 4 micro-batches (llama3-8b shapes, 4 layers, q4_k_m): last-token logits nmse gpu={e:.3e} (oracle reversed-blocks {e_var:.3e}) "
                   f"max|d| gpu={np.max(np.abs(got - ref)):.3e} (variant {np.max(np.abs(var - ref)):.3e}); argmax gpu={int(np.argmax(got))} oracle={int(np.argmax(ref))} margin={top2[-1] - top2[-2]:.3e}; kernels {cnt}")
        assert cnt["wide_launches"] >= 4 * 4 * 3 and cnt["skinny_launches"] == 0, cnt  # 4 micro-batches x 4 layers x (qkv, wo, gate/up [, down])
        assert e <= 1e-3 and e <= max(10.0 * e_var, 1e-10)
        if top2[-1] - top2[-2] > 2.0 * float(np.max(np.abs(var - ref))):
            assert int(np.argmax(got)) == int(np.argmax(ref))
    finally:
        for o in ctxs + [mc, mg]:
            o.free()
