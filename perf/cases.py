"""The work that is measured: prompts and decode steps of the served models, through the host API an engine loop calls.

A pass is one llm_decode() of a prompt, or of one continuous-batching step, with its logits on the host: what llama-box's engine does once
per iteration (llama-box/httpserver.hpp:3539-3623).  The models are the GGUF presets the benchmark names (seeded weights in the exact block
formats; the "-damped" value sets, whose logits are far from ties as a trained model's are) and one model class described by a checkpoint
folder (config.json + model.safetensors, bf16, with expert layers).

A prompt pass clears the cache and decodes `tokens` tokens of one request, the last one's logits wanted.  A step pass decodes 1 + `drafts`
tokens of each of `seqs` requests that hold `past` tokens each, every logits row wanted, and drops the new positions again as a verification
that rejects them does: it can be repeated at the same place.
"""
import ctypes as C
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

import llama_box_amd as L

TINY, LLAMA, QWEN = "tinyllama-1.1b-q8_0", "llama3-8b-q4_k_m", "qwen2-7b-q5_k_m"
CLASS_M, CLASS_L = "nigozen-m", "nigozen-l"

# layers, width, heads, kv heads, head size, ff, vocabulary, rotation base, norm eps, rotation in halves (else neighbours), biases of q / k / v
GGUF = {
    TINY: (22, 2048, 32, 4, 64, 5632, 32000, 1e4, 1e-5, False, False),
    LLAMA: (32, 4096, 32, 8, 128, 14336, 128256, 5e5, 1e-5, False, False),
    QWEN: (28, 3584, 28, 4, 128, 18944, 152064, 1e6, 1e-6, True, True),
}
# the benchmark's sizes of the class: width, layers (dense and expert feed-forward in turn), heads, kv heads, head size, rotated part, chunk of positions,
# dense ff, experts, chosen experts, expert ff, vocabulary
FOLDER = {
    CLASS_M: dict(width=2048, layers=4, heads=16, kv=4, hd=128, rot=64, chunk=1024, ff=8192, experts=8, top=2, eff=2048, vocab=32000),
    CLASS_L: dict(width=4096, layers=2, heads=32, kv=8, hd=128, rot=64, chunk=2048, ff=14336, experts=8, top=2, eff=4096, vocab=32000),
}
UBATCH = 512  # the engine's default micro-batch


def _prompt(name, model, tokens, fa=1, kv="f16"):
    return {"name": name, "model": model, "kind": "prompt", "tokens": tokens, "fa": fa, "kv": kv}


def _step(name, model, seqs, past, drafts=0, fa=1, kv="f16"):
    return {"name": name, "model": model, "kind": "step", "seqs": seqs, "past": past, "drafts": drafts, "fa": fa, "kv": kv}


def listed():
    return [
        _step("tiny decode", TINY, 1, 120),                          # a short greedy generation of the small Q8_0 model: latency and launches
        _prompt("tiny prompt", TINY, 700),                           # a chat turn of ordinary length, not a multiple of the micro-batch
        _step("tiny batch 16", TINY, 16, 150),                       # small model, many users
        _step("llama decode", LLAMA, 1, 2048),                       # the headline: one user behind a 2048-token prompt
        _prompt("llama prompt 2048", LLAMA, 2048),                   # the headline's prompt: the largest matrix products
        _prompt("llama prompt 77", LLAMA, 77, fa=0),                 # a short question with the server's default attention
        _step("llama batch 32", LLAMA, 32, 160),                     # continuous batching with all slots busy
        _step("llama batch 3", LLAMA, 3, 700, fa=0),                 # a few users with the server's default attention
        _step("llama drafts", LLAMA, 1, 1500, drafts=8, kv="q8_0"),  # verification of 8 drafts over a quantised cache
        _step("qwen decode", QWEN, 1, 8000),                         # long context, Q5_K + Q6_K mix
        _prompt("class prompt", CLASS_L, 2000),                      # a folder model's prompt: bf16 products, chunked attention, experts
        _step("class decode", CLASS_M, 2, 900),                      # two users of a folder model
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    model = rng.choice([TINY] * 2 + [LLAMA] * 4 + [QWEN] + [CLASS_M] + [CLASS_L] * 2)
    folder = model in FOLDER
    fa = 1 if folder else rng.choice([0, 1, 1])
    kv = "q8_0" if not folder and fa and rng.random() < 0.25 else "f16"
    if rng.random() < 0.4:
        c = _prompt("", model, log_int(16, 1400 if model == QWEN else 2000), fa, kv)
    else:
        seqs = log_int(1, 4 if folder else 32)
        drafts = rng.randint(1, 8) if seqs <= 4 and rng.random() < 0.25 else 0
        c = _step("", model, seqs, log_int(16, min(2000 if model in (TINY, CLASS_M, CLASS_L) else 8000, 8192 // seqs)), drafts, fa, kv)
    del c["name"]
    return c


# ---------------------------------------------------------------------------------------------- what a program has in hand before the call
class _State:
    """Backend, model, context and the arrays of the call; given back when the last reference (an output's included) goes."""

    backend = model = ctx = None

    def close(self):
        H = L.host()
        if self.ctx:
            H.llm_context_free(self.ctx)
        if self.model:
            H.llm_model_free(self.model)
        if self.backend:
            self.backend.close()
        self.ctx = self.model = self.backend = None

    def __del__(self):
        self.close()


def _ints(v, t=C.c_int32):
    return (t * len(v))(*[int(x) for x in v])


def _tokens(case, seed):
    """int array [requests, tokens of each]: the history first, then what a pass decodes"""
    vocab = FOLDER[case["model"]]["vocab"] if case["model"] in FOLDER else GGUF[case["model"]][6]
    shape = (1, case["tokens"]) if case["kind"] == "prompt" else (case["seqs"], case["past"] + 1 + case["drafts"])
    return np.random.default_rng([int(seed), 7]).integers(0, vocab, shape)


def _gguf_model(case, seed, buft):
    hp = L.HParams()
    if L.host().llm_preset((case["model"] + "-damped").encode(), C.byref(hp)) != 0:
        raise RuntimeError("no preset " + case["model"])
    return L.host().llm_model_synth(C.byref(hp), int(seed) & 0xFFFFFFFF, buft, 0, 1, None)


def _folder_config(z):
    layers = []
    for il in range(z["layers"]):
        mixer = {"heads": z["heads"], "kv_heads": z["kv"], "dim": z["hd"], "vdim": z["hd"], "mask": {"size": z["chunk"]}, "rot": {"base": 1e6, "dims": z["rot"]},
                 "scale": z["hd"] ** -0.5, "v_mix": True}
        mlp = {"kind": "moe", "expert": {"ff": z["eff"]}, "router": {"experts": z["experts"], "top": z["top"]}} if il % 2 else {"kind": "dense", "ff": z["ff"]}
        layers.append({"type": "attention", "mixer": mixer, "mlp": mlp})
    return {"architecture": "Nigozen", "embedding": {"scale": 1.0}, "layers": layers, "norm": {"eps": 1e-5}, "vocab": z["vocab"], "width": z["width"]}


def _folder_weights(z, seed):
    """the checkpoint's tensors (bf16, on the GPU), in file order; matrices [out, in] of gain / sqrt(in)"""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)

    def mat(o, i, gain=1.0):
        return (torch.randn((o, i), generator=g, device="cuda") * (gain / math.sqrt(i))).bfloat16()

    def vec(gain=1.0):
        return (gain * (1.0 + 0.1 * torch.randn(z["width"], generator=g, device="cuda"))).bfloat16()

    E, nq, nkv = z["width"], z["heads"] * z["hd"], z["kv"] * z["hd"]
    yield "embed", mat(z["vocab"], E, math.sqrt(E))
    for il in range(z["layers"]):
        p = "l%d." % il
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            yield p + n, vec(0.05 if n.endswith("b") else 1.0)  # (the norms on the sublayers' outputs: small branches, as the GGUF sets have)
        yield p + "mix.q", mat(nq, E, 2.0)
        yield p + "mix.k", mat(nkv, E, 2.0)
        yield p + "mix.v", mat(nkv, E)
        yield p + "mix.g", mat(nq, E)
        yield p + "mix.o", mat(E, nq)
        yield p + "mix.vmix", torch.tensor(0.5, device="cuda").bfloat16()
        if il % 2:
            for e in range(z["experts"]):
                yield p + "mlp.e%d.up" % e, mat(z["eff"], E, 2.0)
                yield p + "mlp.e%d.down" % e, mat(E, z["eff"])
            yield p + "mlp.router", mat(z["experts"], E, 3.0)
        else:
            yield p + "mlp.up", mat(z["ff"], E)
            yield p + "mlp.down", mat(E, z["ff"])
    yield "final.norm", vec()


def _folder_model(case, seed, buft):
    z = FOLDER[case["model"]]
    with tempfile.TemporaryDirectory() as d:
        with open(os.path.join(d, "config.json"), "w") as f:
            json.dump(_folder_config(z), f)
        head, blobs, at = {}, [], 0
        for name, w in _folder_weights(z, seed):
            raw = w.reshape(-1).view(torch.int16).cpu().numpy()
            head[name] = {"dtype": "BF16", "shape": list(w.shape), "data_offsets": [at, at + raw.nbytes]}
            blobs.append(raw)
            at += raw.nbytes
        hj = json.dumps(head).encode()
        hj += b" " * (-len(hj) % 8)
        with open(os.path.join(d, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(hj)))
            f.write(hj)
            for b in blobs:
                b.tofile(f)
        return L.host().llm_model_load_dir(os.fsencode(d), buft, L.BF16)


def prepare(case, seed):
    H, s = L.host(), _State()
    s.case, s.backend = case, L.Backend(0)
    s.model = (_folder_model if case["model"] in FOLDER else _gguf_model)(case, seed, s.backend.buft)
    if not s.model:
        raise RuntimeError("model creation failed")
    s.n_vocab = H.llm_model_hparams(s.model).contents.n_vocab
    tok = _tokens(case, seed)
    n_seq, per = tok.shape
    folder = case["model"] in FOLDER
    kv = 0 if folder or case["kv"] == "f16" else L.Q8_0  # (a folder model's cache is in the type of its matrices)
    p = L.ContextParams(n_seq * per + 256, UBATCH, case["fa"], 0, 1, kv, kv, max(8, n_seq))
    s.ctx = H.llm_context_new(s.model, s.backend.backend, L.COMPUTE_FN(), C.byref(p))
    if not s.ctx:
        raise RuntimeError("context creation failed")
    past = 0 if case["kind"] == "prompt" else case["past"]
    new = per - past
    for q in range(n_seq if past else 0):  # every request's history, prompt by prompt
        if H.llm_decode(s.ctx, past, _ints(tok[q, :past]), _ints(range(past)), _ints([q] * past), _ints([0] * past, C.c_int8)) != 0:
            raise RuntimeError("prompt failed")
    s.n, s.past = n_seq * new, past
    s.tok, s.pos = _ints(tok[:, past:].reshape(-1)), _ints(list(range(past, per)) * n_seq)
    s.seq = _ints([q for q in range(n_seq) for _ in range(new)])
    s.want = _ints([0] * (new - 1) + [1], C.c_int8) if case["kind"] == "prompt" else None
    s.rows = 1 if case["kind"] == "prompt" else s.n
    s.logits = type("Logits", (C.c_float * (s.rows * s.n_vocab),), {})  # memory of the context's logits; an instance can keep the state alive
    return s


def run(s):
    H = L.host()
    H.llm_kv_seq_rm(s.ctx, -1, s.past, -1)
    rc = H.llm_decode(s.ctx, s.n, s.tok, s.pos, s.seq, s.want)
    if rc != 0 or H.llm_n_outputs(s.ctx) != s.rows:
        raise RuntimeError("llm_decode: %d" % rc)
    mem = s.logits.from_address(C.addressof(H.llm_get_logits(s.ctx).contents))
    mem.state = s
    return np.frombuffer(mem, dtype=np.float32).reshape(s.rows, s.n_vocab)


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _gguf_matrices(model):
    """(bytes, values) of the layers' matrices and of the output matrix"""
    n, E, H, G, D, ff, V = GGUF[model][:7]
    q4, q5, q6, q8 = 144 / 256, 176 / 256, 210 / 256, 34 / 32
    base = {TINY: q8, LLAMA: q4, QWEN: q5}[model]
    byte = val = 0.0
    for il in range(n):
        more = il < n // 8 or il >= 7 * n // 8 or (il - n // 8) % 3 == 2  # layers whose attn_v and ffn_down carry more bits
        high = q8 if model == TINY else q6 if more else base
        byte += base * (2 * E * H * D + E * G * D + 2 * E * ff) + high * (E * G * D + ff * E)
        val += 2 * E * H * D + 2 * E * G * D + 3 * E * ff
    return byte, val, (q8 if model == TINY else q6) * E * V, E * V


def work(case):
    prompt = case["kind"] == "prompt"
    seqs, past, new = (1, 0, case["tokens"]) if prompt else (case["seqs"], case["past"], 1 + case["drafts"])
    T, rows = seqs * new, 1 if prompt else seqs * new
    if case["model"] in FOLDER:
        z = FOLDER[case["model"]]
        n, E, H, G, D, V, chunk = z["layers"], z["width"], z["heads"], z["kv"], z["hd"], z["vocab"], z["chunk"]
        attn = E * D * (3 * H + 2 * G)
        used = min(z["experts"], z["top"] * T)  # experts that a pass touches at the most
        wbytes = 2 * ((n * attn) + (n + 1) // 2 * 2 * E * z["ff"] + n // 2 * (2 * E * z["eff"] * used + 2 * E * z["experts"]))
        val = n * attn + (n + 1) // 2 * 2 * E * z["ff"] + n // 2 * (2 * E * z["eff"] * z["top"] + E * z["experts"])
        obytes, oval, kvb = 2 * E * V, E * V, 2.0
    else:
        n, E, H, G, D, _, V = GGUF[case["model"]][:7]
        wbytes, val, obytes, oval = _gguf_matrices(case["model"])
        chunk, kvb = 1 << 30, 2.0 if case["kv"] == "f16" else 34 / 32
    seen = [min(p % chunk, p) + 1 for p in range(past, past + new)]  # keys that each new position sees
    cells = max(seen)                                                # ... of which each is read once
    return {"bytes": wbytes + obytes + seqs * (cells + new) * n * 2 * G * D * kvb + rows * V * 4 + T * E * 2,
            "flops": 2 * (val * T + oval * rows) + 4 * n * H * D * seqs * sum(seen)}


def tolerance(case):
    # A sum in another order flips 8-bit (GGUF) or bf16 (folder) roundings of the activations behind it.  Measured: the same tokens in micro-batches of 96 and 200 instead of
    # 512, and with the other attention, differ by rel 1.4e-3 .. 2.1e-3, max 6e-3 .. 1.0e-2 (the small model), rel 2.7e-3 .. 3.3e-3, max 1.3e-2 .. 1.8e-2 (the two large ones),
    # rel 6.5e-4 .. 9.5e-4, max 2.6e-3 .. 4.3e-3 (folder models).  Four times that; for folder models room for ONE expert chosen the other way in a near tie besides: it moves
    # its row by up to 0.05 (the output norm's gain) times the two experts' difference, about 0.03 of it.
    if case["model"] in FOLDER:
        return {"rel": 1.5e-2, "max": 0.12}
    return {"rel": 8e-3, "max": 4e-2} if case["model"] == TINY else {"rel": 1.3e-2, "max": 7e-2}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _dequant(raw, kind, rows, cols):
    """packed blocks (uint8, on the GPU) -> float64 [rows, cols]"""
    def half(b):
        return b.contiguous().view(torch.float16).double()

    if kind == L.F32:
        return raw.view(torch.float32).double().view(rows, cols)
    b = raw.view(-1, L.TYPE_SIZE[kind])
    if kind == L.Q8_0:
        return (half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    n = b.shape[0]
    if kind in (L.Q4_K, L.Q5_K):
        d, dmin, sc = half(b[:, 0:2]), half(b[:, 2:4]), b[:, 4:16].int()
        s = torch.cat([sc[:, 0:4] & 63, (sc[:, 8:12] & 15) | ((sc[:, 0:4] >> 6) << 4)], 1).double()
        m = torch.cat([sc[:, 4:8] & 63, (sc[:, 8:12] >> 4) | ((sc[:, 4:8] >> 6) << 4)], 1).double()
        ql = b[:, (48 if kind == L.Q5_K else 16):].view(n, 4, 1, 32)
        q = torch.cat([ql & 15, ql >> 4], 2).view(n, 8, 32).double()
        if kind == L.Q5_K:
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q + 16.0 * ((b[:, 16:48].view(n, 1, 32) >> bit) & 1).double()
        return ((d * s).view(n, 8, 1) * q - (dmin * m).view(n, 8, 1)).view(rows, cols)
    assert kind == L.Q6_K
    ql, qh, sc = b[:, :128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 1, 32), b[:, 192:208].contiguous().view(torch.int8).double()
    low = torch.cat([ql & 15, ql >> 4], 2)  # [n, half, 4, 32]
    high = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], 2)
    q = (low.int() | (high.int() << 4)).double() - 32.0
    return (half(b[:, 208:210]).view(n, 1, 1) * sc.view(n, 16, 1) * q.reshape(n, 16, 16)).view(rows, cols)


def _rotate(x, pos, dims, base, halves):
    """x [S, T, heads, D]"""
    ang = pos.double()[:, None] * float(base) ** (-torch.arange(0, dims, 2, device=x.device, dtype=torch.float64) / dims)
    c, s = ang.cos()[None, :, None, :], ang.sin()[None, :, None, :]
    r = x[..., :dims]
    u, v = (r[..., : dims // 2], r[..., dims // 2:]) if halves else (r[..., 0::2], r[..., 1::2])
    a, b = u * c - v * s, v * c + u * s
    r = torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([r, x[..., dims:]], -1)


def _attend(q, k, v, scale, chunk, sink):
    """q [S, T, H, D], k and v [S, T, G, D], causal, positions 0 .. T - 1 -> [S, T, H * D]"""
    S, T, H, D = q.shape
    G, out = k.shape[2], torch.empty_like(q)
    at = torch.arange(T, device=q.device)
    hidden = at[None, :] > at[:, None]
    if chunk:
        hidden |= (at[None, :] // chunk) != (at[:, None] // chunk)
    for h in range(H):
        kh, vh = k[:, :, h // (H // G)], v[:, :, h // (H // G)]
        s = torch.matmul(q[:, :, h], kh.transpose(1, 2).contiguous()).mul_(scale).masked_fill_(hidden, -math.inf)
        m = s.amax(-1, keepdim=True)
        m = m.clamp(min=0.0) if sink else m
        s = s.sub_(m).exp_()
        z = s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
        out[:, :, h] = torch.matmul(s, vh.contiguous()) / z
    return out.reshape(S, T, H * D)


def _exact_gguf(case, seed, tok, last):
    H, be = L.host(), L.Backend(0)
    model = _gguf_model(case, seed, be.buft)

    def w(name):
        t = H.llm_model_tensor(model, name.encode())
        raw = np.empty(H.ggml_nbytes(t), dtype=np.uint8)
        H.ggml_backend_tensor_get(t, raw.ctypes.data, 0, raw.nbytes)
        x = _dequant(torch.from_numpy(raw).cuda(), t.contents.type, t.contents.ne[1], t.contents.ne[0])
        return x[0] if x.shape[0] == 1 else x

    n, E, nh, ng, D, ff, V, base, eps, halves, biases = GGUF[case["model"]]
    S, T = tok.shape
    pos = torch.arange(T, device="cuda")

    def norm(x, name):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w(name)

    x = w("token_embd.weight")[torch.from_numpy(tok).cuda()]
    for il in range(n):
        p = "blk.%d." % il
        h = norm(x, p + "attn_norm.weight")
        q, k, v = (h @ w(p + "attn_%s.weight" % c).T + (w(p + "attn_%s.bias" % c) if biases else 0.0) for c in "qkv")
        q, k = _rotate(q.view(S, T, nh, D), pos, D, base, halves), _rotate(k.view(S, T, ng, D), pos, D, base, halves)
        x = x + _attend(q, k, v.view(S, T, ng, D), D ** -0.5, 0, False) @ w(p + "attn_output.weight").T
        h = norm(x, p + "ffn_norm.weight")
        x = x + (torch.nn.functional.silu(h @ w(p + "ffn_gate.weight").T) * (h @ w(p + "ffn_up.weight").T)) @ w(p + "ffn_down.weight").T
    out = norm(x[:, T - last:].reshape(S * last, E), "output_norm.weight") @ w("output.weight").T
    H.llm_model_free(model)
    be.close()
    return out


def _exact_folder(case, seed, tok, last):
    z = FOLDER[case["model"]]
    W = {name: w.double() for name, w in _folder_weights(z, seed)}
    S, T = tok.shape
    pos, first = torch.arange(T, device="cuda"), None

    def norm(x, w):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt(d.square().mean(-1, keepdim=True) + 1e-5) * w

    x = W["embed"][torch.from_numpy(tok).cuda()]
    for il in range(z["layers"]):
        p = "l%d." % il
        h = norm(x, W[p + "norm1"])
        q, k, v = (h @ W[p + "mix." + c].T for c in "qkv")
        lam = W[p + "mix.vmix"]
        v = v if first is None else (1.0 - lam) * v + lam * first
        first = v if first is None else first
        q, k = (_rotate(y.view(S, T, -1, z["hd"]), pos, z["rot"], 1e6, False) for y in (q, k))
        a = _attend(q, k, v.view(S, T, -1, z["hd"]), z["hd"] ** -0.5, z["chunk"], True)
        x = x + norm((a * torch.sigmoid(h @ W[p + "mix.g"].T)) @ W[p + "mix.o"].T, W[p + "norm1b"])
        h = norm(x, W[p + "norm2"])
        if il % 2:
            score, pick = (h @ W[p + "mlp.router"].T).topk(z["top"], -1)
            score, f = score.softmax(-1), torch.zeros_like(h)
            for e in range(z["experts"]):
                share = (score * (pick == e)).sum(-1, keepdim=True)
                f += share * ((h @ W[p + "mlp.e%d.up" % e].T).relu().square() @ W[p + "mlp.e%d.down" % e].T)
        else:
            f = torch.nn.functional.gelu(h @ W[p + "mlp.up"].T) @ W[p + "mlp.down"].T
        x = x + norm(f, W[p + "norm2b"])
    return norm(x[:, T - last:].reshape(S * last, -1), W["final.norm"]) @ W["embed"].T


def exact(case, seed):
    tok = _tokens(case, seed)
    last = 1 if case["kind"] == "prompt" else 1 + case["drafts"]
    return (_exact_folder if case["model"] in FOLDER else _exact_gguf)(case, seed, tok, last).cpu().numpy()
