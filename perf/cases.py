"""The work that users of this library have it do, as cases that can be timed and checked.

A case is one call (or the few calls that belong together) of a decoder, a
draft or a matrix product, at widths that the tests and the benchmark use
(Llama-3-8B, Qwen2.5-7B, a small 4-layer decoder), on random weights in the
GGUF block formats, uploaded as a loader would upload them.  Decoders have
few layers where one layer is like the next; one case runs all 32.

listed() names the cases, draw() gives more of the same ranges, prepare()
builds the state from a seed, run() is one pass, exact() the same result in
64 bits from the block bytes alone (no code of this library), work() the bytes
and operations that a pass cannot do without and tolerance() how far two
correct implementations may be apart.
"""
import ctypes
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "abyo-speculate_amd"))
import speculate_hip as S  # noqa: E402

SHAPES = {
    "llama8b": dict(arch=S.ARCH_LLAMA, hidden=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=128256,
                    rope_theta=500000.0, rms_eps=1e-5),
    "qwen7b": dict(arch=S.ARCH_QWEN2, hidden=3584, n_heads=28, n_kv_heads=4, head_dim=128, ffn=18944, vocab=152064,
                   rope_theta=1e6, rms_eps=1e-6),
    "tiny": dict(arch=S.ARCH_LLAMA, hidden=512, n_heads=8, n_kv_heads=8, head_dim=64, ffn=1536, vocab=32000,
                 rope_theta=10000.0, rms_eps=1e-5),
}
FORMATS = {"q4_k": (S.Q4_K, 256, 144), "q5_k": (S.Q5_K, 256, 176), "q6_k": (S.Q6_K, 256, 210), "q8_0": (S.Q8_0, 32, 34)}
MATRICES = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")
KIND = {"token_embd": S.TOK_EMBD, "output": S.OUTPUT, "output_norm": S.OUTPUT_NORM, "attn_q": S.ATTN_Q,
        "attn_k": S.ATTN_K, "attn_v": S.ATTN_V, "attn_output": S.ATTN_OUTPUT, "ffn_gate": S.FFN_GATE,
        "ffn_up": S.FFN_UP, "ffn_down": S.FFN_DOWN, "attn_norm": S.ATTN_NORM, "ffn_norm": S.FFN_NORM,
        "attn_q_bias": S.ATTN_Q_BIAS, "attn_k_bias": S.ATTN_K_BIAS, "attn_v_bias": S.ATTN_V_BIAS}
MATMUL_LAYERS = 8  # layers whose matrix a "matmul" pass multiplies in turn
DRAFT = dict(hidden=4096, n_heads=32, n_kv_heads=8, ffn=14336, draft_vocab=32000, target_vocab=128256, rms_eps=1e-5,
             rope_theta=500000.0, max_pos=2048)


def listed():
    return [
        # one decoded token of the small decoder: launches and host work, hardly any bytes
        dict(name="decode_tiny", kind="decode", shape="tiny", mix="q4_k", layers=4, positions=100, tokens=1),
        # autoregressive decoding, the step that a user without a draft runs for every token
        dict(name="decode_llama8b", kind="decode", shape="llama8b", mix="q4_k_m", layers=8, positions=700, tokens=1),
        # the headline: a whole 32-layer target verifies 4 draft tokens
        dict(name="verify5_llama8b_32l", kind="verify", shape="llama8b", mix="q4_k_m", layers=32, positions=512, tokens=5),
        # 8 drafts on the other architecture: bias, Q5_K attention, Q8_0 FFN, longer context
        dict(name="verify9_qwen7b", kind="verify", shape="qwen7b", mix="q5k_q80", layers=4, positions=2048, tokens=9),
        # EAGLE tree verification with the commit of an accepted path
        dict(name="tree60_llama8b", kind="tree", shape="llama8b", mix="q4_k_m", layers=4, positions=4096, tokens=60),
        # a small, odd tree at a short context on higher-precision weights
        dict(name="tree27_qwen7b", kind="tree", shape="qwen7b", mix="q6_k", layers=4, positions=333, tokens=27),
        # a prompt of ordinary length
        dict(name="prefill512_llama8b", kind="prefill", shape="llama8b", mix="q4_k_m", layers=4, positions=0, tokens=512),
        # a long, ragged prompt: the largest case
        dict(name="prefill2501_qwen7b", kind="prefill", shape="qwen7b", mix="q5k_q80", layers=2, positions=0, tokens=2501),
        # a chat turn appended to a long context
        dict(name="extend100_llama8b", kind="prefill", shape="llama8b", mix="q4_k_m", layers=4, positions=4000, tokens=100),
        # an EAGLE-3 draft chain: fc on the first step, then one midlayer and head per step
        dict(name="draft7_eagle3", kind="draft", positions=600, tokens=7),
        # a weight matrix times caller-owned device rows: a full row batch, and a tree's
        dict(name="matmul128_q4k", kind="matmul", shape="llama8b", matrix="ffn_gate", fmt="q4_k", tokens=128),
        dict(name="matmul40_q6k", kind="matmul", shape="llama8b", matrix="ffn_down", fmt="q6_k", tokens=40),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["decode", "verify", "verify", "tree", "tree", "prefill", "prefill", "prefill", "draft", "matmul"])
    if kind == "draft":
        return dict(kind=kind, positions=_log(rng, 16, 2000), tokens=rng.randint(2, 12))
    shape = rng.choice(["llama8b", "llama8b", "qwen7b", "qwen7b", "tiny"])
    if kind == "matmul":
        matrix = rng.choice(["attn_q", "attn_output", "ffn_gate", "ffn_down"])
        top = min(128, (4 << 20) // (2 * _dims(SHAPES[shape], matrix)[1]))  # the call stages at most 4 MiB of rows
        return dict(kind=kind, shape=shape, matrix=matrix, fmt=rng.choice(sorted(FORMATS)), tokens=_log(rng, 1, top))
    mix = rng.choice(["q4_k_m", "q4_k_m", "q5k_q80", "q4_k", "q5_k", "q6_k", "q8_0"])
    layers = rng.randint(1, 4)
    positions = _log(rng, 16, 6000)
    if kind == "decode":
        tokens = 1
    elif kind == "verify":
        tokens = rng.randint(2, 16)
    elif kind == "tree":
        tokens = _log(rng, 17, 128)
    else:
        tokens = _log(rng, 17, 2400)
        layers = min(layers, max(1, 4000 // tokens))
        positions = rng.choice([0, 0, min(positions, 3000)])
    return dict(kind=kind, shape=shape, mix=mix, layers=layers, positions=positions, tokens=tokens)


# ---- weights: GGUF blocks from a seed -----------------------------------------
def _dims(s, name):
    H, qd, kd = s["hidden"], s["n_heads"] * s["head_dim"], s["n_kv_heads"] * s["head_dim"]
    return {"token_embd": (s["vocab"], H), "output": (s["vocab"], H), "attn_q": (qd, H), "attn_k": (kd, H),
            "attn_v": (kd, H), "attn_output": (H, qd), "ffn_gate": (s["ffn"], H), "ffn_up": (s["ffn"], H),
            "ffn_down": (H, s["ffn"]), "attn_q_bias": (1, qd), "attn_k_bias": (1, kd),
            "attn_v_bias": (1, kd)}.get(name, (1, H))


def _fmt(mix, layers, layer, name):
    """The formats of a quantisation mix (Q4_K_M: Q6_K for some layers' V and down matrices)."""
    if mix == "q4_k_m":
        more = layer >= 0 and (layer < layers // 8 or layer >= 7 * layers // 8 or (layer - layers // 8) % 3 == 2)
        return "q6_k" if more and name in ("attn_v", "ffn_down") else "q4_k"
    if mix == "q5k_q80":
        return "q5_k" if name.startswith("attn") else "q8_0"
    return mix


def _gen(seed, *what):
    h = 1469598103934665603
    for c in repr((seed, what)).encode():
        h = ((h ^ c) * 1099511628211) % (1 << 64)
    return torch.Generator(device="cuda").manual_seed(h >> 1)


def _halves(x):
    return x.to(torch.float16).view(torch.uint8).reshape(x.shape[0], -1)


def _blocks(fmt, rows, K, g):
    """Random blocks [rows * K / block][bytes] whose weights are about N(0, 0.02)-sized, as a model's are."""
    n = rows * K // FORMATS[fmt][1]

    def ints(lo, hi, *shape, dtype=torch.uint8):
        return torch.randint(lo, hi, (n,) + shape, generator=g, device="cuda", dtype=dtype)

    size = 0.8 + 0.4 * torch.rand((n, 1), generator=g, device="cuda")
    if fmt == "q8_0":
        return torch.cat([_halves(size * 2.7e-4), ints(-127, 128, 32, dtype=torch.int8).view(torch.uint8)], 1)
    if fmt == "q6_k":
        sc = ints(40, 120, 16, dtype=torch.int8) * (1 - 2 * ints(0, 2, 16, dtype=torch.int8))
        return torch.cat([ints(0, 256, 128), ints(0, 256, 64), sc.view(torch.uint8), _halves(size * 1.35e-5)], 1)
    sc = ints(32, 64, 8)
    mn = (sc.to(torch.int16) + ints(-3, 4, 8, dtype=torch.int8)).clamp(0, 63).to(torch.uint8)
    packed = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4) << 6, mn[:, :4] | (mn[:, 4:] >> 4) << 6,
                        (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], 1)
    step, mid = (9.0e-5, 7.5) if fmt == "q4_k" else (4.5e-5, 15.5)
    head = [_halves(size * step), _halves(size * step * mid), packed]
    return torch.cat(head + ([ints(0, 256, 32)] if fmt == "q5_k" else []) + [ints(0, 256, 128)], 1)


def _f16(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _dequant(fmt, b):
    """The weights that blocks stand for, in 64 bits: [blocks][elements]."""
    f = torch.float64
    if fmt == "q8_0":
        return _f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(f)
    if fmt == "q6_k":
        ql, qh, sc, d = b[:, :128], b[:, 128:192], b[:, 192:208].contiguous().view(torch.int8).to(f), _f16(b[:, 208:210])
        q = []
        for h in range(2):
            lo, hi = ql[:, 64 * h:64 * h + 64], qh[:, 32 * h:32 * h + 32]
            nib = [lo[:, :32] & 15, lo[:, 32:] & 15, lo[:, :32] >> 4, lo[:, 32:] >> 4]
            q += [x | ((hi >> 2 * i) & 3) << 4 for i, x in enumerate(nib)]
        q = torch.cat(q, 1).to(f) - 32.0
        return (q.reshape(-1, 16, 16) * (d * sc)[:, :, None]).reshape(-1, 256)
    s = b[:, 4:16]
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1).to(f) * _f16(b[:, :2])
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4], 1).to(f) * _f16(b[:, 2:4])
    qs = b[:, -128:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if fmt == "q5_k":
        qh = b[:, 16:48]
        q = q + torch.stack([((qh >> i) & 1) << 4 for i in range(8)], 1)
    return (q.to(f) * sc[:, :, None] - mn[:, :, None]).reshape(-1, 256)


def _weight_bytes(case, seed, layer, name):
    rows, K = _dims(SHAPES[case["shape"]], name)
    fmt = case["fmt"] if case["kind"] == "matmul" else _fmt(case["mix"], case["layers"], layer, name)
    return fmt, _blocks(fmt, rows, K, _gen(seed, layer, name))


def _vector(case, seed, layer, name):
    _, K = _dims(SHAPES[case["shape"]], name)
    v = 0.05 * torch.randn(K, generator=_gen(seed, layer, name), device="cuda")
    return v + 1.0 if name.endswith("norm") else v


def _vectors(case):
    return ["attn_norm", "ffn_norm"] + (["attn_q_bias", "attn_k_bias", "attn_v_bias"] if case["shape"] == "qwen7b" else [])


# ---- inputs ---------------------------------------------------------------------
def _host(seed, *what):
    return np.random.default_rng(abs(hash((int(seed),) + what)) % (1 << 63))


def _ids(seed, what, n, vocab):
    return [int(v) for v in _host(seed, what).integers(0, vocab, n)]


def _tree(seed, n, root, vocab):
    """A BFS-ordered random tree of n nodes, up to 4 children a node, and one root-to-leaf path."""
    r = _host(seed, 3)
    parents, at = [0], 0
    while len(parents) < n:
        kids = min(int(r.integers(1, 5)), n - len(parents))
        parents += [at] * kids
        at += 1
    path, i = [], n - 1
    while i:
        path.append(i)
        i = parents[i]
    return [root] + _ids(seed, 4, n - 1, vocab), parents, [0] + path[::-1]


def _inputs(case, seed):
    """(committed history, new tokens): the decoder has taken in the history when a pass begins."""
    V = SHAPES[case["shape"]]["vocab"]
    return _ids(seed, 1, case["positions"], V), _ids(seed, 2, case["tokens"], V)


def _draft_tensors(seed):
    H, F, V = DRAFT["hidden"], DRAFT["ffn"], DRAFT["draft_vocab"]
    kd = H // DRAFT["n_heads"] * DRAFT["n_kv_heads"]
    mats = {S.D3_FC: (H, 3 * H), S.D3_Q: (H, 2 * H), S.D3_K: (kd, 2 * H), S.D3_V: (kd, 2 * H), S.D3_O: (H, H),
            S.D3_GATE: (F, H), S.D3_UP: (F, H), S.D3_DOWN: (H, F), S.D3_LM_HEAD: (V, H)}
    t = {k: (0.02 * torch.randn(s, generator=_gen(seed, "draft", k), device="cuda")).half() for k, s in mats.items()}
    for k in (S.D3_INPUT_NORM, S.D3_HIDDEN_NORM, S.D3_POST_NORM, S.D3_NORM):
        t[k] = (1.0 + 0.05 * torch.randn(H, generator=_gen(seed, "draft", k), device="cuda")).half()
    return t


def _draft_inputs(case, seed):
    r = _host(seed, 5)
    hidden3 = r.standard_normal(3 * DRAFT["hidden"]).astype(np.float16).astype(np.float32)
    emb = (0.5 * r.standard_normal((case["tokens"], DRAFT["hidden"]))).astype(np.float16).astype(np.float32)
    return hidden3, emb


# ---- one pass ---------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "draft":
        d = S.HipEagle3Draft(**DRAFT)
        for k, v in _draft_tensors(seed).items():
            d.set_tensor(k, v.cpu().numpy())
        d.set_tensor(S.D3_D2T, _host(seed, 6).choice(DRAFT["target_vocab"], DRAFT["draft_vocab"], replace=False))
        return dict(case=case, draft=d, inputs=_draft_inputs(case, seed))
    s = SHAPES[case["shape"]]
    if case["kind"] == "matmul":
        dec = S.HipQuantDecoder(S.Config(n_layers=MATMUL_LAYERS, ctx_len=64, **dict(s, vocab=256)))
        for layer in range(MATMUL_LAYERS):
            fmt, b = _weight_bytes(case, seed, layer, case["matrix"])
            dec.set_tensor(layer, KIND[case["matrix"]], FORMATS[fmt][0], b.cpu().numpy())
        lib = S.load_library()
        lib.sd_model_qmatmul_noalloc.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_int32, ctypes.c_void_p,
                                                 ctypes.c_size_t, ctypes.c_void_p, ctypes.c_void_p]
        lib.sd_model_qmatmul_noalloc.restype = ctypes.c_int32
        rows, K = _dims(s, case["matrix"])
        x = torch.randn((MATMUL_LAYERS, case["tokens"], K), generator=_gen(seed, "x"), device="cuda")
        y = torch.empty((MATMUL_LAYERS, case["tokens"], rows), device="cuda")
        return dict(case=case, dec=dec, lib=lib, x=x, y=y)
    hist, new = _inputs(case, seed)
    ctx = (case["positions"] + case["tokens"] + 64 + 31) // 32 * 32
    dec = S.HipQuantDecoder(S.Config(n_layers=case["layers"], ctx_len=ctx, **s))
    for layer in [-1] + list(range(case["layers"])):
        for name in ("token_embd", "output") if layer < 0 else MATRICES:
            fmt, b = _weight_bytes(case, seed, layer, name)
            dec.set_tensor(layer, KIND[name], FORMATS[fmt][0], b.cpu().numpy())
        for name in ("output_norm",) if layer < 0 else _vectors(case):
            dec.set_tensor(layer, KIND[name], S.F32, _vector(case, seed, layer, name).cpu().numpy())
    if hist:
        dec.observe(hist)
    st = dict(case=case, dec=dec, new=new)
    if case["kind"] == "tree":
        tokens, parents, path = _tree(seed, case["tokens"], hist[-1], s["vocab"])
        st.update(tree=(tokens, parents), path=path)
    return st


@functools.lru_cache(maxsize=None)
def _stream():
    """The one stream that all matrix products of this program go to: they share the library's staging rows."""
    return torch.cuda.Stream()


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "draft":
        d, (hidden3, emb), out = state["draft"], state["inputs"], []
        d.reset()
        h = hidden3
        for i in range(case["tokens"]):
            h, logits = d.forward_hidden(h, emb[i], case["positions"] + i)
            out.append((h, logits))
        return out
    dec = state["dec"]
    if kind == "matmul":
        x, y, n = state["x"], state["y"], case["tokens"]
        stream = _stream().cuda_stream
        for layer in range(MATMUL_LAYERS):
            if state["lib"].sd_model_qmatmul_noalloc(dec._h, layer, KIND[case["matrix"]], x[layer].data_ptr(), n,
                                                     y[layer].data_ptr(), stream):
                raise RuntimeError(state["lib"].sd_last_error().decode())
        return y
    n0 = case["positions"]
    if kind == "verify":
        logits = dec.batched_logits(state["new"][1:])
        dec.rollback_to(n0)
        return logits
    if kind == "tree":
        tree = state["tree"]
        _, hidden = dec.tree_logits_keep_kv(tree, want_logits=False)
        best = dec.last_argmax(case["tokens"])
        dec.commit_tree_path(tree, state["path"])
        dec.rollback_to(n0)
        return hidden, best
    dec.observe(state["new"])
    logits = dec.next_logits()
    dec.rollback_to(n0)
    return logits


# ---- the same in 64 bits ------------------------------------------------------------
def _norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, theta, interleaved):
    """x [heads][tokens][head_dim]"""
    hd = x.shape[-1]
    a = pos[:, None] * theta ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    c, s = a.cos(), a.sin()
    x0, x1 = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., :hd // 2], x[..., hd // 2:])
    y0, y1 = x0 * c - x1 * s, x0 * s + x1 * c
    return torch.stack([y0, y1], -1).reshape(x.shape) if interleaved else torch.cat([y0, y1], -1)


def _exact_decoder(case, seed):
    s, kind = SHAPES[case["shape"]], case["kind"]
    hist, new = _inputs(case, seed)
    eps, hd, nh, nkv = s["rms_eps"], s["head_dim"], s["n_heads"], s["n_kv_heads"]

    def W(layer, name):
        fmt, b = _weight_bytes(case, seed, layer, name)
        return _dequant(fmt, b).reshape(_dims(s, name))

    def V(layer, name):
        return _vector(case, seed, layer, name).double()

    if kind == "tree":
        toks, parents, _ = _tree(seed, case["tokens"], hist[-1], s["vocab"])
        P, ids = len(hist) - 1, hist[:-1] + toks
    elif kind == "verify":
        P, ids, parents = len(hist) - 1, hist + new[1:], None
    else:
        P, ids, parents = len(hist), hist + new, None
    n = len(ids)
    pos = torch.arange(n, device="cuda", dtype=torch.float64)
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
    if parents:
        m = np.zeros((len(parents), len(parents)), bool)
        depth = [0] * len(parents)
        for i, p in enumerate(parents):
            if i:
                m[i], depth[i] = m[p], depth[p] + 1
            m[i, i] = True
        mask[P:, P:] = torch.from_numpy(m).cuda()
        pos[P:] = P + torch.tensor(depth, device="cuda", dtype=torch.float64)
    fmt, b = _weight_bytes(case, seed, -1, "token_embd")
    per_row = s["hidden"] // FORMATS[fmt][1]
    used = b.reshape(s["vocab"], per_row, -1)[torch.tensor(ids, device="cuda")]
    h = _dequant(fmt, used.reshape(n * per_row, -1)).reshape(n, s["hidden"])
    for layer in range(case["layers"]):
        x = _norm(h, V(layer, "attn_norm"), eps)
        q, k, v = (x @ W(layer, "attn_" + c).T + (V(layer, "attn_%s_bias" % c) if case["shape"] == "qwen7b" else 0.0)
                   for c in "qkv")
        q, k, v = (t.reshape(n, -1, hd).transpose(0, 1) for t in (q, k, v))
        q, k = (_rope(t, pos, s["rope_theta"], s["arch"] == S.ARCH_LLAMA) for t in (q, k))
        y = torch.empty(n, nh, hd, device="cuda", dtype=torch.float64)
        for i in range(nh):
            sc = (q[i] @ k[i * nkv // nh].T / math.sqrt(hd)).masked_fill_(~mask, -math.inf)
            y[:, i] = torch.softmax(sc, -1) @ v[i * nkv // nh]
        h = h + y.reshape(n, -1) @ W(layer, "attn_output").T
        x = _norm(h, V(layer, "ffn_norm"), eps)
        g = x @ W(layer, "ffn_gate").T
        h = h + (g * torch.sigmoid(g) * (x @ W(layer, "ffn_up").T)) @ W(layer, "ffn_down").T
    out = _norm(h[P:], V(-1, "output_norm"), eps)
    if kind not in ("verify", "tree"):
        out = out[-1:]
    logits = out @ W(-1, "output").T
    if kind == "tree":
        return out, None
    return logits if kind == "verify" else logits[0]


def _exact_draft(case, seed):
    t = {k: v.double() for k, v in _draft_tensors(seed).items()}
    hidden3, emb = (torch.from_numpy(a).double().cuda() for a in _draft_inputs(case, seed))
    H, nh, nkv, eps = DRAFT["hidden"], DRAFT["n_heads"], DRAFT["n_kv_heads"], DRAFT["rms_eps"]
    hd = H // nh
    # the checkpoint's rotation tables are 16-bit: positions, frequencies and their products
    inv = (1.0 / np.power(np.float32(DRAFT["rope_theta"]), np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd)))
    keys, values, out, h = [], [], [], hidden3
    for i in range(case["tokens"]):
        a = (np.float64(np.float16(case["positions"] + i)) * inv.astype(np.float16).astype(np.float64)).astype(np.float16)
        c, s = (torch.from_numpy(f(a.astype(np.float64)).astype(np.float16)).double().cuda() for f in (np.cos, np.sin))
        p = t[S.D3_FC] @ h if i == 0 else h
        x = torch.cat([_norm(emb[i], t[S.D3_INPUT_NORM], eps), _norm(p, t[S.D3_HIDDEN_NORM], eps)])
        q, k, v = ((t[m] @ x).reshape(-1, hd) for m in (S.D3_Q, S.D3_K, S.D3_V))
        q, k = (torch.cat([z[:, :hd // 2] * c - z[:, hd // 2:] * s, z[:, :hd // 2] * s + z[:, hd // 2:] * c], 1) for z in (q, k))
        keys.append(k)
        values.append(v)
        K, V = (torch.stack(z, 1).repeat_interleave(nh // nkv, 0) for z in (keys, values))
        y = (torch.softmax((K @ q[:, :, None])[..., 0] / math.sqrt(hd), -1)[:, :, None] * V).sum(1)
        after = t[S.D3_O] @ y.reshape(-1) + p
        x = _norm(after, t[S.D3_POST_NORM], eps)
        g = t[S.D3_GATE] @ x
        h = t[S.D3_DOWN] @ (g * torch.sigmoid(g) * (t[S.D3_UP] @ x)) + after
        out.append((h, t[S.D3_LM_HEAD] @ _norm(h, t[S.D3_NORM], eps)))
    return out


def exact(case, seed):
    if case["kind"] == "draft":
        return _exact_draft(case, seed)
    if case["kind"] == "matmul":
        rows, K = _dims(SHAPES[case["shape"]], case["matrix"])
        x = torch.randn((MATMUL_LAYERS, case["tokens"], K), generator=_gen(seed, "x"), device="cuda").double()
        y = []
        for layer in range(MATMUL_LAYERS):
            fmt, b = _weight_bytes(case, seed, layer, case["matrix"])
            y.append(x[layer] @ _dequant(fmt, b).reshape(rows, K).T)
        return torch.stack(y)
    return _exact_decoder(case, seed)


# ---- what a pass cannot do without ----------------------------------------------------
def _matrix_bytes(fmt, rows, K):
    return rows * K // FORMATS[fmt][1] * FORMATS[fmt][2]


def work(case):
    n = case["tokens"]
    if case["kind"] == "draft":
        H, F = DRAFT["hidden"], DRAFT["ffn"]
        kd = H // DRAFT["n_heads"] * DRAFT["n_kv_heads"]
        step = (H + 2 * kd) * 2 * H + H * H + 3 * F * H + DRAFT["draft_vocab"] * H
        weights = 3 * H * H + n * step  # a step begins where the last one ended: each reads the weights
        return {"bytes": 2 * weights + n * 4 * (2 * H + DRAFT["draft_vocab"]), "flops": 2 * weights}
    s = SHAPES[case["shape"]]
    if case["kind"] == "matmul":
        rows, K = _dims(s, case["matrix"])
        return {"bytes": MATMUL_LAYERS * (_matrix_bytes(case["fmt"], rows, K) + 4 * n * (rows + K)),
                "flops": MATMUL_LAYERS * 2 * rows * K * n}
    P = case["positions"] - (case["kind"] in ("verify", "tree"))
    hd, nh, nkv = s["head_dim"], s["n_heads"], s["n_kv_heads"]
    by = fl = 0
    for layer in range(case["layers"]):
        for name in MATRICES:
            rows, K = _dims(s, name)
            by += _matrix_bytes(_fmt(case["mix"], case["layers"], layer, name), rows, K)
            fl += 2 * rows * K * n
        by += 2 * nkv * hd * 2 * (P + n)
        fl += 4 * nh * hd * (n * P + (n * (n + 1) // 2))
    out_rows = n if case["kind"] in ("verify", "tree") else 1
    rows, K = _dims(s, "output")
    by += _matrix_bytes(_fmt(case["mix"], case["layers"], -1, "output"), rows, K)
    by += 4 * out_rows * (K if case["kind"] == "tree" else rows)
    fl += 2 * rows * K * out_rows
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """Activations (above 16 rows weights too) are 16 bits wide at every matrix, sums 32.  Distances from exact(), as
    measured: one matrix 3.5e-4 to 6e-4, a draft chain 1.2e-3, 2 layers 2.5e-3, 4 layers 2.8e-3 to 5.7e-3, 8 layers
    4.1e-3, 32 layers 1.0e-2 (they grow with the root of the layers).  About four times that; of a tree's argmax rows
    a share of near ties may fall to the other token."""
    if case["kind"] == "matmul":
        return {"rel": 2e-3}
    if case["kind"] == "draft":
        return {"rel": 5e-3}
    most = 7e-3 * math.sqrt(case["layers"])
    return {"rel": most, "differ": 0.1} if case["kind"] == "tree" else {"rel": most}
