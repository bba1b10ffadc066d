"""The calls whose time this library is built for, as runnable cases.

Each case is one pass through the public entry points (g4run_amd over
include/g4hip.h), at the sizes of the library's own configurations: the
projections of a decoder layer for one token, for a prompt chunk and for a
large prompt batch; decode and prompt attention over a KV cache; the sampler;
a whole decode step; and a chat turn of a gemma4 model loaded from a GGUF
file.  `listed()` names them, `draw()` makes others of the same ranges,
`prepare()` makes a case's inputs on the GPU and `run()` is the pass.
"""
from __future__ import annotations

import ctypes as C
import math
import os
import struct
import tempfile

import numpy as np
import torch

import g4run_amd as G
from g4run_amd import synth

TYPES = {v: k for k, v in G.TYPE_NAMES.items()}
WEIGHTS = ["q4_0", "q8_0", "q4_K", "q6_K", "q5_K", "q3_K", "q2_K", "tq2_0", "f16", "bf16"]
KV = ["f16", "q8_0", "q4_0"]
MOST_ELEMENTS = 20480 * 2560          # weights of one drawn matrix
MOST_FLOPS = 2 * 509 * 4096 * 11008


def listed():
    return [
        # one token through the smallest matrix of a decode step (a gemma4
        # per-layer input gate): call and launch latency, nothing else
        dict(name="gemv_f16_gate", kind="matmul", wtype="f16", rows=256, cols=2048, nb=1, layers=1, pair=False),
        # one token through the FFN pairs (up, down) of eight decoder layers,
        # replayed from a captured graph as a decode loop does
        dict(name="gemv_q4_0_ffn", kind="matmul", wtype="q4_0", rows=10240, cols=2560, nb=1, layers=8, pair=True),
        # one token through eight K-quant matrices (q4_K_M files)
        dict(name="gemv_q4_K", kind="matmul", wtype="q4_K", rows=4096, cols=11008, nb=1, layers=8, pair=False),
        # a full prompt chunk through a fused gate/up projection
        dict(name="chunk_q4_0_gate_up", kind="matmul", wtype="q4_0", rows=20480, cols=2560, nb=64, layers=1, pair=False),
        # large prompt batches: square projection, K-quant projection with a
        # ragged token count, half-precision projection with an odd one
        dict(name="batch_q8_0", kind="matmul", wtype="q8_0", rows=4096, cols=4096, nb=512, layers=1, pair=False),
        dict(name="batch_q4_K", kind="matmul", wtype="q4_K", rows=4096, cols=11008, nb=509, layers=1, pair=False),
        dict(name="batch_f16", kind="matmul", wtype="f16", rows=4096, cols=4096, nb=201, layers=1, pair=False),
        # one token's attention over a long q8_0 cache
        dict(name="attn_decode_q8_0", kind="attn_decode", kv="q8_0", n_head=8, n_kv=4, hd=256, n_pos=8191),
        # a prompt chunk's attention behind a 4096-position f16 cache
        dict(name="attn_chunk_f16", kind="attn_chunk", n_head=8, n_kv=4, hd=256, pos0=4096, nb=64, window=0),
        # drawing one token from a gemma-sized vocabulary
        dict(name="sample_262144", kind="sample", n_vocab=262144, top_k=40, top_p=0.95, repeat_penalty=1.1, history=128),
        # four decode steps of the 26-layer decoder at the end of 8192 positions
        dict(name="decode_steps", kind="decode", n_layer=26, pos=8160, n_ctx=8192, steps=4),
        # a chat turn of a gemma4 file: a 64-token prompt chunk behind 1024
        # positions, then four decode steps
        dict(name="gemma4_turn", kind="gemma", n_layer=6, pos=1024, nb=64, steps=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matmul"] * 6 + ["attn_decode"] * 2 + ["attn_chunk"] * 2 + ["sample", "decode"])
    if kind == "matmul":
        wt = rng.choice(WEIGHTS)
        step = 16 if wt in ("f16", "bf16") else G.BLCK[TYPES[wt]]
        cols = max(1, _log(rng, 256, 11008) // step) * step
        rows = min(_log(rng, 256, 20480), MOST_ELEMENTS // cols)
        nb = min(_log(rng, 1, 512), max(1, MOST_FLOPS // (2 * rows * cols)))
        one = rows * G.SIZE[TYPES[wt]] * cols // G.BLCK[TYPES[wt]]
        layers = rng.randint(1, max(1, min(8, (200 << 20) // one))) if nb <= 8 else 1
        return dict(kind=kind, wtype=wt, rows=rows, cols=cols, nb=nb, layers=layers, pair=False)
    if kind == "attn_decode":
        n_kv = rng.choice([1, 2, 4])
        return dict(kind=kind, kv=rng.choice(KV), n_head=n_kv * rng.choice([1, 2, 4, 8]), n_kv=n_kv, hd=rng.choice([64, 128, 256]),
                    n_pos=_log(rng, 100, 16384))
    if kind == "attn_chunk":
        n_kv = rng.choice([1, 2, 4])
        return dict(kind=kind, n_head=n_kv * rng.choice([1, 2, 4, 8]), n_kv=n_kv, hd=rng.choice([64, 128, 256, 512]),
                    pos0=_log(rng, 1, 8192), nb=rng.randint(9, 64), window=rng.choice([0, 0, 512]))
    if kind == "sample":
        return dict(kind=kind, n_vocab=4 * _log(rng, 8000, 65536), top_k=rng.choice([0, 20, 40, 64, 100]), top_p=rng.choice([0.9, 0.95, 1.0]),
                    repeat_penalty=rng.choice([1.0, 1.1]), history=rng.randint(0, 512))
    n_ctx = _log(rng, 512, 8192)
    return dict(kind="decode", n_layer=rng.randint(2, 26), pos=rng.randint(64, n_ctx - 8), n_ctx=n_ctx, steps=rng.randint(1, 4))


# ------------------------------------------------------------- the matrices
def _shapes(c):
    """(rows, cols) of every matrix of a pass."""
    one = [(c["rows"], c["cols"])] + ([(c["cols"], c["rows"])] if c["pair"] else [])
    return one * c["layers"]


def _matrices(c, seed):
    """Host GGUF rows and fp32 inputs of every matrix of a pass."""
    t = TYPES[c["wtype"]]
    for i, (rows, cols) in enumerate(_shapes(c)):
        yield t, rows, cols, synth.weights(t, rows, cols, seed=1000 * seed + 2 * i), synth.activations(c["nb"], cols, seed=1000 * seed + 2 * i + 1)


_STREAM = []


def _stream():
    """The one stream of the captured work: a decode loop's passes follow each
    other."""
    if not _STREAM:
        _STREAM.append(G.Stream())
    return _STREAM[0]


def _graph(run):
    """`run(stream)` captured into a graph (after one eager call, which sets up
    any scratch)."""
    s = _stream()
    run(s.ptr)
    s.synchronize()
    return s, G.Graph(s.ptr, lambda: run(s.ptr))


def _prepare_matmul(c, seed):
    W, X, Y = [], [], []
    for t, rows, cols, w, x in _matrices(c, seed):
        W.append(G.Tensor.from_rows(t, w, cols))
        X.append(torch.from_numpy(x).cuda())
        Y.append(torch.empty(c["nb"], rows, device="cuda"))
    st = dict(W=W, X=X, Y=Y, nb=c["nb"], graph=None)
    torch.cuda.synchronize()
    if c["layers"] > 1:
        st["stream"], st["graph"] = _graph(lambda s: _matmuls(st, s))
    return st


def _matmuls(st, stream=None):
    for W, x, y in zip(st["W"], st["X"], st["Y"]):
        G.matmul(W, y.data_ptr(), nb=st["nb"], x=x.data_ptr(), stream=stream)


# ------------------------------------------------------------ the attention
def _prepare_attn(c, seed):
    G.init()
    g = torch.Generator(device="cuda").manual_seed(seed)
    chunk = c["kind"] == "attn_chunk"
    nb, kvt = (c["nb"], G.F16) if chunk else (1, TYPES[c["kv"]])
    H, KVH, hd = c["n_head"], c["n_kv"], c["hd"]
    n_pos = c["pos0"] + nb if chunk else c["n_pos"]
    win = c.get("window", 0)
    # queries whose scores spread by about 2, as a trained model's do
    q = torch.randn(nb, H, hd, device="cuda", generator=g) * (2.0 / math.sqrt(hd))
    raw = [torch.randn(n_pos, KVH, hd, device="cuda", generator=g) for _ in range(2)]
    caches = []
    ring = 576 if win else 0
    for r in raw:
        if ring:                                     # slot p % ring, stored twice
            b = torch.zeros(2 * ring, KVH, hd, device="cuda", dtype=torch.float16)
            p = torch.arange(max(0, n_pos - ring), n_pos, device="cuda")
            b[p % ring] = r[p].half()
            b[p % ring + ring] = r[p].half()
        else:
            b = torch.empty(n_pos * KVH * G.row_size(kvt, hd), device="cuda", dtype=torch.uint8)
            torch.cuda.synchronize()
            G.kv_store(kvt, r.data_ptr(), b.data_ptr(), hd, rows=n_pos * KVH)
        caches.append(b)
    need = G.attn_prefill_workspace_bytes(H, hd, c["pos0"], nb) if chunk else G.attn_workspace_bytes(H, hd, n_pos)
    st = dict(c=c, q=q, k=caches[0], v=caches[1], out=torch.empty(nb, H, hd, device="cuda"), ws=G.Buffer(need), ring=ring, kvt=kvt, raw=raw)
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------- a gemma4 GGUF file
GEMMA = dict(n_embd=2048, n_head=8, hd_full=512, hd_swa=256, n_ff=6144, ple=256, n_vocab=32768, swa=512)


def _sliding(i):
    return i % 2 == 0 or i == 1


def _gguf_str(s):
    return struct.pack("<Q", len(s)) + s.encode()


def _write_gemma(path, n_layer, seed):
    """A gemma4 file of the library's head widths (8 query heads of 512 on full
    layers, 256 on sliding ones, one KV head) with the weight types such files
    mix; the last two layers share their KV."""
    m, rng = GEMMA, np.random.default_rng(seed)
    E, H, F, P, V = m["n_embd"], m["n_head"], m["n_ff"], m["ple"], m["n_vocab"]
    kinds = [int(_sliding(i)) for i in range(n_layer)]
    T = []

    def mat(name, t, cols, rows):
        T.append((name, TYPES[t], [cols, rows], synth.weights(TYPES[t], rows, cols, seed=int(rng.integers(1 << 40)))))

    def vec(name, n, mean=1.0, sd=0.1):
        T.append((name, G.F32, [n], (mean + sd * rng.standard_normal(n)).astype(np.float32)))

    mat("token_embd.weight", "q8_0", E, V)
    mat("per_layer_token_embd.weight", "q4_0", n_layer * P, V)
    mat("per_layer_model_proj.weight", "q8_0", E, n_layer * P)
    vec("per_layer_proj_norm.weight", P)
    vec("output_norm.weight", E)
    vec("rope_freqs.weight", m["hd_full"] // 2, 2.0, 0.2)
    for i in range(n_layer):
        p, hd = f"blk.{i}.", m["hd_swa"] if kinds[i] else m["hd_full"]
        for n in ("attn_norm", "ffn_norm"):
            vec(p + n + ".weight", E)
        for n in ("post_attention_norm", "post_ffw_norm", "post_norm"):    # a layer adds a part of the residual's size
            vec(p + n + ".weight", E, 0.25, 0.02)
        vec(p + "attn_q_norm.weight", hd, 2.0 / math.sqrt(hd), 0.01)       # scores that spread by about 2
        mat(p + "attn_q.weight", "q8_0", E, H * hd)
        if i < n_layer - 2:
            vec(p + "attn_k_norm.weight", hd)
            mat(p + "attn_k.weight", "q4_0", E, hd)
            mat(p + "attn_v.weight", "q8_0", E, hd)
        mat(p + "attn_output.weight", "q4_K", H * hd, E)
        mat(p + "ffn_gate.weight", "q4_0", E, F)
        mat(p + "ffn_up.weight", "q8_0", E, F)
        mat(p + "ffn_down.weight", "q6_K", F, E)
        mat(p + "inp_gate.weight", "f16", E, P)
        mat(p + "proj.weight", "bf16", P, E)
        vec(p + "layer_output_scale.weight", 1, 0.9, 0.05)
    u32, f32, bl, st, ar = 4, 6, 7, 8, 9
    g = "gemma4."
    meta = [("general.architecture", st, "gemma4"), (g + "block_count", u32, n_layer), (g + "context_length", u32, 131072),
            (g + "embedding_length", u32, E), (g + "feed_forward_length", ar, (5, [F] * n_layer)), (g + "attention.head_count", u32, H),
            (g + "attention.head_count_kv", u32, 1), (g + "rope.freq_base", f32, 1e6), (g + "rope.freq_base_swa", f32, 1e4),
            (g + "attention.layer_norm_rms_epsilon", f32, 1e-6), (g + "attention.key_length", u32, m["hd_full"]),
            (g + "attention.key_length_swa", u32, m["hd_swa"]), (g + "final_logit_softcapping", f32, 30.0),
            (g + "attention.sliding_window", u32, m["swa"]), (g + "attention.shared_kv_layers", u32, 2),
            (g + "embedding_length_per_layer_input", u32, P), (g + "rope.dimension_count", u32, m["hd_full"]),
            (g + "rope.dimension_count_swa", u32, m["hd_swa"]), (g + "attention.sliding_window_pattern", ar, (bl, kinds)),
            ("tokenizer.ggml.tokens", ar, (st, ["<t%d>" % i for i in range(V)]))]
    fmt = {4: "<I", 5: "<i", 6: "<f", 7: "<B"}
    head = struct.pack("<IIQQ", 0x46554747, 3, len(T), len(meta))
    for key, t, v in meta:
        head += _gguf_str(key) + struct.pack("<I", t)
        if t == ar:
            head += struct.pack("<IQ", v[0], len(v[1])) + b"".join(_gguf_str(x) if v[0] == st else struct.pack(fmt[v[0]], x) for x in v[1])
        else:
            head += _gguf_str(v) if t == st else struct.pack(fmt[t], v)
    at = 0
    for name, t, ne, a in T:
        head += _gguf_str(name) + struct.pack("<I", len(ne)) + b"".join(struct.pack("<Q", n) for n in ne) + struct.pack("<IQ", t, at)
        at += (a.nbytes + 31) // 32 * 32
    with open(path, "wb") as f:
        f.write(head + b"\0" * (-len(head) % 32))
        for _, _, _, a in T:
            f.write(memoryview(np.ascontiguousarray(a)).cast("B"))
            f.write(b"\0" * (-a.nbytes % 32))


def _ints(a):
    return np.ascontiguousarray(a, np.int32).ctypes.data_as(C.POINTER(C.c_int))


def _prepare_gemma(c, seed):
    fd, path = tempfile.mkstemp(suffix=".gguf")
    os.close(fd)
    try:
        _write_gemma(path, c["n_layer"], seed)
        g = G.Gemma(path, n_ctx=4096)
    finally:
        os.unlink(path)
    rng = np.random.default_rng(seed + 1)
    for p in range(0, c["pos"], 64):                 # the turns before this one
        n = min(64, c["pos"] - p)
        g.prefill(rng.integers(0, g.n_vocab, n), p, want_logits=False)
    toks = np.ascontiguousarray(rng.integers(0, g.n_vocab, c["nb"]), np.int32)
    st = dict(c=c, g=g, toks=toks, ids=_ints(toks), first=int(rng.integers(g.n_vocab)), prompt=torch.empty(g.n_vocab, device="cuda"),
              last=torch.empty(g.n_vocab, device="cuda"), lp=G.lib().g4h_gemma_logits(g.ptr))
    g.set_state(st["first"], c["pos"] + c["nb"])
    st["stream"], st["graph"] = _graph(lambda s: g.step(s))
    torch.cuda.synchronize()
    return st


def _run_gemma(st):
    c, g, s, L = st["c"], st["g"], st["stream"].ptr, G.lib()
    G.check(L.g4h_gemma_prefill(g.ptr, st["ids"], c["nb"], c["pos"], st["prompt"].data_ptr(), s))
    g.set_state(st["first"], c["pos"] + c["nb"], s)
    for _ in range(c["steps"]):
        st["graph"].launch(s)
    G.check(L.g4h_memcpy_d2d(st["last"].data_ptr(), st["lp"], 4 * g.n_vocab, s))
    return {"prompt": st["prompt"], "last": st["last"]}


# ------------------------------------------------------------ the decode step
def _prepare_decode(c, seed):
    m = G.Model(seed=seed, n_layer=c["n_layer"], n_ctx=c["n_ctx"])
    m.fill_kv(seed + 1)
    torch.cuda.synchronize()
    st = dict(c=c, m=m, tok=seed % m.cfg["n_vocab"], logits=torch.empty(m.cfg["n_vocab"], device="cuda"), lp=G.lib().g4h_model_logits(m.ptr))
    m.set_state(st["tok"], c["pos"])
    st["stream"], st["graph"] = _graph(lambda s: m.forward_state(s))
    torch.cuda.synchronize()
    return st


def _run_decode(st):
    c, m, s = st["c"], st["m"], st["stream"].ptr
    m.set_state(st["tok"], c["pos"], s)
    for _ in range(c["steps"]):
        st["graph"].launch(s)
    G.check(G.lib().g4h_memcpy_d2d(st["logits"].data_ptr(), st["lp"], 4 * m.cfg["n_vocab"], s))
    return st["logits"]


# ---------------------------------------------------------------- the sampler
def _prepare_sample(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    fresh = torch.randn(c["n_vocab"], device="cuda", generator=g) * 3.0
    s = G.Sampler(c["n_vocab"], temp=0.8, top_k=c["top_k"], top_p=c["top_p"], repeat_penalty=c["repeat_penalty"], repeat_last_n=256, seed=seed)
    if c["history"]:
        s.accept(np.random.default_rng(seed).integers(0, c["n_vocab"], c["history"]))
    st = dict(s=s, fresh=fresh, logits=torch.empty_like(fresh), id=torch.zeros(1, device="cuda", dtype=torch.int32))
    torch.cuda.synchronize()
    return st


def _run_sample(st):
    st["logits"].copy_(st["fresh"])                  # the head's output of this step
    st["s"].sample(st["logits"].data_ptr(), out=st["id"].data_ptr(), accept=True)
    return {"id": st["id"], "logits": st["logits"]}


# ----------------------------------------------------------------- the passes
def prepare(case, seed):
    G.init()
    return dict({"matmul": _prepare_matmul, "attn_decode": _prepare_attn, "attn_chunk": _prepare_attn, "sample": _prepare_sample,
                 "decode": _prepare_decode, "gemma": _prepare_gemma}[case["kind"]](case, seed), kind=case["kind"])


def run(st):
    k = st["kind"]
    if k == "matmul":
        if st["graph"] is not None:
            st["graph"].launch(st["stream"].ptr)
        else:
            _matmuls(st)
        return st["Y"]
    if k == "attn_decode":
        c = st["c"]
        G.attn_decode(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), st["kvt"], c["n_head"], c["n_kv"], c["hd"], c["n_pos"],
                      st["out"].data_ptr(), ws=st["ws"])
        return st["out"]
    if k == "attn_chunk":
        c = st["c"]
        G.attn_prefill_mm(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), st["kvt"], c["n_head"], c["n_kv"], c["hd"], c["pos0"],
                          c["nb"], st["out"].data_ptr(), window=c["window"], ring=st["ring"], ws=st["ws"])
        return st["out"]
    return {"sample": _run_sample, "decode": _run_decode, "gemma": _run_gemma}[k](st)


def _row_bytes(t, n):
    return n // G.BLCK[t] * G.SIZE[t]


def _kv_positions(c):
    if c["kind"] == "attn_decode":
        return c["n_pos"], c["n_pos"]
    n = c["pos0"] + c["nb"]
    w = c["window"]
    read = n - max(0, c["pos0"] + 1 - w) if w else n
    each = sum(min(c["pos0"] + b + 1, w or n) for b in range(c["nb"]))
    return read, each


def work(case):
    c, k = case, case["kind"]
    if k == "matmul":
        t, by, fl = TYPES[c["wtype"]], 0, 0
        for rows, cols in _shapes(c):
            by += rows * _row_bytes(t, cols) + 4 * c["nb"] * (rows + cols)
            fl += 2 * c["nb"] * rows * cols
        return {"bytes": by, "flops": fl}
    if k in ("attn_decode", "attn_chunk"):
        t = TYPES[c["kv"]] if k == "attn_decode" else G.F16
        nb = c.get("nb", 1)
        read, each = _kv_positions(c)
        return {"bytes": 2 * read * c["n_kv"] * _row_bytes(t, c["hd"]) + 8 * nb * c["n_head"] * c["hd"], "flops": 4 * each * c["n_head"] * c["hd"]}
    if k == "sample":
        return {"bytes": 4 * c["n_vocab"], "flops": c["n_vocab"]}
    if k == "decode":
        m = G.GEMMA_STYLE
        E, F, hd = m["n_embd"], m["n_ff"], m["head_dim"]
        R, Q = (m["n_head"] + 2 * m["n_kv"]) * hd, m["n_head"] * hd
        per = R * E + Q * E + 3 * F * E
        kv = sum(2 * (c["pos"] + i + 1) * m["n_kv"] * hd for i in range(c["steps"]))
        by = c["steps"] * (c["n_layer"] * per * 18 // 32 + m["n_vocab"] * E * 34 // 32 + 4 * m["n_vocab"]) + c["n_layer"] * kv * 2
        fl = 2 * c["steps"] * (c["n_layer"] * per + m["n_vocab"] * E) + c["n_layer"] * kv * 2 * (m["n_head"] // m["n_kv"])
        return {"bytes": by, "flops": fl}
    # gemma: the weights once for the chunk and once per step; the K and V rows of each
    m, by, el, att = GEMMA, 0, 0, 0
    E, H, F, P, V = m["n_embd"], m["n_head"], m["n_ff"], m["ple"], m["n_vocab"]
    for i in range(c["n_layer"]):
        swa = _sliding(i)
        hd = m["hd_swa"] if swa else m["hd_full"]
        own = i < c["n_layer"] - 2
        n = {"q8_0": E * H * hd + (E * hd if own else 0) + E * F, "q4_0": (E * hd if own else 0) + E * F, "q4_K": H * hd * E, "q6_K": F * E,
             "f16": 2 * E * P}
        by += sum(v * G.SIZE[TYPES[t]] // G.BLCK[TYPES[t]] for t, v in n.items())
        el += sum(n.values())
        att += min(c["pos"] + c["nb"], m["swa"] if swa else 1 << 30) * hd
    by += (E * c["n_layer"] * P + E * V) * 34 // 32
    el += E * c["n_layer"] * P
    passes = 1 + c["steps"]
    return {"bytes": passes * (by + 4 * att), "flops": 2 * el * (c["nb"] + c["steps"]) + passes * 2 * E * V + 4 * H * att * (c["nb"] + c["steps"])}


def tolerance(case):
    k = case["kind"]
    if k == "sample":
        return "exact"
    if k == "matmul":
        # exact integer (or f16 / bf16) products, fp32 sums over the row: the two
        # kernel families differ by 1.1e-7 to 2.2e-7
        return {"rel": 2e-6}
    if k in ("attn_decode", "attn_chunk"):
        # a last-bit difference of a score moves single weights to the next
        # fp16 value: the per-token and the prompt kernels differ by 1.2e-5
        # (4e-4 at most)
        return {"rel": 5e-5, "max": 2e-3}
    # whole models: one rounding of a quantized activation travels through all
    # later layers
    return {"rel": 0.03}


# ---------------------------------------------------------- 64-bit reference
def _half(b):
    return b.contiguous().view(torch.float16).double()


def _k4(s):
    """6-bit scales and mins of q4_K / q5_K from their 12 bytes: [..., 8] each."""
    sc = torch.cat([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
    return sc.double(), mn.double()


def _dequant(t, rows, n):
    """GGUF rows (uint8 [r, bytes]) as float64 [r, n]."""
    r = rows.shape[0]
    if t == G.F16:
        return _half(rows)
    if t == G.BF16:
        return rows.contiguous().view(torch.bfloat16).double()
    b = rows.reshape(r, n // G.BLCK[t], G.SIZE[t])
    rep = lambda x, k: x.repeat_interleave(k, -1)  # noqa: E731
    if t == G.Q8_0:
        v = b[..., 2:].contiguous().view(torch.int8).double() * _half(b[..., :2])
    elif t == G.Q4_0:
        q = b[..., 2:]
        v = (torch.cat([q & 15, q >> 4], -1).double() - 8) * _half(b[..., :2])
    elif t == G.TQ2_0:
        q = b[..., :64].reshape(r, -1, 2, 32)
        v = (torch.stack([(q >> (2 * j)) & 3 for j in range(4)], 3).reshape(r, -1, 256).double() - 1) * _half(b[..., 64:66])
    elif t == G.Q2_K:
        q = b[..., 16:80].reshape(r, -1, 2, 32)
        q = torch.stack([(q >> (2 * j)) & 3 for j in range(4)], 3).reshape(r, -1, 256).double()
        v = q * rep((b[..., :16] & 15).double(), 16) * _half(b[..., 80:82]) - rep((b[..., :16] >> 4).double(), 16) * _half(b[..., 82:84])
    elif t == G.Q3_K:
        q = b[..., 32:96].reshape(r, -1, 2, 32)
        lo = torch.stack([(q >> (2 * j)) & 3 for j in range(4)], 3).reshape(r, -1, 256).double()
        hb = torch.stack([(b[..., :32] >> j) & 1 for j in range(8)], 2).reshape(r, -1, 256).double()
        s = b[..., 96:108]
        sc = torch.cat([s[..., :8] & 15, s[..., :8] >> 4], -1) | (torch.cat([(s[..., 8:12] >> (2 * j)) & 3 for j in range(4)], -1) << 4)
        v = (lo - 4 * (1 - hb)) * rep(sc.double() - 32, 16) * _half(b[..., 108:110])
    elif t in (G.Q4_K, G.Q5_K):
        sc, mn = _k4(b[..., 4:16])
        q = b[..., -128:].reshape(r, -1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).reshape(r, -1, 256).double()
        if t == G.Q5_K:
            q = q + 16 * torch.stack([(b[..., 16:48] >> j) & 1 for j in range(8)], 2).reshape(r, -1, 256).double()
        v = q * rep(sc, 32) * _half(b[..., :2]) - rep(mn, 32) * _half(b[..., 2:4])
    else:                                            # q6_K
        ql, qh = b[..., :128].reshape(r, -1, 2, 2, 32), b[..., 128:192].reshape(r, -1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 3)
        hi = torch.cat([(qh >> (2 * j)) & 3 for j in range(4)], 3)
        q = (lo | (hi << 4)).reshape(r, -1, 256).double() - 32
        v = q * rep(b[..., 192:208].contiguous().view(torch.int8).double(), 16) * _half(b[..., 208:210])
    return v.reshape(r, n)


def _activation(t, x):
    """The activation a weight type is multiplied with (x rounded to f16 or
    bf16, or quantized to blocks of 32 or 256 in fp32 arithmetic: host tensors,
    whose divisions are IEEE), as float64."""
    if t == G.F16:
        return x.half().double()
    if t == G.BF16:
        return x.bfloat16().double()
    if t in (G.Q4_0, G.Q8_0):
        b = x.reshape(x.shape[0], -1, 32)
        amax = b.abs().amax(-1, keepdim=True)
        q = torch.round(b * torch.div(torch.tensor(127.0), amax)).double()
        return (q * (amax * np.float32(1 / 127.0)).half().double()).reshape(x.shape)
    b = x.reshape(x.shape[0], -1, 256)
    smax = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    q = torch.round(b.double() * torch.div(torch.tensor(-127.0), smax).double()).clamp(max=127)
    return (q * (smax * np.float32(-1 / 127.0)).double()).reshape(x.shape)


def _exact_attn(c, seed):
    st = _prepare_attn(c, seed)
    chunk, hd, grp = c["kind"] == "attn_chunk", c["hd"], c["n_head"] // c["n_kv"]
    if chunk:
        q = st["q"].half().double()
        k, v = (r.half().double() for r in st["raw"])
    elif st["kvt"] == G.F16:
        q = st["q"].half().double()
        k, v = (r.half().double() for r in st["raw"])
    else:
        q = _activation(G.Q8_0, st["q"].reshape(-1, hd).cpu()).cuda().reshape(st["q"].shape)
        k, v = (_dequant(st["kvt"], st[n].reshape(-1, G.row_size(st["kvt"], hd)), hd).reshape(-1, c["n_kv"], hd) for n in ("k", "v"))
    out = torch.empty_like(q)
    nb, n = q.shape[0], k.shape[0]
    p = torch.arange(n, device="cuda")[None, :]
    at = torch.arange(n - nb, n, device="cuda")[:, None]
    seen = (p <= at) & (p > at - (c.get("window") or n))
    for h in range(c["n_head"]):
        s = (q[:, h] @ k[:, h // grp].T.contiguous()).masked_fill(~seen, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // grp].contiguous()
    return out


def exact(case, seed):
    if case["kind"] in ("attn_decode", "attn_chunk"):
        return _exact_attn(case, seed)
    if case["kind"] != "matmul":
        return None
    Y = []
    for t, rows, cols, w, x in _matrices(case, seed):
        a = _activation(t, torch.from_numpy(x)).cuda()
        y = torch.empty(case["nb"], rows, device="cuda", dtype=torch.float64)
        raw = torch.from_numpy(w)
        for r in range(0, rows, 2048):               # a strip of rows at a time
            y[:, r:r + 2048] = a @ _dequant(t, raw[r:r + 2048].cuda(), cols).T.contiguous()
        Y.append(y)
    return Y
