"""The measured cases: what a program that runs Gemma 4 E4B K-quant models calls.

Single layers and blocks go through the C ABI (include/g4hip.h) by its ctypes
binding, whole prompts and decode steps through the engine.  Sizes are the
E4B shape's (hidden 2560, FFN 10240, 8 query / 2 KV heads of 256 or 512,
window 512, vocabulary 262144), those of the tests, and ragged ones.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "gemma4.c_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "gemma4.c_amd"))
import g4  # noqa: E402
import synth  # noqa: E402

TYPES = {"Q4_K": g4.Q4_K, "Q5_K": g4.Q5_K, "Q6_K": g4.Q6_K, "BF16": g4.BF16}
N_HEADS, N_KV, WINDOW = 8, 2, 512
# the engine cases' model: E4B widths, one period of its layer pattern (five
# sliding-window layers and a global one), a smaller vocabulary
LAYERS, VOCAB, MAX_SEQ = 6, 16384, 1024
CAP = 30.0


def listed():
    return [
        # one token through the per-layer-embedding gate: the smallest matrix of a decode step
        {"name": "mm_ple_gate", "kind": "mm", "type": "Q4_K", "n": 2560, "d": 256},
        # one token through the FFN of six layers: most of a decode step's bytes
        {"name": "ffn_token", "kind": "ffn", "type": "Q4_K", "n": 2560, "hidden": 10240, "layers": 6},
        # the tied LM head of one token, with the greedy pick
        {"name": "lm_head", "kind": "head", "n": 2560, "d": 262144},
        # one token's attention on a sliding-window layer, and on a global layer at a long context
        {"name": "attn_window", "kind": "attn", "hd": 256, "positions": 512},
        {"name": "attn_long", "kind": "attn", "hd": 512, "positions": 32768},
        # a short chat message through eight layers' Q4_K matrices
        {"name": "gemm_short", "kind": "batch", "type": "Q4_K", "n": 2560, "d": 10240, "m": 37, "layers": 8},
        # a whole prompt chunk through four layers' FFN down
        {"name": "gemm_q6k", "kind": "batch", "type": "Q6_K", "n": 10240, "d": 2560, "m": 512, "layers": 4},
        # the same chunk's per-layer-embedding context projection (once per prompt)
        {"name": "gemm_bf16", "kind": "batch", "type": "BF16", "n": 2560, "d": 10752, "m": 511, "layers": 2},
        # a prompt chunk's attention: sliding window after earlier chunks, and global late in a long prompt
        {"name": "attn_rows_window", "kind": "rows", "hd": 256, "m": 511, "p0": 1001, "window": WINDOW},
        {"name": "attn_rows_full", "kind": "rows", "hd": 512, "m": 512, "p0": 7680, "window": 0},
        # a 512-token prompt: 511 tokens in one chunk, the last one with logits
        {"name": "prompt", "kind": "prompt", "tokens": 512},
        # eight decode steps of a conversation, logits read after each
        {"name": "decode", "kind": "decode", "pos": 448, "steps": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mm", "ffn", "head", "attn", "batch", "batch", "rows", "prompt", "decode"])
    if kind == "mm":
        return {"kind": kind, "type": rng.choice(["Q4_K", "Q5_K", "Q6_K", "BF16"]), "n": 256 * rng.randint(1, 40),
                "d": _log(rng, 64, 12288)}
    if kind == "ffn":
        return {"kind": kind, "type": rng.choice(["Q4_K", "Q5_K"]), "n": 256 * rng.randint(4, 16),
                "hidden": 256 * rng.randint(8, 48), "layers": rng.randint(2, 6)}
    if kind == "head":
        return {"kind": kind, "n": 256 * rng.randint(4, 12), "d": _log(rng, 16384, 262144)}
    if kind == "attn":
        return {"kind": kind, "hd": rng.choice([256, 512]), "positions": _log(rng, 8, 32768)}
    if kind == "batch":
        t = rng.choice(["Q4_K", "Q5_K", "Q6_K", "BF16"])
        n, d = rng.choice([(2560, 10240), (2560, 2048), (2560, 10752), (10240, 2560), (4096, 2560), (2048, 2560),
                           (2560, 512), (256, 2560), (1536, 1000)])
        return {"kind": kind, "type": t, "n": n, "d": d, "m": _log(rng, 2, 512), "layers": rng.randint(1, 4)}
    if kind == "rows":
        hd = rng.choice([256, 512])
        return {"kind": kind, "hd": hd, "m": _log(rng, 4, 512), "p0": rng.choice([0, rng.randint(1, 7680)]),
                "window": WINDOW if hd == 256 else 0}
    if kind == "prompt":
        return {"kind": kind, "tokens": _log(rng, 4, 512)}
    return {"kind": kind, "pos": rng.randint(4, 500), "steps": rng.randint(2, 8)}


# ---------------------------------------------------------------------------
# weights: the repository's synthetic K-quant recipe, made on the GPU
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed * 7919 + 17)


def _kquant(g, qtype, rows, n):
    """GGUF bytes [rows, blocks, block bytes] of random blocks"""
    nb, size = n // 256, synth.BLOCK_BYTES[qtype]
    words = torch.randint(-2 ** 31, 2 ** 31 - 1, ((rows * nb * size + 3) // 4,), dtype=torch.int32, device="cuda",
                          generator=g)
    b = words.view(torch.uint8)[: rows * nb * size].reshape(rows, nb, size).clone()

    def half():
        v = torch.randn((rows, nb, 1), device="cuda", generator=g).abs() * 1e-3
        return v.to(torch.float16).view(torch.uint8)

    if qtype == g4.Q6_K:
        b[..., 192:208] = torch.randint(-32, 32, (rows, nb, 16), dtype=torch.int8, device="cuda",
                                        generator=g).view(torch.uint8)
        b[..., 208:210] = half()
    else:
        b[..., 0:2] = half()
        b[..., 2:4] = half()
    return b


def _raw(g, qtype, rows, n):
    if qtype == g4.BF16:
        return (torch.randn((rows, n), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    return _kquant(g, qtype, rows, n)


def _place(lib, raw, qtype, n, d):
    """the tensor as the library keeps it in HBM"""
    if qtype == g4.BF16:
        return raw
    dst = torch.empty(raw.numel(), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    lib.g4_relayout_quant(dst.data_ptr(), raw.data_ptr(), qtype, n, d)
    lib.g4_sync()
    return dst


def _rows(g, m, n):
    """activations as a norm leaves them: unit rms times norm weights"""
    w = torch.rand(n, device="cuda", generator=g) * 0.4 + 0.8
    return torch.randn((m, n), device="cuda", generator=g) * w


def _heads(g, rows, heads, hd, k_norm=False):
    """q or k heads after their norms; the K norm's weights carry hd^-1/2
    (the attention scale itself is 1)"""
    x = torch.randn((rows, heads, hd), device="cuda", generator=g)
    x = x / x.square().mean(-1, keepdim=True).sqrt()
    return (x * (hd ** -0.5 if k_norm else 1.0)).reshape(rows, heads * hd).contiguous()


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _matrix_inputs(case, seed):
    """(raw matrices, x) of an mm, head or batch case"""
    g = _gen(seed)
    t = TYPES[case.get("type", "Q6_K")]
    raws = [_raw(g, t, case["d"], case["n"]) for _ in range(case.get("layers", 1))]
    return t, raws, _rows(g, case.get("m", 1), case["n"])


def _ffn_inputs(case, seed):
    g = _gen(seed)
    t = TYPES[case["type"]]
    n, hidden = case["n"], case["hidden"]
    raws = [(_raw(g, t, hidden, n), _raw(g, t, hidden, n), _raw(g, g4.Q6_K, n, hidden)) for _ in range(case["layers"])]
    return t, raws, _rows(g, case["layers"], n)


def _attn_inputs(case, seed):
    g = _gen(seed)
    hd = case["hd"]
    if case["kind"] == "attn":
        pos, m = case["positions"], 1
    else:
        pos, m = case["p0"] + case["m"], case["m"]
    q = _heads(g, m, N_HEADS, hd)
    return q, _heads(g, pos, N_KV, hd, True), _heads(g, pos, N_KV, hd)


def _shape():
    return synth.ModelShape(n_layers=LAYERS, n_layer_kv=LAYERS, vocab=VOCAB, context=MAX_SEQ)


def _engine(seed):
    """a model file opened by the engine, as a program starts"""
    g = _gen(seed)
    specs = synth.model_tensors(_shape())
    for t in specs:
        if t.qtype in synth.BLOCK_BYTES:
            t.make = lambda r, t=t: _kquant(g, t.qtype, t.ne[1], t.ne[0]).cpu().numpy()
    where = "/dev/shm" if os.path.isdir("/dev/shm") else None
    fd, path = tempfile.mkstemp(suffix=".gguf", dir=where)
    os.close(fd)
    try:
        synth.write_gguf(path, synth.model_kvs(_shape()), specs, seed)
        return g4.Engine(path, max_seq=MAX_SEQ)
    finally:
        os.unlink(path)


def prepare(case, seed):
    kind = case["kind"]
    lib = g4.Lib.get()
    lib.init(0)
    st = {"kind": kind, "lib": lib, "case": case}
    if kind in ("mm", "head", "batch"):
        t, raws, x = _matrix_inputs(case, seed)
        n, d, m = case["n"], case["d"], case.get("m", 1)
        st.update(t=t, x=x, w=[_place(lib, r, t, n, d) for r in raws])
        if kind == "head":
            st.update(logits=_empty(d), token=_empty(1, dtype=torch.int32),
                      part=_empty(lib.L.g4_mm_argmax_part_bytes(d), dtype=torch.uint8))
        else:
            q8 = m * lib.L.g4_q8K_row_stride(n) if kind == "batch" else lib.L.g4_q8K_bytes(n)
            st.update(o=_empty(len(raws), m, d), q8=_empty(q8, dtype=torch.uint8))
    elif kind == "ffn":
        t, raws, x = _ffn_inputs(case, seed)
        n, hidden = case["n"], case["hidden"]
        w = [(_place(lib, a, t, n, hidden), _place(lib, b, t, n, hidden), _place(lib, c, g4.Q6_K, hidden, n))
             for a, b, c in raws]
        st.update(t=t, x=x, w=w, hb=_empty(hidden), y=_empty(len(w), n),
                  q8=_empty(lib.L.g4_q8K_bytes(n), dtype=torch.uint8))
    elif kind == "attn":
        q, k, v = _attn_inputs(case, seed)
        st.update(q=q, k=k, v=v, out=_empty(N_HEADS * case["hd"]))
    elif kind == "rows":
        q, k, v = _attn_inputs(case, seed)
        hd, m, p0, window = case["hd"], case["m"], case["p0"], case["window"]
        kvd = N_KV * hd
        if window:          # a ring holds the window's slots
            ring = window
            kc, vc = _empty(ring, kvd).zero_(), _empty(ring, kvd).zero_()
            lo = max(0, p0 - ring)
            slots = torch.arange(lo, p0, device="cuda") % ring
            kc[slots], vc[slots] = k[lo:p0], v[lo:p0]
        else:
            ring = 0
            kc, vc = k[: max(p0, 1)].clone(), v[: max(p0, 1)].clone()
        span = min(window, p0 + m) if window else p0 + m
        G = min((span + 127) // 128, 16)        # the engine's count of key chunks
        st.update(q=q, kc=kc, vc=vc, kch=k[p0:].contiguous(), vch=v[p0:].contiguous(), ring=ring, G=G,
                  part=_empty(m * lib.L.g4_attn_part_bytes(N_HEADS, hd, G), dtype=torch.uint8),
                  out=_empty(m, N_HEADS * hd))
    else:
        rng = np.random.default_rng(seed)
        st["engine"] = e = _engine(seed)
        if kind == "prompt":
            st["tokens"] = rng.integers(0, VOCAB, case["tokens"], dtype=np.int32)
        else:
            e.prefill(rng.integers(0, VOCAB, case["pos"], dtype=np.int32), 0)
            st["tokens"] = [int(t) for t in rng.integers(0, VOCAB, case["steps"])]
    torch.cuda.synchronize()
    return st


def run(st):
    kind, lib, c = st["kind"], st["lib"], st["case"]
    if kind == "mm":
        lib.g4_mm(st["o"].data_ptr(), st["x"].data_ptr(), st["w"][0].data_ptr(), c["n"], c["d"], st["t"],
                  st["q8"].data_ptr(), 0)
        return st["o"]
    if kind == "batch":
        x, q8 = st["x"].data_ptr(), st["q8"].data_ptr()
        for o, w in zip(st["o"], st["w"]):
            lib.g4_mm_batch(o.data_ptr(), x, w.data_ptr(), c["n"], c["d"], c["m"], st["t"], q8)
        return st["o"]
    if kind == "ffn":
        q8, hb = st["q8"].data_ptr(), st["hb"].data_ptr()
        for x, y, (gate, up, down) in zip(st["x"], st["y"], st["w"]):
            lib.g4_quantize_row_q8_K(x.data_ptr(), q8, c["n"])
            lib.g4_mm_gate_up_gelu(hb, gate.data_ptr(), up.data_ptr(), c["n"], c["hidden"], st["t"], q8)
            lib.g4_mm(y.data_ptr(), hb, down.data_ptr(), c["hidden"], c["n"], g4.Q6_K, None, 0)
        return st["y"]
    if kind == "head":
        lib.g4_mm_argmax_row(st["x"].data_ptr(), st["w"][0].data_ptr(), c["n"], c["d"], st["t"], None, CAP,
                             st["logits"].data_ptr(), st["part"].data_ptr(), st["token"].data_ptr(), None, None)
        return {"logits": st["logits"], "token": st["token"]}
    if kind == "attn":
        lib.g4_attn_decode(st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(), N_KV * c["hd"], 0,
                           c["positions"], N_HEADS, N_KV, c["hd"], 1.0, st["out"].data_ptr())
        return st["out"]
    if kind == "rows":
        lib.g4_attn_decode_rows(st["q"].data_ptr(), st["kc"].data_ptr(), st["vc"].data_ptr(), st["kch"].data_ptr(),
                                st["vch"].data_ptr(), N_KV * c["hd"], st["ring"], c["p0"], c["m"], c["window"],
                                N_HEADS, N_KV, c["hd"], 1.0, st["G"], st["part"].data_ptr(), st["out"].data_ptr(),
                                None)
        return st["out"]
    e, tokens = st["engine"], st["tokens"]
    if kind == "prompt":
        e.prefill(tokens[:-1], 0)
        e.forward(int(tokens[-1]), len(tokens) - 1, 1)
        return e.logits()
    logits = []
    for i, t in enumerate(tokens):
        e.decode_steps(t, c["pos"] + i, 1)
        logits.append(e.logits())
    return logits


def _wbytes(t, n, d):
    return 2 * n * d if t == g4.BF16 else n // 256 * synth.BLOCK_BYTES[t] * d


def work(case):
    kind = case["kind"]
    if kind in ("mm", "head", "batch"):
        n, d, m, layers = case["n"], case["d"], case.get("m", 1), case.get("layers", 1)
        t = TYPES[case.get("type", "Q6_K")]
        return {"bytes": layers * (_wbytes(t, n, d) + 4 * m * d) + 4 * m * n, "flops": 2 * layers * m * n * d}
    if kind == "ffn":
        n, h, layers = case["n"], case["hidden"], case["layers"]
        return {"bytes": layers * (2 * _wbytes(TYPES[case["type"]], n, h) + _wbytes(g4.Q6_K, h, n) + 8 * n),
                "flops": 6 * layers * n * h}
    if kind == "attn":
        p, hd = case["positions"], case["hd"]
        return {"bytes": 8 * p * N_KV * hd + 8 * N_HEADS * hd, "flops": 4 * p * N_HEADS * hd}
    if kind == "rows":
        m, p0, hd, w = case["m"], case["p0"], case["hd"], case["window"]
        keys = sum(min(w, p0 + i + 1) if w else p0 + i + 1 for i in range(m))
        first = max(0, p0 + 1 - w) if w else 0
        return {"bytes": 8 * (p0 + m - first) * N_KV * hd + 8 * m * N_HEADS * hd, "flops": 4 * keys * N_HEADS * hd}
    s = _shape()
    step = synth.decode_weight_bytes(s)
    head = synth.tensor_nbytes(s.v_type, (s.dim, s.vocab))
    per_token = sum(2 * n * d for _, _, n, d in synth.prefill_matmuls(s))
    keys = LAYERS * 4 * N_HEADS * 300       # about the attention's flops per token and head element
    if kind == "prompt":
        m = case["tokens"]
        # the weights once for the chunk and once for the last token, and the head
        chunk = step - head if m > 1 else 0
        return {"bytes": chunk + step, "flops": m * (per_token + keys * 0.5 * m / 256) + 2 * s.dim * s.vocab}
    k = case["steps"]
    return {"bytes": k * (step + 4 * s.vocab), "flops": k * (per_token + 2 * s.dim * s.vocab)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("prompt", "decode"):
        # activations are quantized to 8 bits at five points of each layer: a
        # changed rounding moves a code by one, and six layers carry it on
        # (a prompt in one chunk against the same tokens one by one, whose
        # sums run in another order: rel up to 2.7e-2, max 0.14)
        return {"rel": 0.1, "max": 0.6}
    if kind == "batch":
        # up to 10240 fp32 products and sums in a row: 1.8e-6 off 64 bits
        return {"rel": 8e-6, "max": 8e-5}
    # 32-bit sums: 1e-7 to 7e-7 off 64 bits
    return {"rel": 4e-6, "max": 4e-5}


# ---------------------------------------------------------------------------
# the same in 64 bits, from the GGUF bytes
# ---------------------------------------------------------------------------
def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(raw, t):
    """float64 [rows, n] of GGUF blocks (or bf16 rows)"""
    if t == g4.BF16:
        return raw.double()
    rows, nb, _ = raw.shape
    out = torch.empty((rows, nb, 256), dtype=torch.float64, device=raw.device)
    if t == g4.Q6_K:
        d = _f16(raw[..., 208:210])
        sc = raw[..., 192:208].contiguous().view(torch.int8).double()
        for h in range(2):
            ql = raw[..., 64 * h:64 * h + 64].int()
            qh = raw[..., 128 + 32 * h:160 + 32 * h].int()
            for k in range(4):
                lo = ql[..., 32 * (k & 1):32 * (k & 1) + 32]
                q = ((lo >> (4 * (k >> 1))) & 15 | ((qh >> (2 * k)) & 3) << 4) - 32
                s = sc[..., 8 * h + 2 * k:8 * h + 2 * k + 2].repeat_interleave(16, -1)
                out[..., 128 * h + 32 * k:128 * h + 32 * k + 32] = d * s * q
        return out.reshape(rows, nb * 256)
    d, dmin = _f16(raw[..., 0:2]), _f16(raw[..., 2:4])
    s = raw[..., 4:16].int()
    qs = raw[..., -128:].int()
    for j in range(8):
        if j < 4:
            sc, mn = s[..., j] & 63, s[..., j + 4] & 63
        else:
            sc = s[..., j + 4] & 15 | (s[..., j - 4] >> 6) << 4
            mn = s[..., j + 4] >> 4 | (s[..., j] >> 6) << 4
        q = (qs[..., 32 * (j // 2):32 * (j // 2) + 32] >> (4 * (j & 1))) & 15
        if t == g4.Q5_K:
            q = q + 16 * ((raw[..., 16:48].int() >> j) & 1)
        out[..., 32 * j:32 * j + 32] = d * sc.unsqueeze(-1) * q - dmin * mn.unsqueeze(-1)
    return out.reshape(rows, nb * 256)


def _q8(x):
    """rows as Q8_K holds them (its fp32 steps), in float64"""
    b = x.float().reshape(x.shape[0], -1, 256)
    at = b.abs().argmax(-1, keepdim=True)
    top = torch.gather(b, -1, at)
    inv = torch.where(top == 0, torch.zeros_like(top), -127.0 / top)
    q = torch.clamp(torch.round(inv * b), max=127.0)
    d = torch.where(top == 0, torch.zeros_like(top), 1.0 / inv)
    return (q.double() * d.double()).reshape(x.shape)


def _product(raw, t, x):
    """x [m, n] times the matrix, [m, d]: Q4_K and Q5_K on Q8_K activations"""
    x = x.double() if t in (g4.Q6_K, g4.BF16) else _q8(x)
    step = max(1, (1 << 27) // x.shape[1])
    return torch.cat([x @ _dequant(raw[r:r + step], t).T.contiguous() for r in range(0, raw.shape[0], step)], 1)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * x * (1.0 + 0.044715 * x * x)))


def _attention(q, k, v, hd, first, last):
    """q [m, heads*hd] over keys first[i]..last[i] of row i"""
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    at = torch.arange(k.shape[0], device=q.device)
    hidden = (at < first[:, None]) | (at > last[:, None])
    for h in range(N_HEADS):
        kv = h // (N_HEADS // N_KV)
        kh, vh = (a[:, kv * hd:(kv + 1) * hd].double() for a in (k, v))
        s = q[:, h * hd:(h + 1) * hd].double() @ kh.T.contiguous()
        out[:, h * hd:(h + 1) * hd] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ vh
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("mm", "batch"):
        t, raws, x = _matrix_inputs(case, seed)
        return torch.stack([_product(r, t, x) for r in raws])
    if kind == "head":
        t, raws, x = _matrix_inputs(case, seed)
        logits = CAP * torch.tanh(_product(raws[0], t, x)[0] / CAP)
        return {"logits": logits, "token": None}
    if kind == "ffn":
        t, raws, x = _ffn_inputs(case, seed)
        y = []
        for i, (gate, up, down) in enumerate(raws):
            h = _gelu(_product(gate, t, x[i:i + 1])) * _product(up, t, x[i:i + 1])
            y.append(h @ _dequant(down, g4.Q6_K).T.contiguous())
        return torch.cat(y)
    if kind in ("attn", "rows"):
        q, k, v = _attn_inputs(case, seed)
        last = torch.arange(q.shape[0], device=q.device) + (k.shape[0] - q.shape[0])
        w = case.get("window", 0)
        first = (last + 1 - w).clamp(min=0) if w else torch.zeros_like(last)
        o = _attention(q, k, v, case["hd"], first, last)
        return o[0] if kind == "attn" else o
    return None     # a whole model: its 8-bit activations have no 64-bit counterpart
