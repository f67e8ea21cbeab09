"""The work a program has this framework do, as measurable cases.

Each case is one call (or one short sequence of calls) through the public
entry points (the C-ABI of include/rina_hip.h and include/rina_engine.h,
through the package's ctypes binding), at sizes of the repository's own
configurations: Llama-3.2-1B (2048 wide, 32 / 8 heads of 64, MLP 8192),
DeepSeek-V2-Lite (MLA latent 512 + 64, 64 experts of 1408, top 6, shared
2816, dense MLP 10944, Q2_K) and the RINA Jamba hybrid (10 / 5 heads, 64 + 32).

Kinds:
  linear  rina_hip_linear_fused on one weight matrix, 1 .. 512 rows
  mlp     RMSNorm + W1/W3 + SiLU*up, then W2 + residual, 1 .. 512 rows
  gqa     attention over a KV cache in any of its formats: one decode row,
          or rows that continue (or start) a sequence
  mla     latent attention: one decode row over the cache, or a prompt
  moe     the MoE block: one token, or a prompt's rows
  dq      the RINA-MLA attention of the hybrid: one decode row or a prompt
  model   Inference::forward of a Llama-shaped model: logits of 1 .. 24 rows
          after a prompt
"""
import ctypes as C
import importlib
import json
import math

import numpy as np
import torch

QT = {"q4_0": 5, "fp32": 6, "q4_0f": 7, "q2_k": 10}
EPI = {"store": 0, "add": 1}
KV = {"fp32": 0, "q8": 1, "q4": 2, "q4k_q2v": 3, "q2": 4, "q2k_q1v": 5}
# K and V block formats of the modes (32 values per block): record bytes
FORMATS = {"q8": ("q8", "q8"), "q4": ("q4", "q4"), "q4k_q2v": ("q4", "q2"), "q2": ("q2", "q2"), "q2k_q1v": ("q2", "q1")}
REC = {"q8": 34, "q4": 18, "q2": 10, "q1": 6, "fp32": 128}
EPS = 1e-5
VOCAB = 128256


def _pkg():
    return importlib.import_module("retrieval-is-not-always-needed_amd")


def listed():
    return [
        # the smallest call: one quantized matvec of a decode step
        {"name": "matvec_q4_0_1row", "kind": "linear", "qt": "q4_0", "M": 1, "N": 8192, "K": 2048, "epi": "store"},
        # one greedy step of a chat in its middle, every layer and the LM head
        {"name": "llama_step_p528", "kind": "model", "qt": "q4_0f", "layers": 16, "T": 1, "start": 528},
        # decode attention of a long context over the 8-bit cache
        {"name": "gqa_decode_q8_p4095", "kind": "gqa", "kv": "q8", "H": 32, "Hkv": 8, "T": 1, "start": 4095},
        # decode attention over the latent cache
        {"name": "mla_decode_p2040", "kind": "mla", "qt": "q2_k", "H": 16, "T": 1, "start": 2040},
        # the MoE block of one decoded token
        {"name": "moe_token", "kind": "moe", "T": 1, "E": 64, "k": 6, "d": 2048, "F": 1408, "S": 2816},
        # the MLP over a prompt's rows (the prompt phase's largest products)
        {"name": "mlp_q4_0f_512rows", "kind": "mlp", "qt": "q4_0f", "M": 512, "d": 2048, "ffn": 8192},
        # the dense Q2_K MLP over a prompt of odd length
        {"name": "mlp_q2_k_301rows", "kind": "mlp", "qt": "q2_k", "M": 301, "d": 2048, "ffn": 10944},
        # the next turn of a chat: 512 rows that continue a packed cache
        {"name": "gqa_turn_q8_512_after_1536", "kind": "gqa", "kv": "q8", "H": 32, "Hkv": 8, "T": 512, "start": 1536},
        # a prompt through the latent attention
        {"name": "mla_prompt_1024", "kind": "mla", "qt": "q2_k", "H": 16, "T": 1024, "start": 0},
        # a prompt through the MoE block
        {"name": "moe_prompt_512", "kind": "moe", "T": 512, "E": 64, "k": 6, "d": 2048, "F": 1408, "S": 2816},
        # the hybrid's longest prompt over its packed cache
        {"name": "dq_prompt_1900_q2k_q1v", "kind": "dq", "kv": "q2k_q1v", "H": 10, "Hkv": 5, "db": 32, "T": 1900, "start": 0},
        # a short turn (or a text to score): logits of every new row
        {"name": "llama_rows24_p200", "kind": "model", "qt": "q4_0f", "layers": 16, "T": 24, "start": 200},
    ]


def _log(rng, lo, hi, step=1):
    """A whole number, a multiple of step, spread over the logarithm of [lo, hi]."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(lo, min(hi, int(v) // step * step))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "gqa", "mla", "moe", "dq", "model"])
    one = rng.random() < 0.4               # decode calls are the most frequent ones
    if kind == "linear":
        return {"kind": kind, "qt": rng.choice(["q4_0", "q4_0f", "q2_k", "fp32"]), "M": 1 if one else _log(rng, 2, 512),
                "N": _log(rng, 256, 10944), "K": _log(rng, 256, 8192, 32), "epi": rng.choice(["store", "add"])}
    if kind == "mlp":
        return {"kind": kind, "qt": rng.choice(["q4_0", "q4_0f", "q2_k"]), "M": 1 if one else _log(rng, 2, 512),
                "d": _log(rng, 512, 2048, 128), "ffn": _log(rng, 1024, 8192, 128)}
    if kind == "gqa":
        H, Hkv = rng.choice([(32, 8), (32, 8), (16, 4), (16, 8), (8, 8)])
        return {"kind": kind, "kv": rng.choice(["fp32", "q8", "q4", "q4k_q2v", "q2", "q2k_q1v"]), "H": H, "Hkv": Hkv,
                "T": 1 if one else _log(rng, 2, 512), "start": rng.choice([0, 1, 1]) * _log(rng, 1, 1536) if not one else _log(rng, 16, 4095)}
    if kind == "mla":
        return {"kind": kind, "qt": rng.choice(["q2_k", "q4_0", "q4_0f"]), "H": rng.choice([8, 16]),
                "T": 1 if one else _log(rng, 2, 1024), "start": _log(rng, 16, 2040) if one else 0}
    if kind == "moe":
        E, k = rng.choice([(64, 6), (64, 6), (32, 4), (16, 2)])
        return {"kind": kind, "T": 1 if one else _log(rng, 2, 512), "E": E, "k": k, "d": rng.choice([1024, 2048]),
                "F": rng.choice([704, 1024, 1408]), "S": rng.choice([1408, 2816])}
    if kind == "dq":
        T = 1 if one else _log(rng, 2, 1200)
        return {"kind": kind, "kv": rng.choice(["fp32", "q2k_q1v"]), "H": 10, "Hkv": 5, "db": rng.choice([16, 32]),
                "T": T, "start": _log(rng, 16, 2000) if one else rng.choice([0, 0, 1]) * _log(rng, 1, 600)}
    return {"kind": kind, "qt": rng.choice(["q4_0", "q4_0f"]), "layers": rng.choice([4, 8, 16]),
            "T": 1 if one else _log(rng, 2, 24), "start": _log(rng, 16, 528)}


# ---------------------------------------------------------------------------
# formats: packing (inputs) and 64-bit values (references), in plain torch
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * std


def _nib(q):
    q = q.to(torch.uint8)
    return q[:, 0::2] | (q[:, 1::2] << 4)


def _half(x):
    return x.to(torch.float16).view(-1, 1).view(torch.uint8).view(-1, 2)


def _round(y):
    return torch.sign(y) * torch.floor(y.abs() + 0.5)


def _weight(g, qt, n, std=0.02):
    """n packed weights of N(0, std) (Q2_K: random valid zero-mean blocks)."""
    if qt == "fp32":
        return _randn(g, n, std=std)
    if qt == "q2_k":
        nb = (n + 255) // 256
        blk = torch.randint(0, 256, (nb, 84), dtype=torch.uint8, device="cuda", generator=g)
        sc = blk[:, :16] & 15
        blk[:, :16] = sc | (sc << 4)       # min nibble = scale nibble, dmin = 1.5 d: zero mean
        d = np.float16(std / 9.84)
        dd = np.array([d, np.float16(1.5 * float(d))], np.float16).view(np.uint8)
        blk[:, 80:84] = torch.from_numpy(dd.copy()).cuda()
        return blk.view(-1)
    out = []
    for part in _randn(g, n // 32, 32, std=std).split(1 << 20):
        s = (part.abs().amax(1) / 7).clamp_min(1e-10)
        q = _nib(_round(part / s[:, None]).clamp(-7, 7) + 7)
        sb = _half(s) if qt == "q4_0" else s.view(-1, 1).view(torch.uint8).view(-1, 4)
        out.append(torch.cat([sb, q], 1).view(-1))
    return torch.cat(out)


def _values(qt, w, n):
    """The n weights of a packed tensor in 64 bits."""
    if qt == "fp32":
        return w[:n].double()
    if qt == "q2_k":
        b = w.view(-1, 84)
        dm = b[:, 80:84].contiguous().view(torch.float16).double()
        sc = b[:, :16].long()              # sub-block of page p, group g, half: 8 p + half + 2 g
        qs = b[:, 16:80].long().view(-1, 2, 32)
        v = torch.stack([(qs >> (2 * s)) & 3 for s in range(4)], 2)             # [nb, page, group, 32]
        scv = sc.view(-1, 2, 4, 2).repeat_interleave(16, 3)                     # [nb, page, group, 32]
        v = dm[:, 0, None, None, None] * (scv & 15) * v - dm[:, 1, None, None, None] * (scv >> 4)
        return v.reshape(-1)[:n]
    hb = 2 if qt == "q4_0" else 4
    b = w.view(-1, 16 + hb)
    s = b[:, :hb].contiguous().view(torch.float16 if hb == 2 else torch.float32).double()
    q = b[:, hb:].long()
    return ((torch.stack([q & 15, q >> 4], 2).view(-1, 32) - 7) * s).view(-1)[:n]


def _wbytes(qt, n):
    return {"fp32": 4 * n, "q2_k": (n + 255) // 256 * 84, "q4_0": n // 32 * 18, "q4_0f": n // 32 * 20}[qt]


def _kv_pack(fmt, x):
    """fp32 values (a multiple of 32) as the records of a cache format."""
    if fmt == "fp32":
        return x.reshape(-1).contiguous()
    b = x.reshape(-1, 32)
    amax = b.abs().amax(1)
    if fmt == "q8":
        s = (amax / 127).clamp_min(1e-10)
        q = _round(b / s[:, None]).clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([_half(s), q], 1).view(-1)
    if fmt == "q4":
        s = (amax / 7).clamp_min(1e-10)
        return torch.cat([_half(s), _nib(_round(b / s[:, None]).clamp(-7, 7) + 7)], 1).view(-1)
    if fmt == "q2":
        q = (_round(b / amax[:, None]).clamp(-1, 1) + 1).to(torch.uint8).view(-1, 8, 4)
        q = q[..., 0] | (q[..., 1] << 2) | (q[..., 2] << 4) | (q[..., 3] << 6)
        return torch.cat([_half(amax), q], 1).view(-1)
    bits = (b > 0).long().view(-1, 4, 8) * (1 << torch.arange(8, device=b.device))
    return torch.cat([_half(amax), bits.sum(2).to(torch.uint8)], 1).view(-1)


def _kv_values(fmt, rec, n):
    """The first n values of packed cache records in 64 bits."""
    if fmt == "fp32":
        return rec[:n].double()
    b = rec[:n // 32 * REC[fmt]].view(-1, REC[fmt])
    s = b[:, :2].contiguous().view(torch.float16).double()
    q = b[:, 2:].contiguous()
    if fmt == "q8":
        return (q.view(torch.int8).double() * s).view(-1)
    q = q.long()
    if fmt == "q4":
        v = torch.stack([q & 15, q >> 4], 2).view(-1, 32) - 7
    elif fmt == "q2":
        v = torch.stack([(q >> (2 * i)) & 3 for i in range(4)], 2).view(-1, 32) - 1
    else:
        v = torch.stack([(q >> i) & 1 for i in range(8)], 2).view(-1, 32) * 2 - 1
    return (v * s).view(-1)


def _rope_tables(dim, n, theta):
    a = torch.arange(n, device="cuda", dtype=torch.float32)[:, None] * (1.0 / theta ** (torch.arange(0, dim, 2, device="cuda", dtype=torch.float32) / dim))
    return a.cos().contiguous(), a.sin().contiguous()


def _rope(x, cos, sin, pos, pairs):
    """x [T, H, d] in 64 bits rotated at positions pos ..; pairs: (2i, 2i+1), else (i, i + d/2)."""
    T, _, d = x.shape
    c, s = cos[pos:pos + T].double()[:, None], sin[pos:pos + T].double()[:, None]
    a, b = (x[..., 0::2], x[..., 1::2]) if pairs else (x[..., :d // 2], x[..., d // 2:])
    y = torch.stack([a * c - b * s, a * s + b * c], -1)
    return y.flatten(-2) if pairs else torch.cat([y[..., 0], y[..., 1]], -1)


def _attend(q, K, V, start, scale, own=None):
    """Causal softmax attention in 64 bits: q [T, H, d], K / V [L, Hkv, d];
    own: the rows' own keys and values [T, Hkv, d], used at their position."""
    T, H, _ = q.shape
    rep = H // K.shape[1]
    mask = torch.arange(K.shape[0], device="cuda")[None] > start + torch.arange(T, device="cuda")[:, None]
    out = torch.empty(T, H, V.shape[2], dtype=torch.float64, device="cuda")
    t = torch.arange(T, device="cuda")
    for h in range(H):
        g = h // rep
        s = q[:, h] @ K[:, g].T.contiguous() * scale
        if own is not None:
            s[t, start + t] = (q[:, h] * own[0][:, g]).sum(1) * scale
        p = torch.softmax(s.masked_fill(mask, -math.inf), 1)
        o = p @ V[:, g].contiguous()
        if own is not None:
            o += p[t, start + t, None] * (own[1][:, g] - V[start:start + T, g])
        out[:, h] = o
    return out


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _swiglu(x, wg, wu):
    g = x @ wg.T.contiguous()
    return g * torch.sigmoid(g) * (x @ wu.T.contiguous())


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _inputs(c, seed):
    """The tensors of a case, from the seed alone."""
    g, k = _gen(seed), c["kind"]
    if k == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"w": _weight(g, c["qt"], N * K), "x": _randn(g, M, K), "y": _randn(g, M, N)}
    if k == "mlp":
        d, f, M = c["d"], c["ffn"], c["M"]
        return {"w1": _weight(g, c["qt"], f * d), "w3": _weight(g, c["qt"], f * d), "w2": _weight(g, c["qt"], d * f),
                "ln": 1 + 0.1 * _randn(g, d), "h": _randn(g, M, d), "g": torch.empty(M, f, device="cuda")}
    if k == "gqa":
        T, H, Hkv, P = c["T"], c["H"], c["Hkv"], c["start"]
        n = P + T + 8
        cos, sin = _rope_tables(64, n, 500000.0)
        fk, fv = FORMATS.get(c["kv"], ("fp32", "fp32"))
        return {"q": _randn(g, T, H, 64), "k": _randn(g, T, Hkv, 64), "v": _randn(g, T, Hkv, 64), "cos": cos, "sin": sin,
                "ck": _kv_pack(fk, _randn(g, n, Hkv, 64)), "cv": _kv_pack(fv, _randn(g, n, Hkv, 64)),
                "out": torch.empty(T, H, 64, device="cuda"), "max_seq": n}
    if k == "mla":
        T, H, n = c["T"], c["H"], c["start"] + c["T"] + 8
        cos, sin = _rope_tables(64, n, 10000.0)
        return {"q": _randn(g, T, H * 192), "kva": _randn(g, T, 576), "kn": 1 + 0.1 * _randn(g, 512), "cos": cos, "sin": sin,
                "w": _weight(g, c["qt"], H * 256 * 512, 0.05), "cache": _randn(g, n, 576),
                "out": torch.empty(T, H * 128, device="cuda"), "max_seq": n}
    if k == "moe":
        T, E, d, F, S = c["T"], c["E"], c["d"], c["F"], c["S"]
        return {"h": _randn(g, T, d), "ln": 1 + 0.1 * _randn(g, d), "wr": _randn(g, E, d, std=0.05),
                "sg": _weight(g, "q2_k", S * d), "su": _weight(g, "q2_k", S * d), "sd": _weight(g, "q2_k", d * S),
                "eg": _weight(g, "q2_k", E * F * d), "eu": _weight(g, "q2_k", E * F * d), "ed": _weight(g, "q2_k", E * d * F)}
    if k == "dq":
        T, H, Hkv, db, P = c["T"], c["H"], c["Hkv"], c["db"], c["start"]
        n = P + T + 8
        cos, sin = _rope_tables(db, n, 10000.0)
        K, R, V = _randn(g, n, Hkv, 64), _randn(g, n, Hkv, db), _randn(g, n, Hkv, 64)
        packed = c["kv"] != "fp32"
        return {"qa": _randn(g, T, H, 64), "qb": _randn(g, T, H, db), "ka": _randn(g, T, Hkv, 64), "kb": _randn(g, T, Hkv, db),
                "v": _randn(g, T, Hkv, 64), "cos": cos, "sin": sin,
                "ck": _kv_pack("q2", K) if packed else torch.cat([K, R], 2).view(-1),
                "cv": _kv_pack("q1", V) if packed else V.view(-1), "cr": R.reshape(-1).contiguous() if packed else None,
                "out": torch.empty(T, H, 64, device="cuda"), "max_seq": n}
    d, f, L = 2048, 8192, c["layers"]
    n = 576
    cos, sin = _rope_tables(64, n, 500000.0)
    t = {"wte": _randn(g, VOCAB, d, std=0.02), "ln_f": 1 + 0.1 * _randn(g, d), "cos": cos, "sin": sin, "max_seq": n,
         "ids": torch.randint(0, VOCAB, (c["start"] + c["T"],), device="cuda", generator=g, dtype=torch.int32), "layers": []}
    for _ in range(L):
        t["layers"].append({"attn.w_q.weight": _weight(g, c["qt"], d * d), "attn.w_k.weight": _weight(g, c["qt"], 512 * d),
                            "attn.w_v.weight": _weight(g, c["qt"], 512 * d), "attn.w_o.weight": _weight(g, c["qt"], d * d),
                            "mlp.w1.weight": _weight(g, c["qt"], f * d), "mlp.w2.weight": _weight(g, c["qt"], d * f),
                            "mlp.w3.weight": _weight(g, c["qt"], f * d), "ln1.weight": 1 + 0.1 * _randn(g, d),
                            "ln2.weight": 1 + 0.1 * _randn(g, d)})
    return t


class _Llama:
    """A Llama-shaped engine model over given device tensors, and its Inference."""

    SHAPES = {"attn.w_q.weight": (2048, 2048), "attn.w_k.weight": (512, 2048), "attn.w_v.weight": (512, 2048),
              "attn.w_o.weight": (2048, 2048), "mlp.w1.weight": (8192, 2048), "mlp.w2.weight": (2048, 8192),
              "mlp.w3.weight": (8192, 2048), "ln1.weight": (2048,), "ln2.weight": (2048,)}

    def __init__(self, t, qt):
        self.infer = self.model = None
        rina = _pkg()
        self.eng, self.t = rina.load_engine(), t
        L = len(t["layers"])
        header = {"name": "llama3.2-1b", "dim": 2048, "n_layers": L, "n_heads": 32, "n_kv_heads": 8, "head_dim": 64,
                  "vocab_size": VOCAB, "max_seq_len": t["max_seq"], "hidden_dim": 8192, "weight_tying": True,
                  "kv_quant_mode": "fp32", "layers": [{"type": "standard_attention"}] * L}
        self.model = self.eng.rina_model_create(json.dumps(header).encode())

        def add(name, q, shape, x):
            rina.check(self.eng.rina_model_add_tensor(self.model, name.encode(), q, len(shape), (C.c_int64 * len(shape))(*shape), x.data_ptr()), name)

        add("transformer.wte.weight", QT["fp32"], (VOCAB, 2048), t["wte"])
        add("transformer.ln_f.weight", QT["fp32"], (2048,), t["ln_f"])
        for l, w in enumerate(t["layers"]):
            p = "transformer.h.%d." % l
            for name, x in w.items():
                add(p + name, QT["fp32"] if name.startswith("ln") else QT[qt], self.SHAPES[name], x)
            for name in ("rope_q", "rope"):
                add(p + "attn.%s.cos" % name, QT["fp32"], (t["max_seq"], 32), t["cos"])
                add(p + "attn.%s.sin" % name, QT["fp32"], (t["max_seq"], 32), t["sin"])
        self.infer = self.eng.rina_infer_create(self.model, b"gqa", b"fp32", t["max_seq"])
        if not self.infer:
            raise RuntimeError(self.eng.rina_engine_last_error().decode())

    def __del__(self):
        if self.infer:
            self.eng.rina_infer_destroy(self.infer)
        if self.model:
            self.eng.rina_model_destroy(self.model)


def prepare(case, seed):
    c, rina = case, _pkg()
    hip = rina.load_hip()
    t = _inputs(c, seed)
    st = torch.cuda.current_stream().cuda_stream
    s = {"t": t}                            # calls: (function, its arguments); outs: what they leave
    k = c["kind"]
    p = {n: x.data_ptr() for n, x in t.items() if isinstance(x, torch.Tensor)}
    if k == "linear":
        s["seg"] = rina.LinearSeg(p["w"], None, p["y"], c["N"])
        s["calls"] = [(hip.rina_hip_linear_fused, (C.byref(s["seg"]), 1, QT[c["qt"]], p["x"], c["M"], c["K"], EPI[c["epi"]], 0, None, 0.0, st))]
        s["outs"] = {"y": t["y"]}
    elif k == "mlp":
        d, f, M, qt = c["d"], c["ffn"], c["M"], QT[c["qt"]]
        s["up"], s["down"] = rina.LinearSeg(p["w1"], p["w3"], p["g"], f), rina.LinearSeg(p["w2"], None, p["h"], d)
        s["calls"] = [(hip.rina_hip_linear_fused, (C.byref(s["up"]), 1, qt, p["h"], M, d, 2, 1, p["ln"], EPS, st)),
                      (hip.rina_hip_linear_fused, (C.byref(s["down"]), 1, qt, p["g"], M, f, 1, 0, None, 0.0, st))]
        s["outs"] = {"g": t["g"], "h": t["h"]}
    elif k == "gqa":
        T, H, Hkv, P, n, mode = c["T"], c["H"], c["Hkv"], c["start"], t["max_seq"], KV[c["kv"]]
        wb = hip.rina_hip_gqa_attention_workspace(T, H, 64, n)
        s["ws"] = torch.empty(wb, dtype=torch.uint8, device="cuda")
        w = s["ws"].data_ptr()
        tables = (p["cos"], p["sin"], p["cos"], p["sin"])
        if T == 1:
            s["calls"] = [(hip.rina_hip_gqa_decode_attention, (p["q"], p["k"], p["v"], *tables, p["ck"], p["cv"], mode, H, Hkv, 64, P, None, n,
                                                               p["out"], None, w, wb, st))]
        else:
            s["calls"] = [(hip.rina_hip_rope_append, (p["q"], p["k"], p["v"], *tables, p["ck"], p["cv"], mode, 0, T, H, Hkv, 64, P, None, n, st)),
                          (hip.rina_hip_gqa_attention, (p["q"], p["k"], p["v"], p["ck"], p["cv"], mode, 0, p["cos"], p["sin"], T, H, Hkv, 64, P,
                                                        None, n, p["out"], w, wb, st))]
        s["outs"] = {"out": t["out"], "ck": t["ck"], "cv": t["cv"]}
    elif k == "mla":
        T, H, n = c["T"], c["H"], t["max_seq"]
        wb = hip.rina_hip_mla_attention_workspace(H, 512, 64, n) if T == 1 else hip.rina_hip_mla_prompt_workspace(T, H, 128, 64, 128, 512)
        s["ws"] = torch.empty(wb, dtype=torch.uint8, device="cuda")
        head = (p["q"], p["kva"], p["kn"], EPS, p["cos"], p["sin"], p["w"], QT[c["qt"]], p["cache"], H, 128, 64, 128, 512)
        if T == 1:
            s["calls"] = [(hip.rina_hip_mla_decode_attention, (*head, c["start"], None, n, p["out"], s["ws"].data_ptr(), wb, st))]
        else:
            s["calls"] = [(hip.rina_hip_mla_prompt_attention, (*head, T, n, p["out"], s["ws"].data_ptr(), wb, st))]
        s["outs"] = {"out": t["out"], "cache": t["cache"]}
    elif k == "moe":
        T, E, kk, d, F, S = c["T"], c["E"], c["k"], c["d"], c["F"], c["S"]
        sg, sd = _wbytes("q2_k", F * d), _wbytes("q2_k", d * F)
        wb = hip.rina_hip_moe_block_workspace(d, E, kk, F, S) if T == 1 else hip.rina_hip_moe_rows_workspace(T, d, E, kk, F, S)
        s["ws"] = torch.zeros(wb, dtype=torch.uint8, device="cuda")
        tail = (sg, sd, E, kk, d, F, s["ws"].data_ptr(), wb, st)
        if T == 1:
            s["calls"] = [(hip.rina_hip_moe_block, (p["h"], p["ln"], EPS, p["wr"], QT["fp32"], p["sg"], p["su"], p["sd"], S, p["eg"], p["eu"],
                                                    p["ed"], QT["q2_k"], *tail))]
        else:
            s["calls"] = [(hip.rina_hip_moe_rows, (p["h"], T, p["ln"], EPS, p["wr"], QT["fp32"], p["sg"], p["su"], p["sd"], S, QT["q2_k"],
                                                   p["eg"], p["eu"], p["ed"], QT["q2_k"], *tail))]
        s["outs"] = {"h": t["h"]}
    elif k == "dq":
        T, H, Hkv, db, P, n, mode = c["T"], c["H"], c["Hkv"], c["db"], c["start"], t["max_seq"], KV[c["kv"]]
        head = (p["qa"], p["qb"], p["ka"], p["kb"], p["v"], p["cos"], p["sin"], p["cos"], p["sin"], mode, p["ck"], p["cv"], p.get("cr"),
                H, Hkv, 64, db, 64, P)
        if T == 1:
            wb = hip.rina_hip_dq_attention_workspace(H, 64 + db, n)
            s["ws"] = torch.empty(wb, dtype=torch.uint8, device="cuda")
            s["calls"] = [(hip.rina_hip_dq_decode_attention_kv, (*head, None, n, p["out"], s["ws"].data_ptr(), wb, st))]
        else:
            s["calls"] = [(hip.rina_hip_dq_prompt_attention_kv, (*head, T, n, p["out"], st))]
        s["outs"] = {n_: t[n_] for n_ in ("out", "ck", "cv", "cr") if t[n_] is not None}
    else:
        P, T = c["start"], c["T"]
        s["model"] = m = _Llama(t, c["qt"])
        ids = t["ids"][:P].tolist()         # the prompt before the measured rows
        rina.check(m.eng.rina_infer_generate(m.infer, (C.c_int * P)(*ids), P, 1, (C.c_int * 1)(), 0, st, None), "generate")
        s["logits"] = torch.empty(T, VOCAB, device="cuda")
        s["calls"] = [(m.eng.rina_infer_forward, (m.infer, t["ids"][P:].data_ptr(), s["logits"].data_ptr(), 1, T, P, st))]
        s["outs"] = {"logits": s["logits"]}
    return s


def run(state):
    for f, args in state["calls"]:
        rc = f(*args)
        if rc:
            raise RuntimeError("%s returned %d" % (f.__name__, rc))
    return state["outs"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    c, k = case, case["kind"]
    if k == "linear":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": _wbytes(c["qt"], N * K) + 4 * M * (K + N * (2 if c["epi"] == "add" else 1)), "flops": 2 * M * N * K}
    if k == "mlp":
        M, d, f = c["M"], c["d"], c["ffn"]
        return {"bytes": 3 * _wbytes(c["qt"], d * f) + 4 * M * (2 * d + f), "flops": 6 * M * d * f}
    if k == "gqa":
        T, H, Hkv, P = c["T"], c["H"], c["Hkv"], c["start"]
        rec = sum(REC[f] for f in FORMATS.get(c["kv"], ("fp32", "fp32")))
        return {"bytes": (P + T) * Hkv * 2 * rec + 4 * 64 * T * (2 * H + 2 * Hkv), "flops": 4 * 64 * H * (T * P + T * (T + 1) // 2)}
    if k == "mla":
        T, H, P = c["T"], c["H"], c["start"]
        w = _wbytes(c["qt"], H * 256 * 512)
        if T == 1:
            return {"bytes": w + 4 * 576 * (P + 1) + 4 * H * 320, "flops": 2 * H * (256 * 512 + (P + 1) * (576 + 512))}
        return {"bytes": w + 4 * T * (2 * 576 + H * 320), "flops": 2 * H * (T * 256 * 512 + T * (T + 1) // 2 * 320)}
    if k == "moe":
        T, E, kk, d, F, S = c["T"], c["E"], c["k"], c["d"], c["F"], c["S"]
        used = E * (1 - (1 - kk / E) ** T)  # experts that T rows select
        return {"bytes": 3 * _wbytes("q2_k", S * d) + used * 3 * _wbytes("q2_k", F * d) + 4 * E * d + 8 * T * d,
                "flops": 2 * T * (3 * d * (S + kk * F) + E * d)}
    if k == "dq":
        T, H, Hkv, db, P = c["T"], c["H"], c["Hkv"], c["db"], c["start"]
        rec = 4 * (128 + db) if c["kv"] == "fp32" else 20 + 12 + 4 * db
        return {"bytes": (P + T) * Hkv * rec + 4 * T * (H * (128 + db) + Hkv * (128 + db)), "flops": 2 * H * (128 + db) * (T * P + T * (T + 1) // 2)}
    T, L, P, d = c["T"], c["layers"], c["start"], 2048
    n = d * d * 2 + 2 * 512 * d + 3 * 8192 * d
    return {"bytes": L * (_wbytes(c["qt"], n) + 4096 * (P + T)) + 4 * VOCAB * (d + T),
            "flops": 2 * T * (L * n + VOCAB * d) + L * 8192 * (T * P + T * (T + 1) // 2)}


def tolerance(case):
    """fp32 sums everywhere; whole values are the packed cache records, where
    a row's value can fall on either side of a code's edge.  About four times
    what the paths differ from 64-bit results, per kind."""
    k = case["kind"]
    if k == "model":                        # rounding of a layer travels through the later ones
        return {"rel": 2e-5, "max": 5e-4}
    if k in ("gqa", "dq", "mla"):
        return {"rel": 6e-6, "max": 2e-4, "differ": 1e-5}
    return {"rel": 6e-6, "max": 2e-4}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def exact(case, seed):
    c, k = case, case["kind"]
    t = _inputs(c, seed)
    if k == "linear":
        y = t["x"].double() @ _values(c["qt"], t["w"], c["N"] * c["K"]).view(c["N"], c["K"]).T.contiguous()
        return {"y": y + t["y"].double() if c["epi"] == "add" else y}
    if k == "mlp":
        d, f = c["d"], c["ffn"]
        W = {n: _values(c["qt"], t[n], d * f) for n in ("w1", "w2", "w3")}
        h = t["h"].double()
        g = _swiglu(_norm(h, t["ln"]), W["w1"].view(f, d), W["w3"].view(f, d))
        return {"g": g, "h": h + g @ W["w2"].view(d, f).T.contiguous()}
    if k == "gqa":
        T, Hkv, P = c["T"], c["Hkv"], c["start"]
        fk, fv = FORMATS.get(c["kv"], ("fp32", "fp32"))
        q, kr = (_rope(t[n].double(), t["cos"], t["sin"], P, False) for n in ("q", "k"))
        v = t["v"].double()
        K, V = _kv_values(fk, t["ck"], P * Hkv * 64).view(P, Hkv, 64), _kv_values(fv, t["cv"], P * Hkv * 64).view(P, Hkv, 64)
        out = {"out": _attend(q, torch.cat([K, kr]), torch.cat([V, v]), P, 0.125), "ck": None, "cv": None}
        if c["kv"] == "fp32":
            for n, x in (("ck", kr), ("cv", v)):
                full = t[n].double()
                full[P * Hkv * 64:(P + T) * Hkv * 64] = x.reshape(-1)
                out[n] = full
        return out
    if k == "mla":
        T, H, P = c["T"], c["H"], c["start"]
        q = t["q"].double()
        qr = _rope(q[:, H * 128:].reshape(T, H, 64), t["cos"], t["sin"], P, False)
        kva = t["kva"].double()
        rec = torch.cat([_norm(kva[:, :512], t["kn"]), _rope(kva[:, None, 512:], t["cos"], t["sin"], P, False)[:, 0]], 1)
        cache = t["cache"].double()
        cache[P:P + T] = rec
        W = _values(c["qt"], t["w"], H * 256 * 512).view(H * 256, 512)
        lat = cache[:P + T]
        Kn = (lat[:, :512] @ W[:H * 128].T.contiguous()).view(P + T, H, 128)
        V = (lat[:, :512] @ W[H * 128:].T.contiguous()).view(P + T, H, 128)
        K = torch.cat([Kn, lat[:, None, 512:].expand(P + T, H, 64)], 2)
        out = _attend(torch.cat([q[:, :H * 128].reshape(T, H, 128), qr], 2), K, V, P, 192 ** -0.5)
        return {"out": out.view(T, H * 128), "cache": cache}
    if k == "moe":
        T, E, kk, d, F, S = c["T"], c["E"], c["k"], c["d"], c["F"], c["S"]
        h = t["h"].double()
        a = _norm(h, t["ln"])
        pr, ids = torch.softmax(a @ t["wr"].double().T.contiguous(), 1).topk(kk, 1)
        y = _swiglu(a, _values("q2_k", t["sg"], S * d).view(S, d), _values("q2_k", t["su"], S * d).view(S, d))
        h = h + y @ _values("q2_k", t["sd"], d * S).view(d, S).T.contiguous()
        nb = _wbytes("q2_k", F * d)
        for e in range(E):
            r, j = (ids == e).nonzero(as_tuple=True)
            if not len(r):
                continue
            W = {n: _values("q2_k", t[n][e * nb:(e + 1) * nb], F * d) for n in ("eg", "eu", "ed")}
            y = _swiglu(a[r], W["eg"].view(F, d), W["eu"].view(F, d)) @ W["ed"].view(d, F).T.contiguous()
            h.index_add_(0, r, pr[r, j, None] * y)
        return {"h": h}
    if k == "dq":
        T, Hkv, db, P = c["T"], c["Hkv"], c["db"], c["start"]
        qr, kr = (_rope(t[n].double(), t["cos"], t["sin"], P, True) for n in ("qb", "kb"))
        q = torch.cat([t["qa"].double(), qr], 2)
        kn, v = torch.cat([t["ka"].double(), kr], 2), t["v"].double()
        out = {n: None for n in ("ck", "cv", "cr") if t[n] is not None}
        if c["kv"] == "fp32":
            K, V = t["ck"].double().view(-1, Hkv, 64 + db), t["cv"].double().view(-1, Hkv, 64)
            K[P:P + T], V[P:P + T] = kn, v
            out.update(ck=K.view(-1), cv=V.view(-1))
            K, V = K[:P + T], V[:P + T]
        else:
            R = t["cr"].double().view(-1, Hkv, db)
            R[P:P + T] = kr
            out["cr"] = R.view(-1)
            n = P * Hkv * 64
            Ka = torch.cat([_kv_values("q2", t["ck"], n), _kv_values("q2", _kv_pack("q2", t["ka"]), T * Hkv * 64)]).view(P + T, Hkv, 64)
            V = torch.cat([_kv_values("q1", t["cv"], n), _kv_values("q1", _kv_pack("q1", t["v"]), T * Hkv * 64)]).view(P + T, Hkv, 64)
            K = torch.cat([Ka, R[:P + T]], 2)
        return {"out": _attend(q, K, V, P, (64 + db) ** -0.5, own=(kn, v)), **out}
    h = t["wte"][t["ids"].long()].double()
    n, P = h.shape[0], c["start"]
    for w in t["layers"]:
        W = {m: _values(c["qt"], w[m], math.prod(s)).view(s) for m, s in _Llama.SHAPES.items() if len(s) == 2}
        a = _norm(h, w["ln1.weight"])
        q, kk, v = ((a @ W["attn.w_%s.weight" % x].T.contiguous()).view(n, -1, 64) for x in "qkv")
        q, kk = (_rope(x, t["cos"], t["sin"], 0, False) for x in (q, kk))
        h = h + _attend(q, kk, v, 0, 0.125).reshape(n, 2048) @ W["attn.w_o.weight"].T.contiguous()
        a = _swiglu(_norm(h, w["ln2.weight"]), W["mlp.w1.weight"], W["mlp.w3.weight"])
        h = h + a @ W["mlp.w2.weight"].T.contiguous()
    return {"logits": _norm(h[P:], t["ln_f"]) @ t["wte"].double().T.contiguous()}
