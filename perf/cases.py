"""The work a program has this library do, as cases that can be timed and checked.

Four kinds of case, each through the public entry points:

* "layers": the first transformer blocks of a model through the C ABI
  (include/orc.h): embedding gather, then per block norm + Q|K|V, RoPE + K / V
  store + attention, output projection, gate | up with SwiGLU, down
  projection. One token is a decode step, 2-16 tokens a speculative verify
  pass (both replayed as a captured graph whose position lives on the device,
  as the decode loops do), more tokens a prefill pass launched from the host.
  Several blocks with weights of their own, so that a pass streams its weights
  from HBM as a whole model does.
* "head": final norm, LM head and argmax over the rows of a verify pass.
* "sample" / "spec_round": the sampler on one row of logits, and one round of
  speculative sampling (k draft transforms and draws, k + 1 target rows, the
  acceptance chain).
* "model": a GGUF file loaded by the host library; a prompt is prefilled, then
  tokens are decoded one by one, their logits returned.

Weights are random GGUF blocks whose values are N(0, 0.02^2)-like; every state
has weights of its own.
"""
import ctypes as C
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle-engine_amd", "python"))
import orc  # noqa: E402

EPS = 1e-5
BF16 = 30  # ORC_BF16
TYPES = {"q8_0": orc.Q8_0, "q4_0": orc.Q4_0, "q4_k": orc.Q4_K, "q6_k": orc.Q6_K, "f16": orc.F16, "bf16": BF16,
         "f32": orc.F32}
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210), "f16": (1, 2), "bf16": (1, 2),
         "f32": (1, 4)}
EMBED_ROWS = 2048  # rows of the embedding table of a "layers" case
VERIFY_MAX = 16    # tokens of the largest verify pass; longer passes are prefills


def _layers(name, quant, d_model, heads, kv, hd, ffn, bias, theta, layers, n_tok, pos, ctx):
    return {"name": name, "kind": "layers", "quant": quant, "d_model": d_model, "heads": heads, "kv": kv, "hd": hd,
            "ffn": ffn, "bias": bias, "theta": theta, "layers": layers, "n_tok": n_tok, "pos": pos, "ctx": ctx}


def listed():
    return [
        # a proposal step of the 0.5B-shape Q8_0 draft: the smallest matrices, launches and latency count
        _layers("draft_decode_q8_0", "q8_0", 896, 14, 2, 64, 4864, True, 1e6, 12, 1, 300, 4096),
        # greedy decode of the 3B-shape Q4_K_M target
        _layers("decode_q4_k_m", "q4_k_m", 3072, 24, 8, 128, 8192, False, 5e5, 4, 1, 200, 2048),
        # its verify pass of k = 4 proposals
        _layers("verify_q4_k_m", "q4_k_m", 3072, 24, 8, 128, 8192, False, 5e5, 4, 5, 333, 2048),
        # verify of k = 8 at a long context: the 7B-shape all-Q6_K target after an 8K prompt
        _layers("verify_long_q6_k", "q6_k", 3584, 28, 4, 128, 18944, True, 1e6, 1, 9, 8300, 16384),
        # a short prompt (128 ids, all but the last) on the 3B-shape target
        _layers("prefill_short_q4_k_m", "q4_k_m", 3072, 24, 8, 128, 8192, False, 5e5, 2, 127, 0, 2048),
        # the last pass of an 8K prompt on the 7B-shape target: the largest case
        _layers("prefill_long_q6_k", "q6_k", 3584, 28, 4, 128, 18944, True, 1e6, 1, 1023, 7168, 16384),
        # a prompt pass of the draft
        _layers("prefill_draft_q8_0", "q8_0", 896, 14, 2, 64, 4864, True, 1e6, 4, 1023, 0, 4096),
        # a model that keeps dense weights (1B shape, F16)
        _layers("prefill_f16", "f16", 2048, 32, 8, 64, 8192, False, 5e5, 1, 300, 0, 512),
        # the 7B-shape LM head over the 9 rows of a verify pass, with the greedy argmax
        {"name": "head_verify_q6_k", "kind": "head", "quant": "q6_k", "d_model": 3584, "vocab": 152064, "n_tok": 9},
        # one sampled token (the chat loop without a draft)
        {"name": "sample", "kind": "sample", "vocab": 152064, "top_k": 40, "top_p": 0.95, "temp": 0.8, "pen": 1.1,
         "last": 64},
        # one round of speculative sampling with k = 6
        {"name": "spec_round", "kind": "spec_round", "vocab": 152064, "top_k": 40, "top_p": 0.95, "temp": 0.8,
         "pen": 1.1, "last": 64, "k": 6},
        # a whole small model from its GGUF file: a 512-id prompt, then 8 decoded tokens
        {"name": "model_q8_0", "kind": "model", "quant": "q8_0", "d_model": 896, "heads": 14, "kv": 2, "hd": 64,
         "ffn": 4864, "bias": True, "theta": 1e6, "layers": 8, "vocab": 152064, "n_prompt": 512, "n_gen": 8,
         "ctx": 1024},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "verify", "verify", "prefill", "prefill", "prefill", "head", "sample", "spec_round",
                       "model"])
    if kind == "sample" or kind == "spec_round":
        c = {"kind": kind, "vocab": rng.randint(32000, 152064), "top_k": _log_int(rng, 2, 128),
             "top_p": round(rng.uniform(0.8, 1.0), 3), "temp": round(rng.uniform(0.5, 1.5), 2),
             "pen": rng.choice([1.0, 1.05, 1.1, 1.15]), "last": rng.choice([32, 64, 256])}
        if kind == "spec_round":
            c["k"] = rng.randint(2, 8)
        return c
    if kind == "head":
        q = rng.choice(["q6_k", "q6_k", "q8_0", "q4_k"])
        return {"kind": "head", "quant": q, "d_model": 256 * rng.randint(4, 14), "vocab": rng.randint(32000, 152064),
                "n_tok": rng.choice([1, 1, 2, 5, 7, 9, 16])}
    quant = rng.choice(["q4_k_m", "q4_k_m", "q6_k", "q8_0", "q8_0", "q4_0", "f16", "bf16"])
    if kind == "model" and quant == "q4_k_m":
        quant = "q6_k"  # a file of one type
    hd = rng.choice([64, 128])
    kv = rng.choice([2, 4, 8])
    group = rng.randint(2, 7)
    while kv * group * hd > 4096 or kv * group * hd < 512:
        kv, group = rng.choice([2, 4, 8]), rng.randint(2, 7)
    step = 256 if quant in ("q4_k_m", "q6_k") else 32
    while kv * group * hd % step:
        group += 1
    heads = kv * group
    if group > 8:
        heads = kv * 8
    d_model = step * max(1, _log_int(rng, 768, 3584) // step)
    ffn = step * max(1, int(d_model * rng.uniform(2.0, 5.3)) // step)
    bias, theta = rng.random() < 0.5, rng.choice([5e5, 1e6])
    per_layer = 2 * d_model * (heads + kv) * hd + 3 * d_model * ffn
    if kind == "model":
        return {"kind": "model", "quant": quant, "d_model": d_model, "heads": heads, "kv": kv, "hd": hd, "ffn": ffn,
                "bias": bias, "theta": theta, "layers": max(1, min(6, 100_000_000 // per_layer)), "vocab": 32000,
                "n_prompt": _log_int(rng, 17, 700), "n_gen": rng.randint(1, 8), "ctx": 1024}
    n_tok = {"decode": 1, "verify": rng.randint(2, VERIFY_MAX), "prefill": _log_int(rng, 17, 1023)}[kind]
    pos = 0 if rng.random() < 0.3 else _log_int(rng, 1, 7000)
    layers = 1 if kind == "prefill" else max(1, min(8, 200_000_000 // per_layer))
    ctx = -(-(pos + n_tok + 64) // 256) * 256
    return {k: v for k, v in _layers("", quant, d_model, heads, kv, hd, ffn, bias, theta, layers, n_tok, pos,
                                     ctx).items() if k != "name"}


# ── inputs ───────────────────────────────────────────────────────────────────
class Gen:
    """Random values on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * std

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=self.g) * (hi - lo) + lo

    def ints(self, lo, hi, *shape, dtype=torch.int32):
        return torch.randint(lo, hi, shape, device="cuda", generator=self.g, dtype=dtype)


def _matrix(g, quant, rows, cols):
    """A weight matrix of `rows` rows of `cols` values: its fields as stored in the GGUF blocks."""
    nb = cols // BLOCK[quant][0]
    if quant in ("f16", "bf16", "f32"):
        t = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[quant]
        return {"quant": quant, "w": g.normal(rows, cols, std=0.02).to(t)}
    scale = g.uniform(rows, nb, 1, lo=0.75, hi=1.25)
    if quant == "q8_0":
        q = (g.normal(rows, nb, 32) * 42).round().clamp(-127, 127).to(torch.int8)
        return {"quant": quant, "q": q, "d": (scale * (0.02 / 42)).half()}
    if quant == "q4_0":
        return {"quant": quant, "q": g.ints(0, 16, rows, nb, 32, dtype=torch.uint8), "d": (scale * (0.02 / 4.6)).half()}
    if quant == "q6_k":
        sc = g.ints(64, 128, rows, nb, 2, 4, 2, dtype=torch.int8)
        return {"quant": quant, "q": g.ints(0, 64, rows, nb, 2, 4, 32, dtype=torch.uint8),
                "sc": torch.where(g.uniform(rows, nb, 2, 4, 2) < 0.5, -sc, sc), "d": (scale * (0.02 / 1770)).half()}
    sc = g.ints(32, 64, rows, nb, 8, dtype=torch.uint8)  # q4_k
    mn = (sc.int() + g.ints(-4, 5, rows, nb, 8)).clamp(0, 63).to(torch.uint8)
    return {"quant": quant, "q": g.ints(0, 16, rows, nb, 8, 32, dtype=torch.uint8), "sc": sc, "m": mn,
            "d": (scale * (0.02 / 216)).half(), "dmin": (scale * (0.02 / 216 * 7.5)).half()}


def _pack(m):
    """The GGUF bytes of a matrix."""
    q, t = m["quant"], m.get("q")
    if q in ("f16", "bf16", "f32"):
        return m["w"].contiguous().view(torch.uint8).reshape(-1)
    d = m["d"].contiguous().view(torch.uint8)
    if q == "q8_0":
        parts = [d, t.view(torch.uint8)]
    elif q == "q4_0":
        parts = [d, t[..., :16] | (t[..., 16:] << 4)]
    elif q == "q6_k":
        lo = (t[..., 0:2, :] & 15) | ((t[..., 2:4, :] & 15) << 4)
        hi = t >> 4
        hi = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
        parts = [lo.flatten(2), hi.flatten(2), m["sc"].contiguous().view(torch.uint8).flatten(2), d]
    else:
        s, n = m["sc"], m["m"]
        parts = [d, m["dmin"].contiguous().view(torch.uint8), (s[..., :4] & 63) | ((s[..., 4:] >> 4) << 6),
                 (n[..., :4] & 63) | ((n[..., 4:] >> 4) << 6), (s[..., 4:] & 15) | ((n[..., 4:] & 15) << 4),
                 (t[..., 0::2, :] | (t[..., 1::2, :] << 4)).flatten(2)]
    return torch.cat(parts, -1).contiguous().reshape(-1)


def _w64(m):
    """The values of a matrix in 64 bits."""
    q = m["quant"]
    if q in ("f16", "bf16", "f32"):
        return m["w"].double()
    rows, d = m["q"].shape[0], m["d"].double()
    if q == "q8_0":
        return (m["q"].double() * d).reshape(rows, -1)
    if q == "q4_0":
        return ((m["q"].double() - 8) * d).reshape(rows, -1)
    if q == "q6_k":
        v = (m["q"].double() - 32).reshape(*m["q"].shape[:-1], 2, 16)
        return (v * m["sc"].double()[..., None] * d[:, :, :, None, None, None]).reshape(rows, -1)
    return (m["q"].double() * (d * m["sc"].double())[..., None] -
            (m["dmin"].double() * m["m"].double())[..., None]).reshape(rows, -1)


def _quants(quant):
    """Weight type of each matrix of a block, and of the embedding."""
    base, hi = ("q4_k", "q6_k") if quant == "q4_k_m" else (quant, quant)
    return {"q": base, "k": base, "v": hi, "o": base, "gate": base, "up": base, "down": hi, "embd": hi}


def _shapes(c):
    nq, nk = c["heads"] * c["hd"], c["kv"] * c["hd"]
    return {"q": (nq, c["d_model"]), "k": (nk, c["d_model"]), "v": (nk, c["d_model"]), "o": (c["d_model"], nq),
            "gate": (c["ffn"], c["d_model"]), "up": (c["ffn"], c["d_model"]), "down": (c["d_model"], c["ffn"])}


def _block_weights(c, g):
    ty = _quants(c["quant"])
    w = {n: _matrix(g, ty[n], r, k) for n, (r, k) in _shapes(c).items()}
    w["attn_norm"], w["ffn_norm"] = (1 + g.normal(c["d_model"], std=0.1) for _ in range(2))
    if c["bias"]:
        nq, nk = c["heads"] * c["hd"], c["kv"] * c["hd"]
        w["bq"], w["bk"], w["bv"] = g.normal(nq, std=0.02), g.normal(nk, std=0.02), g.normal(nk, std=0.02)
    return w


def _rope_table(c):
    """(cos, sin) of every position, in the float arithmetic the library documents."""
    half = c["hd"] // 2
    den = np.power(np.float32(c["theta"]), (np.arange(half) * 2).astype(np.float32) / np.float32(c["hd"]))
    th = (np.arange(c["ctx"], dtype=np.float32)[:, None] / den.astype(np.float32)[None]).astype(np.float32)
    return torch.from_numpy(np.stack([np.cos(th), np.sin(th)], -1).astype(np.float32)).cuda()


_dev = None


def _device():
    global _dev
    if _dev is None:
        torch.cuda.init()
        _dev = orc.Device(0)
    return _dev


class Mat:
    """A matrix in device memory; Q8_0 rows of a multiple of 256 values regrouped, as the model loader does."""

    def __init__(self, m, regroup=True):
        self.d = _pack(m)
        self.type = TYPES[m["quant"]]
        shape = m["w"].shape if "w" in m else (m["q"].shape[0], m["q"][0].numel())
        self.n_out, self.n_in = int(shape[0]), int(shape[1])
        if regroup and m["quant"] == "q8_0" and self.n_in % 256 == 0:
            dev = _device()
            torch.cuda.synchronize()
            dev.check(dev.L.orc_q8_0_regroup(self.d.data_ptr(), self.n_out * self.n_in // 256, None))
            dev.sync()
            self.type = orc.Q8_0_X8


def _prepare_layers(c, seed):
    dev, g = _device(), Gen(seed)
    n, D, nq, nk = c["n_tok"], c["d_model"], c["heads"] * c["hd"], c["kv"] * c["hd"]
    s = {"case": c, "dev": dev}
    s["embd"] = Mat(_matrix(g, _quants(c["quant"])["embd"], EMBED_ROWS, D), regroup=False)
    s["ids"] = g.ints(0, EMBED_ROWS, n)
    s["blocks"] = []
    for _ in range(c["layers"]):
        w = _block_weights(c, g)
        s["blocks"].append({k: Mat(v) if isinstance(v, dict) else v for k, v in w.items()})
    # the cache rows of the positions already processed; the rest is written by the passes
    s["k"] = torch.zeros(c["layers"], c["kv"], c["ctx"], c["hd"], device="cuda")
    s["v"] = torch.zeros_like(s["k"])
    for t in (s["k"], s["v"]):
        t[:, :, :c["pos"]] = g.normal(c["layers"], c["kv"], c["pos"], c["hd"])
    s["rope"] = _rope_table(c)
    s["x"], s["qkv"] = torch.empty(n, D, device="cuda"), torch.empty(n, nq + 2 * nk, device="cuda")
    s["att"], s["h"] = torch.empty(n, nq, device="cuda"), torch.empty(n, c["ffn"], device="cuda")
    s["work"] = torch.empty(dev.L.orc_attn_fused_workspace(c["heads"], c["kv"], c["hd"]), dtype=torch.uint8,
                            device="cuda")
    s["pos"] = torch.tensor([c["pos"]], dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    if n <= VERIFY_MAX:  # a step of the decode loop: captured once, replayed for every round
        graph = C.c_void_p()
        dev.check(dev.L.orc_graph_begin(None))
        _run_layers(s)
        dev.check(dev.L.orc_graph_end(None, C.byref(graph)))
        s["graph"] = Graph(dev, graph)
    return s


class Graph:
    def __init__(self, dev, graph):
        self.dev, self.graph = dev, graph

    def launch(self):
        self.dev.check(self.dev.L.orc_graph_launch(self.graph, None))

    def __del__(self):
        try:
            self.dev.L.orc_graph_destroy(self.graph)
        except Exception:
            pass


def _gemm(dev, mats, outs, biases, n, x, ldx, ldy, norm, epi):
    """One fused launch over the matrices; Q4_K and Q6_K segments of different types in a mixed one."""
    segs = (orc.Seg * len(mats))(*[orc.Seg(m.d.data_ptr(), m.n_out, y, b.data_ptr() if b is not None else None)
                                   for m, y, b in zip(mats, outs, biases)])
    npt, eps = (norm.data_ptr(), EPS) if norm is not None else (None, 0.0)
    if len({m.type for m in mats}) > 1:
        ty = (C.c_int32 * len(mats))(*[m.type for m in mats])
        dev.check(dev.L.orc_gemm_fused_mixed(ty, segs, len(mats), n, mats[0].n_in, x, ldx, ldy, npt, C.c_float(eps),
                                             epi, None))
    else:
        dev.check(dev.L.orc_gemm_fused(mats[0].type, segs, len(mats), n, mats[0].n_in, x, ldx, ldy, npt,
                                       C.c_float(eps), epi, None))


def _run_layers(s):
    c, dev = s["case"], s["dev"]
    L, n, D, H, KV, hd, ctx, pos = dev.L, c["n_tok"], c["d_model"], c["heads"], c["kv"], c["hd"], c["ctx"], c["pos"]
    nq, nk = H * hd, KV * hd
    ld = nq + 2 * nk
    x, qkv, att, h = (s[k].data_ptr() for k in ("x", "qkv", "att", "h"))
    e = s["embd"]
    dev.check(L.orc_embed(e.type, e.d.data_ptr(), D, EMBED_ROWS, s["ids"].data_ptr(), n, x, D, None))
    # the bounds of a captured step's positions, as the decode loops declare them
    floor = 512 if pos >= 512 else 0
    limit = min(ctx, max(512, 1 << (pos + n - 1).bit_length()))
    for i, b in enumerate(s["blocks"]):
        kc, vc = s["k"][i].data_ptr(), s["v"][i].data_ptr()
        _gemm(dev, [b["q"], b["k"], b["v"]], [qkv, qkv + 4 * nq, qkv + 4 * (nq + nk)],
              [b.get("bq"), b.get("bk"), b.get("bv")], n, x, D, ld, b["attn_norm"], orc.EPI_STORE)
        if n <= VERIFY_MAX:
            dev.check(L.orc_attn_fused_at(qkv, ld, n, H, KV, hd, s["pos"].data_ptr(), 0, s["rope"].data_ptr(), kc, vc,
                                          ctx, floor, limit, att, nq, s["work"].data_ptr(), None))
        else:
            dev.check(L.orc_attn_prefill(qkv, ld, n, H, KV, hd, pos, s["rope"].data_ptr(), kc, vc, ctx, att, nq,
                                         None))
        _gemm(dev, [b["o"]], [x], [None], n, att, nq, D, None, orc.EPI_ACCUM)
        _gemm(dev, [b["gate"], b["up"]], [h, h], [None, None], n, x, D, c["ffn"], b["ffn_norm"], orc.EPI_SWIGLU)
        _gemm(dev, [b["down"]], [x], [None], n, h, c["ffn"], D, None, orc.EPI_ACCUM)


def _layers_out(s):
    c = s["case"]
    new = slice(c["pos"], c["pos"] + c["n_tok"])
    return {"x": s["x"], "k": s["k"][:, :, new], "v": s["v"][:, :, new]}


def _prepare_head(c, seed):
    dev, g = _device(), Gen(seed)
    s = {"case": c, "dev": dev, "w": Mat(_matrix(g, c["quant"], c["vocab"], c["d_model"]))}
    s["norm"], s["x"] = 1 + g.normal(c["d_model"], std=0.1), g.normal(c["n_tok"], c["d_model"])
    s["logits"] = torch.empty(c["n_tok"], c["vocab"], device="cuda")
    s["ids"] = torch.empty(c["n_tok"], dtype=torch.int32, device="cuda")
    s["work"] = torch.empty(dev.L.orc_argmax_workspace(c["n_tok"], c["vocab"]), dtype=torch.uint8, device="cuda")
    return s


def _run_head(s):
    c, dev = s["case"], s["dev"]
    y, V = s["logits"].data_ptr(), c["vocab"]
    _gemm(dev, [s["w"]], [y], [None], c["n_tok"], s["x"].data_ptr(), c["d_model"], V, s["norm"], orc.EPI_STORE)
    dev.check(dev.L.orc_argmax(y, c["n_tok"], V, V, s["ids"].data_ptr(), s["work"].data_ptr(), None))
    return {"logits": s["logits"], "ids": s["ids"]}


def _sampling_inputs(c, seed):
    """Rows of logits (a few plausible tokens over a wide tail) and the recorded tokens."""
    g = Gen(seed)
    rows = 1 if c["kind"] == "sample" else 2 * c["k"] + 1
    logits = g.normal(rows, c["vocab"], std=2.5)
    hist = g.ints(0, c["vocab"], c["last"])
    if rows > 1:  # the draft's rows resemble the target's
        logits[:c["k"]] = logits[c["k"]:2 * c["k"]] + 0.3 * logits[:c["k"]]
    # some recorded tokens are likely ones
    hist[:8] = torch.topk(logits[-1], 8).indices.to(torch.int32)
    return logits, hist


def _prepare_sampling(c, seed):
    dev = _device()
    logits, hist = _sampling_inputs(c, seed)
    V = c["vocab"]
    s = {"case": c, "dev": dev, "logits": logits, "rows": torch.empty_like(logits)}
    s["state"] = torch.empty(dev.L.orc_sampler_state_bytes(), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    dev.check(dev.L.orc_sampler_init(s["state"].data_ptr(), C.c_float(c["temp"]), C.c_float(c["top_p"]), c["top_k"],
                                     C.c_float(c["pen"]), c["last"], int(seed) & 0xFFFFFFFF, hist.data_ptr(),
                                     c["last"], None))
    dev.sync()
    s["out"] = torch.zeros(c.get("k", 0) + 5, dtype=torch.int32, device="cuda")
    if c["kind"] == "spec_round":
        k = c["k"]
        s["q"], s["p"] = torch.empty(k, V, device="cuda"), torch.empty(k + 1, V, device="cuda")
        s["x"] = torch.zeros(k, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        graph = C.c_void_p()  # rounds are captured once and replayed
        dev.check(dev.L.orc_graph_begin(None))
        _run_spec_round(s)
        dev.check(dev.L.orc_graph_end(None, C.byref(graph)))
        s["graph"] = Graph(dev, graph)
    return s


def _run_sample(s):
    c, dev = s["case"], s["dev"]
    row = s["rows"].data_ptr()  # the sampler rewrites its row: it gets a copy, as of a forward pass
    dev.check(dev.L.orc_memcpy_d2d(row, s["logits"].data_ptr(), 4 * c["vocab"], None))
    dev.check(dev.L.orc_sample(s["state"].data_ptr(), row, c["vocab"], s["out"].data_ptr(), None))
    return {"p": s["rows"], "id": s["out"][:1]}


def _run_spec_round(s):
    c, dev = s["case"], s["dev"]
    L, V, k = dev.L, c["vocab"], c["k"]
    row, q, p, x, st = (s[n].data_ptr() for n in ("rows", "q", "p", "x", "state"))
    dev.check(L.orc_memcpy_d2d(row, s["logits"].data_ptr(), 4 * V * (2 * k + 1), None))
    for i in range(k):
        dev.check(L.orc_transform_draw(st, row + 4 * V * i, V, x if i else None, i, q + 4 * V * i, x + 4 * i, None,
                                       None))
    dev.check(L.orc_transform_probs(st, row + 4 * V * k, V, V, k + 1, x, 0, p, V, None))
    dev.check(L.orc_spec_accept_stochastic(st, p, V, q, V, V, x, k, k + 1, None, s["out"].data_ptr(), None, None,
                                           None))


def _write_gguf(path, c, g):
    """A model file of the case's shape (tied head), with random blocks."""
    def text(v):
        b = v.encode()
        return struct.pack("<Q", len(b)) + b

    ty = c["quant"]
    tensors = [("token_embd.weight", _matrix(g, ty, c["vocab"], c["d_model"]))]
    names = {"q": "attn_q", "k": "attn_k", "v": "attn_v", "o": "attn_output", "gate": "ffn_gate", "up": "ffn_up",
             "down": "ffn_down"}
    for i in range(c["layers"]):
        w = _block_weights(c, g)
        b = "blk.%d." % i
        tensors += [(b + names[n] + ".weight", w[n]) for n in names]
        tensors += [(b + "attn_norm.weight", w["attn_norm"]), (b + "ffn_norm.weight", w["ffn_norm"])]
        if c["bias"]:
            tensors += [(b + "attn_q.bias", w["bq"]), (b + "attn_k.bias", w["bk"]), (b + "attn_v.bias", w["bv"])]
    tensors.append(("output_norm.weight", 1 + g.normal(c["d_model"], std=0.1)))
    arch = "qwen2" if c["bias"] else "llama"
    meta = [("general.architecture", arch)]
    for key, v in (("block_count", c["layers"]), ("context_length", c["ctx"]), ("embedding_length", c["d_model"]),
                   ("feed_forward_length", c["ffn"]), ("attention.head_count", c["heads"]),
                   ("attention.head_count_kv", c["kv"]), ("attention.key_length", c["hd"]),
                   ("attention.value_length", c["hd"]), ("vocab_size", c["vocab"]),
                   ("rope.freq_base", float(c["theta"])), ("attention.layer_norm_rms_epsilon", EPS)):
        meta.append((arch + "." + key, v))
    with open(path, "wb") as f:
        f.write(b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(meta)))
        for key, v in meta:
            f.write(text(key))
            f.write(struct.pack("<I", 8) + text(v) if isinstance(v, str) else
                    struct.pack("<If", 6, v) if isinstance(v, float) else struct.pack("<II", 4, v))
        data, at = [], 0
        for name, m in tensors:
            if isinstance(m, dict):
                raw, t = _pack(m), TYPES[m["quant"]]
                dims = (m["w"].shape[1], m["w"].shape[0]) if "w" in m else (m["q"][0].numel(), m["q"].shape[0])
            else:
                raw, t, dims = m.contiguous().view(torch.uint8).reshape(-1), orc.F32, (m.numel(),)
            f.write(text(name) + struct.pack("<I", len(dims)) + b"".join(struct.pack("<Q", d) for d in dims) +
                    struct.pack("<IQ", t, at))
            raw = raw.cpu().numpy()
            pad = -raw.size % 32
            data.append((raw, pad))
            at += raw.size + pad
        f.write(b"\0" * (-f.tell() % 32))
        for raw, pad in data:
            f.write(raw.data)
            f.write(b"\0" * pad)
    return tensors


def _tokens(c, seed):
    return np.random.default_rng(int(seed)).integers(0, c["vocab"], c["n_prompt"] + c["n_gen"]).astype(np.int32)


def _prepare_model(c, seed):
    _device()
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.gguf")
        _write_gguf(path, c, Gen(seed))
        torch.cuda.empty_cache()
        model = orc.Model(path, c["ctx"])
    return {"case": c, "model": model, "tokens": _tokens(c, seed)}


def _run_model(s):
    c, m, t = s["case"], s["model"], s["tokens"]
    n = c["n_prompt"]
    m.forward_batch(t[:n], 0, logits=False)
    return np.stack([m.forward(t[n + i], n + i) for i in range(c["n_gen"])])


# ── the case interface ───────────────────────────────────────────────────────
def prepare(case, seed):
    return {"layers": _prepare_layers, "head": _prepare_head, "sample": _prepare_sampling,
            "spec_round": _prepare_sampling, "model": _prepare_model}[case["kind"]](case, seed)


def run(state):
    kind = state["case"]["kind"]
    if kind == "layers":
        if "graph" in state:
            state["graph"].launch()
        else:
            _run_layers(state)
        return _layers_out(state)
    if kind == "spec_round":
        state["graph"].launch()
        return {"q": state["q"], "p": state["p"], "x": state["x"], "out": state["out"]}
    return {"head": _run_head, "sample": _run_sample, "model": _run_model}[kind](state)


def _bytes(quant, values):
    per, size = BLOCK[quant]
    return values // per * size


def work(case):
    c, kind = case, case["kind"]
    if kind in ("sample", "spec_round"):
        rows = 1 if kind == "sample" else 2 * c["k"] + 1
        return {"bytes": 8 * rows * c["vocab"], "flops": 8 * rows * c["vocab"]}
    if kind == "head":
        w = c["vocab"] * c["d_model"]
        return {"bytes": _bytes(c["quant"], w) + 4 * c["n_tok"] * (c["d_model"] + c["vocab"]),
                "flops": 2 * c["n_tok"] * w}
    passes = [(c["n_tok"], c["pos"])] if kind == "layers" else \
        [(c["n_prompt"], 0)] + [(1, c["n_prompt"] + i) for i in range(c["n_gen"])]
    ty, sh = _quants(c["quant"]), _shapes(c)
    wb = sum(_bytes(ty[n], r * k) for n, (r, k) in sh.items())
    params = sum(r * k for r, k in sh.values())
    total = {"bytes": 0, "flops": 0}
    for n, pos in passes:
        keys = n * pos + n * (n + 1) // 2  # (query, key) pairs
        total["bytes"] += c["layers"] * (wb + 8 * c["kv"] * c["hd"] * (pos + n)) + 8 * n * c["d_model"]
        total["flops"] += c["layers"] * (2 * n * params + 4 * keys * c["heads"] * c["hd"])
    if kind == "model":
        head = c["vocab"] * c["d_model"]
        total["bytes"] += c["n_gen"] * (_bytes(c["quant"], head) + 4 * c["vocab"])
        total["flops"] += 2 * c["n_gen"] * head
    return total


def tolerance(case):
    # 32-bit products and sums throughout
    return {"rel": 1e-5}


# ── 64-bit references ────────────────────────────────────────────────────────
def _norm64(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g.double()


def _rope64(t, cs, hd):
    """Rotate-half RoPE of [n][heads * hd] rows with the (cos, sin) pairs of their positions."""
    n = t.shape[0]
    t = t.reshape(n, -1, hd)
    a, b = t[..., :hd // 2], t[..., hd // 2:]
    co, si = cs[:, None, :, 0].double(), cs[:, None, :, 1].double()
    return torch.cat([a * co - b * si, a * si + b * co], -1)


def _block64(c, w, x, rope, pos, kc, vc):
    """One transformer block on x [n][D] at positions pos.. over the cache rows kc / vc [kv][pos][hd]."""
    n, hd, KV = x.shape[0], c["hd"], c["kv"]
    group = c["heads"] // KV
    xn = _norm64(x, w["attn_norm"])
    q, k, v = (xn @ _w64(w[m]).T + (w["b" + m].double() if c["bias"] else 0) for m in ("q", "k", "v"))
    cs = rope[pos:pos + n]
    q, k, v = _rope64(q, cs, hd), _rope64(k, cs, hd), v.reshape(n, KV, hd)
    mask = torch.arange(pos + n, device="cuda")[None] > (pos + torch.arange(n, device="cuda"))[:, None]
    att = torch.empty(n, c["heads"], hd, dtype=torch.float64, device="cuda")
    for j in range(KV):
        kk, vv = torch.cat([kc[j], k[:, j]]), torch.cat([vc[j], v[:, j]])
        for i in range(j * group, (j + 1) * group):
            sc = (q[:, i] @ kk.T / math.sqrt(hd)).masked_fill_(mask, -math.inf)
            att[:, i] = torch.softmax(sc, -1) @ vv
    x = x + att.reshape(n, -1) @ _w64(w["o"]).T
    xn = _norm64(x, w["ffn_norm"])
    gate, up = xn @ _w64(w["gate"]).T, xn @ _w64(w["up"]).T
    return x + (gate * torch.sigmoid(gate) * up) @ _w64(w["down"]).T, k.transpose(0, 1), v.transpose(0, 1)


def _exact_layers(c, seed):
    g = Gen(seed)
    e = _matrix(g, _quants(c["quant"])["embd"], EMBED_ROWS, c["d_model"])
    ids = g.ints(0, EMBED_ROWS, c["n_tok"])
    blocks = [_block_weights(c, g) for _ in range(c["layers"])]
    kc, vc = (g.normal(c["layers"], c["kv"], c["pos"], c["hd"]).double() for _ in range(2))
    rope, x, ks, vs = _rope_table(c), _w64(e)[ids.long()], [], []
    for i, w in enumerate(blocks):
        x, k, v = _block64(c, w, x, rope, c["pos"], kc[i], vc[i])
        ks.append(k)
        vs.append(v)
    return {"x": x, "k": torch.stack(ks), "v": torch.stack(vs)}


def _exact_head(c, seed):
    g = Gen(seed)
    w = _matrix(g, c["quant"], c["vocab"], c["d_model"])
    norm, x = 1 + g.normal(c["d_model"], std=0.1), g.normal(c["n_tok"], c["d_model"])
    return {"logits": _norm64(x.double(), norm) @ _w64(w).T, "ids": None}


def _scaled64(c, row, window):
    """A row of logits after the repeat penalty over the window and 1 / temperature."""
    row = row.double().clone()
    if c["pen"] > 1:
        pen = float(np.float32(c["pen"]))
        for i in window[-c["last"]:]:
            row[i] = row[i] / pen if row[i] > 0 else row[i] * pen
    return row / float(np.float32(c["temp"]))


def _transform64(c, row, window):
    """The sampler's distribution of a row: top-k, top-p, kept set renormalised."""
    p = torch.softmax(_scaled64(c, row, window), -1)
    top, ids = torch.sort(p, descending=True, stable=True)
    top, ids = top[:c["top_k"]], ids[:c["top_k"]]
    cut = int((torch.cumsum(top, 0) < float(np.float32(c["top_p"]))).sum()) + 1
    out = torch.zeros_like(p)
    out[ids[:cut]] = top[:cut] / top[:cut].sum()
    return out


def _exact_sample(c, seed):
    logits, hist = _sampling_inputs(c, seed)
    return {"p": torch.softmax(_scaled64(c, logits[0], hist.tolist()), -1)[None], "id": None}


def _exact_spec_round(c, seed):
    logits, hist = _sampling_inputs(c, seed)
    draws, k = np.random.RandomState(int(seed) & 0xFFFFFFFF), c["k"]
    window, q = hist.tolist(), []
    for i in range(k):
        q.append(_transform64(c, logits[i], window))
        u = float(np.float32(draws.randint(0, 1 << 32, dtype=np.uint32)) / np.float32(4294967296.0))
        run = torch.cumsum(q[-1], 0)
        at = int((run < u * run[-1]).sum())
        window.append(min(at, int(torch.nonzero(q[-1])[-1])))
    p = [_transform64(c, logits[k + r], window[:c["last"] + r]) for r in range(k + 1)]
    return {"q": torch.stack(q), "p": torch.stack(p), "x": None, "out": None}


def _exact_model(c, seed):
    g = Gen(seed)
    e = _matrix(g, c["quant"], c["vocab"], c["d_model"])
    blocks = [_block_weights(c, g) for _ in range(c["layers"])]
    norm = 1 + g.normal(c["d_model"], std=0.1)
    ids, rope = torch.from_numpy(_tokens(c, seed)).long().cuda(), _rope_table(c)
    ew = _w64(e)
    x = ew[ids]
    none = torch.empty(c["kv"], 0, c["hd"], dtype=torch.float64, device="cuda")
    for w in blocks:
        x = _block64(c, w, x, rope, 0, none, none)[0]
    return (_norm64(x[c["n_prompt"]:], norm) @ ew.T).cpu().numpy()


def exact(case, seed):
    return {"layers": _exact_layers, "head": _exact_head, "sample": _exact_sample, "spec_round": _exact_spec_round,
            "model": _exact_model}[case["kind"]](case, seed)
