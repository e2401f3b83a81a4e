"""Performance cases of the quantized compute path: what each stands for, its inputs, one pass, its cost and accuracy.

A case is a dict of plain values with a "kind":

  matvec        one matrix-vector product through the engine entry point on host buffers (x in, y out)
  ffn_gemv      one token's feed-forward products (up, then down) of several layers, batch 1
  layer_decode  one decoder layer for one token over its Q8_0 KV cache, replayed as a captured graph (the position is
                in device memory, as a decode loop keeps it)
  attn_decode   one token's attention over a long Q8_0 KV cache
  gemm          the product of a prompt (or of a few drafted or batched tokens) with one weight matrix
  layer_prefill one decoder layer over a prompt chunk behind a cached context
  attn_prefill  a prompt chunk's attention over the Q8_0 KV cache
  moe           the routed expert feed-forward layer
  head          final norm, output head and top-k of one token

Weights are drawn as a quantizer of zero-mean Gaussian matrices of standard deviation 1 / sqrt(cols) leaves them
(every format's bytes are made here), activations are N(0, 1), cache rows are quantized N(0, 1).
"""
import ctypes
import math

import numpy as np
import torch

from desireeia_amd import _lib, ops

Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14  # GGUF type ids
TYPES = {"q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K}
BLOCK = {Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}
# matrix types of a layer: the common 4-bit mix (6-bit values and down projection) and the plain formats
MIXES = {"q4_k_m": {"v": "q6_k", "down": "q6_k", "*": "q4_k"}, "q8_0": {"*": "q8_0"}, "q4_0": {"*": "q4_0"},
         "q6_k": {"*": "q6_k"}}
THETA, EPS = 500000.0, 1e-5


def listed():
    return [
        # an engine that offloads single products calls with host vectors: the smallest call, all latency
        {"name": "matvec_q8_0_4096", "kind": "matvec", "fmt": "q8_0", "rows": 4096, "cols": 4096},
        # the feed-forward products of a decoded token, 4 layers of an 8B model
        {"name": "ffn_gemv_q4_k", "kind": "ffn_gemv", "fmt": "q4_k", "n_embd": 4096, "n_ff": 14336, "layers": 4},
        # decoding with an 8B model at a 4096-token context
        {"name": "layer_decode_8b_4096", "kind": "layer_decode", "mix": "q4_k_m", "n_embd": 4096, "n_head": 32,
         "n_head_kv": 8, "head_dim": 128, "n_ff": 14336, "pos": 4096, "style": "plain"},
        # decoding with a small 8-bit model early in a conversation: biases and QK-norm, 64-value heads
        {"name": "layer_decode_small_300", "kind": "layer_decode", "mix": "q8_0", "n_embd": 1024, "n_head": 16,
         "n_head_kv": 4, "head_dim": 64, "n_ff": 2048, "pos": 300, "style": "qwen"},
        # decoding with a long document in the context
        {"name": "attn_decode_32k", "kind": "attn_decode", "n_head": 32, "n_head_kv": 8, "head_dim": 128,
         "pos": 32767},
        # a prompt chunk's product with the gate or up matrix
        {"name": "gemm_q4_k_512", "kind": "gemm", "fmt": "q4_k", "rows": 14336, "cols": 4096, "n_tok": 512},
        # a short follow-up question (or drafted tokens) against the 6-bit down matrix
        {"name": "gemm_q6_k_29", "kind": "gemm", "fmt": "q6_k", "rows": 4096, "cols": 14336, "n_tok": 29},
        # the second chunk of a long prompt: the largest chunk the engine sends
        {"name": "layer_prefill_2048", "kind": "layer_prefill", "mix": "q4_k_m", "n_embd": 4096, "n_head": 32,
         "n_head_kv": 8, "head_dim": 128, "n_ff": 14336, "pos0": 2048, "n_tok": 2048, "style": "plain"},
        # a follow-up turn's attention behind a cached conversation
        {"name": "attn_prefill_512_3584", "kind": "attn_prefill", "n_head": 32, "n_head_kv": 8, "head_dim": 128,
         "pos0": 3584, "n_tok": 512, "n_swa": 0},
        # a mixture-of-experts layer: a batch of tokens, and one decoded token
        {"name": "moe_64", "kind": "moe", "n_expert": 8, "k": 2, "n_embd": 4096, "n_ff": 14336, "n_tok": 64},
        {"name": "moe_1", "kind": "moe", "n_expert": 8, "k": 2, "n_embd": 4096, "n_ff": 14336, "n_tok": 1},
        # the last step of every decoded token: the head of a 128256-token vocabulary and its candidates
        {"name": "head_q6_k_128256", "kind": "head", "fmt": "q6_k", "rows": 128256, "cols": 4096, "kk": 104},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    return step * rng.randint(-(-lo // step), hi // step)


def _layer_shape(rng):
    hd = rng.choice((64, 128, 128, 256))
    per = rng.choice((1, 2, 4, 4, 8))
    n_kv = rng.choice([n for n in (1, 2, 4, 8) if n * per * hd % 256 == 0 and n * per * hd <= 4096])
    return {"mix": rng.choice(("q4_k_m", "q4_k_m", "q8_0", "q4_0", "q6_k")), "n_embd": _mult(rng, 512, 4096, 256),
            "n_head": n_kv * per, "n_head_kv": n_kv, "head_dim": hd, "n_ff": _mult(rng, 1024, 14336, 256)}


def draw(rng):
    kind = rng.choice(("matvec", "ffn_gemv", "layer_decode", "layer_decode", "attn_decode", "gemm", "gemm", "gemm",
                       "layer_prefill", "attn_prefill", "moe", "head"))
    fmt = rng.choice(("q4_k", "q4_k", "q6_k", "q8_0", "q4_0"))
    if kind == "matvec":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 64, 16384), "cols": _mult(rng, 512, 14336, 256)}
    if kind == "ffn_gemv":
        e, f = _mult(rng, 1024, 4096, 256), _mult(rng, 2048, 14336, 256)
        return {"kind": kind, "fmt": fmt, "n_embd": e, "n_ff": f, "layers": rng.randint(2, 4)}
    if kind == "layer_decode":
        return dict(_layer_shape(rng), kind=kind, pos=_log(rng, 1, 8192),
                    style=rng.choice(("plain", "qwen", "gemma", "gate")))
    if kind in ("attn_decode", "attn_prefill"):
        hd = rng.choice((64, 128, 128, 256))
        n_kv, per = rng.choice((2, 4, 8)), rng.choice((2, 4, 4, 8))
        c = {"kind": kind, "n_head": n_kv * per, "n_head_kv": n_kv, "head_dim": hd}
        if kind == "attn_decode":
            return dict(c, pos=_log(rng, 64, 32767))
        return dict(c, pos0=_log(rng, 1, 4096) - 1, n_tok=_log(rng, 8, 1024), n_swa=rng.choice((0, 0, 0, 1024)))
    if kind == "gemm":
        rows, cols = _log(rng, 256, 14336), _mult(rng, 1024, 14336, 256)
        return {"kind": kind, "fmt": fmt, "rows": rows, "cols": cols, "n_tok": _log(rng, 4, 1024)}
    if kind == "layer_prefill":
        return dict(_layer_shape(rng), kind=kind, pos0=_log(rng, 1, 2048) - 1, n_tok=_log(rng, 8, 1024),
                    style=rng.choice(("plain", "plain", "qwen")))
    if kind == "moe":
        n_expert = rng.choice((4, 8, 16, 32, 64))
        return {"kind": kind, "n_expert": n_expert, "k": rng.choice((2, 2, 4)), "n_embd": _mult(rng, 1024, 4096, 256),
                "n_ff": _mult(rng, 512, 14336 * 8 // max(8, n_expert), 256), "n_tok": _log(rng, 1, 512)}
    return {"kind": kind, "fmt": fmt, "rows": _log(rng, 8000, 152000), "cols": _mult(rng, 1024, 4096, 256),
            "kk": rng.randint(1, 256)}


# ------------------------------------------------------------------ inputs --

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Gen:
    """Seeded draws on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=_dev()).manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, device=_dev(), generator=self.g)

    def uniform(self, lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, device=_dev(), generator=self.g)

    def weights(self, qtype, rows, cols, std=None):
        """GGUF bytes [rows][row bytes] of a Gaussian matrix, made in pieces of 4096 rows."""
        std = cols ** -0.5 if std is None else std
        return torch.cat([self._piece(qtype, min(4096, rows - r), cols, std) for r in range(0, rows, 4096)])

    def _piece(self, qtype, rows, cols, std):
        qk, sz = BLOCK[qtype]
        nb = rows * cols // qk

        def half(v):
            return v.half().view(torch.uint8).reshape(nb, 2)

        def ints(sd, mid, lo, hi):
            return (self.normal(nb, qk) * sd + mid).round_().clamp_(lo, hi)

        blk = torch.empty(nb, sz, dtype=torch.uint8, device=_dev())
        jitter = self.uniform(0.8, 1.25, nb)
        if qtype == Q8_0:
            blk[:, :2] = half(std / 42 * jitter)
            blk[:, 2:] = ints(42, 0, -127, 127).to(torch.int8).view(torch.uint8)
        elif qtype == Q4_0:
            q = ints(2.8, 8, 0, 15).to(torch.uint8)
            blk[:, :2] = half(std / 2.8 * jitter)
            blk[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
        elif qtype == Q4_K:
            q = ints(3, 7.5, 0, 15).to(torch.uint8).view(nb, 4, 2, 32)
            sc = self.uniform(28, 63, nb, 8).round_()
            mn = (sc * (7.5 / 8)).round_().to(torch.uint8)
            sc = sc.to(torch.uint8)
            d = std / 3 / 45 * jitter
            blk[:, 0:2], blk[:, 2:4] = half(d), half(8 * d)
            blk[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
            blk[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
            blk[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
            blk[:, 16:] = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128)
        else:
            q = ints(10, 32, 0, 63).to(torch.uint8).view(nb, 2, 4, 32)  # [half][quarter][32]
            lo, hi = q & 15, q >> 4
            ql = torch.stack((lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)), 2)
            blk[:, :128] = ql.reshape(nb, 128)
            blk[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(nb, 64)
            sign = 1 - 2 * (self.uniform(0, 1, nb, 16) < 0.5).float()
            blk[:, 192:208] = (self.uniform(64, 127, nb, 16).round_() * sign).to(torch.int8).view(torch.uint8)
            blk[:, 208:] = half(std / 10 / 96 * jitter)
        return blk.view(rows, cols // qk * sz)

    def cache(self, n_pos, n_head_kv, hd):
        """Rows of a Q8_0 cache: N(0, 1) rows, quantized per 32."""
        v = self.normal(n_pos * n_head_kv * hd // 32, 32)
        d = v.abs().amax(1, keepdim=True) / 127
        blk = torch.empty(len(v), 34, dtype=torch.uint8, device=_dev())
        blk[:, :2] = d.half().view(torch.uint8)
        blk[:, 2:] = (v / d).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        return blk.view(n_pos, n_head_kv * hd // 32 * 34)


def _layer_shapes(c):
    mix, e, f = MIXES[c["mix"]], c["n_embd"], c["n_ff"]
    qd, kvd = c["n_head"] * c["head_dim"], c["n_head_kv"] * c["head_dim"]
    s = {"q": (qd, e), "k": (kvd, e), "v": (kvd, e), "o": (e, qd), "gate": (f, e), "up": (f, e), "down": (e, f)}
    if c["style"] == "gate":
        s["ag"] = (c["n_head"], e)
    return {n: (TYPES["q8_0" if n == "ag" else mix.get(n, mix["*"])],) + rc for n, rc in s.items()}


def _inputs(c, seed):
    """The raw inputs of a case, the same for prepare() and exact()."""
    g, kind, s = _Gen(seed), c["kind"], {}
    if kind in ("matvec", "gemm", "head"):
        s["w"] = g.weights(TYPES[c["fmt"]], c["rows"], c["cols"])
        s["x"] = g.normal(c["n_tok"], c["cols"]) if kind == "gemm" else g.normal(c["cols"])
        if kind == "head":
            s["norm"] = 1 + 0.1 * g.normal(c["cols"])
    elif kind == "ffn_gemv":
        t, e, f = TYPES[c["fmt"]], c["n_embd"], c["n_ff"]
        s["up"] = [g.weights(t, f, e) for _ in range(c["layers"])]
        s["down"] = [g.weights(t, e, f) for _ in range(c["layers"])]
        s["x"], s["h"] = g.normal(c["layers"], e), g.normal(c["layers"], f)
    elif kind in ("layer_decode", "layer_prefill"):
        e, hd, kvd = c["n_embd"], c["head_dim"], c["n_head_kv"] * c["head_dim"]
        s["w"] = {n: g.weights(t, r, k) for n, (t, r, k) in _layer_shapes(c).items()}
        n_prior = c["pos"] if kind == "layer_decode" else c["pos0"]
        n_new = 1 if kind == "layer_decode" else c["n_tok"]
        s["k"], s["v"] = (g.cache(n_prior, c["n_head_kv"], hd) for _ in range(2))
        s["x"] = g.normal(n_new, e)
        s["norms"] = [1 + 0.1 * g.normal(e) for _ in range(4)]
        s["bias"] = [0.3 * g.normal(n) for n in (c["n_head"] * hd, kvd, kvd)]
        s["qk"] = [1 + 0.1 * g.normal(hd) for _ in range(2)]
    elif kind in ("attn_decode", "attn_prefill"):
        n_pos = c["pos"] + 1 if kind == "attn_decode" else c["pos0"] + c["n_tok"]
        s["k"], s["v"] = (g.cache(n_pos, c["n_head_kv"], c["head_dim"]) for _ in range(2))
        s["q"] = g.normal(c.get("n_tok", 1), c["n_head"] * c["head_dim"])
    else:
        n, e, f = c["n_expert"], c["n_embd"], c["n_ff"]
        s["gate"], s["up"] = g.weights(Q4_K, n * f, e), g.weights(Q4_K, n * f, e)
        s["down"] = g.weights(Q4_K, n * e, f)
        s["x"], s["logits"] = g.normal(c["n_tok"], e), g.normal(c["n_tok"], n)
    return s


# -------------------------------------------------------------- the passes --

class _Uploaded:
    """A matrix uploaded through the engine entry point, freed with its owner."""

    def __init__(self, fmt, data, rows, cols):
        self.fmt, self.qs, self.scale = fmt, ctypes.c_void_p(), ctypes.c_void_p()
        host = data.cpu().numpy()
        if not _lib.load().cuda_upload_weights(fmt, host.ctypes.data_as(ctypes.c_void_p), rows, cols,
                                               ctypes.byref(self.qs), ctypes.byref(self.scale)):
            raise RuntimeError("cuda_upload_weights failed")

    def __del__(self):
        _lib.load().cuda_free_device(self.qs)


def _layer(c, s, n_ctx):
    mats = {n: ops.QuantMatrix.from_gguf(t, s["w"][n], r, k) for n, (t, r, k) in _layer_shapes(c).items()}
    style = c["style"]
    layer = ops.DecoderLayer(mats, s["norms"][0], s["norms"][1], c["n_head"], c["n_head_kv"], c["head_dim"], n_ctx,
                             rms_eps=EPS, rope_theta=THETA, bias=s["bias"] if style == "qwen" else None,
                             qk_norm=s["qk"] if style == "qwen" else None, act_gelu=style == "gemma",
                             post_norms=s["norms"][2:] if style == "gemma" else None, attn_gate=mats.get("ag"))
    for own, given in ((layer.cache.k, s["k"]), (layer.cache.v, s["v"])):
        own[:given.numel()].copy_(given.reshape(-1))
    return layer


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    kind, st = c["kind"], {"case": case}
    if kind == "matvec":
        t = TYPES[c["fmt"]]
        st["m"] = _Uploaded(ops.FMT_OF_TYPE[t], s["w"], c["rows"], c["cols"])
        st["x"], st["y"] = s["x"].cpu().numpy(), np.empty(c["rows"], np.float32)
    elif kind == "ffn_gemv":
        t, e, f = TYPES[c["fmt"]], c["n_embd"], c["n_ff"]
        st["up"] = [ops.QuantMatrix.from_gguf(t, w, f, e) for w in s["up"]]
        st["down"] = [ops.QuantMatrix.from_gguf(t, w, e, f) for w in s["down"]]
        st["x"], st["h"] = s["x"], s["h"]
        st["y_up"], st["y_down"] = torch.empty_like(s["h"]), torch.empty_like(s["x"])
    elif kind == "layer_decode":
        layer = st["layer"] = _layer(c, s, c["pos"] + 1)
        st["x"], st["y"] = s["x"].reshape(-1), torch.empty_like(s["x"].reshape(-1))
        layer.set_rope(c["pos"])
        st["pos"] = torch.tensor([c["pos"]], dtype=torch.int32, device="cuda")
        layer.decode(st["x"], st["pos"], out=st["y"])
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            layer.decode(st["x"], st["pos"], out=st["y"])
    elif kind == "gemm":
        st["m"] = ops.QuantMatrix.from_gguf(TYPES[c["fmt"]], s["w"], c["rows"], c["cols"])
        st["x"], st["work"] = s["x"], ops.gemm_workspace(st["m"], c["n_tok"])
        st["y"] = torch.empty(c["n_tok"], c["rows"], device="cuda")
    elif kind == "layer_prefill":
        layer = st["layer"] = _layer(c, s, c["pos0"] + c["n_tok"])
        st["x"], st["y"], st["work"] = s["x"], torch.empty_like(s["x"]), layer.prefill_workspace(c["n_tok"])
        st["rope"] = torch.stack([ops.rope_cache(c["head_dim"], c["pos0"] + t, THETA)
                                  for t in range(c["n_tok"])]).cuda()
    elif kind in ("attn_decode", "attn_prefill"):
        n_pos = len(s["k"])
        st["cache"] = ops.KVCache(n_pos, c["n_head_kv"], c["head_dim"])
        st["cache"].k.copy_(s["k"].reshape(-1))
        st["cache"].v.copy_(s["v"].reshape(-1))
        if kind == "attn_decode":
            st["q"] = s["q"].reshape(-1)
            st["work"] = ops.attn_workspace(c["n_head"], c["n_head_kv"], c["head_dim"], n_pos)
        else:
            st["q"] = s["q"]
            st["work"] = ops.attn_prefill_workspace(c["n_tok"], c["n_head"], c["n_head_kv"], c["head_dim"])
        st["y"] = torch.empty_like(st["q"])
    elif kind == "moe":
        n, e, f = c["n_expert"], c["n_embd"], c["n_ff"]
        gate, up = (ops.QuantMatrix.from_gguf(Q4_K, s[k], n * f, e) for k in ("gate", "up"))
        st["layer"] = ops.MoeLayer(gate, up, ops.QuantMatrix.from_gguf(Q4_K, s["down"], n * e, f), n, c["k"])
        st["x"], st["logits"], st["y"] = s["x"], s["logits"], torch.empty_like(s["x"])
    else:
        st["m"] = ops.QuantMatrix.from_gguf(TYPES[c["fmt"]], s["w"], c["rows"], c["cols"])
        st["x"], st["norm"], st["y"] = s["x"], s["norm"], torch.empty(c["rows"], device="cuda")
    return st


def run(state):
    st, c = state, state["case"]
    kind = c["kind"]
    if kind == "matvec":
        m, lib = st["m"], _lib.load()
        x, y = st["x"].ctypes.data, st["y"].ctypes.data
        if m.scale:
            rc = lib.matmul_q8_0_cuda_resident(m.qs, m.scale, c["rows"], c["cols"], x, y)
        else:
            rc = lib.matmul_kquant_cuda_resident(m.fmt, m.qs, c["rows"], c["cols"], x, y)
        _lib.check(rc, "matvec")
        return st["y"]
    if kind == "ffn_gemv":
        for i, (up, down) in enumerate(zip(st["up"], st["down"])):
            ops.matmul(up, st["x"][i], out=st["y_up"][i])
            ops.matmul(down, st["h"][i], out=st["y_down"][i])
        return st["y_up"], st["y_down"]
    if kind == "layer_decode":
        st["graph"].replay()
        return st["y"], st["layer"].cache.k, st["layer"].cache.v
    if kind == "gemm":
        return ops.gemm(st["m"], st["x"], out=st["y"], work=st["work"])
    if kind == "layer_prefill":
        y = st["layer"].prefill(st["x"], c["pos0"], out=st["y"], work=st["work"], rope=st["rope"])
        return y, st["layer"].cache.k, st["layer"].cache.v
    if kind == "attn_decode":
        return ops.attention_decode(st["q"], st["cache"], c["n_head"], c["pos"], out=st["y"], work=st["work"])
    if kind == "attn_prefill":
        return ops.attention_prefill(st["q"], st["cache"], c["n_head"], c["pos0"], n_swa=c["n_swa"], out=st["y"],
                                     work=st["work"])
    if kind == "moe":
        return st["layer"](st["x"], st["logits"], out=st["y"])
    logits = ops.head_logits(st["m"], st["x"], st["norm"], eps=EPS, out=st["y"])
    ids, vals = ops.topk(logits, c["kk"])
    return logits, ids, vals


# -------------------------------------------------------- cost and accuracy --

def _row_bytes(qtype, cols):
    return cols // BLOCK[qtype][0] * BLOCK[qtype][1]


def _attn_pairs(pos0, n_tok, n_swa):
    """(query token, key) pairs and the number of distinct keys read."""
    if not n_swa:
        return n_tok * (pos0 + 1) + n_tok * (n_tok - 1) // 2, pos0 + n_tok
    pairs = sum(min(n_swa, pos0 + t + 1) for t in range(n_tok))
    return pairs, min(pos0 + n_tok, n_swa + n_tok - 1)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("matvec", "gemm", "head"):
        t, n = TYPES[c["fmt"]], c.get("n_tok", 1)
        b = c["rows"] * _row_bytes(t, c["cols"]) + 4 * n * (c["rows"] + c["cols"])
        return {"bytes": b + (4 * c["cols"] + 8 * c["kk"] if kind == "head" else 0),
                "flops": 2 * n * c["rows"] * c["cols"]}
    if kind == "ffn_gemv":
        t, e, f = TYPES[c["fmt"]], c["n_embd"], c["n_ff"]
        return {"bytes": c["layers"] * (f * _row_bytes(t, e) + e * _row_bytes(t, f) + 8 * (e + f)),
                "flops": c["layers"] * 4 * e * f}
    if kind == "moe":
        e, f, n = c["n_embd"], c["n_ff"], c["n_tok"]
        used = c["n_expert"] * (1 - (1 - c["k"] / c["n_expert"]) ** n)  # experts with a token, on average
        return {"bytes": int(used * (2 * f * _row_bytes(Q4_K, e) + e * _row_bytes(Q4_K, f)) + 8 * n * e),
                "flops": 6 * n * c["k"] * e * f}
    hd, nh, nkv = c["head_dim"], c["n_head"], c["n_head_kv"]
    pos_bytes = 2 * nkv * hd // 32 * 34
    pos0, n = c.get("pos0", c.get("pos")), c.get("n_tok", 1)
    pairs, keys = _attn_pairs(pos0, n, c.get("n_swa", 0))
    if kind in ("attn_decode", "attn_prefill"):
        return {"bytes": keys * pos_bytes + 8 * n * nh * hd, "flops": 4 * hd * nh * pairs}
    shapes = _layer_shapes(c).values()
    return {"bytes": sum(r * _row_bytes(t, k) for t, r, k in shapes) + (keys + n) * pos_bytes + 8 * n * c["n_embd"],
            "flops": 2 * n * sum(r * k for _, r, k in shapes) + 4 * hd * nh * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind in ("matvec", "ffn_gemv"):
        return {"rel": 2e-6}  # the same integers, 32-bit sums in another order
    if kind == "head":
        return {"rel": 1e-5, "differ": 0.1}  # the norm's scale may move an activation across a rounding tie
    if kind in ("attn_decode", "attn_prefill"):
        return {"rel": 2e-5}  # operands split into two 16-bit parts: 4e-6 to 7e-6 from the 64-bit form
    if kind == "gemm":
        return {"rel": 4e-3}  # 16-bit matrix operands of zero-mean weights: up to 1.2e-3 each
    if kind == "moe":
        return {"rel": 1.5e-2}  # the same operands, then the product re-quantized: rounding ties fall otherwise (7e-3)
    if kind == "layer_decode":
        return {"rel": 2e-3, "differ": 0.02}  # 8-bit activations re-quantized: a rounding tie may fall otherwise
    return {"rel": 2e-2, "differ": 0.15}  # the products' 16-bit operands and four re-quantizations, cache rows among them


# -------------------------------------------------------------- 64-bit form --

def _f64(qtype, data, rows, cols):
    """The matrix of GGUF bytes, in 64 bits: (weights, minimums per 32 or None)."""
    qk, sz = BLOCK[qtype]
    b = data.reshape(-1, sz)

    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if qtype == Q8_0:
        return (half(0) * b[:, 2:].view(torch.int8).double()).reshape(rows, cols), None
    if qtype == Q4_0:
        q = torch.cat((b[:, 2:] & 15, b[:, 2:] >> 4), 1).double() - 8
        return (half(0) * q).reshape(rows, cols), None
    if qtype == Q4_K:
        s = b[:, 4:16]
        sc = torch.cat((s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)), 1).double()
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)), 1).double()
        qs = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat((qs & 15, qs >> 4), 2).reshape(-1, 8, 32).double()
        return ((half(0) * sc)[..., None] * q).reshape(rows, cols), (half(2) * mn).reshape(rows, cols // 32)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
    q = torch.stack(((ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)), 2)
    sc = b[:, 192:208].view(torch.int8).double()
    return ((half(208) * sc)[..., None] * (q.double() - 32).reshape(-1, 16, 16)).reshape(rows, cols), None


def _quantized(x, per):
    """x [n][cols] (32-bit) as the path quantizes it per 32 or per 256 values, in 64 bits."""
    b = x.float().reshape(len(x), -1, per)
    amax = b.abs().amax(2, keepdim=True)
    d = amax / 127
    inv = torch.where(d > 0, 1 / d if per == 32 else 127 / amax, torch.zeros_like(d))
    return ((b * inv).round().clamp(-127, 127).double() * d.double()).reshape(x.shape)


def _product(qtype, data, rows, x, act):
    """x [n][cols] times the matrix: act "gemv" (the decode products' activations), "gemm" (per 32, minimums against
    the exact block sums) or None (activations as they are)."""
    cols = x.shape[1]
    w, mn = _f64(qtype, data, rows, cols)
    xq = x.double() if act is None else _quantized(x, 256 if act == "gemv" and qtype in (Q4_K, Q6_K) else 32)
    y = xq @ w.t()
    if mn is not None:
        y -= (x.double() if act == "gemm" else xq).reshape(len(x), -1, 32).sum(2) @ mn.t()
    return y


def _heads(cache, n_head_kv, hd):
    """Cache rows as [head][pos][hd] in 64 bits."""
    return _f64(Q8_0, cache, len(cache), n_head_kv * hd)[0].reshape(len(cache), n_head_kv, hd).transpose(0, 1)


def _attention(q, k, v, pos0, n_swa=0):
    """q [head][tok][hd], k / v [kv head][pos][hd]; token t sees positions up to pos0 + t."""
    per = len(q) // len(k)
    key = torch.arange(k.shape[1], device=q.device)
    at = pos0 + torch.arange(q.shape[1], device=q.device)
    seen = key[None] <= at[:, None]
    if n_swa:
        seen &= key[None] > at[:, None] - n_swa
    out = torch.empty_like(q)
    for h in range(len(q)):
        s = (q[h] @ k[h // per].t()) / math.sqrt(q.shape[2])
        out[h] = torch.softmax(s.masked_fill(~seen, -math.inf), 1) @ v[h // per]
    return out


def _norm(x, w):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * w.double()


def _exact_layer(c, s):
    shapes, style, hd = _layer_shapes(c), c["style"], c["head_dim"]
    decode = c["kind"] == "layer_decode"
    pos0, x = c["pos"] if decode else c["pos0"], s["x"].double()
    n = len(x)

    def mul(name, v):
        t, r, _ = shapes[name]
        return _product(t, s["w"][name], r, v, None)

    xn = _norm(x, s["norms"][0])
    q, k, v = (mul(name, xn) for name in "qkv")
    if style == "qwen":
        q, k, v = (a + b.double() for a, b in zip((q, k, v), s["bias"]))
    q, k, v = (a.reshape(n, -1, hd).transpose(0, 1) for a in (q, k, v))
    if style == "qwen":
        q, k = _norm(q, s["qk"][0]), _norm(k, s["qk"][1])
    freq = THETA ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)
    ang = (pos0 + torch.arange(n, device=x.device, dtype=torch.float64))[:, None] * freq
    cos, sin = ang.cos(), ang.sin()

    def rope(a):
        lo, hi = a[..., :hd // 2], a[..., hd // 2:]
        return torch.cat((lo * cos - hi * sin, lo * sin + hi * cos), -1)

    keys = torch.cat((_heads(s["k"], c["n_head_kv"], hd), rope(k)), 1)
    vals = torch.cat((_heads(s["v"], c["n_head_kv"], hd), v), 1)
    a = _attention(rope(q), keys, vals, pos0).transpose(0, 1)
    if style == "gate":
        a = a * torch.sigmoid(mul("ag", xn))[..., None]
    o = mul("o", a.reshape(n, -1))
    x2 = x + (_norm(o, s["norms"][2]) if style == "gemma" else o)
    fn = _norm(x2, s["norms"][1])
    act = (lambda z: torch.nn.functional.gelu(z, approximate="tanh")) if style == "gemma" else torch.nn.functional.silu
    d = mul("down", act(mul("gate", fn)) * mul("up", fn))
    y = x2 + (_norm(d, s["norms"][3]) if style == "gemma" else d)
    return (y.reshape(-1) if decode else y), None, None


def _exact_moe(c, s):
    n, e, f = c["n_expert"], c["n_embd"], c["n_ff"]
    wts, ids = torch.softmax(s["logits"].double(), 1).topk(c["k"], 1)
    wts = wts / wts.sum(1, keepdim=True)
    y = torch.zeros(c["n_tok"], e, dtype=torch.float64, device=s["x"].device)
    for i in range(n):
        tok, slot = (ids == i).nonzero(as_tuple=True)
        if len(tok):
            x = s["x"][tok]
            h = torch.nn.functional.silu(_product(Q4_K, s["gate"][i * f:(i + 1) * f], f, x, "gemv"))
            h = h * _product(Q4_K, s["up"][i * f:(i + 1) * f], f, x, "gemv")
            y[tok] += wts[tok, slot, None] * _product(Q4_K, s["down"][i * e:(i + 1) * e], e, h, "gemv")
    return y


def exact(case, seed):
    """run()'s outputs in 64 bits. Single products take the path's quantized activations (they are part of what it
    computes); whole layers are compared with the layer of real numbers that their 8-bit activations stand for."""
    c, s, kind = case, _inputs(case, seed), case["kind"]
    if kind == "matvec":
        return _product(TYPES[c["fmt"]], s["w"], c["rows"], s["x"][None], "gemv")[0]
    if kind == "ffn_gemv":
        t, e, f = TYPES[c["fmt"]], c["n_embd"], c["n_ff"]
        return (torch.cat([_product(t, w, f, x[None], "gemv") for w, x in zip(s["up"], s["x"])]),
                torch.cat([_product(t, w, e, x[None], "gemv") for w, x in zip(s["down"], s["h"])]))
    if kind == "gemm":
        return _product(TYPES[c["fmt"]], s["w"], c["rows"], s["x"], "gemm")
    if kind in ("layer_decode", "layer_prefill"):
        return _exact_layer(c, s)
    if kind in ("attn_decode", "attn_prefill"):
        hd, n = c["head_dim"], len(s["q"])
        q = s["q"].double().reshape(n, -1, hd).transpose(0, 1)
        pos0 = c["pos"] if kind == "attn_decode" else c["pos0"]
        a = _attention(q, _heads(s["k"], c["n_head_kv"], hd), _heads(s["v"], c["n_head_kv"], hd), pos0,
                       c.get("n_swa", 0)).transpose(0, 1).reshape(n, -1)
        return a.reshape(-1) if kind == "attn_decode" else a
    if kind == "moe":
        return _exact_moe(c, s)
    x = s["x"]
    scale = 1 / (x.square().double().sum() / len(x) + EPS).float().sqrt()
    y = torch.cat([_product(TYPES[c["fmt"]], s["w"][r:r + 16384], min(16384, c["rows"] - r),
                            (x * scale * s["norm"])[None], "gemv")[0] for r in range(0, c["rows"], 16384)])
    return y, None, y.topk(c["kk"])[0]
