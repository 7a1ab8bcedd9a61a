"""The work a user of this framework has it do, as cases that can be timed.

A case is one call sequence through the public entry points of
include/mynah_asr_hip.h at one size:

  linear       one product of a resident weight             mynah_asr_hip_qgemm_dev
  ffn          SiLU feed-forward, two products              mynah_asr_hip_qffn_dev
  attention    relative-position attention core             mynah_asr_hip_relpos_attention_dev
  layer        one FastConformer encoder layer              mynah_asr_hip_encoder_layer_dev
  subsampling  mel features to encoder rows                 mynah_asr_hip_subsampling_dev
  decoder      AED greedy decoding, then the logits of the
               decoded tokens (their confidences)           mynah_asr_hip_aed_decode_dev, _aed_forced_dev
  host_ffn     the feed-forward on the caller's host arrays mynah_asr_hip_qffn

Sizes are the FastConformer-0.6B / Canary-style ones of the benchmark
configurations (d 1024, 8 heads, FFN 4096, conv kernel 9, vocabulary 16384,
60 s = 750 encoder frames) and the smaller width the tests use. Weights are
N(0, 0.02) in the named block format, activations N(0, 1); everything is made
from the seed.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mynah-asr_amd"))
import mynah_hip as M  # noqa: E402

FORMATS = {"F32": M.F32, "INT8": M.INT8, "INT4": M.INT4, "Q8_0": M.Q8_0, "Q4_K": M.Q4_K, "Q6_K": M.Q6_K}
CONV_K = 9

_lib = None
_stream = None


def lib():
    global _lib
    if _lib is None:
        _lib = M.HipLib()
    return _lib


def stream():
    """The one stream all device calls run on: a thread's calls share its workspaces, so they are ordered."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one decoder position's feed-forward: the smallest call, launches and latency
        {"name": "ffn_1row", "kind": "ffn", "fmt": "Q8_0", "rows": 1, "d": 1024, "f": 4096},
        # the vocabulary projection of four beams: one pass over the largest matrix
        {"name": "vocab_head_4rows", "kind": "linear", "fmt": "Q8_0", "rows": 4, "k": 1024, "n": 16384, "int8act": False},
        # a 5 s utterance through one encoder layer
        {"name": "layer_5s", "kind": "layer", "fmt": "Q8_0", "T": 63, "nseq": 1, "d": 1024, "H": 8, "stream": False},
        # a 60 s utterance through one encoder layer (single-file transcription)
        {"name": "layer_60s", "kind": "layer", "fmt": "Q8_0", "T": 750, "nseq": 1, "d": 1024, "H": 8, "stream": False},
        # the batch of the encoder-forward configuration: 16 x 60 s, the largest
        {"name": "layer_16x60s", "kind": "layer", "fmt": "Q8_0", "T": 750, "nseq": 16, "d": 1024, "H": 8, "stream": False},
        # a streaming model's layer ([70, 13] context, causal conv, layer-norm conv norm, biases), odd length
        {"name": "layer_stream_4x20s", "kind": "layer", "fmt": "Q6_K", "T": 251, "nseq": 4, "d": 1024, "H": 8, "stream": True},
        # the feed-forward of the row-stable batch (8 x 750 frames) with K-quant weights
        {"name": "ffn_q4k_6000", "kind": "ffn", "fmt": "Q4_K", "rows": 6000, "d": 1024, "f": 4096},
        # the int8-activation product of the qmat INT8 format over the same batch
        {"name": "linear_int8_6000", "kind": "linear", "fmt": "INT8", "rows": 6000, "k": 1024, "n": 4096, "int8act": True},
        # the attention core of a streaming model's batch, 16 x 60 s
        {"name": "attention_stream_16x60s", "kind": "attention", "T": 750, "nseq": 16, "d": 1024, "H": 8, "left": 70, "right": 13},
        # the convolutional front end, 4 x 60 s of 80 mel features
        {"name": "subsampling_4x60s", "kind": "subsampling", "frames": 6000, "nseq": 4, "mels": 80, "C": 256, "d": 1024, "causal": False},
        # 24 tokens decoded and scored over one 60 s utterance
        {"name": "decoder_24", "kind": "decoder", "fmt": "Q8_0", "T": 750, "tokens": 24, "layers": 4, "d": 1024, "H": 8,
         "f": 4096, "vocab": 16384},
        # the drop-in call of a C caller that keeps its activations in host memory, 20 s
        {"name": "host_ffn_250", "kind": "host_ffn", "fmt": "Q8_0", "rows": 250, "d": 1024, "f": 4096},
    ]


def _between(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "ffn", "ffn", "layer", "layer", "layer", "attention", "subsampling", "decoder",
                       "host_ffn"])
    if kind == "linear":
        int8act = rng.random() < 0.25
        fmt = rng.choice(["INT8", "INT4", "Q8_0"] if int8act else ["F32", "INT8", "Q8_0", "Q8_0", "Q4_K", "Q4_K", "Q6_K"])
        k, n = rng.choice([(1024, 1024), (1024, 4096), (4096, 1024), (1024, 2048), (1024, 16384), (512, 2048), (640, 1024)])
        if k == 640 and fmt not in ("F32", "INT8", "INT4", "Q8_0"):
            k = 512   # (super-blocks of 256)
        return {"kind": kind, "fmt": fmt, "rows": _between(rng, 1, 1500 if n == 16384 else 6000), "k": k, "n": n,
                "int8act": int8act}
    if kind == "ffn":
        d = rng.choice([1024, 1024, 512])
        return {"kind": kind, "fmt": rng.choice(["Q8_0", "Q8_0", "Q4_K", "Q6_K", "INT8"]), "rows": _between(rng, 1, 6000),
                "d": d, "f": 4 * d}
    if kind == "layer":
        d, H = rng.choice([(1024, 8), (1024, 8), (512, 8), (512, 4)])
        T = _between(rng, 14, 1500)
        return {"kind": kind, "fmt": rng.choice(["Q8_0", "Q8_0", "Q4_K", "Q6_K"]), "T": T,
                "nseq": _between(rng, 1, max(1, min(16, 6000 // T))), "d": d, "H": H, "stream": rng.random() < 0.3}
    if kind == "attention":
        stream = rng.random() < 0.5
        T = _between(rng, 30, 3000 if stream else 1500)
        left, right = rng.choice([(70, 13), (70, 6), (140, 27)]) if stream else (-1, 0)
        d, H = rng.choice([(1024, 8), (512, 8)])
        return {"kind": kind, "T": T, "nseq": _between(rng, 1, max(1, min(16, 6000 // T))), "d": d, "H": H, "left": left,
                "right": right}
    if kind == "subsampling":
        frames = _between(rng, 200, 6000)
        return {"kind": kind, "frames": frames, "nseq": _between(rng, 1, max(1, min(4, 12000 // frames))),
                "mels": rng.choice([80, 128]), "C": 256, "d": rng.choice([1024, 512]), "causal": rng.random() < 0.3}
    if kind == "decoder":
        return {"kind": kind, "fmt": rng.choice(["Q8_0", "Q8_0", "Q4_K"]), "T": _between(rng, 40, 750),
                "tokens": _between(rng, 4, 23), "layers": rng.choice([2, 4]), "d": 1024, "H": 8, "f": 4096,
                "vocab": rng.choice([16384, 5248])}
    return {"kind": kind, "fmt": rng.choice(["Q8_0", "Q4_K", "INT8"]), "rows": _between(rng, 1, 750), "d": 1024, "f": 4096}


# ------------------------------------------------------- weights in their formats
# Each maker returns the host bytes (and scales) the framework takes and the
# values they stand for, in 64 bits.
def _f16(x):
    return x.to(torch.float16)


def _nonzero(x):
    return torch.where(x == 0, torch.ones_like(x), x)


def _bytes(*parts):
    return torch.cat([p.contiguous().view(torch.uint8).reshape(*p.shape[:2], -1) for p in parts], dim=2)


def _make_q8_0(w):
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    d = _f16(b.abs().amax(2, keepdim=True) / 127.0)
    q = torch.round(b / _nonzero(d.float())).clamp(-127, 127).to(torch.int8)
    return _bytes(d, q), None, (d.double() * q.double()).view(n, k)


def _make_q4_k(w):
    n, k = w.shape
    b = w.view(n, k // 256, 8, 32)
    mn = (-b.amin(3)).clamp_min(0.0)
    sc = (b.amax(3) + mn) / 15.0
    d, dm = _f16(sc.amax(2, keepdim=True) / 63.0), _f16(mn.amax(2, keepdim=True) / 63.0)
    ls = torch.round(sc / _nonzero(d.float())).clamp(0, 63).to(torch.int32)
    lm = torch.round(mn / _nonzero(dm.float())).clamp(0, 63).to(torch.int32)
    step = (d.float() * ls)[..., None]
    low = (dm.float() * lm)[..., None]
    q = torch.round((b + low) / _nonzero(step)).clamp(0, 15).to(torch.int32)
    a, c = ls[..., :4] | ((ls[..., 4:] >> 4) << 6), lm[..., :4] | ((lm[..., 4:] >> 4) << 6)
    e = (ls[..., 4:] & 15) | ((lm[..., 4:] & 15) << 4)
    scales = torch.cat([a, c, e], 2).to(torch.uint8)
    qs = (q[:, :, 0::2] | (q[:, :, 1::2] << 4)).to(torch.uint8).reshape(n, k // 256, 128)
    val = d.double()[..., None] * ls.double()[..., None] * q.double() - dm.double()[..., None] * lm.double()[..., None]
    return _bytes(d, dm, scales, qs), None, val.reshape(n, k)


def _make_q6_k(w):
    n, k = w.shape
    b = w.view(n, k // 256, 16, 16)
    sc = b.abs().amax(3) / 31.0
    d = _f16(sc.amax(2, keepdim=True) / 127.0)
    s = torch.round(sc / _nonzero(d.float())).clamp(0, 127).to(torch.int32)
    q = torch.round(b / _nonzero(d.float() * s)[..., None]).clamp(-32, 31).to(torch.int32)
    val = (d.double() * s.double())[..., None] * q.double()
    u = (q + 32).reshape(n, k // 256, 2, 4, 32)   # [half of 128][quarter][32]
    ql = torch.stack([(u[..., 0, :] & 15) | ((u[..., 2, :] & 15) << 4), (u[..., 1, :] & 15) | ((u[..., 3, :] & 15) << 4)], 3)
    qh = (u[..., 0, :] >> 4) | ((u[..., 1, :] >> 4) << 2) | ((u[..., 2, :] >> 4) << 4) | ((u[..., 3, :] >> 4) << 6)
    return _bytes(ql.to(torch.uint8).reshape(n, k // 256, 128), qh.to(torch.uint8).reshape(n, k // 256, 64),
                  s.to(torch.int8), d), None, val.reshape(n, k)


def _make_int8(w):
    s = _nonzero(w.abs().amax(1, keepdim=True)) / 127.0
    q = torch.round(w / s).clamp(-127, 127).to(torch.int8)
    return q, s.view(-1), s.double() * q.double()


def _make_int4(w):
    n, k = w.shape
    b = w.view(n, k // 32, 32)
    s = _nonzero(b.abs().amax(2, keepdim=True)) / 7.0
    q = torch.round(b / s).clamp(-7, 7).to(torch.int32)
    u = (q + 8).view(n, k)
    return (u[:, 0::2] | (u[:, 1::2] << 4)).to(torch.uint8), s.view(n, k // 32), (s.double() * q.double()).view(n, k)


def _make_f32(w):
    return w, None, w.double()


_MAKE = {"F32": _make_f32, "INT8": _make_int8, "INT4": _make_int4, "Q8_0": _make_q8_0, "Q4_K": _make_q4_k,
         "Q6_K": _make_q6_k}


class Draws:
    """A seeded stream of normal arrays; the same sequence for prepare and exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))

    def normal(self, *shape, sigma=1.0, mean=0.0):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, 1.0, generator=self.g)
        return t.mul_(sigma).add_(mean)

    def weight(self, fmt, n, k, sigma=0.02):
        """(fmt, host data, host scales, the values in 64 bits)"""
        data, scales, val = _MAKE[fmt](self.normal(n, k, sigma=sigma))
        return fmt, data, scales, val


def host_weight(w):
    fmt, data, scales, val = w
    return M.Weight(FORMATS[fmt], val.shape[0], val.shape[1], data.cpu().numpy(),
                    None if scales is None else scales.cpu().numpy())


def device_weight(w):
    return M.DeviceWeight(lib(), host_weight(w))


# --------------------------------------------------------------------- products
def _weights(case, r):
    if case["kind"] == "linear":
        return [r.weight(case["fmt"], case["n"], case["k"])]
    return [r.weight(case["fmt"], case["f"], case["d"]), r.weight(case["fmt"], case["d"], case["f"])]


class Linear:
    def __init__(self, case, seed):
        r = Draws(seed)
        self.w = device_weight(_weights(case, r)[0])
        self.rows, self.mode = case["rows"], M.INT8ACT if case["int8act"] else M.EXACT
        self.x = r.normal(case["rows"], case["k"])
        self.y = torch.empty(case["rows"], case["n"], device="cuda")
        self.stream = stream().cuda_stream

    def run(self):
        if self.mode != M.EXACT:
            lib().set_numerics(self.mode)
        self.w.gemm(self.x.data_ptr(), self.y.data_ptr(), self.rows, 0, self.stream)
        if self.mode != M.EXACT:
            lib().set_numerics(M.EXACT)
        return self.y


class Ffn:
    def __init__(self, case, seed):
        r = Draws(seed)
        self.w1, self.w2 = (device_weight(w) for w in _weights(case, r))
        self.rows = case["rows"]
        self.x = r.normal(case["rows"], case["d"])
        self.y = torch.empty(case["rows"], case["d"], device="cuda")
        self.stream = stream().cuda_stream

    def run(self):
        M.ffn_dev(lib(), self.w1, self.w2, self.x.data_ptr(), self.y.data_ptr(), self.rows, self.stream)
        return self.y


class HostFfn:
    def __init__(self, case, seed):
        r = Draws(seed)
        self.w1, self.w2 = (host_weight(w) for w in _weights(case, r))
        self.rows = case["rows"]
        self.x = r.normal(case["rows"], case["d"]).cpu().numpy()
        self.y = np.empty((case["rows"], case["d"]), np.float32)

    def run(self):
        rc = lib().L.mynah_asr_hip_qffn(ctypes.byref(self.w1.desc), ctypes.byref(self.w2.desc), self.x.ctypes.data,
                                        self.y.ctypes.data, self.rows)
        if rc != 0:
            raise RuntimeError(lib().last_error())
        return self.y

    def __del__(self):   # the resident copies are keyed by the host arrays' addresses
        for w in (getattr(self, "w1", None), getattr(self, "w2", None)):
            if w is not None:
                M.evict(lib(), w)


def _silu64(x):
    return x * torch.sigmoid(x)


def _quantized64(x):
    """The reference's per-row int8 activations (src/qmat.c:186-202), as the values they stand for."""
    x = x.cpu().numpy()
    amax = np.abs(x).max(1, keepdims=True)
    inv = np.divide(np.float32(127.0), amax, out=np.zeros_like(amax), where=amax > 0)
    t = x * inv
    q = np.clip(np.trunc(np.where(t >= 0, t + np.float32(0.5), t - np.float32(0.5))), -127, 127)
    return torch.from_numpy(q.astype(np.float64) * (amax / np.float32(127.0)).astype(np.float64)).cuda()


def _exact_linear(case, seed):
    r = Draws(seed)
    w = _weights(case, r)[0][3]
    x = r.normal(case["rows"], case["k"])
    return (_quantized64(x) if case["int8act"] else x.double()) @ w.T


def _exact_ffn(case, seed):
    r = Draws(seed)
    w1, w2 = (w[3] for w in _weights(case, r))
    y = _silu64(r.normal(case["rows"], case["d"]).double() @ w1.T) @ w2.T
    return y.cpu().numpy() if case["kind"] == "host_ffn" else y


# -------------------------------------------------------------------- attention
def _attention_inputs(case, r):
    T, n, d = case["T"], case["nseq"], case["d"]
    return [r.normal(n, T, d) for _ in range(3)] + [r.normal(2 * T - 1, d), r.normal(d, sigma=0.1), r.normal(d, sigma=0.1)]


class Attention:
    def __init__(self, case, seed):
        self.case = case
        self.inputs = _attention_inputs(case, Draws(seed))
        self.ctx = torch.empty(case["nseq"], case["T"], case["d"], device="cuda")
        self.stream = stream().cuda_stream

    def run(self):
        c = self.case
        M.relpos_attention_dev(lib(), *[t.data_ptr() for t in self.inputs], self.ctx.data_ptr(), c["T"], c["d"], c["H"],
                               c["left"], c["right"], c["nseq"], self.stream)
        return self.ctx


def _visible(T, left, right):
    """[T] first and one-past-last key of each row's window (src/encoder.c:373-381)."""
    t = torch.arange(T)
    if left < 0:
        return torch.zeros(T, dtype=torch.long), torch.full((T,), T)
    chunk = right + 1
    return ((t // chunk - left // chunk) * chunk).clamp_min(0), ((t // chunk + 1) * chunk).clamp_max(T)


def _attend64(q, k, v, rk, bu, bv, H, left, right):
    """src/encoder.c:315-410 / 220-313 on [nseq, T, d] in 64 bits."""
    q, k, v, rk, bu, bv = (t.double() for t in (q, k, v, rk, bu, bv))
    n, T, d = q.shape
    dk = d // H
    j0, j1 = (a.cuda()[:, None] for a in _visible(T, left, right))
    j = torch.arange(T, device="cuda")[None]
    shift = T - 1 + j - j.T
    mask = (j >= j0) & (j < j1)
    out = torch.empty_like(q)
    for s in range(n):
        for h in range(H):
            c = slice(h * dk, (h + 1) * dk)
            score = (q[s, :, c] + bu[c]) @ k[s, :, c].T.contiguous()
            score += ((q[s, :, c] + bv[c]) @ rk[:, c].T.contiguous()).gather(1, shift)
            p = torch.softmax((score / math.sqrt(dk)).masked_fill(~mask, -math.inf), 1)
            out[s, :, c] = p @ v[s, :, c]
    return out


def _exact_attention(case, seed):
    return _attend64(*_attention_inputs(case, Draws(seed)), case["H"], case["left"], case["right"])


# ---------------------------------------------------------------- encoder layer
LINEARS = ("ff1_w1", "ff1_w2", "q_w", "k_w", "v_w", "o_w", "relk_w", "pw1_w", "pw2_w", "ff2_w1", "ff2_w2")


def _layer_params(case, r):
    """The layer's tensors: linears as `Draws.weight` gives them, the rest f32 arrays. A streaming model has linear
    biases and a layer norm in its conv module, the others neither."""
    d, fmt = case["d"], case["fmt"]
    f = 4 * d
    p = {}
    for n in ("ff1", "att", "conv", "ff2", "out"):
        p[f"ln_{n}_w"], p[f"ln_{n}_b"] = r.normal(d, sigma=0.1, mean=1.0), r.normal(d, sigma=0.1)
    shapes = {"ff1_w1": (f, d), "ff1_w2": (d, f), "ff2_w1": (f, d), "ff2_w2": (d, f), "pw1_w": (2 * d, d)}
    for n in LINEARS:
        p[n] = r.weight("F32" if n == "relk_w" else fmt, *shapes.get(n, (d, d)))
    p["bias_u"], p["bias_v"] = r.normal(d, sigma=0.1), r.normal(d, sigma=0.1)
    p["dw_w"] = r.normal(d, CONV_K, sigma=0.3)
    if case["stream"]:
        for n, m in (("ff1_b1", f), ("ff1_b2", d), ("ff2_b1", f), ("ff2_b2", d), ("q_b", d), ("k_b", d), ("v_b", d),
                     ("o_b", d), ("pw1_b", 2 * d), ("dw_b", d), ("pw2_b", d)):
            p[n] = r.normal(m, sigma=0.1)
        p["cnorm_w"], p["cnorm_b"] = r.normal(d, sigma=0.1, mean=1.0), r.normal(d, sigma=0.1)
    else:
        p["cnorm_scale"], p["cnorm_shift"] = r.normal(d, sigma=0.1, mean=1.0), r.normal(d, sigma=0.1)
    return p


def _context(case):
    return (70, 13) if case["stream"] else (-1, 0)


def _positions(T, d):
    """The relative positional embedding (src/encoder.c:201-212), f32."""
    pos = (T - 1 - np.arange(2 * T - 1, dtype=np.float64))[:, None]
    a = pos * np.power(10000.0, -2.0 * np.arange(d // 2, dtype=np.float64)[None] / d)
    pe = np.empty((2 * T - 1, d), np.float32)
    pe[:, 0::2], pe[:, 1::2] = np.sin(a), np.cos(a)
    return torch.from_numpy(pe).cuda()


class Layer:
    def __init__(self, case, seed):
        r = Draws(seed)
        self.case, self.keep, self.c = case, [], M.EncLayerC()
        for n, t in _layer_params(case, r).items():
            if n in LINEARS:
                t = device_weight(t)
            self.keep.append(t)
            setattr(self.c, n, t.h if n in LINEARS else t.data_ptr())
        self.pe = _positions(case["T"], case["d"])
        self.x0 = r.normal(case["nseq"] * case["T"], case["d"])
        self.x = torch.empty_like(self.x0)
        self.stream = stream()

    def run(self):
        c, (left, right) = self.case, _context(self.case)
        with torch.cuda.stream(self.stream):   # the layer works in place: its input is laid out first
            self.x.copy_(self.x0)
        rc = lib().L.mynah_asr_hip_encoder_layer_dev(
            ctypes.byref(self.c), self.x.data_ptr(), c["T"], c["nseq"], self.pe.data_ptr(), c["d"], c["H"], CONV_K,
            int(c["stream"]), left, right, self.stream.cuda_stream)
        if rc != 0:
            raise RuntimeError(lib().last_error())
        return self.x


def _layer_norm64(x, w, b):
    m = x.mean(1, keepdim=True)
    v = ((x - m) ** 2).mean(1, keepdim=True)
    return (x - m) / torch.sqrt(v + 1e-5) * w + b


def _exact_layer(case, seed):
    r = Draws(seed)
    p = {n: t[3] if n in LINEARS else t.double() for n, t in _layer_params(case, r).items()}
    T, n, d = case["T"], case["nseq"], case["d"]
    pe, x = _positions(T, d).double(), r.normal(n * T, d).double()

    def lin(a, name, bias=None):
        y = a @ p[name].T
        return y + p[bias] if bias in p else y

    def ffn(a, k):
        h = _layer_norm64(a, p[f"ln_{k}_w"], p[f"ln_{k}_b"])
        return lin(_silu64(lin(h, f"{k}_w1", f"{k}_b1")), f"{k}_w2", f"{k}_b2")

    x = x + 0.5 * ffn(x, "ff1")
    h = _layer_norm64(x, p["ln_att_w"], p["ln_att_b"])
    q, k, v = (lin(h, f"{c}_w", f"{c}_b").view(n, T, d) for c in "qkv")
    ctx = _attend64(q, k, v, pe @ p["relk_w"].T, p["bias_u"], p["bias_v"], case["H"], *_context(case)).view(n * T, d)
    x = x + lin(ctx, "o_w", "o_b")
    h = lin(_layer_norm64(x, p["ln_conv_w"], p["ln_conv_b"]), "pw1_w", "pw1_b")
    g = (h[:, :d] * torch.sigmoid(h[:, d:])).view(n, T, d)
    pc = CONV_K - 1 if case["stream"] else (CONV_K - 1) // 2
    pad = torch.zeros(n, T + CONV_K - 1, d, dtype=torch.float64, device="cuda")
    pad[:, pc:pc + T] = g
    c = sum(pad[:, j:j + T] * p["dw_w"][:, j] for j in range(CONV_K)) + (p["dw_b"] if "dw_b" in p else 0.0)
    c = c.reshape(n * T, d)
    c = _layer_norm64(c, p["cnorm_w"], p["cnorm_b"]) if case["stream"] else c * p["cnorm_scale"] + p["cnorm_shift"]
    x = x + lin(_silu64(c), "pw2_w", "pw2_b")
    x = x + 0.5 * ffn(x, "ff2")
    return _layer_norm64(x, p["ln_out_w"], p["ln_out_b"])


# ------------------------------------------------------------------ subsampling
def _out_len(n, causal):
    return (n + (3 if causal else 2) - 3) // 2 + 1


def _sub_sizes(case):
    t, f = [case["frames"]], [case["mels"]]
    for _ in range(3):
        t.append(_out_len(t[-1], case["causal"]))
        f.append(_out_len(f[-1], case["causal"]))
    return t, f


def _sub_params(case, r):
    C, (_, f) = case["C"], _sub_sizes(case)
    p = {"conv_in_w": r.normal(C, 1, 3, 3, sigma=0.3), "conv_in_b": r.normal(C, sigma=0.1)}
    for i in range(2):
        p[f"dw_w{i}"], p[f"dw_b{i}"] = r.normal(C, 1, 3, 3, sigma=0.3), r.normal(C, sigma=0.1)
        p[f"pw_w{i}"], p[f"pw_b{i}"] = r.normal(C, C, sigma=0.05), r.normal(C, sigma=0.1)
    p["lin_w"], p["lin_b"] = r.normal(case["d"], C * f[3], sigma=0.02), r.normal(case["d"], sigma=0.1)
    return p


class Subsampling:
    def __init__(self, case, seed):
        r = Draws(seed)
        self.case = case
        self.ss = M.DeviceSubsampling(lib(), {n: t.cpu().numpy() for n, t in _sub_params(case, r).items()},
                                      int(case["causal"]))
        self.mel = r.normal(case["nseq"] * case["frames"], case["mels"])
        self.out = torch.empty(case["nseq"] * _sub_sizes(case)[0][3], case["d"], device="cuda")
        self.stream = stream().cuda_stream

    def run(self):
        c = self.case
        self.ss.run(self.mel.data_ptr(), c["frames"], c["nseq"], c["mels"], self.out.data_ptr(), 1.0, self.stream)
        return self.out


def _exact_subsampling(case, seed):
    r = Draws(seed)
    p = {n: t.double() for n, t in _sub_params(case, r).items()}
    mel = r.normal(case["nseq"] * case["frames"], case["mels"]).double()
    pl, pr = (2, 1) if case["causal"] else (1, 1)

    def conv(x, w, b):   # 3x3, stride 2, each output channel from its own input channel (or from the only one)
        x = torch.nn.functional.pad(x, (pl, pr, pl, pr))
        to, fo = (x.shape[1] - 3) // 2 + 1, (x.shape[2] - 3) // 2 + 1
        y = b[:, None, None].expand(-1, to, fo).clone()
        for i in range(3):
            for j in range(3):
                y += w[:, 0, i, j][:, None, None] * x[:, i:i + 2 * to - 1:2, j:j + 2 * fo - 1:2]
        return y

    out = []
    for s in range(case["nseq"]):
        a = torch.relu(conv(mel[s * case["frames"]:(s + 1) * case["frames"]][None], p["conv_in_w"], p["conv_in_b"]))
        for i in range(2):
            a = conv(a, p[f"dw_w{i}"], p[f"dw_b{i}"])
            a = torch.relu((p[f"pw_w{i}"] @ a.flatten(1)).view_as(a) + p[f"pw_b{i}"][:, None, None])
        out.append(a.permute(1, 0, 2).flatten(1) @ p["lin_w"].T + p["lin_b"])
    return torch.cat(out)


# ---------------------------------------------------------------------- decoder
PROMPT = 4   # prompt tokens


def _decoder_params(case, r):
    d, f, v, fmt = case["d"], case["f"], case["vocab"], case["fmt"]
    layers = []
    for _ in range(case["layers"]):
        p = {n: r.weight(fmt, d, d) for n in ("sq", "sk", "sv", "so", "cq", "ck", "cv", "co")}
        p["ff1"], p["ff2"] = r.weight(fmt, f, d), r.weight(fmt, d, f)
        for n in list(p):
            p[n + "_b"] = r.normal(p[n][3].shape[0], sigma=0.02)
        for n in ("self", "cross", "ffn"):
            p[f"ln_{n}_w"], p[f"ln_{n}_b"] = r.normal(d, sigma=0.02, mean=1.0), r.normal(d, sigma=0.02)
        layers.append(p)
    top = {"emb": r.normal(v, d), "pos": r.normal(PROMPT + case["tokens"], d, sigma=0.3),
           "embln_w": r.normal(d, sigma=0.02, mean=1.0), "embln_b": r.normal(d, sigma=0.02),
           "fin_w": r.normal(d, sigma=0.02, mean=1.0), "fin_b": r.normal(d, sigma=0.02), "head": r.weight(fmt, v, d),
           "head_b": r.normal(v, sigma=0.02)}
    enc = r.normal(case["T"], d)
    prompt = torch.randint(0, v, (PROMPT,), device="cuda", generator=r.g, dtype=torch.int64)
    return top, layers, enc, prompt


class Decoder:
    def __init__(self, case, seed):
        top, layers, self.enc, prompt = _decoder_params(case, Draws(seed))
        self.T, self.cap, self.keep = case["T"], case["tokens"], []
        self.tokens = np.zeros(PROMPT + self.cap, np.int32)   # the prompt, then what is decoded
        self.tokens[:PROMPT] = prompt.cpu().numpy()
        self.layers = (M.AedLayerC * len(layers))()
        for c, p in zip(self.layers, layers):
            for n, t in p.items():
                setattr(c, n, self._dev(t))
        self.c = M.AedC(case["layers"], case["d"], case["H"], case["f"], case["vocab"], PROMPT + self.cap)
        for n, t in top.items():
            setattr(self.c, n, self._dev(t))
        self.c.layers = self.layers
        self.logits = torch.empty(PROMPT + self.cap - 1, case["vocab"], device="cuda")
        self.stream = stream().cuda_stream

    def _dev(self, t):
        t = device_weight(t) if isinstance(t, tuple) else t
        self.keep.append(t)
        return t.h if isinstance(t, M.DeviceWeight) else t.data_ptr()

    def run(self):
        L, c, t = lib().L, ctypes.byref(self.c), self.tokens
        n = L.mynah_asr_hip_aed_decode_dev(c, self.enc.data_ptr(), self.T, t.ctypes.data, PROMPT, -1,
                                           t[PROMPT:].ctypes.data, self.cap, self.stream)
        if n != self.cap or L.mynah_asr_hip_aed_forced_dev(c, self.enc.data_ptr(), self.T, t.ctypes.data,
                                                           PROMPT + n - 1, self.logits.data_ptr(), self.stream) != 0:
            raise RuntimeError(lib().last_error())
        return t[PROMPT:], self.logits


def _exact_decoder(case, seed):
    """src/decoder_aed.c:139-232 in 64 bits: the prompt's positions and each token's, over all tokens so far."""
    top, layers, enc, tokens = _decoder_params(case, Draws(seed))
    val = lambda t: t[3] if isinstance(t, tuple) else t.double()  # noqa: E731
    top, layers, enc = {n: val(t) for n, t in top.items()}, [{n: val(t) for n, t in p.items()} for p in layers], enc.double()
    H, dk = case["H"], case["d"] // case["H"]
    lin = lambda a, p, n: a @ p[n].T + p[n + "_b"]  # noqa: E731
    cross = [(lin(enc, p, "ck"), lin(enc, p, "cv")) for p in layers]

    def attend(q, k, v, mask):
        out = torch.empty_like(q)
        for h in range(H):
            c = slice(h * dk, (h + 1) * dk)
            s = q[:, c] @ k[:, c].T.contiguous() / math.sqrt(dk)
            out[:, c] = torch.softmax(s.masked_fill(mask, -math.inf) if mask is not None else s, 1) @ v[:, c]
        return out

    def logits(tokens):
        i = torch.arange(len(tokens), device="cuda")
        x = _layer_norm64(top["emb"][tokens] + top["pos"][i], top["embln_w"], top["embln_b"])
        for p, kv in zip(layers, cross):
            h = _layer_norm64(x, p["ln_self_w"], p["ln_self_b"])
            x = x + lin(attend(lin(h, p, "sq"), lin(h, p, "sk"), lin(h, p, "sv"), i[None] > i[:, None]), p, "so")
            h = _layer_norm64(x, p["ln_cross_w"], p["ln_cross_b"])
            x = x + lin(attend(lin(h, p, "cq"), *kv, None), p, "co")
            x = x + lin(torch.relu(lin(_layer_norm64(x, p["ln_ffn_w"], p["ln_ffn_b"]), p, "ff1")), p, "ff2")
        return _layer_norm64(x, top["fin_w"], top["fin_b"]) @ top["head"].T + top["head_b"]

    for _ in range(case["tokens"]):
        out = logits(tokens)
        tokens = torch.cat([tokens, out[-1:].argmax(1)])
    return tokens[PROMPT:].to(torch.int32), out


# ------------------------------------------------------------------- the contract
_STATE = {"linear": Linear, "ffn": Ffn, "attention": Attention, "layer": Layer, "subsampling": Subsampling,
          "decoder": Decoder, "host_ffn": HostFfn}
_EXACT = {"linear": _exact_linear, "ffn": _exact_ffn, "attention": _exact_attention, "layer": _exact_layer,
          "subsampling": _exact_subsampling, "decoder": _exact_decoder, "host_ffn": _exact_ffn}


def prepare(case, seed):
    state = _STATE[case["kind"]](case, seed)
    torch.cuda.synchronize()   # the inputs are ready before a call on another stream reads them
    return state


def run(state):
    return state.run()


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _pairs(T, left, right):
    j0, j1 = _visible(T, left, right)
    return int((j1 - j0).sum())


def work(case):
    kind, wb = case["kind"], lambda n, k: M.weight_bytes(FORMATS[case["fmt"]], n, k)
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": 4 * m * (n + k) + wb(n, k), "flops": 2 * m * n * k}
    if kind in ("ffn", "host_ffn"):
        m, d, f = case["rows"], case["d"], case["f"]
        return {"bytes": 8 * m * d + 2 * wb(f, d), "flops": 4 * m * d * f}
    if kind == "attention":
        T, n, d = case["T"], case["nseq"], case["d"]
        return {"bytes": 16 * n * T * d + 4 * (2 * T - 1) * d,
                "flops": 6 * d * n * _pairs(T, case["left"], case["right"])}
    if kind == "layer":
        T, n, d = case["T"], case["nseq"], case["d"]
        f, m = 4 * d, n * T
        return {"bytes": 8 * m * d + 4 * (2 * T - 1) * d + 4 * d * d + 4 * wb(f, d) + 7 * wb(d, d),
                "flops": 2 * m * d * (4 * f + 7 * d + CONV_K) + 2 * (2 * T - 1) * d * d +
                6 * d * n * _pairs(T, *_context(case))}
    if kind == "subsampling":
        t, f = _sub_sizes(case)
        n, C, d = case["nseq"], case["C"], case["d"]
        return {"bytes": 4 * n * (t[0] * f[0] + t[3] * d) + 4 * (C * f[3] * d + 2 * C * C),
                "flops": 2 * n * C * (9 * (t[1] * f[1] + t[2] * f[2] + t[3] * f[3]) + C * (t[2] * f[2] + t[3] * f[3]) +
                                      t[3] * f[3] * d)}
    d, f, v, T, s = case["d"], case["f"], case["vocab"], case["T"], case["tokens"]
    n, per = PROMPT + s - 1, case["layers"] * (6 * wb(d, d) + 2 * wb(f, d))
    # decoding reads the linears and the cross keys and values once a position, scoring once in all
    return {"bytes": n * (per + wb(v, d) + case["layers"] * 8 * T * d) + per + wb(v, d) + 4 * n * v +
            2 * case["layers"] * (2 * wb(d, d) + 8 * T * d) + 8 * T * d,
            "flops": 2 * (2 * n * (case["layers"] * (6 * d * d + 2 * d * f + 2 * d * T + d * n) + v * d) +
                          case["layers"] * 4 * T * d * d)}


def tolerance(case):
    """About four times the distance from 64 bits that each path measures (the products 1e-7 to 3e-7, the K-quant
    feed-forward 8e-7, the attention core 4e-7, a layer, which ends in a layer norm, 1e-7, the rest 2e-7): f32 sums of
    products whose operands carry 22 bits."""
    rel = {"linear": 1e-6, "ffn": 3e-6, "host_ffn": 3e-6, "attention": 2e-6, "layer": 6e-7}.get(case["kind"], 1e-6)
    return {"rel": rel, "max": 12 * rel}
