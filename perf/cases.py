"""Workloads of the backend that its speed is measured on.

Each case is one pass of work that a program on this backend does, at the
sizes of the model configurations in `bobcat_amd.lfm2` and
`bobcat_amd.qwen35`: the matrix-vector launches of a decode step, attention
against a long cache, the mixture of experts and the DeltaNet block, the
GEMM blocks of a prefill batch, sampling, and the model drivers as a whole.
`listed()` names the fixed cases, `draw()` gives others of the same ranges.
`exact()` restates a case in float64 with plain torch.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from bobcat_amd import lfm2, qwen35
from bobcat_amd._lib import DeltaShape, Sampling, check, lib
from bobcat_amd.backend import (Format, Hip, NormSpec, Store, attention_decode_scratch_floats, row_bytes)
from bobcat_amd.synth import pack_q4k_scales

EPS = 1e-5
THETA = 1e6
F64 = torch.float64
FORMATS = {"q4k": Format.Q4K, "q6k": Format.Q6K, "q8_0": Format.Q8_0, "f16": Format.F16}
EMBED_ROWS = 512  # rows of the token embedding that feeds a block


# --- device memory --------------------------------------------------------

_HIP: Hip | None = None


def _hip() -> Hip:
    """The process's one device context, as a program opens it."""
    global _HIP
    if _HIP is None:
        torch.cuda.init()
        _HIP = Hip()
    return _HIP


class _Memory:
    """A device buffer's memory for torch (the array interface), which keeps the buffer."""

    def __init__(self, view, shape: tuple, typestr: str):
        self.buffer = view.buffer
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, strides=None, version=3,
                                             data=(view.buffer.device_ptr + view.offset, False))


class State:
    """What a program keeps between calls: device buffers and plain values."""

    def __init__(self, case: dict):
        self.case, self.hip = case, _hip()

    def _view(self, buffer):
        # A buffer is freed with its last view, not with the context.
        self.hip._buffers.remove(buffer)
        return buffer.at(0)

    def put(self, array: np.ndarray):
        return self._view(self.hip.buffer_from(array))

    def zeros(self, count: int, width: int = 4):
        return self._view(self.hip.new_buffer(count * width))

    @staticmethod
    def tensor(view, shape: tuple, typestr: str = "<f4") -> torch.Tensor:
        return torch.as_tensor(_Memory(view, shape, typestr), device="cuda")


# --- weights in block formats ---------------------------------------------

def _weights(rng: np.random.Generator, fmt: str, rows: int, cols: int, std: float = 0.02) -> np.ndarray:
    """Zero-centred random weights of about `std`, as the bytes of `fmt`."""
    if fmt == "f16":
        return (std * rng.standard_normal((rows, cols), np.float32)).astype(np.float16).view(np.uint8).reshape(-1)
    if fmt == "q8_0":
        n = rows * cols // 32
        w = rng.integers(0, 256, (n, 34), np.uint8)
        w[:, :2] = rng.uniform(0.5, 1.5, n).astype(np.float32).__mul__(std / 74).astype(np.float16).view(np.uint8).reshape(n, 2)
        return w.reshape(-1)
    n = rows * cols // 256
    if fmt == "q6k":
        w = rng.integers(0, 256, (n, 210), np.uint8)
        w[:, 192:208] = rng.integers(20, 64, (n, 16), np.uint8)
        w[:, 208:] = (rng.uniform(0.5, 1.5, n) * std / (18.5 * 42)).astype(np.float16).view(np.uint8).reshape(n, 2)
        return w.reshape(-1)
    w = rng.integers(0, 256, (n, 144), np.uint8)
    d = rng.uniform(0.5, 1.5, n) * std / (4.6 * 42)
    w[:, :4] = np.stack([d, 7.5 * d], 1).astype(np.float16).view(np.uint8).reshape(n, 4)
    sc = rng.integers(20, 64, (n, 8), np.uint8)
    w[:, 4:16] = pack_q4k_scales(sc, sc)
    return w.reshape(-1)


def _f64(array: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(array)).cuda().to(F64)


def _dense(fmt: str, data: np.ndarray, rows: int, cols: int) -> torch.Tensor:
    """The matrix of a block format's bytes in float64."""
    if fmt == "f16":
        return _f64(data.view(np.float16)).reshape(rows, cols)
    if fmt == "f32":
        return _f64(data.view(np.float32)).reshape(rows, cols)
    if fmt == "q8_0":
        b = data.reshape(-1, 34)
        return (_f64(b[:, :2].copy().view(np.float16)) * _f64(b[:, 2:].view(np.int8))).reshape(rows, cols)
    if fmt == "q6k":
        b = torch.from_numpy(data.reshape(-1, 210)).cuda()
        d = _f64(data.reshape(-1, 210)[:, 208:].copy().view(np.float16))
        ql, qh = b[:, :128].reshape(-1, 2, 64).int(), b[:, 128:192].reshape(-1, 2, 32).int()
        lo, hi = torch.cat([ql & 15, ql >> 4], 2).reshape(-1, 2, 4, 32), torch.stack([qh >> s & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | hi << 4) - 32
        sc = b[:, 192:208].view(torch.int8).to(F64).reshape(-1, 2, 4, 2).repeat_interleave(16, 3)
        return (d.reshape(-1, 1, 1, 1) * sc * q).reshape(rows, cols)
    b = torch.from_numpy(data.reshape(-1, 144)).cuda()
    d = _f64(data.reshape(-1, 144)[:, :4].copy().view(np.float16))
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6) << 4], 1).to(F64)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6) << 4], 1).to(F64)
    q = b[:, 16:].reshape(-1, 4, 1, 32).int()
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).to(F64)
    return (d[:, :1, None] * sc[:, :, None] * q - d[:, 1:, None] * mn[:, :, None]).reshape(rows, cols)


def _rms(x: torch.Tensor, w: torch.Tensor, eps: float = EPS) -> torch.Tensor:
    return w * x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _norm_weight(rng, n: int) -> np.ndarray:
    return (1 + 0.1 * rng.uniform(-1, 1, n)).astype(np.float32)


def _silu(x: torch.Tensor) -> torch.Tensor:
    return x * torch.sigmoid(x)


def _rope(x: torch.Tensor, pos: torch.Tensor, n_rot: int, theta: float) -> torch.Tensor:
    """NeoX rotation of the first n_rot elements of x [..., tokens, head_dim] for positions pos [tokens]."""
    half = n_rot // 2
    f = theta ** (-torch.arange(half, dtype=F64, device=x.device) * 2 / n_rot)
    a = pos.to(F64)[:, None] * f
    x0, x1 = x[..., :half], x[..., half:n_rot]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos(), x[..., n_rot:]], -1)


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, first: int) -> torch.Tensor:
    """Causal attention of queries [tokens, heads, hd] at positions first.. over k, v [keys, kv, hd]."""
    heads, kv = q.shape[1], k.shape[1]
    visible = torch.arange(k.shape[0], device=q.device)[None] <= first + torch.arange(q.shape[0], device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(heads):
        s = q[:, h] @ k[:, h * kv // heads].T.contiguous() / math.sqrt(q.shape[2])
        out[:, h] = torch.softmax(s.masked_fill(~visible, -math.inf), 1) @ v[:, h * kv // heads].contiguous()
    return out


def _short_conv(bcx: torch.Tensor, taps: torch.Tensor, hist: torch.Tensor):
    """The gated short convolution of bcx [tokens, 3n]: (outputs, new history)."""
    b, c, x = bcx.chunk(3, 1)
    k = taps.shape[1]
    bx = torch.cat([hist, b * x])
    return c * sum(taps[:, j] * bx[j:j + b.shape[0]] for j in range(k)), bx[-(k - 1):]


# --- the kinds of work ----------------------------------------------------
#
# Each kind has draw(rng) (the case's values), inputs(case, rng) (host arrays),
# prepare(state, arrays), run(state), exact(case, arrays) and work(case).

def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _blocks(rng, lo: int, hi: int) -> int:
    return 256 * rng.randint(lo, hi)


class Gemv:
    """One projection of one token, with the norm of its input fused in: the shortest call a program makes."""

    @staticmethod
    def draw(rng):
        return dict(fmt=rng.choice(["q4k", "q4k", "q6k", "q8_0", "f16"]), rows=_log_int(rng, 256, 16384),
                    cols=_blocks(rng, 2, 42), norm=rng.random() < 0.5)

    @staticmethod
    def inputs(c, rng):
        return dict(w=_weights(rng, c["fmt"], c["rows"], c["cols"]), x=rng.standard_normal(c["cols"], np.float32),
                    norm=_norm_weight(rng, c["cols"]))

    @staticmethod
    def prepare(s, a):
        s.w, s.x, s.norm = s.put(a["w"]), s.put(a["x"]), NormSpec(s.put(a["norm"]), EPS)
        s.y = s.zeros(s.case["rows"])
        s.out = s.tensor(s.y, (s.case["rows"],))

    @staticmethod
    def run(s):
        c = s.case
        s.hip.begin()
        s.hip.matvec(FORMATS[c["fmt"]], s.w, c["rows"], c["cols"], s.x, s.y, norm=s.norm if c["norm"] else None)
        s.hip.end()
        return s.out

    @staticmethod
    def exact(c, a):
        x = _f64(a["x"])
        return _dense(c["fmt"], a["w"], c["rows"], c["cols"]) @ (_rms(x, _f64(a["norm"])) if c["norm"] else x)

    @staticmethod
    def work(c):
        return dict(bytes=c["rows"] * row_bytes(FORMATS[c["fmt"]], c["cols"]) + 4 * (c["rows"] + 2 * c["cols"]),
                    flops=2 * c["rows"] * c["cols"])

    tolerance = {"rel": 4e-6}


class DecodeLayers:
    """One token through some convolution layers (projection with the short convolution, output projection, SwiGLU
    block), recorded together as a decode step records its launches."""
    TAPS = 3

    @staticmethod
    def draw(rng):
        return dict(fmt=rng.choice(["q4k", "q4k", "q4k", "q6k", "q8_0"]), n=_blocks(rng, 2, 8), n_ff=_blocks(rng, 6, 42),
                    layers=rng.randint(1, 4))

    @staticmethod
    def shapes(c):
        n, f = c["n"], c["n_ff"]
        return dict(in_proj=(3 * n, n), out_proj=(n, n), gate=(f, n), up=(f, n), down=(n, f))

    @classmethod
    def inputs(cls, c, rng):
        n = c["n"]
        layer = lambda: dict({k: _weights(rng, c["fmt"], *s) for k, s in cls.shapes(c).items()},  # noqa: E731
                             taps=rng.uniform(-0.5, 0.5, (n, cls.TAPS)).astype(np.float32),
                             hist=rng.standard_normal((cls.TAPS - 1, n), np.float32),
                             norm=_norm_weight(rng, n), ffn_norm=_norm_weight(rng, n))
        return dict(embed=_weights(rng, "q4k", EMBED_ROWS, n, 1.0), token=rng.integers(0, EMBED_ROWS, 1).astype(np.uint32),
                    layers=[layer() for _ in range(c["layers"])])

    @staticmethod
    def prepare(s, a):
        c = s.case
        s.layers = [{k: s.put(v) for k, v in layer.items()} for layer in a["layers"]]
        s.embed, s.token = s.put(a["embed"]), s.put(a["token"])
        s.hidden, s.conv, s.ffn = s.zeros(c["n"]), s.zeros(c["n"]), s.zeros(c["n_ff"])
        s.out = [s.tensor(s.hidden, (c["n"],))] + [s.tensor(layer["hist"], (DecodeLayers.TAPS - 1, c["n"]))
                                                   for layer in s.layers]

    @staticmethod
    def run(s):
        c, h, f = s.case, s.hip, FORMATS[s.case["fmt"]]
        n, n_ff = c["n"], c["n_ff"]
        h.begin()
        h.embed(Format.Q4K, s.embed, EMBED_ROWS, s.token, s.hidden, n, 1)
        for w in s.layers:
            h.matvec_conv(f, w["in_proj"], n, s.hidden, NormSpec(w["norm"], EPS), w["taps"], w["hist"], s.conv, n,
                          DecodeLayers.TAPS)
            h.matvec(f, w["out_proj"], n, n, s.conv, s.hidden, accumulate=True)
            h.matvec_swiglu(f, w["gate"], w["up"], n_ff, n, s.hidden, NormSpec(w["ffn_norm"], EPS), s.ffn)
            h.matvec(f, w["down"], n, n_ff, s.ffn, s.hidden, accumulate=True)
        h.end()
        return s.out

    @classmethod
    def exact(cls, c, a):
        x = _dense("q4k", a["embed"], EMBED_ROWS, c["n"])[int(a["token"][0])][None]
        hists = []
        for layer in a["layers"]:
            w = {k: _dense(c["fmt"], layer[k], *s) for k, s in cls.shapes(c).items()}
            y, hist = _short_conv(_rms(x, _f64(layer["norm"])) @ w["in_proj"].T, _f64(layer["taps"]), _f64(layer["hist"]))
            x = x + y @ w["out_proj"].T
            t = _rms(x, _f64(layer["ffn_norm"]))
            x = x + (_silu(t @ w["gate"].T) * (t @ w["up"].T)) @ w["down"].T
            hists.append(hist)
        return [x[0]] + hists

    @classmethod
    def work(cls, c):
        n, f = c["n"], FORMATS[c["fmt"]]
        return dict(bytes=c["layers"] * (sum(r * row_bytes(f, k) for r, k in cls.shapes(c).values()) + 4 * n * (2 + cls.TAPS
                                         + 2 * (cls.TAPS - 1))) + 5 * n,
                    flops=2 * c["layers"] * sum(r * k for r, k in cls.shapes(c).values()))

    tolerance = {"rel": 1e-5}


class AttnDecode:
    """The attention of one new token over the cache of its context."""

    @staticmethod
    def draw(rng):
        kv, hd = rng.choice([2, 4, 8]), rng.choice([64, 64, 128, 256])
        return dict(heads=kv * rng.choice([1, 2, 4]), kv=kv, hd=hd, half=rng.random() < 0.8, pos=_log_int(rng, 1, 32767))

    @staticmethod
    def inputs(c, rng):
        kvd, dt = c["kv"] * c["hd"], np.float16 if c["half"] else np.float32
        cache = lambda: np.concatenate([rng.standard_normal((c["pos"], kvd), np.float32),  # noqa: E731
                                        np.zeros((1, kvd), np.float32)]).astype(dt)
        normal = lambda n: rng.standard_normal(n, np.float32)  # noqa: E731
        return dict(q=2 * normal(c["heads"] * c["hd"]), k=2 * normal(kvd), v=normal(kvd), q_norm=_norm_weight(rng, c["hd"]),
                    k_norm=_norm_weight(rng, c["hd"]), kc=cache(), vc=cache())

    @staticmethod
    def prepare(s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        s.scratch = s.zeros(attention_decode_scratch_floats(c["heads"], c["hd"], c["pos"] + 1, c["half"]))
        s.o = s.zeros(c["heads"] * c["hd"])
        row, t = c["pos"] * c["kv"] * c["hd"] * (2 if c["half"] else 4), "<f2" if c["half"] else "<f4"
        s.out = [s.tensor(s.o, (c["heads"], c["hd"])), s.tensor(s.kc.buffer.at(row), (c["kv"], c["hd"]), t),
                 s.tensor(s.vc.buffer.at(row), (c["kv"], c["hd"]), t)]

    @staticmethod
    def run(s):
        c = s.case
        s.hip.begin()
        s.hip.attention_decode(s.q, s.k, s.v, s.q_norm, s.k_norm, EPS, THETA, c["hd"], s.kc, s.vc, c["half"], s.scratch,
                               s.o, c["heads"], c["kv"], c["hd"], c["pos"], c["pos"] + 1)
        s.hip.end()
        return s.out

    @staticmethod
    def exact(c, a):
        pos = torch.tensor([c["pos"]], device="cuda")
        turn = lambda x, w, n: _rope(_rms(_f64(x).reshape(n, 1, c["hd"]), _f64(w)), pos, c["hd"], THETA)  # noqa: E731
        q, k, v = turn(a["q"], a["q_norm"], c["heads"]), turn(a["k"], a["k_norm"], c["kv"]), _f64(a["v"])
        kc, vc = (_f64(a[n]).reshape(-1, c["kv"], c["hd"]) for n in ("kc", "vc"))
        kc[-1], vc[-1] = k[:, 0], v.reshape(c["kv"], c["hd"])
        if c["half"]:
            kc[-1], vc[-1] = kc[-1].half().to(F64), vc[-1].half().to(F64)
        return [_attend(q.transpose(0, 1), kc, vc, c["pos"])[0], kc[-1], vc[-1]]

    @staticmethod
    def work(c):
        row = c["kv"] * c["hd"]
        return dict(bytes=(2 * c["pos"] + 2) * row * (2 if c["half"] else 4) + 4 * (2 * c["heads"] * c["hd"] + 2 * row),
                    flops=4 * c["heads"] * c["hd"] * (c["pos"] + 1))

    tolerance = {"rel": 1e-3}  # the stored key's rounding to f16; the output itself is far closer


class SampleHead:
    """The end of a sampled decode step: the output projection of the last token and a draw from its logits."""

    @staticmethod
    def draw(rng):
        return dict(fmt=rng.choice(["q4k", "q6k", "f16"]), n=_blocks(rng, 2, 8), vocab=_log_int(rng, 4096, 65536),
                    top_k=rng.choice([0, 20, 40, 64, 200]), top_p=rng.choice([0.8, 0.9, 0.95, 1.0]),
                    min_p=rng.choice([0.0, 0.05]), temperature=rng.choice([0.3, 0.7, 1.0]), penalty=rng.choice([1.0, 1.1]))

    @staticmethod
    def inputs(c, rng):
        return dict(w=_weights(rng, c["fmt"], c["vocab"], c["n"], 0.06), x=3 * rng.standard_normal(c["n"], np.float32),
                    norm=_norm_weight(rng, c["n"]), recent=rng.integers(0, c["vocab"], 64).astype(np.uint32),
                    u=np.float32(rng.uniform(0, 0.999)))

    @staticmethod
    def prepare(s, a):
        c = s.case
        s.w, s.x, s.norm, s.recent = s.put(a["w"]), s.put(a["x"]), NormSpec(s.put(a["norm"]), EPS), s.put(a["recent"])
        s.u, s.settings = float(a["u"]), Sampling(c["temperature"], c["top_k"], c["top_p"], c["min_p"], c["penalty"])
        s.logits, s.token = s.zeros(c["vocab"]), s.zeros(1)
        s.out = [s.tensor(s.logits, (c["vocab"],)), s.tensor(s.token, (1,), "<i4")]

    @staticmethod
    def run(s):
        c = s.case
        s.hip.begin()
        s.hip.matvec(FORMATS[c["fmt"]], s.w, c["vocab"], c["n"], s.x, s.logits, norm=s.norm)
        s.hip.sample_draw(s.logits, c["vocab"], s.recent, 64, s.settings, s.u, s.token)
        s.hip.end()
        return s.out

    @staticmethod
    def exact(c, a):
        y = _dense(c["fmt"], a["w"], c["vocab"], c["n"]) @ _rms(_f64(a["x"]), _f64(a["norm"]))
        r = torch.from_numpy(np.unique(a["recent"]).astype(np.int64)).cuda()
        y[r] = torch.where(y[r] > 0, y[r] / c["penalty"], y[r] * c["penalty"])
        return [y, None]

    @staticmethod
    def work(c):
        return dict(bytes=c["vocab"] * (row_bytes(FORMATS[c["fmt"]], c["n"]) + 4) + 8 * c["n"], flops=2 * c["vocab"] * c["n"])

    tolerance = {"rel": 4e-6}


class Ffn:
    """The SwiGLU block of a prefill batch."""

    @staticmethod
    def draw(rng):
        return dict(fmt=rng.choice(["q4k", "q4k", "q6k", "q8_0"]), n=_blocks(rng, 2, 8), n_ff=_blocks(rng, 6, 42),
                    tokens=_log_int(rng, 2, 512))

    @staticmethod
    def inputs(c, rng):
        n, f = c["n"], c["n_ff"]
        return dict(embed=_weights(rng, "q4k", EMBED_ROWS, n, 1.0),
                    tokens=rng.integers(0, EMBED_ROWS, c["tokens"]).astype(np.uint32), norm=_norm_weight(rng, n),
                    gate=_weights(rng, c["fmt"], f, n), up=_weights(rng, c["fmt"], f, n), down=_weights(rng, c["fmt"], n, f))

    @staticmethod
    def prepare(s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        s.hidden, s.normed, s.ffn = (s.zeros(c["tokens"] * w) for w in (c["n"], c["n"], c["n_ff"]))
        s.out = s.tensor(s.hidden, (c["tokens"], c["n"]))

    @staticmethod
    def run(s):
        c, h, f = s.case, s.hip, FORMATS[s.case["fmt"]]
        n, n_ff, t = c["n"], c["n_ff"], c["tokens"]
        h.begin()
        h.embed(Format.Q4K, s.embed, EMBED_ROWS, s.tokens, s.hidden, n, t)
        h.rms_norm(s.hidden, s.norm, s.normed, n, t, EPS)
        h.matmul(f, s.gate, n_ff, n, s.normed, s.ffn, t, Store.OVERWRITE)
        h.matmul(f, s.up, n_ff, n, s.normed, s.ffn, t, Store.SWIGLU)
        h.matmul(f, s.down, n, n_ff, s.ffn, s.hidden, t, Store.ACCUMULATE)
        h.end()
        return s.out

    @staticmethod
    def exact(c, a):
        n, f = c["n"], c["n_ff"]
        x = _dense("q4k", a["embed"], EMBED_ROWS, n)[torch.from_numpy(a["tokens"].astype(np.int64)).cuda()]
        t = _rms(x, _f64(a["norm"]))
        y = _silu(t @ _dense(c["fmt"], a["gate"], f, n).T) * (t @ _dense(c["fmt"], a["up"], f, n).T)
        return x + y @ _dense(c["fmt"], a["down"], n, f).T

    @staticmethod
    def work(c):
        n, f, t, m = c["n"], c["n_ff"], c["tokens"], FORMATS[c["fmt"]]
        return dict(bytes=2 * f * row_bytes(m, n) + n * row_bytes(m, f) + 8 * t * n, flops=6 * t * n * f)

    tolerance = {"rel": 1.6e-3}


class ConvBlock:
    """The gated short convolution block of a prefill batch."""
    TAPS = 3

    @staticmethod
    def draw(rng):
        return dict(fmt=rng.choice(["q4k", "q4k", "q6k", "q8_0", "f16"]), n=_blocks(rng, 2, 8), tokens=_log_int(rng, 2, 512))

    @classmethod
    def inputs(cls, c, rng):
        n = c["n"]
        return dict(embed=_weights(rng, "q4k", EMBED_ROWS, n, 1.0),
                    tokens=rng.integers(0, EMBED_ROWS, c["tokens"]).astype(np.uint32), norm=_norm_weight(rng, n),
                    in_proj=_weights(rng, c["fmt"], 3 * n, n), out_proj=_weights(rng, c["fmt"], n, n),
                    taps=rng.uniform(-0.5, 0.5, (n, cls.TAPS)).astype(np.float32),
                    hist=rng.standard_normal((cls.TAPS - 1, n), np.float32))

    @staticmethod
    def prepare(s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        s.hidden, s.normed, s.bcx, s.conv = (s.zeros(c["tokens"] * w * c["n"]) for w in (1, 1, 3, 1))
        s.out = [s.tensor(s.hidden, (c["tokens"], c["n"])), s.tensor(s.hist, (ConvBlock.TAPS - 1, c["n"]))]

    @staticmethod
    def run(s):
        c, h, f = s.case, s.hip, FORMATS[s.case["fmt"]]
        n, t = c["n"], c["tokens"]
        h.begin()
        h.embed(Format.Q4K, s.embed, EMBED_ROWS, s.tokens, s.hidden, n, t)
        h.rms_norm(s.hidden, s.norm, s.normed, n, t, EPS)
        h.matmul(f, s.in_proj, 3 * n, n, s.normed, s.bcx, t, Store.OVERWRITE)
        h.short_conv_batch(s.bcx, s.taps, s.hist, s.conv, n, ConvBlock.TAPS, t)
        h.matmul(f, s.out_proj, n, n, s.conv, s.hidden, t, Store.ACCUMULATE)
        h.end()
        return s.out

    @staticmethod
    def exact(c, a):
        n = c["n"]
        x = _dense("q4k", a["embed"], EMBED_ROWS, n)[torch.from_numpy(a["tokens"].astype(np.int64)).cuda()]
        y, hist = _short_conv(_rms(x, _f64(a["norm"])) @ _dense(c["fmt"], a["in_proj"], 3 * n, n).T, _f64(a["taps"]),
                              _f64(a["hist"]))
        return [x + y @ _dense(c["fmt"], a["out_proj"], n, n).T, hist]

    @staticmethod
    def work(c):
        n, t = c["n"], c["tokens"]
        return dict(bytes=4 * n * row_bytes(FORMATS[c["fmt"]], n) + 8 * t * n, flops=8 * t * n * n)

    tolerance = {"rel": 1.6e-3}


class Moe:
    """A mixture-of-experts block: grouped by expert for a batch, expert by expert for one token."""

    @staticmethod
    def draw(rng):
        used = rng.choice([2, 4])
        return dict(n=_blocks(rng, 2, 8), n_ff=_blocks(rng, 1, 7), experts=rng.choice([8, 16, 32]), used=used,
                    tokens=rng.choice([1, _log_int(rng, 2, 512), _log_int(rng, 2, 512)]))

    @staticmethod
    def inputs(c, rng):
        n, f, e = c["n"], c["n_ff"], c["experts"]
        return dict(embed=_weights(rng, "q4k", EMBED_ROWS, n, 1.0),
                    tokens=rng.integers(0, EMBED_ROWS, c["tokens"]).astype(np.uint32), norm=_norm_weight(rng, n),
                    router=(rng.standard_normal((e, n), np.float32) / np.sqrt(n)).astype(np.float32),
                    bias=rng.uniform(-0.05, 0.05, e).astype(np.float32), gate=_weights(rng, "q4k", e * f, n),
                    up=_weights(rng, "q4k", e * f, n), down=_weights(rng, "q4k", e * n, f))

    @staticmethod
    def prepare(s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        t, u = c["tokens"], c["used"]
        s.hidden, s.normed = s.zeros(t * c["n"]), s.zeros(t * c["n"])
        s.route, s.offsets, s.entries = s.zeros(2 * u * t), s.zeros(c["experts"] + 1), s.zeros(u * t)
        s.ffn, s.rows = s.zeros(u * t * c["n_ff"]), s.zeros(u * t * c["n"])
        s.out = s.tensor(s.hidden, (t, c["n"]))

    @staticmethod
    def run(s):
        c, h, q = s.case, s.hip, Format.Q4K
        n, f, e, u, t = c["n"], c["n_ff"], c["experts"], c["used"], c["tokens"]
        h.begin()
        h.embed(q, s.embed, EMBED_ROWS, s.tokens, s.hidden, n, t)
        h.moe_route(s.hidden, NormSpec(s.norm, EPS), s.normed, s.router, s.bias, s.route, n, e, u, t)
        if t == 1:
            h.matvec_experts_swiglu(q, s.gate, s.up, f, n, e, s.normed, s.route, u, s.ffn, 1)
            h.matvec_experts_down(q, s.down, n, f, e, s.ffn, s.route, u, s.hidden, 1)
        else:
            h.moe_group(s.route, s.offsets, s.entries, e, u, t)
            h.matmul_experts(q, s.gate, s.up, f, n, e, s.normed, True, s.offsets, s.entries, u, s.ffn, t)
            h.matmul_experts(q, s.down, None, n, f, e, s.ffn, False, s.offsets, s.entries, u, s.rows, t)
            h.moe_combine(s.rows, s.route, s.hidden, n, u, t)
        h.end()
        return s.out

    @staticmethod
    def exact(c, a):
        n, f, e = c["n"], c["n_ff"], c["experts"]
        x = _dense("q4k", a["embed"], EMBED_ROWS, n)[torch.from_numpy(a["tokens"].astype(np.int64)).cuda()]
        t = _rms(x, _f64(a["norm"]))
        score = torch.sigmoid(t @ _f64(a["router"]).T)
        pick = torch.topk(score + _f64(a["bias"]), c["used"], 1).indices
        weight = score.gather(1, pick)
        weight = torch.zeros_like(score).scatter_(1, pick, weight / (weight.sum(1, keepdim=True) + 1e-6))
        y = x.clone()
        for i in range(e):
            at = weight[:, i].nonzero()[:, 0]
            part = lambda k, r, w: _dense("q4k", a[k].reshape(e, -1)[i], r, w)  # noqa: E731
            if at.numel():
                g = _silu(t[at] @ part("gate", f, n).T) * (t[at] @ part("up", f, n).T)
                y[at] += weight[at, i:i + 1] * (g @ part("down", n, f).T)
        return y

    @staticmethod
    def work(c):
        n, f, t, u = c["n"], c["n_ff"], c["tokens"], c["used"]
        busy = min(c["experts"], u * t)
        return dict(bytes=busy * (2 * f * row_bytes(12, n) + n * row_bytes(12, f)) + 4 * c["experts"] * n + 8 * t * n,
                    flops=6 * t * u * n * f)

    tolerance = {"rel": 8e-4}  # the batch's inputs and weights in f16


class DeltaNet:
    """The Gated DeltaNet mixer of a prefill batch after its projections: convolution, gates, chunked recurrence and
    gated output norm."""
    TAPS = 4

    @staticmethod
    def draw(rng):
        nk = rng.choice([2, 4, 8, 16])
        return dict(nk=nk, nv=nk * rng.choice([1, 2]), dk=rng.choice([64, 128, 128]), dv=rng.choice([64, 128, 128]),
                    tokens=_log_int(rng, 2, 1024))

    @staticmethod
    def dims(c):
        return 2 * c["nk"] * c["dk"] + c["nv"] * c["dv"], c["nv"] * c["dv"]

    @classmethod
    def inputs(cls, c, rng):
        conv, value = cls.dims(c)
        t, nv = c["tokens"], c["nv"]
        normal = lambda *s: rng.standard_normal(s, np.float32)  # noqa: E731
        step = np.exp(rng.uniform(math.log(1e-3), math.log(0.1), nv))
        return dict(x=normal(t, conv), taps=0.4 * normal(conv, cls.TAPS), hist=normal(conv, cls.TAPS - 1), z=normal(t, value),
                    raw_beta=normal(t, nv), raw_alpha=normal(t, nv), a=-rng.uniform(1, 16, nv).astype(np.float32),
                    dt_bias=np.log(np.expm1(step)).astype(np.float32), norm=_norm_weight(rng, c["dv"]),
                    state=0.1 * normal(nv, c["dk"], c["dv"]))

    @classmethod
    def prepare(cls, s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        conv, value = cls.dims(c)
        t = c["tokens"]
        s.shape = DeltaShape(c["nk"], c["nv"], c["dk"], c["dv"])
        s.y, s.beta, s.alpha, s.o = s.zeros(t * conv), s.zeros(t * c["nv"]), s.zeros(t * c["nv"]), s.zeros(t * value)
        s.scratch = s.zeros(lib().bch_gdn_chunk_scratch_floats(C.byref(s.shape), t))
        s.out = [s.tensor(s.o, (t, value)), s.tensor(s.state, (c["nv"], c["dk"], c["dv"])),
                 s.tensor(s.hist, (conv, cls.TAPS - 1))]

    @classmethod
    def run(cls, s):
        c, h, L = s.case, s.hip, lib()
        conv, value = cls.dims(c)
        t, nv = c["tokens"], c["nv"]
        h.begin()
        h.copy(s.raw_beta, s.beta, t * nv)
        h.copy(s.raw_alpha, s.alpha, t * nv)
        check(L.bch_gdn_conv(h.handle, s.x.c(), s.taps.c(), s.hist.c(), s.y.c(), conv, cls.TAPS, t))
        check(L.bch_gdn_gates(h.handle, s.beta.c(), s.alpha.c(), s.a.c(), s.dt_bias.c(), nv, t * nv))
        check(L.bch_gdn_recurrence_chunked(h.handle, s.y.c(), s.beta.c(), s.alpha.c(), s.state.c(), s.o.c(),
                                           C.byref(s.shape), t, 1 / math.sqrt(c["dk"]), s.scratch.c()))
        check(L.bch_gdn_gated_norm(h.handle, s.o.c(), s.norm.c(), s.z.c(), c["dv"], t * nv, 1e-6))
        h.end()
        return s.out

    @classmethod
    def exact(cls, c, a):
        conv, value = cls.dims(c)
        t, nk, nv, dk, dv = c["tokens"], c["nk"], c["nv"], c["dk"], c["dv"]
        x, taps = torch.cat([_f64(a["hist"]).T, _f64(a["x"])]), _f64(a["taps"])
        y = _silu(sum(taps[:, j] * x[j:j + t] for j in range(cls.TAPS)))
        q, k, v = y.split([nk * dk, nk * dk, value], 1)
        unit = lambda m: m / torch.sqrt((m * m).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = (unit(m.reshape(t, nk, dk)).repeat(1, nv // nk, 1) for m in (q, k))
        q, v = q / math.sqrt(dk), v.reshape(t, nv, dv)
        beta = torch.sigmoid(_f64(a["raw_beta"]))
        decay = torch.exp(_f64(a["a"]) * torch.nn.functional.softplus(_f64(a["raw_alpha"]) + _f64(a["dt_bias"])))
        S, out = _f64(a["state"]), torch.empty(t, nv, dv, dtype=F64, device="cuda")
        for i in range(t):
            S = S * decay[i, :, None, None]
            delta = (v[i] - (S * k[i, :, :, None]).sum(1)) * beta[i, :, None]
            S = S + k[i, :, :, None] * delta[:, None]
            out[i] = (S * q[i, :, :, None]).sum(1)
        out = _rms(out, _f64(a["norm"]), 1e-6) * _silu(_f64(a["z"]).reshape(t, nv, dv))
        return [out.reshape(t, value), S, x[-(cls.TAPS - 1):].T.contiguous()]

    @classmethod
    def work(cls, c):
        conv, value = cls.dims(c)
        t, nv, dk, dv = c["tokens"], c["nv"], c["dk"], c["dv"]
        return dict(bytes=4 * (t * (conv + 2 * value + 2 * nv) + 2 * nv * dk * dv + conv * (3 * cls.TAPS - 2)),
                    flops=t * (6 * nv * dk * dv + 2 * conv * cls.TAPS))

    tolerance = {"rel": 4e-6}


class AttnPrefill:
    """The attention of a prefill batch over the cache of its context."""

    @staticmethod
    def draw(rng):
        kv, hd = rng.choice([2, 4, 8]), rng.choice([64, 64, 128, 256])
        first = rng.choice([0, _log_int(rng, 1, 7680)])
        return dict(heads=kv * rng.choice([1, 2, 4]), kv=kv, hd=hd, first=first, tokens=_log_int(rng, 2, 512))

    @staticmethod
    def inputs(c, rng):
        keys, kvd = c["first"] + c["tokens"], c["kv"] * c["hd"]
        return dict(q=2 * rng.standard_normal((c["tokens"], c["heads"] * c["hd"]), np.float32),
                    kc=rng.standard_normal((keys, kvd), np.float32).astype(np.float16),
                    vc=rng.standard_normal((keys, kvd), np.float32).astype(np.float16))

    @staticmethod
    def prepare(s, a):
        c = s.case
        for k, v in a.items():
            setattr(s, k, s.put(v))
        s.o = s.zeros(c["tokens"] * c["heads"] * c["hd"])
        s.out = s.tensor(s.o, (c["tokens"], c["heads"], c["hd"]))

    @staticmethod
    def run(s):
        c = s.case
        s.hip.begin()
        s.hip.attention_prefill(s.q, s.kc, s.vc, s.o, c["heads"], c["kv"], c["hd"], c["first"], c["tokens"],
                                c["first"] + c["tokens"])
        s.hip.end()
        return s.out

    @staticmethod
    def exact(c, a):
        q = _f64(a["q"]).reshape(-1, c["heads"], c["hd"])
        return _attend(q, *(_f64(a[n]).reshape(-1, c["kv"], c["hd"]) for n in ("kc", "vc")), c["first"])

    @staticmethod
    def work(c):
        t, q, first = c["tokens"], c["heads"] * c["hd"], c["first"]
        return dict(bytes=4 * (first + t) * c["kv"] * c["hd"] + 8 * t * q, flops=4 * q * (t * first + t * (t + 1) // 2))

    tolerance = {"rel": 4e-6}


MODELS = {c.name: c for c in (lfm2.LFM2_350M, lfm2.LFM2_2_6B, qwen35.QWEN35_0_8B)}


def _lfm2_logits(w: "lfm2.Lfm2Weights", tokens) -> torch.Tensor:
    """The logits after `tokens` in float64."""
    cfg, a = w.cfg, w.arrays
    name = {int(v): k for k, v in FORMATS.items()}
    mat = lambda key, rows, cols, fmt: _dense(name[int(fmt)], a[key], rows, cols)  # noqa: E731
    n, hd, t, lf = cfg.n_embd, cfg.head_dim, len(tokens), cfg.layer_format
    embed = mat("token_embd", cfg.n_vocab, n, cfg.embd_format)
    x = embed[torch.as_tensor(np.asarray(tokens, np.int64)).cuda()]
    for il in range(cfg.n_layers):
        y = _rms(x, _f64(a[f"{il}.attn_norm"]), cfg.norm_eps)
        if il in cfg.attention_layers:
            pos = torch.arange(t, device="cuda")
            split = lambda m, h: (y @ mat(f"{il}.{m}", h * hd, n, lf).T).reshape(t, h, hd)  # noqa: E731
            turn = lambda m, h, v: _rope(_rms(split(m, h), _f64(a[f"{il}.{v}"]), cfg.norm_eps).transpose(0, 1), pos,  # noqa: E731
                                         hd, cfg.rope_theta).transpose(0, 1)
            o = _attend(turn("wq", cfg.n_heads, "q_norm"), turn("wk", cfg.n_kv_heads, "k_norm"), split("wv", cfg.n_kv_heads), 0)
            x = x + o.reshape(t, -1) @ mat(f"{il}.wo", n, cfg.n_heads * hd, lf).T
        else:
            y = y @ mat(f"{il}.in_proj", 3 * n, n, lf).T
            hist = torch.zeros(cfg.conv_kernel - 1, n, dtype=F64, device="cuda")
            y = _short_conv(y, _f64(a[f"{il}.taps"]).reshape(n, -1), hist)[0]
            x = x + y @ mat(f"{il}.out_proj", n, n, lf).T
        y = _rms(x, _f64(a[f"{il}.ffn_norm"]), cfg.norm_eps)
        y = _silu(y @ mat(f"{il}.gate", cfg.n_ff, n, lf).T) * (y @ mat(f"{il}.up", cfg.n_ff, n, lf).T)
        x = x + y @ mat(f"{il}.down", n, cfg.n_ff, lf).T
    return embed @ _rms(x[-1], _f64(a["output_norm"]), cfg.norm_eps)


class Model:
    """What the model drivers' cases share."""

    @staticmethod
    def inputs(c, rng):
        cfg = MODELS[c["model"]]
        kind = qwen35.Qwen35Weights if isinstance(cfg, qwen35.Qwen35Config) else lfm2.Lfm2Weights
        return dict(weights=kind(cfg, seed=int(rng.integers(1 << 30))),
                    prompt=rng.integers(0, cfg.n_vocab, c["prompt"]).astype(np.uint32))

    @staticmethod
    def open(s, a, n_ctx):
        kind = qwen35.Qwen35Hip if isinstance(a["weights"].cfg, qwen35.Qwen35Config) else lfm2.Lfm2Hip
        s.model, s.prompt = kind(s.hip, a["weights"], n_ctx=n_ctx), a["prompt"]

    @staticmethod
    def matrices(c):
        """(bytes, weights) that a decode step reads, the output projection apart from the layers."""
        cfg = MODELS[c["model"]]
        w = cfg.weight_bytes()
        each = 256 / 144
        out = cfg.n_vocab * cfg.n_embd
        return w["layers"], w["layers"] * each, w["output"], out


class ModelPrefill(Model):
    """A new prompt through a model: its first logits."""

    @staticmethod
    def draw(rng):
        model = rng.choice(sorted(MODELS))
        return dict(model=model, prompt=_log_int(rng, 2, 512 if model == lfm2.LFM2_2_6B.name else 1024))

    @classmethod
    def prepare(cls, s, a):
        cls.open(s, a, s.case["prompt"] + 64)

    @staticmethod
    def run(s):
        s.model.reset()
        return s.model.prefill(s.prompt)

    @staticmethod
    def exact(c, a):
        return _lfm2_logits(a["weights"], a["prompt"]) if c["model"].startswith("lfm2") else None

    @classmethod
    def work(cls, c):
        lb, lw, ob, ow = cls.matrices(c)
        return dict(bytes=lb + ob, flops=2 * (c["prompt"] * lw + ow))

    tolerance = {"rel": 4e-3}  # the rounding of the f16 cache and inputs travels through the layers


class ModelDecode(Model):
    """Greedy tokens after a prompt, from a checkpoint of it, and the logits after the last."""

    @staticmethod
    def draw(rng):
        return dict(model=rng.choice([lfm2.LFM2_350M.name, qwen35.QWEN35_0_8B.name]), prompt=_log_int(rng, 2, 1500),
                    tokens=rng.randint(2, 32))

    @classmethod
    def prepare(cls, s, a):
        cls.open(s, a, s.case["prompt"] + s.case["tokens"] + 64)
        s.model.prefill(s.prompt, logits=False)
        s.blob = s.model.checkpoint()

    @staticmethod
    def run(s):
        s.model.restore(s.blob)
        tokens = s.model.generate_next(s.case["tokens"] - 1)
        return [tokens.astype(np.int64), s.model.step(int(tokens[-1]))]

    @staticmethod
    def exact(c, a):
        if not c["model"].startswith("lfm2") or c["tokens"] * c["prompt"] > 10000:
            return None
        tokens = list(a["prompt"])
        for _ in range(c["tokens"] + 1):
            logits = _lfm2_logits(a["weights"], tokens)
            tokens.append(int(logits.argmax()))
        first = len(a["prompt"])
        return [np.asarray(tokens[first + 1:first + c["tokens"]], np.int64), logits]

    @classmethod
    def work(cls, c):
        lb, lw, ob, ow = cls.matrices(c)
        return dict(bytes=c["tokens"] * (lb + ob), flops=2 * c["tokens"] * (lw + ow))

    tolerance = {"rel": 4e-3}


KINDS = dict(gemv=Gemv, decode_layers=DecodeLayers, attn_decode=AttnDecode, sample_head=SampleHead, ffn=Ffn,
             conv=ConvBlock, moe=Moe, deltanet=DeltaNet, attn_prefill=AttnPrefill, model_prefill=ModelPrefill,
             model_decode=ModelDecode)


def listed() -> list[dict]:
    return [
        # The input projection of a 2048-wide layer for one token: one launch.
        dict(name="gemv_norm", kind="gemv", fmt="q4k", rows=8192, cols=2048, norm=True),
        # Four layers of a decode step at the sizes of the 2.6B model.
        dict(name="decode_layers", kind="decode_layers", fmt="q4k", n=2048, n_ff=10752, layers=4),
        # One token's experts of the 8B mixture (4 of 32).
        dict(name="moe_decode", kind="moe", n=2048, n_ff=1792, experts=32, used=4, tokens=1),
        # One attention layer of a decode step after a 32K prompt.
        dict(name="attn_decode_32k", kind="attn_decode", heads=32, kv=8, hd=64, half=True, pos=32767),
        # The last launches of a sampled step with the usual sampler settings.
        dict(name="sample_head", kind="sample_head", fmt="q4k", n=2048, vocab=65536, top_k=40, top_p=0.95, min_p=0.05,
             temperature=0.7, penalty=1.1),
        # The feed-forward block of a full prefill batch at the sizes of the 2.6B model.
        dict(name="ffn_512", kind="ffn", fmt="q4k", n=2048, n_ff=10752, tokens=512),
        # The tail batch of a prompt through a convolution layer of a mixed-format file.
        dict(name="conv_q6k_137", kind="conv", fmt="q6k", n=2048, tokens=137),
        # The experts of a full prefill batch.
        dict(name="moe_512", kind="moe", n=2048, n_ff=1792, experts=32, used=4, tokens=512),
        # A DeltaNet layer of a full prefill batch at the sizes of the 0.8B model.
        dict(name="deltanet_512", kind="deltanet", nk=16, nv=16, dk=128, dv=128, tokens=512),
        # A prefill batch of a long prompt: 512 queries over 8,192 keys.
        dict(name="attn_prefill_8k", kind="attn_prefill", heads=32, kv=8, hd=64, first=7680, tokens=512),
        # The headline prompt: 512 tokens through the 2.6B model.
        dict(name="prefill_2.6b_512", kind="model_prefill", model=lfm2.LFM2_2_6B.name, prompt=512),
        # A short reply of the 350M model.
        dict(name="decode_350m", kind="model_decode", model=lfm2.LFM2_350M.name, prompt=300, tokens=16),
    ]


def draw(rng) -> dict:
    kind = rng.choice(sorted(KINDS))
    return dict(kind=kind, **KINDS[kind].draw(rng))


def _inputs(case: dict, seed: int) -> dict:
    return KINDS[case["kind"]].inputs(case, np.random.default_rng(seed))


def prepare(case: dict, seed: int) -> State:
    state = State(case)
    KINDS[case["kind"]].prepare(state, _inputs(case, seed))
    return state


def run(state: State):
    return KINDS[state.case["kind"]].run(state)


def work(case: dict) -> dict:
    return KINDS[case["kind"]].work(case)


def tolerance(case: dict) -> dict:
    if case["kind"] == "moe" and case["tokens"] == 1:
        return {"rel": 4e-6}  # one token's products stay in f32
    return KINDS[case["kind"]].tolerance


def exact(case: dict, seed: int):
    return KINDS[case["kind"]].exact(case, _inputs(case, seed))
