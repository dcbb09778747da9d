"""What is measured of this framework: the fp8 linear path of the DiT blocks, called through
the package's public entry points over the sizes that its workloads, tests and benchmark use.

Widths are those of the two DiTs that the workloads name (hidden 5120 with a GELU FFN of
13824; H3's hidden 5376, 56 heads of 128, SwiGLU FFN of 14336); row counts run from a short
prompt over whole latent frames (1560 tokens each) to the 32760 tokens of 21 frames, with
13107 as one rank's share of a sequence. Draws add odd row counts and generic odd widths.
"""
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vdn-minimax-h3_amd"))

from vdn_fp8 import (Fp8Linear, fast_block_forward, fast_ff_forward, gelu_quantize, pre_quantize,  # noqa: E402
                     quantize_activation, requantize_weight)
from vdn_fp8.softmax_attention import qkv  # noqa: E402

DEV = "cuda:0"
BF16 = torch.bfloat16
FRAME = 1560                    # tokens of one latent frame (30 x 52 patches)
MOST_FLOPS = 2.0 * 32760 * 15360 * 5120

# (N, K) of the linears of the two DiTs, as they are called alone.
WIDTHS = ((15360, 5120), (13824, 5120), (5120, 13824), (5120, 5120), (7168, 5376), (5376, 7168), (28672, 5376),
          (5376, 14336), (5376, 5120), (1024, 1024))
# hidden, heads, FFN width
H3 = (5376, 56, 14336)
HEAD_DIM = 128
EPS = 1e-6


def listed():
    return [
        # the smallest linear of the workloads: two launches, so latency counts
        {"name": "linear_1024", "kind": "linear", "M": 1024, "N": 1024, "K": 1024, "dtype": "bf16"},
        # the context embedder on an encoded prompt (821 tokens)
        {"name": "prompt_embed", "kind": "linear", "M": 821, "N": 5376, "K": 5120, "dtype": "bf16"},
        # the token refiner's SwiGLU feed-forward on a prompt of 1299 tokens
        {"name": "refiner_ff", "kind": "ff", "M": 1299, "C": 5376, "I": 14336},
        # the fused QKV projection of 21 latent frames: the largest single layer
        {"name": "dit_qkv", "kind": "linear", "M": 32760, "N": 15360, "K": 5120, "dtype": "bf16"},
        # attention-out with the AdaLN gate of each frame and the residual, six frames
        {"name": "dit_out_gate", "kind": "gated", "M": 6 * FRAME, "N": 5120, "K": 5120, "T": 6},
        # a GELU feed-forward with a broadcast gate, three frames
        {"name": "dit_gelu_ffn", "kind": "gelu", "M": 3 * FRAME, "C": 5120, "I": 13824},
        # the attention's input: three projections of one quantization, QK-norm and rope
        {"name": "h3_qkv", "kind": "qkv", "M": 13107, "C": 5376, "heads": 56},
        # one whole block (attention core aside) on one rank's share of a sequence
        {"name": "h3_block", "kind": "block", "M": 13107, "C": 5376, "heads": 56, "I": 14336, "T": 9},
        # the block's pre-norm and modulation, quantized for the projections
        {"name": "h3_prenorm", "kind": "prenorm", "M": 13107, "K": 5376, "T": 9},
        # assembling a model: a LoRA folded into a weight, which is then quantized
        {"name": "lora_qkv", "kind": "requant", "N": 15360, "K": 5120, "rank": 64},
        {"name": "lora_h3_down", "kind": "requant", "N": 5376, "K": 14336, "rank": 64},
        # a float16 model with widths that no tile divides
        {"name": "f16_odd", "kind": "linear", "M": 1111, "N": 4100, "K": 4112, "dtype": "f16"},
    ]


def _log(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def _rows(rng, flops_a_row, most=MOST_FLOPS):
    """A row count from 64 to 32760 (as far as `most` allows): whole frames now and then, odd ones otherwise."""
    high = max(65, min(32760, int(most / flops_a_row)))
    m = _log(rng, 64, high)
    if m > FRAME and rng.random() < 0.3:
        m = m // FRAME * FRAME
    return m


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "gated", "gelu", "ff", "qkv", "block", "prenorm", "requant",
                       "requant", "odd"))
    if kind == "linear":
        N, K = rng.choice(WIDTHS)
        return {"kind": kind, "M": _rows(rng, 2.0 * N * K), "N": N, "K": K, "dtype": "bf16"}
    if kind == "odd":
        N, K = 4 * (_log(rng, 1024, 8192) // 4), 16 * (_log(rng, 1024, 8192) // 16)
        return {"kind": "linear", "M": _rows(rng, 2.0 * N * K, MOST_FLOPS / 16), "N": N, "K": K,
                "dtype": rng.choice(("bf16", "f16", "f32"))}
    if kind == "gated":
        N, K = rng.choice(((5120, 5120), (5376, 7168), (5120, 13824), (5376, 14336)))
        return {"kind": kind, "M": _rows(rng, 2.0 * N * K), "N": N, "K": K, "T": rng.randint(1, 21)}
    if kind == "gelu":
        return {"kind": kind, "M": _rows(rng, 4.0 * 5120 * 13824), "C": 5120, "I": 13824}
    if kind == "ff":
        return {"kind": kind, "M": _rows(rng, 6.0 * H3[0] * H3[2]), "C": H3[0], "I": H3[2]}
    if kind == "qkv":
        return {"kind": kind, "M": _rows(rng, 6.0 * H3[0] * H3[1] * HEAD_DIM), "C": H3[0], "heads": H3[1]}
    if kind == "block":
        return {"kind": kind, "M": _rows(rng, 7.9e8, 2 * MOST_FLOPS), "C": H3[0], "heads": H3[1], "I": H3[2],
                "T": rng.randint(1, 12)}
    if kind == "prenorm":
        return {"kind": kind, "M": _rows(rng, 1.0), "K": rng.choice((1024, 4096, 5120, 5376, 7168)),
                "T": rng.randint(1, 21)}
    N, K = rng.choice(WIDTHS)
    return {"kind": kind, "N": N, "K": K, "rank": rng.choice((0, 8, 16, 32, 48, 64, 128))}


# ---------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------

DTYPES = {"bf16": BF16, "f16": torch.float16, "f32": torch.float32}


class _Draw:
    """Seeded normal draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(DEV).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=BF16):
        t = torch.empty(*shape, device=DEV).normal_(mean, std, generator=self.g)
        return t.to(dtype)

    def rows(self, M, K, dtype=BF16):
        """Activations: N(0, 1), 0.1% of the channels (at least one) 20 times as large."""
        x = torch.empty(M, K, device=DEV).normal_(generator=self.g)
        x[:, torch.randperm(K, generator=self.g, device=DEV)[:max(1, K // 1000)]] *= 20.0
        return x.to(dtype)

    def linear(self, N, K, bias=True, dtype=BF16):
        w = self.normal(N, K, std=0.02, dtype=dtype)
        return w, self.normal(N, std=0.01, dtype=dtype) if bias else None

    def frames(self, M, T):
        """Table row of each token: T runs of whole frames, as near as M allows."""
        return (torch.arange(M, device=DEV) * T // max(M, 1)).to(torch.int32)

    def table(self, T, K, mean=0.0):
        return self.normal(T, K, std=0.3, mean=mean)


def _layer(wb):
    """The framework's layer of a weight and a bias, as a user's program makes it of its Linear."""
    w, b = wb
    lin = nn.Linear(w.shape[1], w.shape[0], bias=b is not None, dtype=w.dtype, device="meta")
    lin.weight = nn.Parameter(w, requires_grad=False)
    if b is not None:
        lin.bias = nn.Parameter(b, requires_grad=False)
    return Fp8Linear(lin)


class _Norm(nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight, self.eps = weight, EPS


class _Proj(nn.Module):
    def __init__(self, proj):
        super().__init__()
        self.proj = proj


class _FeedForward(nn.Module):
    """SwiGLU projection, dropout (none at inference), down projection."""

    def __init__(self, proj, down):
        super().__init__()
        self.net = nn.ModuleList([_Proj(proj), nn.Identity(), down])

    forward = fast_ff_forward


class _Attention(nn.Module):
    """The attention around its core, which is not this package's: projections, QK-norm, rope
    and the output projection, with the sum of q, k and v in the core's place."""

    def __init__(self, q, k, v, out, heads, norm_q, norm_k):
        super().__init__()
        self.q, self.k, self.v, self.out = q, k, v, out
        self.heads, self.norm_q, self.norm_k = heads, norm_q, norm_k

    def forward(self, x, rotary_emb, attention_mask=None):
        query, key, value, _ = qkv(x.reshape(-1, x.shape[-1]), self.q, self.k, self.v, self.heads, self.norm_q,
                                   self.norm_k, rotary_emb)
        return self.out(((query + key) + value).flatten(1)).reshape(x.shape)


class _Block(nn.Module):
    def __init__(self, tables, norm1, norm2, attn, ff):
        super().__init__()
        self.tables, self.norm1, self.norm2, self.attn, self.ff = tables, norm1, norm2, attn, ff

    def adaln_proj(self, temb):
        return self.tables

    forward = fast_block_forward


def _rope(M):
    pos = torch.arange(M, device=DEV, dtype=torch.float32)[:, None]
    inv = 10000.0 ** (-torch.arange(0, HEAD_DIM, 2, device=DEV, dtype=torch.float32) / HEAD_DIM)
    ang = (pos * inv).repeat(1, 2)
    return ang.cos(), ang.sin()


def _inputs(case, seed):
    """The plain tensors of a case, of the seed alone."""
    d, kind = _Draw(seed), case["kind"]
    if kind == "linear":
        t = DTYPES[case["dtype"]]
        return {"x": d.rows(case["M"], case["K"], t), "w": d.linear(case["N"], case["K"], dtype=t)}
    if kind == "gated":
        M, N, K, T = case["M"], case["N"], case["K"], case["T"]
        return {"x": d.rows(M, K), "w": d.linear(N, K, bias=False), "gate": d.table(T, N, 1.0),
                "idx": d.frames(M, T), "res": d.normal(M, N)}
    if kind == "gelu":
        M, C, I = case["M"], case["C"], case["I"]
        return {"x": d.rows(M, C), "up": d.linear(I, C), "down": d.linear(C, I, bias=False),
                "gate": d.table(1, C, 1.0).reshape(C)}
    if kind == "ff":
        M, C, I = case["M"], case["C"], case["I"]
        return {"x": d.rows(M, C), "proj": d.linear(2 * I, C, bias=False), "down": d.linear(C, I, bias=False)}
    if kind in ("qkv", "block"):
        M, C, H = case["M"], case["C"], case["heads"]
        E = H * HEAD_DIM
        s = {"x": d.rows(M, C) if kind == "qkv" else d.normal(1, M, C), "rope": _rope(M),
             "q": d.linear(E, C, bias=False), "k": d.linear(E, C, bias=False), "v": d.linear(E, C, bias=False),
             "nq": d.normal(HEAD_DIM, std=0.1, mean=1.0), "nk": d.normal(HEAD_DIM, std=0.1, mean=1.0)}
        if kind == "block":
            I, T = case["I"], case["T"]
            s.update(out=d.linear(C, E, bias=False), proj=d.linear(2 * I, C, bias=False),
                     down=d.linear(C, I, bias=False), n1=d.normal(C, std=0.1, mean=1.0),
                     n2=d.normal(C, std=0.1, mean=1.0), tables=tuple(d.table(T, C) for _ in range(6)),
                     idx=d.frames(M, T))
        return s
    if kind == "prenorm":
        M, K, T = case["M"], case["K"], case["T"]
        return {"x": d.rows(M, K), "w": d.normal(K, std=0.1, mean=1.0), "scale": d.table(T, K),
                "shift": d.table(T, K), "idx": d.frames(M, T)}
    N, K, r = case["N"], case["K"], case["rank"]
    s = {"w": d.normal(N, K, std=0.02)}
    if r:
        s.update(a=d.normal(r, K, std=0.01), b=d.normal(N, r, std=0.01))
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s["kind"] = kind
    if kind in ("linear", "gated"):
        s["layer"] = _layer(s.pop("w"))
    elif kind == "gelu":
        s["up"], s["down"] = _layer(s["up"]), _layer(s["down"])
    elif kind == "ff":
        s["ff"] = _FeedForward(_layer(s.pop("proj")), _layer(s.pop("down")))
    elif kind in ("qkv", "block"):
        s["heads"] = case["heads"]
        s["q"], s["k"], s["v"] = _layer(s["q"]), _layer(s["k"]), _layer(s["v"])
        s["nq"], s["nk"] = _Norm(s["nq"]), _Norm(s["nk"])
        if kind == "block":
            attn = _Attention(s["q"], s["k"], s["v"], _layer(s.pop("out")), s["heads"], s["nq"], s["nk"])
            ff = _FeedForward(_layer(s.pop("proj")), _layer(s.pop("down")))
            s["block"] = _Block(s["tables"], _Norm(s["n1"]), _Norm(s["n2"]), attn, ff)
    elif kind == "requant":
        s["lora"] = (s["a"], s["b"], 1.0) if case["rank"] else None
    return s


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["layer"](s["x"])
    if kind == "gated":
        return s["layer"](s["x"], epilogue="gate", gate=s["gate"], gate_index=s["idx"], residual=s["res"])
    if kind == "gelu":
        h = s["up"].forward_quantized(*quantize_activation(s["x"]))
        return s["down"].forward_quantized(*gelu_quantize(h), epilogue="gate", gate=s["gate"])
    if kind == "ff":
        return s["ff"](s["x"])
    if kind == "qkv":
        q, k, v, raw = qkv(s["x"], s["q"], s["k"], s["v"], s["heads"], s["nq"], s["nk"], s["rope"])
        return [q, k, v, raw[0], raw[1]]
    if kind == "block":
        return s["block"](s["x"], None, s["idx"], s["rope"])
    if kind == "prenorm":
        codes, scale = pre_quantize(s["x"], s["w"], EPS, s["scale"], s["shift"], s["idx"])
        return [codes.view(torch.uint8), scale]
    codes, scale = requantize_weight(s["w"], lora=s["lora"])
    return [codes.view(torch.uint8), scale]


# ---------------------------------------------------------------------------------------
# what a pass cannot do without, and how far two right answers may be apart
# ---------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        e = 4 if case["dtype"] == "f32" else 2
        return {"bytes": e * M * K + N * K + 4 * N + e * N + e * M * N, "flops": 2.0 * M * N * K}
    if kind == "gated":
        M, N, K, T = case["M"], case["N"], case["K"], case["T"]
        return {"bytes": 2 * M * K + N * K + 4 * N + 2 * T * N + 4 * M + 4 * M * N, "flops": 2.0 * M * N * K}
    if kind in ("gelu", "ff"):
        M, C, I = case["M"], case["C"], case["I"]
        parts = 2 if kind == "gelu" else 3
        return {"bytes": 4 * M * C + parts * C * I + 4 * (C + (parts - 1) * I), "flops": 2.0 * parts * M * C * I}
    if kind == "qkv":
        M, C, E = case["M"], case["C"], case["heads"] * HEAD_DIM
        return {"bytes": 2 * M * C + 3 * E * C + 12 * E + 8 * M * HEAD_DIM + 5 * 2 * M * E, "flops": 6.0 * M * E * C}
    if kind == "block":
        M, C, E, I, T = case["M"], case["C"], case["heads"] * HEAD_DIM, case["I"], case["T"]
        return {"bytes": 4 * M * C + 4 * E * C + 3 * C * I + 12 * T * C + 8 * M * HEAD_DIM + 4 * M,
                "flops": 2.0 * M * (4 * E * C + 3 * C * I)}
    if kind == "prenorm":
        M, K, T = case["M"], case["K"], case["T"]
        return {"bytes": 2 * M * K + M * K + 4 * M + 2 * K + 4 * T * K + 4 * M, "flops": 8.0 * M * K}
    N, K, r = case["N"], case["K"], case["rank"]
    return {"bytes": 3 * N * K + 4 * N + 2 * r * (N + K), "flops": 2.0 * r * N * K + 2.0 * N * K}


def tolerance(case):
    kind = case["kind"]
    if kind == "requant":
        if not case["rank"]:
            return "exact"          # the same codes and scales, whatever the order of a maximum
        # a bf16 rounding of a merged element that falls the other way moves a code, or a row's scale
        return {"rel": 1e-3, "max": 8e-3, "differ": 1e-3}
    if kind == "prenorm":
        return {"rel": 1e-3, "max": 8e-3, "differ": 1e-3}
    if kind == "linear" and case["dtype"] == "f32":
        return {"rel": 1e-4, "max": 2e-3}      # the matrix cores align the products of a step: 2.4e-5 measured
    if kind == "linear" and case["dtype"] == "f16":
        return {"rel": 4e-3, "max": 2e-2}
    if kind in ("gelu", "ff", "block"):
        # a rounding that falls the other way in one layer moves codes of the next
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------------------
# the same in 64 bits (plain torch)
# ---------------------------------------------------------------------------------------

def _codes(x):
    """Rows of binary32 or narrower values as the path quantizes them: e4m3 codes by the row's
    scale max(absmax / 448, 1e-12). The scale and the quotient are the path's own in binary32
    (the codes are whole numbers, the same whatever computes them)."""
    scale = _scale(x)
    return _over(x.float(), scale).to(torch.float8_e4m3fn), scale


def _weight_codes(w):
    scale = _scale(w)
    return _over(w, scale.to(w.dtype)).to(torch.float8_e4m3fn), scale


def _scale(x):
    return (x.abs().amax(1, keepdim=True).double() / 448.0).float().clamp_min(1e-12)


def _over(x, scale):
    """x / scale rounded once to x's type, by row blocks (a 64-bit quotient rounded again is the
    correctly rounded one for these types)."""
    return torch.cat([(x[i:i + 8192].double() / scale[i:i + 8192].double()).to(x.dtype)
                      for i in range(0, x.shape[0], 8192)])


def _mm(xq, xs, w):
    """x_scale * w_scale * (codes of x @ codes of the weight), by row blocks."""
    wq, ws = _weight_codes(w)
    w64 = wq.float().double().t().contiguous()
    out = torch.empty(xq.shape[0], w.shape[0], device=xq.device, dtype=torch.float64)
    for i in range(0, xq.shape[0], 4096):
        out[i:i + 4096] = xq[i:i + 4096].float().double() @ w64
    return out.mul_(xs.double()).mul_(ws.double().t())


def _norm(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _mod(x, w, scale, shift, idx):
    return _norm(x, w) * (1.0 + scale.double()[idx.long()]) + shift.double()[idx.long()]


def _qk(t, w, rope, heads):
    """QK-norm, then the rotation of the two halves by bf16 tables."""
    t = _norm(t.unflatten(-1, (heads, -1)), w)
    cos, sin = (c.to(BF16).double()[:, None] for c in rope)
    lo, hi = t.chunk(2, -1)
    return t * cos + torch.cat((-hi, lo), -1) * sin


def _qkv64(xq, xs, s, heads):
    """Query and key (normed, rotated), value, and the raw query and key: the projections are
    bf16 tensors on the path, so what follows them reads bf16 values."""
    q, k, v = (_mm(xq, xs, s[n][0]) for n in ("q", "k", "v"))
    split = lambda t: t.unflatten(-1, (heads, -1))  # noqa: E731
    return [_qk(q.to(BF16), s["nq"], s["rope"], heads), _qk(k.to(BF16), s["nk"], s["rope"], heads), split(v), split(q),
            split(k)]


def _swiglu64(h, I):
    h = h.to(BF16).double()
    return h[:, :I] * F.silu(h[:, I:])


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "linear":
        w, b = s["w"]
        return _mm(*_codes(s["x"]), w) + b.double()
    if kind == "gated":
        v = _mm(*_codes(s["x"]), s["w"][0])
        return s["res"].double() + s["gate"].double()[s["idx"].long()] * v
    if kind == "gelu":
        h = _mm(*_codes(s["x"]), s["up"][0]) + s["up"][1].double()
        g = F.gelu(h.to(BF16).double(), approximate="tanh").to(BF16)
        return _mm(*_codes(g), s["down"][0]) * s["gate"].double()
    if kind == "ff":
        act = _swiglu64(_mm(*_codes(s["x"]), s["proj"][0]), case["I"])
        return _mm(*_codes(act), s["down"][0])
    if kind == "qkv":
        return _qkv64(*_codes(s["x"]), s, case["heads"])
    if kind == "block":
        shift1, scale1, gate1, shift2, scale2, gate2 = s["tables"]
        idx = s["idx"].long()
        x = s["x"][0]
        normed = _mod(x, s["n1"], scale1, shift1, idx).to(BF16)
        q, k, v, _, _ = _qkv64(*_codes(normed), s, case["heads"])
        a = ((q.to(BF16) + k.to(BF16)) + v.to(BF16)).flatten(1)
        attn = _mm(*_codes(a), s["out"][0]).to(BF16)
        x = (x.double() + gate1.double()[idx] * attn.double()).to(BF16)
        normed = _mod(x, s["n2"], scale2, shift2, idx).to(BF16)
        act = _swiglu64(_mm(*_codes(normed), s["proj"][0]), case["I"])
        v = _mm(*_codes(act), s["down"][0])
        return (x.double() + gate2.double()[idx] * v)[None]
    if kind == "prenorm":
        y = _mod(s["x"], s["w"], s["scale"], s["shift"], s["idx"])
        return [None, y.abs().amax(1, keepdim=True) / 448.0]
    w = s["w"].double()
    if case["rank"]:
        w = w + s["b"].double() @ s["a"].double()
    return [None, w.abs().amax(1) / 448.0]
