"""Workloads of the attention library, called through its C ABI on torch tensors.

listed() holds the calls that users of the library make: the shapes of bench.py
and torch_compare.py (the reference's harness shapes among them), one query row
against a long key cache, ragged lengths, and the pre-pass pipeline.  draw()
gives further calls of the same ranges.  prepare() makes the inputs, run() is
one call, exact() the same result in float64, work() the bytes and operations
the call cannot do without.

Cases: dtype "f32" or "bf16"; B, H, Lq, Lk, D as in the C ABI; pe "none",
"rope" (interleaved pairs), "rope_half" (rotate-half) or "sinusoidal"; rot the
rotated width (0: all of D); call "ex" (atn_attention_fwd_ex), "dropin" (the
synchronous attention_forward_optimized / attention_forward_bf16) or
"separate" (attention_forward_separate_rope: Q and K rotated by a pre-pass
with the caller's caches, then attention).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "accelerated-final-project_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import attn_mi355x as am  # noqa: E402  (after torch: both then use one HIP runtime)


def _case(name, dtype, B, H, Lq, Lk, D, pe="none", rot=0, sigma=1.0, call="ex"):
    c = {"dtype": dtype, "B": B, "H": H, "Lq": Lq, "Lk": Lk, "D": D, "pe": pe, "rot": rot,
         "sigma": sigma, "call": call}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call of the benchmark, through the reference's own synchronous entry point:
        # what one call costs when there is nothing to compute
        _case("tiny_f32_dropin", "f32", 1, 1, 4, 4, 8, call="dropin"),
        # short self-attention with large heads, the reference's headline shape
        _case("short_f32", "f32", 1, 4, 64, 64, 2048),
        # short cross-attention with the largest heads
        _case("cross_bf16", "bf16", 1, 4, 32, 128, 8192),
        # long sequences, large heads, RoPE inside the call: the largest job
        _case("long_rope_bf16", "bf16", 8, 8, 1024, 1024, 4096, pe="rope_half"),
        # cross-attention onto a longer context, sinusoidal positions
        _case("cross_sin_bf16", "bf16", 4, 16, 256, 2048, 1024, pe="sinusoidal", sigma=0.5),
        # a batch of prompts at the usual head size, fp32: the reference's long-sequence shape
        _case("prompt_f32", "f32", 4, 32, 512, 512, 128),
        # the same batch in bf16 with rotate-half RoPE
        _case("prompt_rope_bf16", "bf16", 4, 32, 512, 512, 128, pe="rope_half"),
        # one long document
        _case("long_bf16", "bf16", 1, 8, 4096, 4096, 128),
        # decoding: one new query row against a long key cache
        _case("decode_bf16", "bf16", 1, 32, 1, 8192, 128),
        # longer sequences with large heads in fp32
        _case("large_head_f32", "f32", 1, 4, 512, 512, 2048),
        # lengths and a head size that fit no tile, interleaved RoPE
        _case("ragged_rope_f32", "f32", 4, 8, 1000, 999, 100, pe="rope"),
        # the pre-pass pipeline: Q and K rotated into buffers of the caller's, then attention
        _case("separate_rope_f32", "f32", 4, 32, 512, 512, 128, pe="rope", call="separate"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _up(x, m):
    return max(m, (x + m - 1) // m * m)


def draw(rng):
    kind = rng.choice(("short", "short", "prompt", "prompt", "prompt", "decode", "large_bf16",
                       "large_bf16", "large_f32", "large_f32", "separate"))
    dtype = rng.choice(("f32", "bf16"))
    pe = rng.choice(("none", "none", "rope", "rope_half", "sinusoidal"))
    rot = 0
    sigma = rng.choice((1.0, 1.0, 0.5))
    call = "ex"
    if kind == "short":
        B, H = rng.choice((1, 1, 2)), rng.choice((1, 2, 4, 8))
        Lq, Lk = _log(rng, 1, 64), _log(rng, 4, 128)
        D = _up(_log(rng, 8, 8192), 8)
        if rng.random() < 0.25:
            call, pe = "dropin", "none"
    elif kind == "decode":
        B, H = rng.choice((1, 2, 4)), rng.choice((8, 16, 32))
        Lq, Lk = rng.choice((1, 1, 2, 4, 8, 16)), _log(rng, 256, 16384)
        D = rng.choice((64, 80, 96, 128, 128, 256))
    elif kind == "prompt":
        B, H = rng.choice((1, 2, 4, 8)), rng.choice((4, 8, 16, 32))
        Lq = _log(rng, 65, 4096)
        Lk = Lq if rng.random() < 0.6 else _log(rng, 130, 4096)
        D = rng.choice((32, 40, 64, 64, 72, 80, 96, 100, 128, 128, 128, 160, 192, 256))
    elif kind == "separate":
        B, H = rng.choice((1, 2, 4)), rng.choice((4, 8, 16, 32))
        Lq = Lk = _log(rng, 130, 2048)
        D = rng.choice((64, 96, 128, 256, 512, 1024))
        dtype, pe, call = "f32", "rope", "separate"
        if rng.random() < 0.3:
            rot = D // 2
    else:
        dtype = "bf16" if kind == "large_bf16" else "f32"
        B, H = rng.choice((1, 2, 4)), rng.choice((2, 4, 8, 16))
        Lq = _log(rng, 65, 1024)
        Lk = Lq if rng.random() < 0.5 else _log(rng, 130, 2048)
        D = _up(_log(rng, 264, 8192), 8)
        if rng.random() < 0.15:
            D += rng.choice((1, 2, 4))  # a head size that is no whole number of vectors
    if pe.startswith("rope") and D % 2:
        D += 1
    if pe == "rope" and rot == 0 and rng.random() < 0.2:
        rot = max(2, D // 4 * 2)
    # no drawn call costs more than the largest listed one
    limit = 1.0e12 if dtype == "bf16" else 6.0e10
    if D % 8:
        limit /= 10
    while 4.0 * B * H * Lq * Lk * D > limit or B * H * (Lq + Lk) * D > 2 ** 29:
        if B > 1:
            B //= 2
        elif H > 1:
            H //= 2
        else:
            Lq, Lk = max(1, Lq // 2), max(4, Lk // 2)
    return _case(None, dtype, B, H, Lq, Lk, D, pe, rot, sigma, call)


# ------------------------------------------------------------------ inputs
def _inputs(case, seed):
    """Q, K, V on the GPU: N(0, sigma), as activations and projections are."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    B, H, D = case["B"], case["H"], case["D"]
    out = []
    for L in (case["Lq"], case["Lk"], case["Lk"]):
        x = torch.randn((B, H, L, D), generator=g, device="cuda", dtype=torch.float32)
        out.append(x.mul_(case["sigma"]).to(dt))
    return out


def _rotary(case):
    return case["rot"] or case["D"]


def _angles(npos, n, width):
    """pos * (1 / 10000^(2i / width)) for i < n, in the float32 steps that the C ABI states."""
    i = np.arange(n, dtype=np.float32)
    e = (np.float32(2.0) * i) / np.float32(width)
    p = np.power(10000.0, e.astype(np.float64)).astype(np.float32)
    freq = np.float32(1.0) / p
    return np.arange(npos, dtype=np.float32)[:, None] * freq[None, :]


def _caches(case):
    """The reference's cos and sin caches [pos][rotary] (pairs hold one value twice)."""
    r = _rotary(case)
    a = np.repeat(_angles(max(case["Lq"], case["Lk"]), r // 2, r), 2, axis=1).astype(np.float64)
    return [torch.from_numpy(f(a).astype(np.float32)).cuda() for f in (np.cos, np.sin)]


def prepare(case, seed):
    lib = am.lib()
    q, k, v = _inputs(case, seed)
    out = torch.empty_like(q)
    dims = [case[n] for n in ("B", "H", "Lq", "Lk", "D")]
    state = {"keep": (q, k, v), "out": out}
    ptr = [t.data_ptr() for t in (q, k, v, out)]
    if case["call"] == "dropin":
        state["call"] = (lib.attention_forward_optimized if case["dtype"] == "f32"
                         else lib.attention_forward_bf16)
        state["args"] = ptr + dims
    elif case["call"] == "separate":
        qr, kr, cs = torch.empty_like(q), torch.empty_like(k), _caches(case)
        state["keep"] += tuple(cs)
        state["out"] = [qr, kr, out]
        state["call"] = lib.attention_forward_separate_rope
        state["args"] = (ptr[:3] + [qr.data_ptr(), kr.data_ptr(), out.data_ptr()] +
                         [t.data_ptr() for t in cs] + dims + [_rotary(case)])
    else:
        pe = None
        if case["pe"] == "sinusoidal":
            pe = am.make_pe("sinusoidal")
        elif case["pe"] != "none":
            pe = am.make_pe("rope", "half" if case["pe"] == "rope_half" else "interleaved",
                            case["rot"])
        if pe is not None:  # the angle tables, built once for all calls of these sizes
            am.lib().atn_prepare_pe_ex(ctypes.byref(pe), case["D"], max(case["Lq"], case["Lk"]))
        stream = torch.cuda.current_stream().cuda_stream
        state["pe"] = pe
        state["call"] = lib.atn_attention_fwd_ex
        state["args"] = ([am.ATN_DTYPE_F32 if case["dtype"] == "f32" else am.ATN_DTYPE_BF16] + ptr +
                         dims + [ctypes.byref(pe) if pe is not None else None, None, 0, stream])
    return state


def run(state):
    status = state["call"](*state["args"])
    if status:  # (the drop-ins return nothing)
        raise RuntimeError("status %d" % status)
    return state["out"]


# ------------------------------------------------------------------ the same in float64
def _rotate(x, case):
    """RoPE over the rows of x [B, H, L, D] in x's type (float64)."""
    r = _rotary(case)
    a = torch.from_numpy(_angles(x.shape[2], r // 2, r).astype(np.float64)).to(x.device)
    if case["call"] == "separate":  # the caches hold float32 values
        c, s = torch.cos(a).float().to(x.dtype), torch.sin(a).float().to(x.dtype)
    else:
        c, s = torch.cos(a), torch.sin(a)
    y = x.clone()
    if case["pe"] == "rope_half":
        x0, x1 = x[..., :r // 2], x[..., r // 2:r]
        y[..., :r // 2], y[..., r // 2:r] = x0 * c - x1 * s, x0 * s + x1 * c
    else:
        x0, x1 = x[..., 0:r:2], x[..., 1:r:2]
        y[..., 0:r:2], y[..., 1:r:2] = x0 * c - x1 * s, x0 * s + x1 * c
    return y


def _add_positions(x):
    D = x.shape[-1]
    a = np.repeat(_angles(x.shape[2], (D + 1) // 2, D), 2, axis=1)[:, :D].astype(np.float64)
    t = np.sin(a)
    t[:, 1::2] = np.cos(a[:, 1::2])
    return x + torch.from_numpy(t).to(x.device)


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    qr, kr = ([torch.empty(t.shape, dtype=torch.float64, device=q.device) for t in (q, k)]
              if case["call"] == "separate" else (None, None))
    for b in range(case["B"]):
        for h in range(case["H"]):
            x, y = q[b:b + 1, h:h + 1].double(), k[b:b + 1, h:h + 1].double()
            if case["pe"] == "sinusoidal":
                x, y = _add_positions(x), _add_positions(y)
            elif case["pe"] != "none":
                x, y = _rotate(x, case), _rotate(y, case)
            if qr is not None:
                qr[b, h], kr[b, h] = x[0, 0], y[0, 0]
            s = torch.mm(x[0, 0], y[0, 0].t().contiguous()) / math.sqrt(case["D"])
            o[b, h] = torch.mm(torch.softmax(s, dim=-1), v[b, h].double())
    return o if qr is None else [qr, kr, o]


# ------------------------------------------------------------------ cost and tolerance
def work(case):
    B, H, Lq, Lk, D = (case[n] for n in ("B", "H", "Lq", "Lk", "D"))
    es = 4 if case["dtype"] == "f32" else 2
    byts = B * H * (2 * Lq + 2 * Lk) * D * es
    if case["call"] == "separate":  # the rotated copies, written, and the caches
        byts += B * H * (Lq + Lk) * D * es + 2 * max(Lq, Lk) * _rotary(case) * 4
    return {"bytes": byts, "flops": 4 * B * H * Lq * Lk * D}


def tolerance(case):
    # the largest errors against float64 over the listed and 150 drawn calls, times about four:
    # f32 2.2e-6 normwise and 2.8e-5 of the larger of value and rms (sinusoidal encodings at
    # head_d 5218, peaked rows), bf16 2.4e-3 and 2.1e-2
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1.1e-4}
    return {"rel": 1e-2, "max": 8e-2}
