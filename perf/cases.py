"""What a user of this library has it do, as cases that can be timed and checked.

A caller is an inference engine on one MI355X: its weights are GGUF tensors pinned once, its activations stay
on the GPU between calls, and every call goes through one context (one stream) of ``qxotic_amd.jam.HipJAM``.
Four kinds of case:

* ``mm``: one matmul through the device entry point, R = W @ A^T, with an optional bias.
* ``host``: the same through ``HipJAM.mm`` with host activations and host result (the call an engine makes that
  keeps its activations in host memory), the weight pinned.
* ``moe``: one gpt-oss-shaped mixture-of-experts block: router, top-k, routing, grouped gate|up with the gather
  folded in, gated activation, grouped down projection, weighted combine.
* ``step``: a stack of Llama-shaped decoder layers' projections and the output head, as one decode step (or a
  small batch of sequences) runs them: q|k|v, attention output into the residual, gate|up, gated activation, down
  projection into the residual. Attention itself and the norms belong to the caller and are left out: the output
  projection reads the q part of q|k|v.

``exact`` is the operation's own definition in 64 bits: the activations go through the int8 block quantization
that the operation prescribes (its rounding is part of the result), and everything after that is exact.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from qxotic_amd.jam import JAM, HipJAM, Segment

CODES = {"F32": JAM.F32, "F16": JAM.F16, "BF16": JAM.BF16, "Q8_0": JAM.Q8_0, "Q4_0": JAM.Q4_0, "Q4_K": JAM.Q4_K,
         "Q5_K": JAM.Q5_K, "Q6_K": JAM.Q6_K, "MXFP4": JAM.MXFP4}
BLOCK = {"F32": (1, 4), "F16": (1, 2), "BF16": (1, 2), "Q8_0": (32, 34), "Q4_0": (32, 18), "Q4_K": (256, 144),
         "Q5_K": (256, 176), "Q6_K": (256, 210), "MXFP4": (32, 17)}   # elements, bytes


def listed():
    return [
        # the smallest call: one token through a 4096-wide Q8_0 projection
        {"name": "decode_q8_0_4096x4096", "kind": "mm", "dtype": "Q8_0", "m": 4096, "k": 4096, "n": 1, "bias": False},
        # one token through Llama-3-8B's gate or up projection, the library's headline shape
        {"name": "decode_q4_k_14336x4096", "kind": "mm", "dtype": "Q4_K", "m": 14336, "k": 4096, "n": 1, "bias": False},
        # a few tokens at once (several sequences, or drafted tokens being checked) through a down projection
        {"name": "few_q4_0_4096x14336_n4", "kind": "mm", "dtype": "Q4_0", "m": 4096, "k": 14336, "n": 4, "bias": False},
        # batched decode: sixteen sequences' next tokens
        {"name": "batch_q4_k_14336x4096_n16", "kind": "mm", "dtype": "Q4_K", "m": 14336, "k": 4096, "n": 16, "bias": False},
        # a short prompt of odd length through gpt-oss's attention output projection with its bias
        {"name": "prompt_q8_0_2880x4096_n77", "kind": "mm", "dtype": "Q8_0", "m": 2880, "k": 4096, "n": 77, "bias": True},
        # prefill of 512 tokens, the two shapes of Llama-3-8B's FFN in a Q4_K_M file
        {"name": "prefill_q4_k_14336x4096_n512", "kind": "mm", "dtype": "Q4_K", "m": 14336, "k": 4096, "n": 512, "bias": False},
        {"name": "prefill_q6_k_4096x14336_n512", "kind": "mm", "dtype": "Q6_K", "m": 4096, "k": 14336, "n": 512, "bias": False},
        # prefill of an unquantized model
        {"name": "prefill_f16_14336x4096_n512", "kind": "mm", "dtype": "F16", "m": 14336, "k": 4096, "n": 512, "bias": False},
        # the drop-in host call of an engine whose activations live in host memory, one token
        {"name": "host_q4_k_14336x4096", "kind": "host", "dtype": "Q4_K", "m": 14336, "k": 4096, "n": 1},
        # gpt-oss-20B's MoE block: a 512-token prompt, and one token's decode
        {"name": "moe_prompt_512", "kind": "moe", "tokens": 512, "experts": 32, "topk": 4, "dim": 2880, "ff": 2880},
        {"name": "moe_decode_1", "kind": "moe", "tokens": 1, "experts": 32, "topk": 4, "dim": 2880, "ff": 2880},
        # four Llama-3-8B layers and its output head in a Q4_K_M file, one token
        {"name": "step_llama_4_layers", "kind": "step", "tokens": 1, "layers": 4, "dim": 4096, "qkv": 6144, "ff": 14336,
         "vocab": 128256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["mm", "host", "moe", "step"], [12, 1, 3, 2])[0]
    if kind in ("mm", "host"):
        dtype = rng.choice(["Q4_K", "Q6_K", "Q8_0", "Q4_0", "MXFP4", "Q5_K", "F16", "BF16"])
        unit = BLOCK[dtype][0] if BLOCK[dtype][0] > 32 else 32
        k = max(2, _log(rng, 1024, 14336) // unit) * unit
        m = _log(rng, 512, min(28672, 14336 * 4096 // k))
        m -= m % rng.choice([1, 16, 32, 128])   # most tensors have round row counts, views of them may not
        case = {"kind": kind, "dtype": dtype, "m": m, "k": k, "n": _log(rng, 1, 512 if kind == "mm" else 16)}
        if kind == "mm":
            case["bias"] = rng.random() < 0.25
        return case
    if kind == "moe":
        return {"kind": "moe", "tokens": _log(rng, 1, 512), "experts": rng.choice([8, 16, 32]), "topk": rng.choice([2, 4]),
                "dim": 32 * _log(rng, 16, 90), "ff": 32 * _log(rng, 16, 90)}
    heads = rng.choice([4, 8, 16, 32])
    return {"kind": "step", "tokens": _log(rng, 1, 8), "layers": rng.randint(1, 4), "dim": 128 * heads,
            "qkv": 128 * (heads + 2 * max(1, heads // 4)), "ff": 256 * _log(rng, 4, 56), "vocab": _log(rng, 4000, 128256)}


# ------------------------------------------------------------------------------------------ weights
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _half_bytes(x):
    return x.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _scale_min_bytes(sc, mn):   # 6-bit scales and mins of 8 sub-blocks in 12 bytes
    return torch.cat([sc[..., :4] | (sc[..., 4:] >> 4 << 6), mn[..., :4] | (mn[..., 4:] >> 4 << 6),
                      (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], -1)


def _safe_div(a, b):
    return torch.where(b > 0, a / b.clamp_min(1e-30), torch.zeros_like(a))


def _quantize(dtype, x):
    """[m, k] f32 on the GPU -> [m, row bytes] uint8 in the GGUF block layout."""
    m, k = x.shape
    u8 = torch.uint8
    if dtype in ("F32", "F16", "BF16"):
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[dtype]
        return x.to(t).view(u8).reshape(m, -1)
    be = BLOCK[dtype][0]
    b = x.view(m, k // be, be)
    if dtype == "Q8_0":
        d = b.abs().amax(-1) / 127
        q = _safe_div(b, d[..., None]).round().clamp(-127, 127).to(torch.int8).view(u8)
        out = torch.cat([_half_bytes(d), q], -1)
    elif dtype == "Q4_0":
        at = b.abs().argmax(-1, keepdim=True)
        d = b.gather(-1, at)[..., 0] / -8
        q = torch.where(d[..., None] != 0, b / d[..., None] + 8.5, torch.full_like(b, 8)).floor().clamp(0, 15).to(u8)
        out = torch.cat([_half_bytes(d), q[..., :16] | (q[..., 16:] << 4)], -1)
    elif dtype == "MXFP4":
        e = (b.abs().amax(-1).clamp_min(2.0 ** -100).log2().floor() - 2)
        v = b * torch.exp2(-e)[..., None]
        edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=x.device)
        q = torch.bucketize(v.abs().contiguous(), edges).to(u8) | ((v < 0).to(u8) << 3)
        out = torch.cat([(e + 127).to(u8)[..., None], q[..., :16] | (q[..., 16:] << 4)], -1)
    elif dtype in ("Q4_K", "Q5_K"):
        top = 15 if dtype == "Q4_K" else 31
        s = b.reshape(m, k // 256, 8, 32)
        lo = s.amin(-1).clamp_max(0)
        sub, off = (s.amax(-1) - lo) / top, -lo
        d, dmin = (sub.amax(-1) / 63).half(), (off.amax(-1) / 63).half()
        sc = _safe_div(sub, d.float()[..., None]).round().clamp(0, 63)
        mn = _safe_div(off, dmin.float()[..., None]).round().clamp(0, 63)
        ds = (d.float()[..., None] * sc)[..., None]
        q = _safe_div(s + (dmin.float()[..., None] * mn)[..., None], ds).round().clamp(0, top).to(u8)
        low = q & 15
        head = [_half_bytes(d), _half_bytes(dmin), _scale_min_bytes(sc.to(u8), mn.to(u8))]
        if dtype == "Q5_K":
            bit = torch.zeros_like(q[..., 0, :])
            for i in range(8):
                bit |= (q[..., i, :] >> 4) << i
            head.append(bit)
        out = torch.cat(head + [(low[..., 0::2, :] | (low[..., 1::2, :] << 4)).reshape(m, k // 256, 128)], -1)
    else:   # Q6_K
        s = b.reshape(m, k // 256, 16, 16)
        sub = s.abs().amax(-1) / 31
        d = (sub.amax(-1) / 127).half()
        sc = _safe_div(sub, d.float()[..., None]).round().clamp(0, 127)
        q = (_safe_div(s, (d.float()[..., None] * sc)[..., None]).round().clamp(-32, 31) + 32).to(u8)
        q = q.reshape(m, k // 256, 2, 4, 32)   # half, run of 32, element
        ql = torch.cat([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4), (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], -1)
        qh = (q[..., 0, :] >> 4) | ((q[..., 1, :] >> 4) << 2) | ((q[..., 2, :] >> 4) << 4) | ((q[..., 3, :] >> 4) << 6)
        out = torch.cat([ql.flatten(2), qh.flatten(2), sc.to(u8), _half_bytes(d)], -1)
    return out.reshape(m, -1)


def _weight(dtype, m, k, gen, std=0.02):
    return _quantize(dtype, torch.randn((m, k), generator=gen, device="cuda") * std)


def _activations(n, k, gen, outliers):
    """N(0, 1); prompts also hold a few large values, as hidden states of language models do."""
    x = torch.randn((n, k), generator=gen, device="cuda")
    if outliers:
        hit = torch.rand((n, k), generator=gen, device="cuda") < 0.01
        x = torch.where(hit, x.sign() * 20, x)
    return x


# --------------------------------------------------------------------------------------------- state
_JAM = None


def _jam():
    """The program's one context: every state is served by it, in order, on its stream."""
    global _JAM
    if _JAM is None:
        _JAM = HipJAM(0)
    return _JAM


class _Pinned:
    """A weight as the program holds it: GGUF bytes in host memory, resident on the GPU while this lives."""

    def __init__(self, dtype, m, k, raw):
        self.dtype, self.code, self.m, self.k = dtype, CODES[dtype], m, k
        self.host = raw.cpu().numpy()
        self.seg = Segment.of(self.host)
        if _jam().pin(self.seg, self.code, k, m) != JAM.OK:
            raise RuntimeError(_jam().last_error())

    def __del__(self):
        try:
            _jam().evict(self.seg)
        except Exception:
            pass   # the context went first


def _ok(status):
    if status != JAM.OK:
        raise RuntimeError(_jam().last_error())


def _inputs(case, seed):
    """Everything a case starts from, on the GPU: weights as GGUF bytes, activations and biases."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("mm", "host"):
        m, k, n = case["m"], case["k"], case["n"]
        got = {"w": _weight(case["dtype"], m, k, g), "a": _activations(n, k, g, n >= 8)}
        if case.get("bias"):
            got["bias"] = torch.randn(m, generator=g, device="cuda") * 0.5
        return got
    if kind == "moe":
        e, d, ff, n = case["experts"], case["dim"], case["ff"], case["tokens"]
        return {"router": _weight("F32", e, d, g),
                "router_bias": -1.1 * torch.log(torch.arange(1, e + 1, device="cuda", dtype=torch.float32)),   # popularity
                "gate_up": _weight("MXFP4", e * 2 * ff, d, g), "down": _weight("MXFP4", e * d, ff, g),
                "gate_up_bias": torch.randn((e, 2 * ff), generator=g, device="cuda") * 0.1,
                "down_bias": torch.randn((e, d), generator=g, device="cuda") * 0.1,
                "x": _activations(n, d, g, n >= 8)}
    d, ff, L = case["dim"], case["ff"], case["layers"]
    out_std = 0.02 / math.sqrt(2 * L)   # projections into the residual
    got = {"x": _activations(case["tokens"], d, g, False)}
    for i in range(L):
        got["qkv%d" % i] = _weight("Q4_K", case["qkv"], d, g)
        got["o%d" % i] = _weight("Q4_K", d, d, g, out_std)
        got["gate_up%d" % i] = _weight("Q4_K", 2 * ff, d, g)
        got["down%d" % i] = _weight("Q6_K", d, ff, g, out_std / 4)
    got["head"] = _weight("Q6_K", case["vocab"], d, g)
    return got


def prepare(case, seed):
    x = _inputs(case, seed)
    kind, s = case["kind"], {"case": case}
    empty = lambda *shape: torch.empty(shape, dtype=torch.float32, device="cuda")   # noqa: E731
    if kind == "host":
        s["w"] = _Pinned(case["dtype"], case["m"], case["k"], x["w"])
        s["a"] = x["a"].cpu().numpy()
        s["c"] = np.zeros((case["n"], case["m"]), np.float32)
        s["a_seg"], s["c_seg"] = Segment.of(s["a"]), Segment.of(s["c"])
    elif kind == "mm":
        s["w"] = _Pinned(case["dtype"], case["m"], case["k"], x["w"])
        s["a"], s["bias"], s["c"] = x["a"], x.get("bias"), empty(case["n"], case["m"])
    elif kind == "moe":
        e, d, ff, n, topk = (case[v] for v in ("experts", "dim", "ff", "tokens", "topk"))
        i32 = lambda size: torch.zeros(size, dtype=torch.int32, device="cuda")   # noqa: E731
        s["router"] = _Pinned("F32", e, d, x["router"])
        s["gate_up"] = _Pinned("MXFP4", e * 2 * ff, d, x["gate_up"])
        s["down"] = _Pinned("MXFP4", e * d, ff, x["down"])
        for name in ("x", "router_bias", "gate_up_bias", "down_bias"):
            s[name] = x[name]
        s["logits"], s["select"], s["prob"] = empty(n, e), empty(n, e), empty(n * topk)
        s["route_expert"], s["counts"], s["offsets"] = i32(n * topk), i32(e), i32(e + 1)
        s["slot_route"], s["route_slot"] = i32(n * topk), i32(n * topk)
        s["h"], s["y"], s["out"] = empty(n * topk, 2 * ff), empty(n * topk, d), empty(n, d)
    else:
        d, n = case["dim"], case["tokens"]
        for name, raw in x.items():
            if name != "x":
                dtype = "Q6_K" if name.startswith(("down", "head")) else "Q4_K"
                k = case["ff"] if name.startswith("down") else d
                s[name] = _Pinned(dtype, raw.shape[0], k, raw)
        s["embedding"], s["x"], s["qkv"] = x["x"], empty(n, d), empty(n, case["qkv"])
        s["gu"], s["logits"] = empty(n, 2 * case["ff"]), empty(n, case["vocab"])
    s["stream"] = torch.cuda.ExternalStream(_jam().stream())
    torch.cuda.synchronize()   # the inputs were made on torch's own stream
    return s


# ----------------------------------------------------------------------------------------------- run
def _mm(jam, w, a, lda, c, ldc, n, bias=None, accumulate=False):
    if bias is None and not accumulate:
        _ok(jam.mm_device(w.seg, w.code, w.k, a, lda, c, ldc, w.m, n, w.k))
    else:
        _ok(jam.mm_device_ex(w.seg, w.code, w.k, a, lda, c, ldc, w.m, n, w.k, bias, accumulate))


def run(s):
    jam, case = _jam(), s["case"]
    kind = case["kind"]
    if kind == "host":
        w = s["w"]
        _ok(jam.mm_contiguous(w.seg, s["a_seg"], s["c_seg"], w.code, w.m, case["n"], w.k))
        return s["c"]
    if kind == "mm":
        bias = s["bias"].data_ptr() if s["bias"] is not None else None
        _mm(jam, s["w"], s["a"].data_ptr(), case["k"], s["c"].data_ptr(), case["m"], case["n"], bias)
        return s["c"]
    if kind == "moe":
        e, d, ff, n, topk = (case[v] for v in ("experts", "dim", "ff", "tokens", "topk"))
        x, h, counts = s["x"].data_ptr(), s["h"].data_ptr(), s["counts"].data_ptr()
        _mm(jam, s["router"], x, d, s["logits"].data_ptr(), e, n, s["router_bias"].data_ptr())
        with torch.cuda.stream(s["stream"]):
            s["select"].copy_(s["logits"])   # top-k consumes its input
        _ok(jam.moe_select_topk(s["select"].data_ptr(), None, n, e, e, topk, jam.TOPK_SOFTMAX, s["route_expert"].data_ptr(),
                                s["prob"].data_ptr()))
        _ok(jam.moe_route(s["route_expert"].data_ptr(), n, topk, e, counts, s["offsets"].data_ptr(), s["slot_route"].data_ptr(),
                          s["route_slot"].data_ptr()))
        _ok(jam.mm_grouped_gather(s["gate_up"].seg, JAM.MXFP4, d, 2 * ff, e, counts, x, d, s["slot_route"].data_ptr(), topk, h,
                                  2 * ff, d, n * topk, None, s["gate_up_bias"].data_ptr()))
        _ok(jam.glu_device(jam.ACT_SWIGLU_OAI, h, 2 * ff, h + 4 * ff, 2 * ff, n * topk, ff))
        _ok(jam.mm_grouped_ex(s["down"].seg, JAM.MXFP4, ff, d, e, counts, h, 2 * ff, s["y"].data_ptr(), d, ff, n * topk, None,
                              s["down_bias"].data_ptr()))
        _ok(jam.moe_combine(s["y"].data_ptr(), d, s["route_expert"].data_ptr(), s["prob"].data_ptr(), s["route_slot"].data_ptr(),
                            n, topk, e, d, s["out"].data_ptr(), d))
        return {"logits": s["logits"], "out": s["out"]}
    d, ff, n, x, gu = case["dim"], case["ff"], case["tokens"], s["x"].data_ptr(), s["gu"].data_ptr()
    with torch.cuda.stream(s["stream"]):
        s["x"].copy_(s["embedding"])   # the residual stream starts at the token's embedding
    for i in range(case["layers"]):
        _mm(jam, s["qkv%d" % i], x, d, s["qkv"].data_ptr(), case["qkv"], n)
        _mm(jam, s["o%d" % i], s["qkv"].data_ptr(), case["qkv"], x, d, n, accumulate=True)
        _mm(jam, s["gate_up%d" % i], x, d, gu, 2 * ff, n)
        _ok(jam.glu_device(jam.ACT_SWIGLU, gu, 2 * ff, gu + 4 * ff, 2 * ff, n, ff))
        _mm(jam, s["down%d" % i], gu, 2 * ff, x, d, n, accumulate=True)
    _mm(jam, s["head"], x, d, s["logits"].data_ptr(), case["vocab"], n)
    return {"logits": s["logits"], "hidden": s["x"]}


# ----------------------------------------------------------------------------------- work, tolerance
def _bytes(dtype, m, k):
    return m * (k // BLOCK[dtype][0]) * BLOCK[dtype][1]


def work(case):
    """Each weight, input and output once; two operations per multiply-add."""
    if case["kind"] in ("mm", "host"):
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": _bytes(case["dtype"], m, k) + 4 * n * (m + k), "flops": 2 * m * k * n}
    if case["kind"] == "moe":
        e, d, ff, n, topk = (case[v] for v in ("experts", "dim", "ff", "tokens", "topk"))
        busy = min(e, n * topk)
        per_row = 3 * d * ff
        return {"bytes": busy * (_bytes("MXFP4", 2 * ff, d) + _bytes("MXFP4", d, ff)) + 4 * e * d + 8 * n * d,
                "flops": 2 * n * (topk * per_row + e * d)}
    d, ff, n, L, v = (case[x] for x in ("dim", "ff", "tokens", "layers", "vocab"))
    layer = _bytes("Q4_K", case["qkv"] + d + 2 * ff, d) + _bytes("Q6_K", d, ff)
    return {"bytes": L * layer + _bytes("Q6_K", v, d) + 4 * n * (d + v),
            "flops": 2 * n * (L * ((case["qkv"] + d + 2 * ff) * d + d * ff) + v * d)}


def tolerance(case):
    # f32 sums of exact block products: 7e-8 to 6e-7 seen against 64 bits (max 8e-6).
    if case["kind"] in ("mm", "host"):
        return {"rel": 3e-6, "max": 3e-5}
    # Between two matmuls the activations are quantized again, so a last-bit difference moves an int8 code here and
    # there: up to 2e-4 seen (max 6e-3) behind one such step, 1e-2 (max 5e-2) at the end of four layers.
    return {"rel": 1e-3, "max": 2e-2} if case["kind"] == "moe" else {"rel": 5e-2, "max": 2e-1}


# --------------------------------------------------------------------------------------------- exact
def _f64(raw, dtype):
    """(code part [m, k], offset per run [m, k / run], run) in 64 bits: the weight is code part - offset."""
    m = raw.shape[0]
    if dtype in ("F32", "F16", "BF16"):
        t = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[dtype]
        return raw.contiguous().view(t).double(), None, 1
    b = raw.view(m, -1, BLOCK[dtype][1])
    half = lambda at: b[..., at:at + 2].contiguous().view(torch.float16)[..., 0].double()   # noqa: E731
    if dtype == "Q8_0":
        return (half(0)[..., None] * b[..., 2:].contiguous().view(torch.int8).double()).reshape(m, -1), None, 1
    if dtype == "Q4_0":
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).double()
        return (half(0)[..., None] * q).reshape(m, -1), 8 * half(0), 32
    if dtype == "MXFP4":
        values = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12], dtype=torch.float64, device=raw.device)
        values = torch.cat([values, -values])
        q = values[torch.cat([b[..., 1:] & 15, b[..., 1:] >> 4], -1).long()]
        return (torch.exp2(b[..., 0].double() - 128)[..., None] * q).reshape(m, -1), None, 1
    if dtype in ("Q4_K", "Q5_K"):
        s = b[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)], -1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)], -1).double()
        nib = b[..., -128:].reshape(m, -1, 4, 32)
        q = torch.stack([nib & 15, nib >> 4], -2).reshape(m, -1, 8, 32)
        if dtype == "Q5_K":
            q = q | torch.stack([(b[..., 16:48] >> i & 1) << 4 for i in range(8)], -2)
        return ((half(0)[..., None] * sc)[..., None] * q.double()).reshape(m, -1), (half(2)[..., None] * mn).reshape(m, -1), 32
    ql, qh, sc = b[..., :128].reshape(m, -1, 2, 2, 32), b[..., 128:192].reshape(m, -1, 2, 32), b[..., 192:208]
    low = torch.stack([ql[..., 0, :] & 15, ql[..., 1, :] & 15, ql[..., 0, :] >> 4, ql[..., 1, :] >> 4], -2)
    q = (low | torch.stack([(qh >> (2 * i) & 3) << 4 for i in range(4)], -2)).reshape(m, -1, 16, 16).double()
    scale = half(208)[..., None] * sc.contiguous().view(torch.int8).double()
    return (scale[..., None] * q).reshape(m, -1), (32 * scale).reshape(m, -1), 16


def _exact_mm(raw, dtype, x):
    """[n, m] in 64 bits, x [n, k] f32: the operation's int8 activations (per 32 elements; from 8 tokens on the
    weights' offsets meet the unquantized sums, and the last m % 16 rows the unquantized activations)."""
    n, k = x.shape
    code, off, run = _f64(raw, dtype)
    if dtype in ("F32", "F16", "BF16"):
        return (x.bfloat16().double() if dtype == "BF16" else x.double()) @ code.T
    b = x.view(n, k // 32, 32)
    top = b.abs().amax(-1)
    c127 = torch.full_like(top, 127)   # tensor by tensor: torch multiplies by a scalar divisor's reciprocal
    d = top / c127
    inv = torch.where(top > 0, torch.ones_like(d) / d if n < 8 else c127 / top, torch.zeros_like(top))
    q = (b * inv[..., None]).round().clamp(-128, 127)
    xq = (q.double() * d.double()[..., None]).view(n, k)
    sums = lambda v: v.view(n, k // run, run).sum(-1)   # noqa: E731
    out = xq @ code.T
    if off is not None:
        out -= sums(xq if n < 8 else x.double()) @ off.T
    tail = raw.shape[0] % 16
    if n >= 8 and tail:
        out[:, -tail:] = x.double() @ code[-tail:].T - (sums(x.double()) @ off[-tail:].T if off is not None else 0)
    return out


def exact(case, seed):
    x = _inputs(case, seed)
    if case["kind"] in ("mm", "host"):
        out = _exact_mm(x["w"], case["dtype"], x["a"])
        return out + x["bias"].double() if "bias" in x else out
    if case["kind"] == "moe":
        e, d, ff, n, topk = (case[v] for v in ("experts", "dim", "ff", "tokens", "topk"))
        logits = _exact_mm(x["router"], "F32", x["x"]) + x["router_bias"].double()
        top, pick = logits.topk(topk, -1)
        prob = torch.softmax(top, -1)
        out = torch.zeros((n, d), dtype=torch.float64, device="cuda")
        for i in range(e):
            tok, at = (pick == i).nonzero(as_tuple=True)
            if not tok.numel():
                continue
            h = _exact_mm(x["gate_up"][i * 2 * ff:(i + 1) * 2 * ff], "MXFP4", x["x"][tok]) + x["gate_up_bias"][i].double()
            gate, up = h[:, :ff].clamp_max(7), h[:, ff:].clamp(-7, 7)
            act = gate * torch.sigmoid(1.702 * gate) * (up + 1)
            y = _exact_mm(x["down"][i * d:(i + 1) * d], "MXFP4", act.float()) + x["down_bias"][i].double()
            out[tok] += prob[tok, at][:, None] * y
        return {"logits": logits, "out": out}
    if case["layers"] > 1:
        return None   # one moved int8 code spreads through the next layers: which side moves it is chance
    ff, h = case["ff"], x["x"].double()
    for i in range(case["layers"]):
        qkv = _exact_mm(x["qkv%d" % i], "Q4_K", h.float())
        h = h + _exact_mm(x["o%d" % i], "Q4_K", qkv[:, :case["dim"]].float().contiguous())
        gu = _exact_mm(x["gate_up%d" % i], "Q4_K", h.float())
        act = gu[:, :ff] * torch.sigmoid(gu[:, :ff]) * gu[:, ff:]
        h = h + _exact_mm(x["down%d" % i], "Q6_K", act.float())
    return {"logits": _exact_mm(x["head"], "Q6_K", h.float()), "hidden": h}
