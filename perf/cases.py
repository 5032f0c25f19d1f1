"""Workloads of the quantized-linear library, as a program that serves GGUF models makes them.

Four kinds of case, each through the library's public entry points:

  linear   QMatMul::forward (qmm_qmatmul_forward): one weight, `rows` activation rows, every route of it -- a single
           decode row, the few rows of a small decode batch or a speculative step, a prompt's prefill
  layers   the linear layers of some decoder layers at one decode step: q/k/v, o, gate/up, down, each layer with weights
           of its own, so that a pass streams more than the last-level cache holds.  Up to two rows the launches that
           quantize their own input (launch_mmvq_gguf_*_quantize*), above QMatMul::forward and fused_ffn
  ffn      fused_ffn (qmm_fused_ffn): a decoder layer's feed-forward block over a prompt
  moe      the experts block (qmm_moe_forward): the routed decode form at a few tokens, the grouped form above

Weights are N(0, 0.02) quantized to the case's GGUF type, activations N(0, 1), routing the softmax top-k of N(0, 1)
logits.  The handles (weights on the GPU) and the output buffers are what such a program keeps.
"""
import ctypes
import math
import os
import sys

import torch

_PKG = os.path.abspath("inference.rs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import qmm  # noqa: E402

TYPES = {"q4_0": qmm.Q4_0, "q5_0": qmm.Q5_0, "q8_0": qmm.Q8_0, "q4_k": qmm.Q4K, "q5_k": qmm.Q5K, "q6_k": qmm.Q6K}
DTYPES = {"f32": (torch.float32, qmm.F32), "f16": (torch.float16, qmm.F16), "bf16": (torch.bfloat16, qmm.BF16)}


def _weight_bytes(t, n, k):
    return n * k // qmm.BLOCK_SIZE[TYPES[t]] * qmm.TYPE_SIZE[TYPES[t]]


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # an attention output projection at one decode row: the smallest call, where launches and latency count
        dict(name="decode_o_q4k", kind="linear", wtype="q4_k", n=4096, k=4096, rows=1, dtype="f32"),
        # the linear layers of four decoder layers (the Q4_K_M mix: Q6_K for v and down) at one decode row
        dict(name="layers_b1", kind="layers", hidden=4096, kv=1024, inter=14336, layers=4, rows=1),
        # the same at a decode batch of eight sequences
        dict(name="layers_b8", kind="layers", hidden=4096, kv=1024, inter=14336, layers=4, rows=8),
        # an FFN up projection at a decode batch of 16 in bf16
        dict(name="rows16_q4k_bf16", kind="linear", wtype="q4_k", n=14336, k=4096, rows=16, dtype="bf16"),
        # a speculative step's few rows on a Q8_0 model, f16
        dict(name="rows5_q8_0_f16", kind="linear", wtype="q8_0", n=11008, k=4096, rows=5, dtype="f16"),
        # a short prompt on an odd-sized Q5_K weight
        dict(name="rows77_q5k", kind="linear", wtype="q5_k", n=5003, k=2560, rows=77, dtype="f32"),
        # a prompt of 512 tokens: the up projection (Q4_K) and the down projection (Q6_K)
        dict(name="prefill_q4k", kind="linear", wtype="q4_k", n=14336, k=4096, rows=512, dtype="f32"),
        dict(name="prefill_q6k", kind="linear", wtype="q6_k", n=4096, k=14336, rows=512, dtype="f32"),
        # a ragged prompt on a 32-value type, f16
        dict(name="prefill_q4_0_f16", kind="linear", wtype="q4_0", n=8192, k=4096, rows=333, dtype="f16"),
        # the feed-forward block over a prompt of 1024 tokens: the largest call
        dict(name="ffn_1024", kind="ffn", gate="q4_k", down="q6_k", hidden=4096, inter=14336, rows=1024),
        # eight experts, top-2: four tokens (the indexed decode form), 64 tokens (the grouped form)
        dict(name="moe_4tok", kind="moe", gate="q4_k", down="q4_k", experts=8, topk=2, hidden=4096, inter=14336,
             rows=4),
        dict(name="moe_64tok", kind="moe", gate="q4_k", down="q4_k", experts=8, topk=2, hidden=4096, inter=14336,
             rows=64),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "linear", "layers", "ffn", "moe"])
    if kind == "linear":
        t = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q4_0", "q5_0", "q5_k"])
        return dict(kind=kind, wtype=t, n=_log_uniform(rng, 1000, 16384), k=256 * _log_uniform(rng, 4, 56),
                    rows=rng.choice([1, _log_uniform(rng, 2, 32), _log_uniform(rng, 2, 32),
                                     _log_uniform(rng, 33, 1024)]), dtype=rng.choice(["f32", "f16", "bf16"]))
    if kind == "layers":
        hidden = 256 * rng.randint(8, 16)
        return dict(kind=kind, hidden=hidden, kv=hidden // rng.choice([1, 2, 4]),
                    inter=256 * rng.randint(hidden // 128, hidden // 72), layers=rng.randint(2, 4),
                    rows=rng.choice([1, 2, rng.randint(3, 32)]))
    if kind == "ffn":
        return dict(kind=kind, gate=rng.choice(["q4_k", "q8_0", "q6_k"]), down=rng.choice(["q4_k", "q8_0", "q6_k"]),
                    hidden=256 * rng.randint(8, 16), inter=256 * rng.randint(20, 56), rows=_log_uniform(rng, 1, 1024))
    return dict(kind=kind, gate=rng.choice(["q4_k", "q8_0", "q6_k"]), down=rng.choice(["q4_k", "q8_0", "q6_k"]),
                experts=rng.choice([4, 8, 16]), topk=rng.choice([1, 2, 4]), hidden=256 * rng.randint(8, 16),
                inter=256 * rng.randint(6, 24), rows=_log_uniform(rng, 1, 256))


# ------------------------------------------------------------------------------------------------ inputs

def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


def _f16(x):
    return x.to(torch.float16)


def _halves(h):
    """f16 [n] as its two bytes [n, 2]."""
    return h.contiguous().view(torch.uint8).reshape(-1, 2)


def _scales_min(sc, m):
    """The 12 bytes that hold a Q4_K / Q5_K super-block's eight 6-bit scales and mins."""
    out = torch.empty(sc.shape[0], 12, dtype=torch.uint8, device=sc.device)
    out[:, 0:4] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 4:8] = (m[:, :4] | ((m[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 8:12] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
    return out


def _quantize_weight(t, w, values):
    """w [blocks, block size] f32 -> the GGUF blocks of type t (uint8 [blocks, bytes]) and, if asked, their values in
    float64: round-to-nearest on each sub-block's range."""
    val = None
    if t == "q8_0":
        d = _f16(w.abs().amax(1, keepdim=True) / 127)
        q = torch.round(w / d.float().clamp_min(1e-30)).clamp(-127, 127)
        blocks = torch.cat([_halves(d), q.to(torch.int8).view(torch.uint8)], 1)
        if values:
            val = d.double() * q.double()
    elif t in ("q4_0", "q5_0"):
        half = 8 if t == "q4_0" else 16
        big = torch.gather(w, 1, w.abs().argmax(1, keepdim=True))
        d = _f16(big / -half)
        dd = torch.where(d == 0, torch.ones_like(d), d).float()
        q = (torch.round(w / dd) + half).clamp(0, 2 * half - 1).to(torch.int64)
        qs = ((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4)).to(torch.uint8)
        parts = [_halves(d)]
        if t == "q5_0":
            bit = ((q >> 4) << torch.arange(32, device=w.device)).sum(1, keepdim=True)
            parts.append(torch.cat([(bit >> s) & 255 for s in (0, 8, 16, 24)], 1).to(torch.uint8))
        blocks = torch.cat(parts + [qs], 1)
        if values:
            val = d.double() * (q - half).double()
    elif t in ("q4_k", "q5_k"):
        top = 15 if t == "q4_k" else 31
        s = w.reshape(-1, 8, 32)
        low = (-s.amin(2)).clamp_min(0)
        scale = (s.amax(2) + low) / top
        d, dmin = _f16(scale.amax(1, keepdim=True) / 63), _f16(low.amax(1, keepdim=True) / 63)
        sc = torch.round(scale / d.float().clamp_min(1e-30)).clamp(0, 63)
        m = torch.round(low / dmin.float().clamp_min(1e-30)).clamp(0, 63)
        step, off = (d.float() * sc)[:, :, None], (dmin.float() * m)[:, :, None]
        q = torch.round((s + off) / step.clamp_min(1e-30)).clamp(0, top).to(torch.uint8)
        lo, hi = q[:, 0::2, :], q[:, 1::2, :]
        qs = ((lo & 15) | ((hi & 15) << 4)).reshape(-1, 128)
        parts = [_halves(d), _halves(dmin), _scales_min(sc.to(torch.int64), m.to(torch.int64))]
        if t == "q5_k":
            qh = torch.zeros(s.shape[0], 32, dtype=torch.uint8, device=w.device)
            for j in range(8):
                qh |= (q[:, j, :] >> 4) << j
            parts.append(qh)
        blocks = torch.cat(parts + [qs], 1)
        if values:
            val = (d.double() * sc.double())[:, :, None] * q.double() - (dmin.double() * m.double())[:, :, None]
            val = val.reshape(-1, 256)
    else:  # q6_k
        s = w.reshape(-1, 16, 16)
        scale = s.abs().amax(2) / 31
        d = _f16(scale.amax(1, keepdim=True) / 127)
        sc = torch.round(scale / d.float().clamp_min(1e-30)).clamp(-128, 127)
        q = torch.round(s / (d.float() * sc)[:, :, None].clamp_min(1e-30)).clamp(-32, 31).to(torch.int64)
        u = (q + 32).to(torch.uint8).reshape(-1, 2, 4, 32)  # half, quarter, value
        ql = torch.cat([(u[:, :, 0] & 15) | ((u[:, :, 2] & 15) << 4), (u[:, :, 1] & 15) | ((u[:, :, 3] & 15) << 4)], 2)
        qh = (u[:, :, 0] >> 4) | ((u[:, :, 1] >> 4) << 2) | ((u[:, :, 2] >> 4) << 4) | ((u[:, :, 3] >> 4) << 6)
        blocks = torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _halves(d)],
                           1)
        if values:
            val = ((d.double() * sc.double())[:, :, None] * q.double()).reshape(-1, 256)
    return blocks, val


def _weight(t, n, k, seed, salt, values=False):
    """The blocks of an [n, k] weight (and its values), made in pieces of whole rows to bound the scratch memory."""
    g = _gen(seed, salt)
    bs = qmm.BLOCK_SIZE[TYPES[t]]
    blocks, vals = [], []
    step = max(1, (1 << 26) // k)
    for r0 in range(0, n, step):
        rows = min(step, n - r0)
        w = torch.randn(rows * k // bs, bs, device="cuda", generator=g) * 0.02
        b, v = _quantize_weight(t, w, values)
        blocks.append(b.reshape(-1))
        vals.append(v)
    return torch.cat(blocks), torch.cat(vals).reshape(n, k) if values else None


def _acts(rows, k, dtype, seed, salt):
    return torch.randn(rows, k, device="cuda", generator=_gen(seed, salt)).to(DTYPES[dtype][0])


def _routing(case, seed):
    logits = torch.randn(case["rows"], case["experts"], device="cuda", generator=_gen(seed, 900))
    p, ids = torch.topk(torch.softmax(logits, 1), case["topk"], dim=1)
    return ids.to(torch.int32).contiguous(), (p / p.sum(1, keepdim=True)).contiguous()


class _Tensor:
    """A QTensor handle of the host layer, freed with its owner."""

    def __init__(self, t, n, k, blocks, experts=1):
        data = blocks.cpu()
        self.handle = ctypes.c_void_p()
        _check(qmm.host().qmm_qtensor_from_data(TYPES[t], data.data_ptr(), data.numel(), experts, n, k, 0,
                                                ctypes.byref(self.handle)))
        self.ptr = qmm.host().qmm_qtensor_device_ptr(self.handle)

    def __del__(self):
        if self.handle:
            qmm.host().qmm_qtensor_free(self.handle)


class _Moe:
    def __init__(self, gate, up, down):
        self.weights = (gate, up, down)
        self.handle = ctypes.c_void_p()
        _check(qmm.host().qmm_moe_new(gate.handle, up.handle, down.handle, 0, ctypes.byref(self.handle)))

    def __del__(self):
        if self.handle:
            qmm.host().qmm_moe_free(self.handle)


def _host():
    h = qmm.host()
    h.qmm_fused_ffn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int64, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p]
    return h


def _check(rc):
    if rc != 0:
        raise RuntimeError(qmm.host().qmm_host_last_error().decode())


# a layer's projections: name, weight type, output and input width
def _projections(c):
    h, kv, f = c["hidden"], c["kv"], c["inter"]
    return (("q", "q4_k", h, h), ("k", "q4_k", kv, h), ("v", "q6_k", kv, h), ("o", "q4_k", h, h),
            ("gate", "q4_k", f, h), ("up", "q4_k", f, h), ("down", "q6_k", h, f))


def _experts(t, n, k, experts, seed, salt):
    return torch.cat([_weight(t, n, k, seed, salt + e)[0] for e in range(experts)])


def prepare(case, seed):
    H, L = _host(), qmm.lib()
    kind, rows = case["kind"], case["rows"]
    st = {"keep": [], "calls": [], "out": []}

    def empty(n, dtype="f32"):
        t = torch.empty(rows, n, device="cuda", dtype=DTYPES[dtype][0])
        st["keep"].append(t)
        return t

    if kind == "linear":
        w = _Tensor(case["wtype"], case["n"], case["k"], _weight(case["wtype"], case["n"], case["k"], seed, 1)[0])
        x, y = _acts(rows, case["k"], case["dtype"], seed, 500), empty(case["n"], case["dtype"])
        st["keep"] += [w, x]
        st["calls"].append((H.qmm_qmatmul_forward, (w.handle, x.data_ptr(), DTYPES[case["dtype"]][1], rows,
                                                    y.data_ptr())))
        st["out"].append(y)
    elif kind == "layers":
        h, kv, f = case["hidden"], case["kv"], case["inter"]
        xa, xo, xf = (_acts(rows, h, "f32", seed, 500 + i) for i in range(3))
        st["keep"] += [xa, xo, xf]
        for layer in range(case["layers"]):
            w = {name: _Tensor(t, n, k, _weight(t, n, k, seed, 10 * layer + i)[0])
                 for i, (name, t, n, k) in enumerate(_projections(case))}
            st["keep"].append(w)
            q, k_, v, o, d = empty(h), empty(kv), empty(kv), empty(h), empty(h)
            st["out"] += [q, k_, v, o]
            if rows <= 2:  # the launches that quantize their own input
                mid = empty(f)
                st["out"].append(mid)
                st["calls"] += [
                    (L.launch_mmvq_gguf_q4_k_q6_k_f32_fused_qkv_quantize,
                     (w["q"].ptr, w["k"].ptr, w["v"].ptr, xa.data_ptr(), q.data_ptr(), k_.data_ptr(), v.data_ptr(), h,
                      h, kv, kv, h, rows)),
                    (L.launch_mmvq_gguf_q4_k_f32_quantize_plain,
                     (w["o"].ptr, xo.data_ptr(), o.data_ptr(), h, h, h, h, rows)),
                    (L.launch_mmvq_gguf_q4_k_f32_fused_glu_quantize,
                     (w["gate"].ptr, w["up"].ptr, xf.data_ptr(), mid.data_ptr(), h, f, h, f, rows, 0))]
                if rows == 1:
                    st["calls"].append((L.launch_mmvq_gguf_q6_k_f32_quantize_plain,
                                        (w["down"].ptr, mid.data_ptr(), d.data_ptr(), f, h, f, h, 1)))
                else:
                    st["calls"].append((H.qmm_qmatmul_forward, (w["down"].handle, mid.data_ptr(), 0, rows,
                                                                d.data_ptr())))
            else:
                for name, x, y in (("q", xa, q), ("k", xa, k_), ("v", xa, v), ("o", xo, o)):
                    st["calls"].append((H.qmm_qmatmul_forward, (w[name].handle, x.data_ptr(), 0, rows, y.data_ptr())))
                st["calls"].append((H.qmm_fused_ffn, (w["gate"].handle, w["up"].handle, w["down"].handle,
                                                      xf.data_ptr(), rows, 0, d.data_ptr())))
            st["out"].append(d)
    elif kind == "ffn":
        h, f = case["hidden"], case["inter"]
        g, u, d = (_Tensor(t, n, k, _weight(t, n, k, seed, i)[0])
                   for i, (t, n, k) in enumerate(((case["gate"], f, h), (case["gate"], f, h), (case["down"], h, f))))
        x, y = _acts(rows, h, "f32", seed, 500), empty(h)
        st["keep"] += [g, u, d, x]
        st["calls"].append((H.qmm_fused_ffn, (g.handle, u.handle, d.handle, x.data_ptr(), rows, 0, y.data_ptr())))
        st["out"].append(y)
    else:
        h, f, e = case["hidden"], case["inter"], case["experts"]
        ws = [_Tensor(t, n, k, _experts(t, n, k, e, seed, 100 * i), e)
              for i, (t, n, k) in enumerate(((case["gate"], f, h), (case["gate"], f, h), (case["down"], h, f)))]
        moe = _Moe(*ws)
        ids, p = _routing(case, seed)
        x, y = _acts(rows, h, "f32", seed, 500), empty(h)
        st["keep"] += [moe, ids, p, x]
        st["moe"] = (moe.handle, x.data_ptr(), rows, ids.data_ptr(), p.data_ptr(), case["topk"], y.data_ptr())
        st["out"].append(y)
    return st


def run(state):
    stream = torch.cuda.current_stream().cuda_stream
    if "moe" in state:
        _check(qmm.host().qmm_moe_forward(*state["moe"], stream, 0))
    for fn, args in state["calls"]:
        if fn(*args, stream):  # 0, or None from the launchers, whose errors are read once below
            raise RuntimeError(qmm.host().qmm_host_last_error().decode())
    qmm.check()
    return state["out"]


# ------------------------------------------------------------------------------------------------ work and tolerance

def work(case):
    kind, m = case["kind"], case["rows"]
    if kind == "linear":
        n, k, e = case["n"], case["k"], DTYPES[case["dtype"]][0].itemsize
        return {"bytes": _weight_bytes(case["wtype"], n, k) + m * (n + k) * e, "flops": 2 * m * n * k}
    if kind == "layers":
        p, h, f = _projections(case), case["hidden"], case["inter"]
        acts = 3 * h + sum(n for _, _, n, _ in p if n != f) + (f if m <= 2 else 0)
        return {"bytes": case["layers"] * (sum(_weight_bytes(t, n, k) for _, t, n, k in p) + 4 * m * acts),
                "flops": case["layers"] * sum(2 * m * n * k for _, _, n, k in p)}
    h, f = case["hidden"], case["inter"]
    per = 2 * _weight_bytes(case["gate"], f, h) + _weight_bytes(case["down"], h, f)
    if kind == "ffn":
        return {"bytes": per + 8 * m * h, "flops": 6 * m * h * f}
    e, topk = case["experts"], min(case["topk"], case["experts"])
    used = e * (1 - (1 - topk / e) ** m)  # experts that some token is routed to, on average
    return {"bytes": int(used * per) + 8 * m * h + 8 * m * topk, "flops": 6 * m * topk * h * f}


def tolerance(case):
    # about four times the distance measured to `exact`: 0.8 to 2e-7 for f32 outputs (sums of up to 14336 products in
    # f32), 2.1e-4 and 1.7e-3 for f16 and bf16 (the output's own rounding); 0.6 to 3e-4 where an intermediate is quantized
    # to 8 bits again, since a few of its values land on the other side of a rounding step
    if case["kind"] == "linear":
        return {"rel": {"f32": 1e-6, "f16": 8e-4, "bf16": 7e-3}[case["dtype"]]}
    return {"rel": 1.2e-3}


# ------------------------------------------------------------------------------------------------ 64-bit results

def _round_away(p):
    return torch.where(p < 0, -torch.floor(0.5 - p), torch.floor(0.5 + p))


def _quantize_acts(t, x):
    """The activations x [rows, k] as the type's dot product reads them, in float64: Q8_0 blocks of 32 for the 32-value
    types, Q8_K blocks of 256 for the super-block types.  The roundings to 8 bits are the format's: every step one f32
    operation (the divisions in float64 and then rounded, which gives f32's own result)."""
    x = x.float()
    rows, k = x.shape
    if qmm.BLOCK_SIZE[TYPES[t]] == 32:
        b = x.reshape(-1, 32)
        d = (b.abs().amax(1, keepdim=True).double() / 127).float()
        inv = torch.where(d > 0, (1 / d.double()).float(), torch.zeros_like(d))
        return (_round_away((b * inv).double()) * d.half().double()).reshape(rows, k)
    b = torch.nn.functional.pad(x, (0, -k % 256)).reshape(-1, 256)
    a, at = b.abs(), torch.arange(256, device=b.device)
    first = torch.where(a == a.amax(1, keepdim=True), at, 256).amin(1, keepdim=True)  # the first of largest magnitude
    big = torch.gather(b, 1, first)
    inv = torch.where(big != 0, (-127 / big.double()).float(), torch.zeros_like(big))
    q = _round_away((b * inv).double()).clamp(-128, 127)
    d = torch.where(big != 0, (1 / inv.double()).float(), torch.zeros_like(big))
    return (q * d.double()).reshape(rows, -1)[:, :k]


def _matmul(t, x, w):
    return _quantize_acts(t, x) @ w.t()


def _glu(t_gate, t_down, x, g, u, d):
    xq = _quantize_acts(t_gate, x)
    gate = xq @ g.t()
    mid = gate / (1 + torch.exp(-gate)) * (xq @ u.t())
    return mid, _matmul(t_down, mid, d)


def exact(case, seed):
    kind, rows = case["kind"], case["rows"]
    if kind == "linear":
        t = case["wtype"]
        w = _weight(t, case["n"], case["k"], seed, 1, True)[1]
        return [_matmul(t, _acts(rows, case["k"], case["dtype"], seed, 500), w)]
    if kind == "layers":
        h = case["hidden"]
        xa, xo, xf = (_acts(rows, h, "f32", seed, 500 + i) for i in range(3))
        out = []
        for layer in range(case["layers"]):
            w = {name: _weight(t, n, k, seed, 10 * layer + i, True)[1]
                 for i, (name, t, n, k) in enumerate(_projections(case))}
            out += [_matmul("q4_k", xa, w["q"]), _matmul("q4_k", xa, w["k"]), _matmul("q6_k", xa, w["v"]),
                    _matmul("q4_k", xo, w["o"])]
            mid, d = _glu("q4_k", "q6_k", xf, w["gate"], w["up"], w["down"])
            out += [mid, d] if rows <= 2 else [d]
        return out
    h, f = case["hidden"], case["inter"]
    shapes = ((case["gate"], f, h), (case["gate"], f, h), (case["down"], h, f))
    x = _acts(rows, h, "f32", seed, 500)
    if kind == "ffn":
        g, u, d = (_weight(t, n, k, seed, i, True)[1] for i, (t, n, k) in enumerate(shapes))
        return [_glu(case["gate"], case["down"], x, g, u, d)[1]]
    ids, p = _routing(case, seed)
    out = torch.zeros(rows, h, device="cuda", dtype=torch.float64)
    for e in range(case["experts"]):
        tok, slot = torch.nonzero(ids == e, as_tuple=True)
        if tok.numel() == 0:
            continue
        g, u, d = (_weight(t, n, k, seed, 100 * i + e, True)[1] for i, (t, n, k) in enumerate(shapes))
        y = _glu(case["gate"], case["down"], x[tok], g, u, d)[1]
        out.index_add_(0, tok, y * p[tok, slot].double()[:, None])
    return [out]
