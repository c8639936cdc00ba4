"""The work that a user of libqwhip has it do, as cases to time.

Every case is a chain of the library's own doors as a serving program calls them, on the library's stream, over weights that were
quantized once and buffers that such a program keeps:

- `block`: the quantized part of a dense transformer block: embedding gather, norm, q/k/v projection, output projection of the
  attention's rows (attention itself is not the library's), norm with residual, gate|up with its gated activation, down.  One row is a
  decode step, 2 to 16 rows a verify window of speculative decoding (the GEMV doors), more rows are prefill (the GEMM doors).
- `moe`: a mixture-of-experts layer: norm, router, expert choice, routed gate|up and down projections, weighted sum, with or without a
  shared expert.  Up to 8 rows take the routed GEMV doors, more rows the sorted, grouped GEMM doors, as `qw::QWMoEOperator` decides.
- `head`: final norm, vocabulary projection, argmax.
- `f32`: a projection of fp32 activations (the f32 operator family), with its rotation.
- `load`: what happens once per weight matrix when a checkpoint is loaded: quantize, or repack of an affine checkpoint.
"""
from __future__ import annotations

import ctypes as C
import math

import torch

from qwegn_amd import qwhip

EPS = 1e-6
VOCAB_ROWS = 8192                # rows of the embedding table that a block case keeps
PLANES = 64 << 20                # bytes of GEMM workspace behind the activation copy (what the library's split-K planes may take)

# container: (kind, bits, group); the names are those of the tests and of bench.py
FORMATS = {
    "hq4_g32_m5": (qwhip.KIND_HQ4_G32_M5, 4, 32),
    "hq4_g64": (qwhip.KIND_ROTATED_HQ, 4, 64), "hq4_g128": (qwhip.KIND_ROTATED_HQ, 4, 128),
    "hq8_g32": (qwhip.KIND_ROTATED_HQ, 8, 32), "hq8_g64": (qwhip.KIND_ROTATED_HQ, 8, 64),
    "hq6_g32": (qwhip.KIND_ROTATED_HQ, 6, 32), "hq3_g32": (qwhip.KIND_ROTATED_HQ, 3, 32),
    "aq4_g32": (qwhip.KIND_NATIVE_AFFINE, 4, 32), "aq4_g64": (qwhip.KIND_NATIVE_AFFINE, 4, 64),
    "aq8_g64": (qwhip.KIND_NATIVE_AFFINE, 8, 64), "aq6_g64": (qwhip.KIND_NATIVE_AFFINE, 6, 64),
    "aq2_g64": (qwhip.KIND_NATIVE_AFFINE, 2, 64),
}


def listed():
    m5 = "hq4_g32_m5"
    return [
        # a token of a small dense model: short blocks, where launches and latency count
        {"name": "decode_small", "kind": "block", "rows": 1, "layers": 4, "hidden": 2048, "qkv": 3072, "inter": 6144,
         "attn": m5, "up": m5, "down": m5, "x": "f16"},
        # a token of a 27B-class dense model on the default container (the shapes of the benchmark's decode and MLP workloads)
        {"name": "decode_dense", "kind": "block", "rows": 1, "layers": 1, "hidden": 5120, "qkv": 7168, "inter": 17408,
         "attn": m5, "up": m5, "down": m5, "x": "f16"},
        # a verify window of four draft tokens on the mixed containers of the benchmark's small-M configuration
        {"name": "verify_mixed", "kind": "block", "rows": 4, "layers": 1, "hidden": 5120, "qkv": 7168, "inter": 17408,
         "attn": "hq8_g32", "up": m5, "down": "hq4_g64", "x": "f16"},
        # the widest verify window, on a checkpoint in the standard basis (4-bit affine, 8-bit attention)
        {"name": "verify_wide", "kind": "block", "rows": 16, "layers": 1, "hidden": 4096, "qkv": 6144, "inter": 12288,
         "attn": "aq8_g64", "up": "aq4_g64", "down": "aq4_g64", "x": "bf16"},
        # a short prompt of odd length on a mixed-width checkpoint
        {"name": "prefill_ragged", "kind": "block", "rows": 333, "layers": 1, "hidden": 2560, "qkv": 3584, "inter": 9728,
         "attn": "hq6_g32", "up": "hq3_g32", "down": "hq4_g64", "x": "bf16"},
        # a long prompt on the 27B-class model: the largest call
        {"name": "prefill_dense", "kind": "block", "rows": 4096, "layers": 1, "hidden": 5120, "qkv": 7168, "inter": 17408,
         "attn": m5, "up": m5, "down": m5, "x": "bf16"},
        # a token of an A3B-style mixture of experts
        {"name": "moe_decode", "kind": "moe", "rows": 1, "layers": 4, "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8, "shared": 0, "fmt": m5},
        # four draft tokens on an affine 4-bit mixture with a shared expert
        {"name": "moe_verify", "kind": "moe", "rows": 4, "layers": 2, "hidden": 2048, "inter": 512, "experts": 256, "top_k": 8, "shared": 512,
         "fmt": "aq4_g64"},
        # a long prompt through the mixture
        {"name": "moe_prefill", "kind": "moe", "rows": 2048, "layers": 1, "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8, "shared": 0, "fmt": m5},
        # the vocabulary projection of one token
        {"name": "head", "kind": "head", "rows": 1, "hidden": 5120, "vocab": 151936, "fmt": m5},
        # fp32 activations, four rows
        {"name": "f32_rows", "kind": "f32", "rows": 4, "n": 17408, "k": 5120, "fmt": m5, "epi": 0},
        # one matrix of a bf16 checkpoint quantized at load time
        {"name": "load", "kind": "load", "op": "quantize", "n": 17408, "k": 5120, "fmt": m5},
    ]


def _log(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step) * step))


def _enough(case):
    """Decode and verify passes over small layers take up to four of them: a model's next layer is not in the caches."""
    if case["rows"] <= 16:
        case["layers"] = max(1, min(4, round(9e7 / work(case)["bytes"])))
    return case


def _draw(rng):
    pick = rng.random()
    default = rng.random() < 0.4                      # the default container throughout
    fmt = lambda: "hq4_g32_m5" if default else rng.choice(sorted(FORMATS))  # noqa: E731
    if pick < 0.6:
        rows = 1 if pick < 0.2 else rng.randint(2, 16) if pick < 0.4 else _log(rng, 17, 4096, 1)
        hidden = _log(rng, 1024, 6144, 256)
        inter = round(hidden * rng.uniform(1.5, 4.0) / 128) * 128
        return _enough({"kind": "block", "rows": rows, "layers": 1, "hidden": hidden, "qkv": hidden + 256 * rng.randint(1, 8), "inter": inter,
                        "attn": fmt(), "up": fmt(), "down": fmt(), "x": rng.choice(["f16", "bf16"])})
    if pick < 0.85:
        rows = 1 if pick < 0.67 else rng.randint(2, 8) if pick < 0.73 else _log(rng, 9, 2048, 1)
        experts = rng.choice([16, 32, 64, 128, 256])
        return _enough({"kind": "moe", "rows": rows, "layers": 1, "hidden": _log(rng, 1024, 4096, 256),
                        "inter": _log(rng, 384, min(1536, 196608 // experts), 128), "experts": experts, "top_k": rng.choice([2, 4, 6, 8]),
                        "shared": rng.choice([0, 0, 512, 1024]), "fmt": fmt()})
    if pick < 0.90:
        return {"kind": "head", "rows": rng.choice([1, 1, rng.randint(2, 16)]), "hidden": _log(rng, 1024, 5120, 256),
                "vocab": _log(rng, 32000, 151936, 1), "fmt": fmt()}
    if pick < 0.95:
        return {"kind": "f32", "rows": _log(rng, 1, 256, 1), "n": _log(rng, 1024, 17408, 32), "k": _log(rng, 1024, 8192, 128),
                "fmt": fmt(), "epi": rng.choice([0, 1, 3])}
    op = rng.choice(["quantize", "repack"])
    return {"kind": "load", "op": op, "n": _log(rng, 1024, 34816, 1), "k": _log(rng, 1024, 8192, 256),
            "fmt": rng.choice(["aq4_g32", "aq4_g64", "aq8_g64", "aq6_g64", "aq2_g64"]) if op == "repack" else fmt()}


def draw(rng):
    most = max((work(c) for c in listed()), key=lambda w: w["flops"])
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= most["flops"] and w["bytes"] <= 4 * most["bytes"]:
            return case


# ---- what the cases are made of ---------------------------------------------------------------------------------------------


_DEVICE = []


def _device():
    """The program's one device and stream."""
    if not _DEVICE:
        _DEVICE.append(qwhip.Device(0))
    return _DEVICE[0]


def _rotated(fmt):
    return FORMATS[fmt][0] != qwhip.KIND_NATIVE_AFFINE


def _bank_bytes(fmt, n, k):
    _, bits, group = FORMATS[fmt]
    return n * (k // group) * (4 + group * bits // 8)


class _Maker:
    """Inputs from one seed, and banks quantized by the library."""

    def __init__(self, seed):
        self.dev = _device()
        self.lib, self.stream = self.dev.lib, self.dev.stream.handle
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.keep = []

    def randn(self, *shape, dtype=torch.float16, std=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=dtype)
        return x.mul_(std) if std != 1.0 else x

    def rows(self, m, k, dtype=torch.float16):
        """Activations N(0, 1) with 0.1 % outliers twenty times as large."""
        x = self.randn(m, k, dtype=torch.float32)
        x[torch.rand((m, k), generator=self.g, device="cuda") < 0.001] *= 20.0
        return x.to(dtype)

    def empty(self, *shape, dtype=torch.float16):
        return torch.zeros(shape, device="cuda", dtype=dtype)

    def bank(self, fmt, n, k):
        """(view, blocks) of N(0, 0.02) weights [n, k]."""
        kind, bits, group = FORMATS[fmt]
        blocks = torch.empty(_bank_bytes(fmt, n, k), device="cuda", dtype=torch.uint8)
        step = max(1, (1 << 28) // k)
        for r in range(0, n, step):
            m = min(step, n - r)
            src = self.randn(m, k, dtype=torch.bfloat16, std=0.02)
            torch.cuda.synchronize()
            self._quantize(fmt, src, m, k, blocks.data_ptr() + _bank_bytes(fmt, r, k))
            self.dev.stream.sync()
        view = qwhip.WeightView(blocks.data_ptr(), blocks.numel(), n, k, kind, bits, group)
        self.keep += [blocks, view]
        return C.byref(view)

    def _quantize(self, fmt, src, n, k, out):
        _, bits, group = FORMATS[fmt]
        rot = 1 if _rotated(fmt) else 0
        if fmt == "hq4_g32_m5":
            qwhip.check(self.lib.qwhip_quantize_hq4_g32(self.stream, src.data_ptr(), qwhip.BF16, n, k, rot, out))
        else:
            qwhip.check(self.lib.qwhip_quantize_blocks(self.stream, src.data_ptr(), qwhip.BF16, n, k, bits, group, rot, 2, out))


def _dt(t):
    return {torch.float16: qwhip.F16, torch.bfloat16: qwhip.BF16, torch.float32: qwhip.F32}[t.dtype]


def _state(mk, calls, out):
    """A list of doors with their arguments, the buffers behind them, and what the pass computes."""
    torch.cuda.synchronize()
    return {"calls": [(getattr(mk.lib, name), args) for name, *args in calls], "out": out, "keep": mk.keep}


def _block(c, mk):
    m, h, qkv, inter = c["rows"], c["hidden"], c["qkv"], c["inter"]
    s, x_dtype = mk.stream, torch.bfloat16 if c["x"] == "bf16" else torch.float16
    table = mk.bank("aq8_g64", VOCAB_ROWS, h)
    tokens = torch.randint(0, VOCAB_ROWS, (m,), generator=mk.g, device="cuda", dtype=torch.int32)
    e32, res = mk.empty(m, h, dtype=torch.float32), mk.empty(m, h)
    xn, xn2, o, act, mlp = mk.empty(m, h), mk.empty(m, h), mk.empty(m, h), mk.empty(m, inter), mk.empty(m, h)
    mk.keep += [tokens, e32, xn, xn2, o, act]
    pre_attn, pre_up, pre_down = (qwhip.X_PREROTATED if _rotated(c[k]) else 0 for k in ("attn", "up", "down"))
    decode = m <= 16
    ws = None if decode else mk.empty(m * max(h, inter) + PLANES // 2)
    mk.keep.append(ws)
    calls = [("qwhip_embed_aq_f32", s, table, tokens.data_ptr(), m, 1, e32.data_ptr()),
             ("qwhip_cast_f32_to_f16", s, e32.data_ptr(), res.data_ptr(), m * h)]

    def project(w, x, flags, y, n):
        if decode:
            return ("qwhip_gemv", s, w, x.data_ptr(), _dt(x), m, flags, y.data_ptr(), None)
        return ("qwhip_gemm", s, w, x.data_ptr(), _dt(x), m, 0, y.data_ptr(), qwhip.F16, 0, flags, ws.data_ptr(), ws.numel() * 2)

    qkvs = []
    for layer in range(c["layers"]):
        wq, wo = mk.bank(c["attn"], qkv, h), mk.bank(c["attn"], h, h)
        wu, wd = mk.bank(c["up"], 2 * inter, h), mk.bank(c["down"], h, inter)
        g1, g2 = mk.randn(h, std=0.1), mk.randn(h, std=0.1)
        attn, q = mk.rows(m, h, x_dtype), mk.empty(m, qkv)
        mk.keep += [g1, g2, attn]
        qkvs.append(q)
        first = layer == 0
        calls.append(("qwhip_rmsnorm", s, (res if first else mlp).data_ptr(), g1.data_ptr(), None if first else res.data_ptr(), m, h, EPS,
                      1 if pre_attn else 0, xn.data_ptr()))
        calls.append(project(wq, xn, pre_attn, q, qkv))
        calls.append(project(wo, attn, 0, o, h))          # the attention's rows are not in the rotated basis: the door rotates them
        calls.append(("qwhip_rmsnorm", s, o.data_ptr(), g2.data_ptr(), res.data_ptr(), m, h, EPS, 1 if pre_up else 0, xn2.data_ptr()))
        if decode:
            # one row: the header's advice, the activation stays plain and the down projection rotates its input itself
            rot_act = 1 if pre_down and m > 1 else 0
            calls.append(("qwhip_gemv_silu_pair", s, wu, xn2.data_ptr(), qwhip.F16, m, pre_up, rot_act, act.data_ptr()))
            calls.append(project(wd, act, pre_down if m > 1 else 0, mlp, h))
        else:
            calls.append(("qwhip_gemm_swiglu", s, wu, xn2.data_ptr(), qwhip.F16, m, 0, 1 if pre_down else 0, act.data_ptr(), 0, pre_up,
                          ws.data_ptr(), ws.numel() * 2))
            calls.append(project(wd, act, pre_down, mlp, h))
    return _state(mk, calls, {"qkv": qkvs, "attn_out": o, "mlp": mlp, "residual": res})


def _moe(c, mk):
    calls, outs = [], []
    for _ in range(c["layers"]):
        outs.append(_moe_layer(c, mk, calls))
    return _state(mk, calls, outs)


def _moe_layer(c, mk, calls):
    m, h, inter, e, k, fmt, sh = c["rows"], c["hidden"], c["inter"], c["experts"], c["top_k"], c["fmt"], c["shared"]
    s, rot, pairs = mk.stream, _rotated(fmt), m * k
    pre = qwhip.X_PREROTATED if rot else 0
    f32, i32 = torch.float32, torch.int32
    x, gamma, wr = mk.rows(m, h), mk.randn(h, std=0.1), mk.randn(e, h, dtype=torch.bfloat16, std=h ** -0.5)
    wgu, wdn = mk.bank(fmt, e * 2 * inter, h), mk.bank(fmt, e * h, inter)
    xn, plain, logits = mk.empty(m, h), mk.empty(m, h, dtype=f32), mk.empty(m, e, dtype=f32)
    idx, wts, act = mk.empty(m, k, dtype=i32), mk.empty(m, k, dtype=f32), mk.empty(pairs, inter)
    out = mk.empty(m, h)
    mk.keep += [x, gamma, wr, xn, plain, logits, act]
    calls.append(("qwhip_rmsnorm", s, x.data_ptr(), gamma.data_ptr(), None, m, h, EPS, 1 if rot else 0, xn.data_ptr()))
    xr = xn
    if rot:                                               # the router reads the rows in the standard basis
        calls.append(("qwhip_moe_bridge_f16_to_f32", s, xn.data_ptr(), None, plain.data_ptr(), m, h))
        xr = plain
    shared, gate = None, None
    if sh:
        gw, gate_t, sh32 = mk.randn(h, dtype=f32, std=h ** -0.5), mk.empty(m, dtype=f32), mk.empty(m, h, dtype=f32)
        wsu, wsd, sact = mk.bank(fmt, 2 * sh, h), mk.bank(fmt, h, sh), mk.empty(m, sh)
        mk.keep += [gw, gate_t, sh32, sact]
        shared, gate = sh32.data_ptr(), gate_t.data_ptr()
        calls.append(("qwhip_router_gemm_shared_gate", s, xr.data_ptr(), _dt(xr), wr.data_ptr(), qwhip.BF16, m, e, h, logits.data_ptr(),
                      gw.data_ptr(), gate))
        if m <= 16:
            rot_act = 1 if rot and m > 1 else 0
            calls.append(("qwhip_gemv_silu_pair", s, wsu, xn.data_ptr(), qwhip.F16, m, pre, rot_act, sact.data_ptr()))
            calls.append(("qwhip_gemv", s, wsd, sact.data_ptr(), qwhip.F16, m, pre if m > 1 else 0, None, shared))
        else:
            ws = mk.empty(m * max(h, sh) + PLANES // 2)
            mk.keep.append(ws)
            calls.append(("qwhip_gemm_swiglu", s, wsu, xn.data_ptr(), qwhip.F16, m, 0, 1 if rot else 0, sact.data_ptr(), 0, pre, ws.data_ptr(),
                          ws.numel() * 2))
            calls.append(("qwhip_gemm", s, wsd, sact.data_ptr(), qwhip.F16, m, 0, shared, qwhip.F32, 0, pre, ws.data_ptr(), ws.numel() * 2))
    else:
        calls.append(("qwhip_router_gemm", s, xr.data_ptr(), _dt(xr), wr.data_ptr(), qwhip.BF16, m, e, h, logits.data_ptr()))
    if m <= 8:
        calls.append(("qwhip_moe_route_gateup_decode", s, wgu, e, xn.data_ptr(), qwhip.F16, pre, logits.data_ptr(), m, k, 1, 1.0, idx.data_ptr(),
                      wts.data_ptr(), act.data_ptr()))
        calls.append(("qwhip_moe_down_decode", s, wdn, e, act.data_ptr(), idx.data_ptr(), wts.data_ptr(), m, k, shared, gate, out.data_ptr(),
                      qwhip.F16))
    else:
        tiles = max(1, mk.lib.qwhip_moe_max_tiles(e, pairs))
        off, sp, tok, inv = (mk.empty(n, dtype=i32) for n in (e + 1, pairs, pairs, pairs))
        te, tr, tc = (mk.empty(n, dtype=i32) for n in (tiles, tiles, 1))
        dn = mk.empty(pairs, h)
        mk.keep += [off, sp, tok, inv, te, tr, tc, dn]
        plan = (off.data_ptr(), te.data_ptr(), tr.data_ptr(), tc.data_ptr(), tiles, pairs)
        calls += [
            ("qwhip_moe_route", s, logits.data_ptr(), m, e, k, 1, 1.0, idx.data_ptr(), wts.data_ptr()),
            ("qwhip_moe_group_pairs", s, idx.data_ptr(), e, pairs, k, off.data_ptr(), sp.data_ptr(), tok.data_ptr(), inv.data_ptr(), te.data_ptr(),
             tr.data_ptr(), tc.data_ptr(), 1),
            ("qwhip_moe_grouped_gemm_swiglu", s, wgu, e, xn.data_ptr(), qwhip.F16, 0, tok.data_ptr(), *plan, 1 if rot else 0, act.data_ptr(), 0),
            ("qwhip_moe_grouped_gemm", s, wdn, e, act.data_ptr(), qwhip.F16, 0, None, *plan, dn.data_ptr(), qwhip.F16, 0),
            ("qwhip_moe_combine", s, dn.data_ptr(), qwhip.F16, inv.data_ptr(), wts.data_ptr(), m, k, h, shared, gate, out.data_ptr(), qwhip.F16)]
    return {"out": out, "experts": idx, "weights": wts}


def _head(c, mk):
    m, h, n, s, rot = c["rows"], c["hidden"], c["vocab"], mk.stream, _rotated(c["fmt"])
    x, gamma, xn = mk.rows(m, h), mk.randn(h, std=0.1), mk.empty(m, h)
    w = mk.bank(c["fmt"], n, h)
    logits, tokens = mk.empty(m, n, dtype=torch.float32), mk.empty(m, dtype=torch.int32)
    mk.keep += [x, gamma, xn]
    return _state(mk, [("qwhip_rmsnorm", s, x.data_ptr(), gamma.data_ptr(), None, m, h, EPS, 1 if rot else 0, xn.data_ptr()),
                       ("qwhip_head_argmax", s, w, xn.data_ptr(), qwhip.F16, m, qwhip.X_PREROTATED if rot else 0, logits.data_ptr(),
                        tokens.data_ptr())], {"logits": logits, "tokens": tokens})


def _f32(c, mk):
    m, n, k, s = c["rows"], c["n"], c["k"], mk.stream
    x, y = mk.rows(m, k, torch.float32), mk.empty(m, n, dtype=torch.float32)
    w, calls, xr = mk.bank(c["fmt"], n, k), [], x
    if _rotated(c["fmt"]):
        xr = mk.empty(m, k, dtype=torch.float32)
        calls.append(("qwhip_h32_f32", s, x.data_ptr(), xr.data_ptr(), m, k))
    calls.append(("qwhip_gemv_f32", s, w, xr.data_ptr(), m, c["epi"], 1.0, y.data_ptr()))
    mk.keep += [x, xr]
    return _state(mk, calls, {"y": y})


def _load(c, mk):
    n, k, s = c["n"], c["k"], mk.stream
    _, bits, group = FORMATS[c["fmt"]]
    blocks = torch.zeros(_bank_bytes(c["fmt"], n, k), device="cuda", dtype=torch.uint8)
    if c["op"] == "quantize":
        src = mk.randn(n, k, dtype=torch.bfloat16, std=0.02)
        mk.keep.append(src)
        rot = 1 if _rotated(c["fmt"]) else 0
        if c["fmt"] == "hq4_g32_m5":
            call = ("qwhip_quantize_hq4_g32", s, src.data_ptr(), qwhip.BF16, n, k, rot, blocks.data_ptr())
        else:
            call = ("qwhip_quantize_blocks", s, src.data_ptr(), qwhip.BF16, n, k, bits, group, rot, 2, blocks.data_ptr())
        return _state(mk, [call], {"blocks": blocks})
    codes = torch.randint(0, 256, (n * k * bits // 8,), generator=mk.g, device="cuda", dtype=torch.uint8)
    scale = (torch.rand(n * k // group, generator=mk.g, device="cuda") * 0.05 + 1e-3).to(torch.bfloat16)
    bias = (-torch.rand(n * k // group, generator=mk.g, device="cuda") * 0.3 - 1e-2).to(torch.bfloat16)
    refused = mk.empty(1, dtype=torch.int32)
    mk.keep += [codes, scale, bias]
    return _state(mk, [("qwhip_repack_mlx_affine", s, codes.data_ptr(), scale.data_ptr(), bias.data_ptr(), qwhip.BF16, n, k, bits, group,
                        blocks.data_ptr(), refused.data_ptr())], {"blocks": blocks, "refused": refused})


_PREPARE = {"block": _block, "moe": _moe, "head": _head, "f32": _f32, "load": _load}


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, _Maker(seed))


def run(state):
    for door, args in state["calls"]:
        qwhip.check(door(*args))
    return state["out"]


def work(case):
    """Weights, inputs and outputs once each; two operations for each weight and row."""
    c = case
    if c["kind"] == "block":
        m, h, qkv, inter = c["rows"], c["hidden"], c["qkv"], c["inter"]
        weights = _bank_bytes(c["attn"], qkv + h, h) + _bank_bytes(c["up"], 2 * inter, h) + _bank_bytes(c["down"], h, inter)
        layer = weights + m * (h + qkv) * 2 + 4 * h
        # per pass: the embedding rows in; the output projection, the block's output and the residual out
        return {"bytes": c["layers"] * layer + m * (_bank_bytes("aq8_g64", 1, h) + 3 * h * 2),
                "flops": c["layers"] * 2 * m * ((qkv + h) * h + 3 * inter * h)}
    if c["kind"] == "moe":
        m, h, inter, e, k, sh = c["rows"], c["hidden"], c["inter"], c["experts"], c["top_k"], c["shared"]
        used = e * (1 - (1 - k / e) ** m)                 # experts that some row takes
        size = lambda width: _bank_bytes(c["fmt"], 2 * width, h) + _bank_bytes(c["fmt"], h, width)  # noqa: E731
        return {"bytes": c["layers"] * (used * size(inter) + (size(sh) + 4 * h if sh else 0) + e * h * 2 + m * (4 * h + 8 * k) + 2 * h),
                "flops": c["layers"] * 2 * m * (3 * h * (k * inter + sh) + e * h)}
    if c["kind"] == "head":
        return {"bytes": _bank_bytes(c["fmt"], c["vocab"], c["hidden"]) + c["rows"] * (2 * c["hidden"] + 4 * c["vocab"] + 4) + 2 * c["hidden"],
                "flops": 2 * c["rows"] * c["vocab"] * c["hidden"]}
    if c["kind"] == "f32":
        return {"bytes": _bank_bytes(c["fmt"], c["n"], c["k"]) + 4 * c["rows"] * (c["k"] + c["n"]), "flops": 2 * c["rows"] * c["n"] * c["k"]}
    _, bits, group = FORMATS[c["fmt"]]
    blocks = _bank_bytes(c["fmt"], c["n"], c["k"])
    return {"bytes": blocks + (2 * c["n"] * c["k"] if c["op"] == "quantize" else blocks), "flops": 0}


def tolerance(case):
    """About four times what the chain measured against itself in 64 bits on the same f16 weights."""
    if case["kind"] == "load":
        return "exact"                                    # the blocks are the packer's bytes
    if case["kind"] == "f32":
        return {"rel": 1e-5}                              # fp32 sums of up to 8192 products
    if case["kind"] == "head":
        return {"rel": 1.2e-3, "differ": 0.002}           # 2.8e-4: the f16 rounding of the normed row
    if case["kind"] == "block":
        return {"rel": 4e-3}                              # up to 1.1e-3: an f16 rounding after each of a block's six steps
    if case["rows"] <= 8:
        return {"rel": 2.5e-3, "differ": 0.002}           # 6.4e-4
    # an expert at the edge of the top-k may change with the last bits of the normed row, and that row's output with it:
    # 0.2 % of the choices, 1.4e-2 over all rows and 1.2 in the largest difference against 64 bits; 5e-4 where no choice changes
    return {"rel": 1e-2, "max": 0.99, "differ": 0.005}
