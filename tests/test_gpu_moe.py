"""GPU parity of the MoE pieces (router, routing, pair sort + tile list, grouped GEMM, combine, decode
GEMVs) and of the whole routed block against the CPU oracle, through the C ABI."""
import ctypes as C

import numpy as np
import pytest

from oracle import qworacle as qo
from qwegn_amd import qwhip
from tests import helpers as H

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.fixture(scope="module")
def dev():
    return qwhip.Device(0)


def _route(dev, logits, k, norm=True, scale=1.0):
    t, e = logits.shape
    lb, ib, wb = dev.put(logits.astype(np.float32)), dev.alloc(t * k * 4), dev.alloc(t * k * 4)
    qwhip.check(dev.lib.qwhip_moe_route(dev.stream.handle, lb.ptr, t, e, k, 1 if norm else 0, scale, ib.ptr, wb.ptr))
    return ib.download(np.int32, (t, k)), wb.download(np.float32, (t, k))


@pytest.mark.parametrize("t,e,k", [(64, 128, 8), (5, 8, 2), (33, 512, 16), (7, 100, 3)])
def test_moe_route_matches_oracle(dev, t, e, k):
    rng = np.random.default_rng(e + k)
    logits = rng.standard_normal((t, e)).astype(np.float32)
    idx, wts = _route(dev, logits, k, norm=True, scale=2.5)
    ridx, rwts = qo.moe_route(logits, k, norm_topk=True, routed_scale=2.5)
    assert np.array_equal(idx, ridx)
    np.testing.assert_allclose(wts, rwts, rtol=2e-6, atol=1e-9)
    idx2, wts2 = _route(dev, logits, k, norm=False)
    ridx2, rwts2 = qo.moe_route(logits, k, norm_topk=False)
    assert np.array_equal(idx2, ridx2)
    np.testing.assert_allclose(wts2, rwts2, rtol=2e-6, atol=1e-9)


def test_moe_route_ties_and_non_finite(dev):
    logits = np.zeros((3, 64), dtype=np.float32)          # all tied: lowest indices win, in order
    logits[1, 10] = np.inf                                 # non-finite never wins
    logits[1, 11] = np.nan
    logits[2, :] = -np.inf                                 # nothing to select
    logits[2, 5] = 1.0
    idx, wts = _route(dev, logits, 4)
    assert idx[0].tolist() == [0, 1, 2, 3]
    assert 10 not in idx[1] and 11 not in idx[1] and idx[1].tolist() == [0, 1, 2, 3]
    assert idx[2].tolist() == [5, -1, -1, -1]
    assert wts[2].tolist() == [1.0, 0.0, 0.0, 0.0]
    np.testing.assert_allclose(wts[0], 0.25, rtol=1e-6)


# one to eight experts a lane, the last lanes without one; a single expert; a full last lane
@pytest.mark.parametrize("e", [1, 63, 64, 65, 128, 129, 256, 257, 511])
def test_route_edges_of_the_expert_count(dev, e):
    """Rows of ties, of one candidate, of none, of the lowest finite logits and of infinities: ids and weights as the oracle's; the fused
    projection, whose later row blocks stop at their own rank, leaves the same ids, weights and activations."""
    k, hidden, inter = min(e, 8), 256, 96
    rng = np.random.default_rng(e)
    logits = rng.standard_normal((8, e)).astype(np.float32)
    logits[1] = 0.25
    logits[2, : e - 1] = np.nan
    logits[3] = -np.inf
    logits[4] = -np.finfo(np.float32).max
    logits[4, e // 2] = -3.0e38
    logits[5, ::2] = np.inf
    logits[6, e - 1] = np.finfo(np.float32).max
    logits[7] = np.round(logits[7] * 2)              # ties between some
    idx, wts = _route(dev, logits, k, scale=1.5)
    with np.errstate(over="ignore"):
        ridx, rwts = qo.moe_route(logits, k, True, 1.5)
    assert np.array_equal(idx, ridx)
    np.testing.assert_allclose(wts, rwts, rtol=2e-6, atol=1e-9)
    lib, st = dev.lib, dev.stream.handle
    blocks, _, _, _ = _moe_banks(e, hidden, inter, seed=3, fmt="hq4_g32")
    bank, xb, lb = dev.put(blocks), dev.put(rng.standard_normal((8, hidden)).astype(np.float16)), dev.put(logits)
    view = H.view_of(dev, bank, "hq4_g32", e * 2 * inter, hidden)
    ib, wb, ab, a2 = dev.alloc(8 * k * 4 + 256), dev.alloc(8 * k * 4 + 256), dev.alloc(8 * k * inter * 2), dev.alloc(8 * k * inter * 2)
    qwhip.check(lib.qwhip_moe_route_gateup_decode(st, C.byref(view), e, xb.ptr, qwhip.F16, 0, lb.ptr, 8, k, 1, 1.5, ib.ptr, wb.ptr, ab.ptr))
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(view), e, xb.ptr, qwhip.F16, 0, ib.ptr, 8, k, a2.ptr))
    dev.stream.sync()
    assert np.array_equal(ib.download(np.int32, (8, k)), idx)
    assert np.array_equal(wb.download(np.uint32, (8, k)), wts.view(np.uint32))
    assert np.array_equal(ab.download(np.uint16, (8, k, inter)), a2.download(np.uint16, (8, k, inter)))


@pytest.mark.parametrize("xdt", ["f32", "bf16", "f16"])
def test_router_gemm(dev, xdt):
    t, e, h = 19, 128, 2048
    rng = np.random.default_rng(1)
    x = rng.standard_normal((t, h)).astype(np.float32)
    wr = (rng.standard_normal((e, h)) * 0.05).astype(np.float32)
    if xdt == "f32":
        xh, code, xv = x, qwhip.F32, x
    elif xdt == "bf16":
        xh, code, xv = qo.f32_to_bf16_bits(x), qwhip.BF16, qo.round_bf16(x)
    else:
        xh, code = x.astype(np.float16), qwhip.F16
        xv = xh.astype(np.float32)
    xb, wb, lb = dev.put(xh), dev.put(wr), dev.alloc(t * e * 4)
    qwhip.check(dev.lib.qwhip_router_gemm(dev.stream.handle, xb.ptr, code, wb.ptr, qwhip.F32, t, e, h, lb.ptr))
    got = lb.download(np.float32, (t, e))
    ref = xv.astype(np.float64) @ wr.astype(np.float64).T
    assert qo.normalized_error(got, ref) <= 1e-5


@pytest.mark.parametrize("t,e,h,wdt", [(19, 128, 2048, "f32"), (5, 64, 4096, "bf16"), (33, 40, 5120, "f32"), (3, 8, 16384, "f16")])
def test_router_gemm_shared_gate_and_wide_rows(dev, t, e, h, wdt):
    """The shared-expert gate column sigmoid(x . w) beside the logits, on hidden sizes up to the largest; the logits are those of
    the plain door bit for bit."""
    rng = np.random.default_rng(4)
    x = rng.standard_normal((t, h)).astype(np.float32)
    wr = (rng.standard_normal((e, h)) * 0.05).astype(np.float32)
    shw = (rng.standard_normal(h) * 0.03).astype(np.float32)
    if wdt == "f32":
        wh, wcode, wv = wr, qwhip.F32, wr
    elif wdt == "bf16":
        wh, wcode, wv = qo.f32_to_bf16_bits(wr), qwhip.BF16, qo.round_bf16(wr)
    else:
        wh, wcode = wr.astype(np.float16), qwhip.F16
        wv = wh.astype(np.float32)
    xb, wb, sb = dev.put(x), dev.put(wh), dev.put(shw)
    l1, l2, go = dev.alloc(t * e * 4), dev.alloc(t * e * 4), dev.alloc(t * 4)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_router_gemm_shared_gate(st, xb.ptr, qwhip.F32, wb.ptr, wcode, t, e, h, l1.ptr, sb.ptr, go.ptr))
    qwhip.check(lib.qwhip_router_gemm(st, xb.ptr, qwhip.F32, wb.ptr, wcode, t, e, h, l2.ptr))
    dev.stream.sync()
    got, plain, gate = l1.download(np.float32, (t, e)), l2.download(np.float32, (t, e)), go.download(np.float32, (t,))
    assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))
    assert qo.normalized_error(got, x.astype(np.float64) @ wv.astype(np.float64).T) <= 1e-5
    np.testing.assert_allclose(gate, qo.router_shared_gate_f64(x, shw), rtol=0, atol=2e-6)
    assert lib.qwhip_router_gemm_shared_gate(st, xb.ptr, qwhip.F32, wb.ptr, wcode, t, e, h, l1.ptr, sb.ptr, None) == qwhip.E_NULL
    assert lib.qwhip_router_gemm(st, xb.ptr, qwhip.F32, wb.ptr, wcode, t, e, 16388, l1.ptr) == qwhip.E_BAD_SHAPE


@pytest.mark.parametrize("xdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("wdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("t,e,h", [(1, 1, 32), (1, 65, 2080), (2, 16, 64), (16, 17, 2048), (17, 33, 1056), (300, 130, 544), (1025, 257, 96)])
def test_router_gemm_tiles(dev, t, e, h, xdt, wdt):
    """One row, the edges of the 16-row tiles, both tile widths and hidden sizes that leave a wave without a chunk, with the gate
    column.  Every product and sum is fp32 (bf16 products hold all bits of the activations).  A chain has at most 40 terms at
    h = 2080; roundings of 2^-24 that fall either way leave sqrt(40) 2^-24 = 4e-7 of the result, and the bar is five times that
    (all the same way they would leave 40 2^-24 = 2.4e-6)."""
    rng = np.random.default_rng(t + e + h)
    cast = {"f32": (lambda v: (v, qwhip.F32, v)), "f16": (lambda v: (v.astype(np.float16), qwhip.F16, v.astype(np.float16).astype(np.float32))),
            "bf16": (lambda v: (qo.f32_to_bf16_bits(v), qwhip.BF16, qo.round_bf16(v)))}
    xh, xcode, xv = cast[xdt](rng.standard_normal((t, h)).astype(np.float32))
    wh, wcode, wv = cast[wdt]((rng.standard_normal((e, h)) * 0.05).astype(np.float32))
    shw = (rng.standard_normal(h) * 0.03).astype(np.float32)
    xb, wb, sb = dev.put(xh), dev.put(wh), dev.put(shw)
    lb, go = dev.alloc(t * e * 4), dev.alloc(t * 4)
    qwhip.check(dev.lib.qwhip_router_gemm_shared_gate(dev.stream.handle, xb.ptr, xcode, wb.ptr, wcode, t, e, h, lb.ptr, sb.ptr, go.ptr))
    got, gate = lb.download(np.float32, (t, e)), go.download(np.float32, (t,))
    assert qo.normalized_error(got, xv.astype(np.float64) @ wv.astype(np.float64).T) <= 2e-6
    np.testing.assert_allclose(gate, qo.router_shared_gate_f64(xv, shw), rtol=0, atol=2e-6)
    for b in (xb, wb, sb, lb, go):
        b.free()


def _router_operands(rng, t, e, h, xdt, wdt):
    cast = {"f32": (lambda v: (v, qwhip.F32, v)), "f16": (lambda v: (v.astype(np.float16), qwhip.F16, v.astype(np.float16).astype(np.float32))),
            "bf16": (lambda v: (qo.f32_to_bf16_bits(v), qwhip.BF16, qo.round_bf16(v)))}
    return cast[xdt](rng.standard_normal((t, h)).astype(np.float32)), cast[wdt]((rng.standard_normal((e, h)) * 0.05).astype(np.float32))


@pytest.mark.parametrize("xdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("wdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("t,e,h", [(2048, 128, 2048), (1025, 257, 1056), (1024, 161, 2080)])
def test_router_gemm_trips_of_the_wide_tile(dev, t, e, h, xdt, wdt):
    """From 160 tiles of 64 weight rows on: whole trips of the unrolled loop, a trip that ends early, a second one; same bar as above."""
    (xh, xcode, xv), (wh, wcode, wv) = _router_operands(np.random.default_rng(e), t, e, h, xdt, wdt)
    xb, wb, lb = dev.put(xh), dev.put(wh), dev.alloc(t * e * 4)
    qwhip.check(dev.lib.qwhip_router_gemm(dev.stream.handle, xb.ptr, xcode, wb.ptr, wcode, t, e, h, lb.ptr))
    assert qo.normalized_error(lb.download(np.float32, (t, e)), xv.astype(np.float64) @ wv.astype(np.float64).T) <= 2e-6
    for b in (xb, wb, lb):
        b.free()


@pytest.mark.parametrize("xdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("wdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("t", [1, 2, 3, 9])
@pytest.mark.parametrize("h,skew", [(100, 0), (1000, 0), (1056, 1)])
def test_router_gemm_of_any_hidden_size_and_alignment(dev, h, skew, t, xdt, wdt):
    """Hidden sizes that are no multiple of 32 and rows that begin one element past a 16-byte boundary, in tiles of one to eight token
    rows, with the gate; chains of up to 17 terms a lane, 64 lanes."""
    e = 37
    rng = np.random.default_rng(h + t)
    (xh, xcode, xv), (wh, wcode, wv) = _router_operands(rng, t, e, h, xdt, wdt)
    shw = (rng.standard_normal(h) * 0.03).astype(np.float32)
    put = lambda a: dev.put(np.concatenate([np.zeros(skew, a.dtype), a.ravel()]))  # noqa: E731
    xb, wb, sb, lb, gb = put(xh), put(wh), put(shw), dev.alloc(t * e * 4), dev.alloc(t * 4)
    qwhip.check(dev.lib.qwhip_router_gemm_shared_gate(dev.stream.handle, xb.ptr + skew * xh.itemsize, xcode, wb.ptr + skew * wh.itemsize, wcode, t, e, h,
                                                      lb.ptr, sb.ptr + 4 * skew, gb.ptr))
    assert qo.normalized_error(lb.download(np.float32, (t, e)), xv.astype(np.float64) @ wv.astype(np.float64).T) <= 2e-6
    np.testing.assert_allclose(gb.download(np.float32, (t,)), qo.router_shared_gate_f64(xv, shw), rtol=0, atol=2e-6)
    for b in (xb, wb, sb, lb, gb):
        b.free()


@pytest.mark.parametrize("xdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("wdt", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("h", [96, 100, 1056, 2048])
def test_router_rows_do_not_depend_on_the_call(dev, h, xdt, wdt):
    """A token's logits and gate bit for bit: alone, in windows of 2 to 17 rows, in a prefill that takes the wide tile (65 x 5 tiles of 64
    weight rows), with fewer experts beside it, and wherever the gate's weights begin."""
    rng = np.random.default_rng(h)
    t, e = 1025, 257
    cast = {"f32": (lambda v: (v.astype(np.float32), qwhip.F32, 4)), "f16": (lambda v: (v.astype(np.float16), qwhip.F16, 2)),
            "bf16": (lambda v: (qo.f32_to_bf16_bits(v.astype(np.float32)), qwhip.BF16, 2))}
    xh, xcode, xs = cast[xdt](rng.standard_normal((t, h)))
    wh, wcode, _ = cast[wdt](rng.standard_normal((e, h)) * 0.05)
    sb = dev.put(np.concatenate([[7.0], rng.standard_normal(h) * 0.03, np.zeros(8)]).astype(np.float32))
    xb, wb, lb, gb = dev.put(xh), dev.put(wh), dev.alloc(t * e * 4), dev.alloc(t * 4)

    def run(row, n, experts, skew):
        # the gate's weights from element 1 on, moved to a 16-byte boundary unless `skew`
        gate = sb.ptr + 4
        if not skew:
            qwhip.check(dev.lib.qwhip_memcpy_d2d(dev.stream.handle, ab.ptr, gate, h * 4))
            gate = ab.ptr
        qwhip.check(dev.lib.qwhip_router_gemm_shared_gate(dev.stream.handle, xb.ptr + row * h * xs, xcode, wb.ptr, wcode, n, experts, h, lb.ptr, gate, gb.ptr))
        return lb.download(np.uint32, (n, experts)), gb.download(np.uint32, (n,))

    ab = dev.alloc(h * 4)
    want, gate = run(0, t, e, False)
    for row, n, experts, skew in [(0, 1, e, False), (700, 1, e, True), (1, 2, e, False), (9, 3, e, True), (40, 4, e, False), (1019, 5, e, False),
                                  (16, 17, e, True), (0, t, 20, False), (0, t, e, True), (3, 1, 1, False)]:
        if xdt != "f32" and h % 8 != 0 and row % 2:
            continue   # f16 rows of 100 columns begin at other boundaries
        got, g = run(row, n, experts, skew)
        assert np.array_equal(got, want[row : row + n, :experts]), (row, n, experts, skew)
        assert np.array_equal(g, gate[row : row + n]), (row, n, experts, skew)
    for b in (xb, wb, sb, ab, lb, gb):
        b.free()


@pytest.mark.parametrize("t,e,k", [(33, 128, 8), (5, 40, 4), (9, 512, 16), (7, 100, 3)])
@pytest.mark.parametrize("mode", ["bias", "split", "bias+split", "softmax+scale"])
@pytest.mark.parametrize("norm", [0, 1])
def test_route_modes_match_oracle(dev, t, e, k, mode, norm):
    """qwhip_moe_route_ex: sigmoid scoring with a selection bias and / or split-feature logits, and the per-expert scale;
    the choice is the oracle's exactly (ties and non-finite logits included), the weights within 2e-6."""
    rng = np.random.default_rng(t * 7 + e)
    split = "split" in mode
    lg = rng.standard_normal((t, 2 * e if split else e)).astype(np.float32)
    lg[0, 1] = lg[0, 0]                                        # a tie
    lg[t - 1, 2] = np.nan
    lg[t - 1, 3] = -np.inf
    bias = (rng.standard_normal(e) * 0.5).astype(np.float32) if "bias" in mode else None
    scale = (rng.random(e) + 0.5).astype(np.float32) if "scale" in mode else None
    lb, ib, wb = dev.put(lg), dev.alloc(t * k * 4), dev.alloc(t * k * 4)
    bb = dev.put(bias) if bias is not None else None
    sb = dev.put(scale) if scale is not None else None
    qwhip.check(dev.lib.qwhip_moe_route_ex(dev.stream.handle, lb.ptr, t, e, k, norm, 1.5, 1 if split else 0, bb.ptr if bb else None,
                                           sb.ptr if sb else None, ib.ptr, wb.ptr))
    dev.stream.sync()
    idx, wts = ib.download(np.int32, (t, k)), wb.download(np.float32, (t, k))
    ridx, rwts = qo.moe_route_ex(lg, k, bool(norm), 1.5, bias=bias, split_feature=split, scale_param=scale)
    assert np.array_equal(idx, ridx)
    np.testing.assert_allclose(wts, rwts, rtol=2e-6, atol=1e-9)


def _group(dev, ids, experts, top_k, compact=True):
    pairs = ids.size
    mt = max(1, dev.lib.qwhip_moe_max_tiles(experts, pairs))
    b = dict(ids=dev.put(ids.astype(np.int32)), off=dev.alloc((experts + 1) * 4), sp=dev.alloc(pairs * 4), stok=dev.alloc(pairs * 4),
             inv=dev.alloc(pairs * 4), te=dev.alloc(mt * 4), tr=dev.alloc(mt * 4), tc=dev.alloc(16))
    qwhip.check(dev.lib.qwhip_moe_group_pairs(dev.stream.handle, b["ids"].ptr, experts, pairs, top_k, b["off"].ptr, b["sp"].ptr,
                                              b["stok"].ptr, b["inv"].ptr, b["te"].ptr, b["tr"].ptr, b["tc"].ptr, 1 if compact else 0))
    dev.stream.sync()
    out = dict(off=b["off"].download(np.int32, (experts + 1,)), sp=b["sp"].download(np.int32, (pairs,)),
               stok=b["stok"].download(np.int32, (pairs,)), inv=b["inv"].download(np.int32, (pairs,)),
               tc=int(b["tc"].download(np.int32, (1,))[0]))
    out["te"] = b["te"].download(np.int32, (mt,))[: out["tc"]]
    out["tr"] = b["tr"].download(np.int32, (mt,))[: out["tc"]]
    out["bufs"], out["max_tiles"] = b, mt
    return out


@pytest.mark.parametrize("t,e,k,compact", [(300, 128, 8, True), (300, 128, 8, False), (3, 16, 2, True), (2048, 128, 8, True), (50, 512, 16, True)])
def test_moe_group_pairs_invariants_and_tiles(dev, t, e, k, compact):
    """Sort invariants (Tests/QWFlashNextMetalTests/MoE/FNMetalMoEGroupTests.swift:80-92) and the tile list
    against the closed forms of QWGemmMoE.swift:24-62 / qw_moe_tile.metalh."""
    rng = np.random.default_rng(t + e)
    ids = np.stack([rng.choice(e, size=k, replace=False) for _ in range(t)]).astype(np.int32)
    ids[rng.random(ids.shape) < 0.02] = -1                     # a few empty routes
    g = _group(dev, ids, e, k, compact)
    ref = qo.moe_group_pairs(ids, e, k, compact_tail=compact)
    valid = int((ids >= 0).sum())
    assert g["off"][0] == 0 and g["off"][e] == valid and np.all(np.diff(g["off"]) >= 0)
    assert np.array_equal(g["off"], ref["expertOff"])
    sp = g["sp"][:valid]
    assert np.array_equal(np.sort(sp), np.flatnonzero(ids.ravel() >= 0))           # each valid pair exactly once
    assert np.array_equal(g["stok"][:valid], sp // k)
    assert np.array_equal(g["inv"][sp], np.arange(valid))                           # invPerm o sortedPairIdx = id
    assert np.all(g["inv"][ids.ravel() < 0] == -1)
    flat = ids.ravel()
    for ex in range(e):                                                             # slots of expert ex hold its pairs
        assert np.all(flat[sp[g["off"][ex]:g["off"][ex + 1]]] == ex)
    assert g["tc"] == ref["tileCount"] <= g["max_tiles"]
    assert np.array_equal(g["te"], ref["tileE"]) and np.array_equal(g["tr"], ref["tileR"])


def _moe_banks(experts, hidden, inter, seed, fmt="hq4_g32_m5"):
    gu_blocks, gu16 = H.make_bank(fmt, experts * 2 * inter, hidden, seed)
    dn_blocks, dn16 = H.make_bank(fmt, experts * hidden, inter, seed + 1)
    return gu_blocks, gu16.reshape(experts, 2 * inter, hidden), dn_blocks, dn16.reshape(experts, hidden, inter)


def _hidden_rows(rng, t, hidden, xdt):
    """Hidden rows in the experts' basis as the device takes them (f16 values, or bf16 bit patterns), their dtype code, and
    the values they hold."""
    x32 = rng.standard_normal((t, hidden)).astype(np.float32)
    if xdt == "f16":
        xh = qo.rotate_activation_f16(x32)
        return xh, qwhip.F16, xh.astype(np.float32)
    bits = qo.f32_to_bf16_bits(qo.fwht32_ortho(x32))
    return bits, qwhip.BF16, qo.bf16_bits_to_f32(bits)


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
@pytest.mark.parametrize("t,experts,hidden,inter,k", [(40, 8, 256, 128, 2), (130, 16, 512, 192, 4)])
def test_moe_prefill_chain_matches_oracle(dev, t, experts, hidden, inter, k, xdt):
    """route -> pair sort -> grouped gate_up GEMM -> SwiGLU+FWHT -> grouped down GEMM -> combine; f16 and bf16 hidden rows."""
    fmt = "hq4_g32_m5"
    gu_blocks, gu16, dn_blocks, dn16 = _moe_banks(experts, hidden, inter, seed=11)
    rng = np.random.default_rng(5)
    x16, xcode, xval = _hidden_rows(rng, t, hidden, xdt)                                     # rotated hidden rows
    logits = rng.standard_normal((t, experts)).astype(np.float32)
    idx, wts = _route(dev, logits, k)
    g = _group(dev, idx, experts, k)
    pairs = t * k
    lib, st, b = dev.lib, dev.stream.handle, g["bufs"]
    gub, dnb, xb = dev.put(gu_blocks), dev.put(dn_blocks), dev.put(x16)
    gu_out, act, dn_out, out = dev.alloc(pairs * 2 * inter * 2), dev.alloc(pairs * inter * 2), dev.alloc(pairs * hidden * 4), dev.alloc(t * hidden * 4)
    wb = dev.put(wts)
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    vdn = H.view_of(dev, dnb, fmt, experts * hidden, inter)
    qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vgu), experts, xb.ptr, xcode, 0, b["stok"].ptr, b["off"].ptr, b["te"].ptr,
                                           b["tr"].ptr, b["tc"].ptr, g["max_tiles"], pairs, gu_out.ptr, qwhip.F16, 0))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu_out.ptr, qwhip.F16, act.ptr, pairs, inter, 1))
    qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vdn), experts, act.ptr, qwhip.F16, 0, None, b["off"].ptr, b["te"].ptr,
                                           b["tr"].ptr, b["tc"].ptr, g["max_tiles"], pairs, dn_out.ptr, qwhip.F32, 0))
    qwhip.check(lib.qwhip_moe_combine(st, dn_out.ptr, qwhip.F32, b["inv"].ptr, wb.ptr, t, k, hidden, None, None, out.ptr, qwhip.F32))
    dev.stream.sync()
    got = out.download(np.float32, (t, hidden))
    ref = qo.moe_forward_f64(xval, idx, wts, gu16, dn16, act_f16=True, rotate_act=True)
    assert qo.normalized_error(got, ref) <= TOL
    assert np.allclose(qo.moe_forward_grouped_f64(xval, idx, wts, gu16, dn16, act_f16=True, rotate_act=True), ref, rtol=1e-3, atol=1e-5)


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g32", "hq4_g64", "hq8_g32", "aq2_g64", "hq3_g32", "hq6_g32"])
@pytest.mark.parametrize("t,experts,hidden,inter,k,rot", [(40, 8, 256, 128, 2, 1), (130, 16, 512, 192, 4, 1), (300, 4, 128, 64, 2, 0),
                                                          (64, 8, 192, 448, 3, 1)])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_fused_gate_up_swiglu_equals_the_two_step_chain(dev, fmt, t, experts, hidden, inter, k, rot, xdt):
    """qwhip_moe_grouped_gemm_swiglu == qwhip_moe_grouped_gemm (f16 out) + qwhip_swiglu_fwht, bit for bit, on the rows of the
    sorted list (intermediate sizes with a partial 128-column tile included), and the chain built on it meets the oracle;
    f16 and bf16 hidden rows on every container."""
    gu_blocks, gu16, dn_blocks, dn16 = _moe_banks(experts, hidden, inter, seed=13, fmt=fmt)
    rng = np.random.default_rng(9)
    x16, xcode, xval = _hidden_rows(rng, t, hidden, xdt)
    logits = rng.standard_normal((t, experts)).astype(np.float32)
    idx, wts = _route(dev, logits, k)
    g = _group(dev, idx, experts, k)
    pairs = t * k
    lib, st, b = dev.lib, dev.stream.handle, g["bufs"]
    gub, xb = dev.put(gu_blocks), dev.put(x16)
    gu_out = dev.alloc(pairs * 2 * inter * 2)
    act2, act1 = dev.put(np.zeros((pairs, inter), np.float16)), dev.put(np.zeros((pairs, inter), np.float16))
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vgu), experts, xb.ptr, xcode, 0, b["stok"].ptr, b["off"].ptr, b["te"].ptr,
                                           b["tr"].ptr, b["tc"].ptr, g["max_tiles"], pairs, gu_out.ptr, qwhip.F16, 0))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu_out.ptr, qwhip.F16, act2.ptr, pairs, inter, rot))
    qwhip.check(lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(vgu), experts, xb.ptr, xcode, 0, b["stok"].ptr, b["off"].ptr,
                                                  b["te"].ptr, b["tr"].ptr, b["tc"].ptr, g["max_tiles"], pairs, rot, act1.ptr, 0))
    dev.stream.sync()
    valid = int(g["off"][experts])
    two, one = act2.download(np.float16, (pairs, inter))[:valid], act1.download(np.float16, (pairs, inter))[:valid]
    assert np.array_equal(one.view(np.uint16), two.view(np.uint16))
    # against the oracle: act of sorted slot p = swiglu(x[tok] . gate_e, x[tok] . up_e), rotated
    e_of = np.repeat(np.arange(experts), np.diff(g["off"]))
    xs = xval[g["stok"][:valid]].astype(np.float64)
    gu = np.einsum("pk,pnk->pn", xs, gu16[e_of].astype(np.float64)).astype(np.float16).astype(np.float32)
    want = qo.swiglu_fwht_f16(gu[:, :inter], gu[:, inter:], rotate=bool(rot)).astype(np.float32)
    assert qo.normalized_error(one.astype(np.float32), want) <= TOL


_SPANS_FEW = [1, 16, 17, 0, 32, 33, 63, 64, 65, 2]                  # at most 48 rows an expert: spans of 64
_SPANS_MANY = [31, 64, 96, 97, 0, 128, 129, 160, 161, 225, 300]     # spans of 128 (96 on the 6- and 8-bit containers) on wide enough banks


_SPANS_M5 = [3000, 2725]                                            # HQ4_G32_M5 takes them on K past 1536 only


@pytest.mark.parametrize("fmt,counts,k,inter,xdt,compact", [
    (fmt, *case) for fmt in sorted(H.FORMATS)
    for case in [(_SPANS_FEW, 128, 96, "f16", True), (_SPANS_FEW, 768, 32, "bf16", False), (_SPANS_MANY, 384, 96, "f16", False)]
    + ([(_SPANS_M5, 2176, 2144, "f16", True)] if fmt == "hq4_g32_m5" else [(_SPANS_MANY, 128, 6688, "bf16", True)])]
    + [(fmt, _SPANS_MANY, 384, 6688, "f16", False) for fmt in ("hq4_g64", "hq3_g32", "hq6_g32")])
def test_grouped_gemm_spans(dev, fmt, counts, k, inter, xdt, compact):
    """Experts of every span shape (fragment edges, the last row of a span, empty experts), one, three and six pairs of K-steps (up to
    five of them 8-bit banks this small take the 64-row kernel), partial column tiles: fp32 sums of k exact products against fp64, f16 and bf16 as their roundings, the fused gate|up bit for bit."""
    if fmt in ("aq8_g256",):
        k = 256 * (k // 128)                                          # whole groups; takes the 64-row kernel
    e, n = len(counts), 2 * inter
    rng = np.random.default_rng(k + inter)
    blocks, w16 = H.make_bank(fmt, min(e * n, 3001), k, seed=21)
    if e * n > 3001:
        pick = rng.integers(0, 3001, e * n)                           # a large bank's rows are drawn from fewer
        blocks, w16 = blocks[pick], w16[pick]
    ids = rng.permutation(np.repeat(np.arange(e), counts)).astype(np.int32).reshape(-1, 1)
    pairs = ids.size
    x, xcode, xval = _hidden_rows(rng, pairs, k, xdt)
    g = _group(dev, ids, e, 1, compact)
    lib, st, b = dev.lib, dev.stream.handle, g["bufs"]
    bank, xb = dev.put(blocks), dev.put(x)
    view = H.view_of(dev, bank, fmt, e * n, k)
    plan = (b["stok"].ptr, b["off"].ptr, b["te"].ptr, b["tr"].ptr, b["tc"].ptr, g["max_tiles"], pairs)
    y32, y16, yb = dev.alloc(pairs * n * 4), dev.alloc(pairs * n * 2), dev.alloc(pairs * n * 2)
    act1, act2 = dev.alloc(pairs * inter * 2), dev.alloc(pairs * inter * 2)
    for y, dt in ((y32, qwhip.F32), (y16, qwhip.F16), (yb, qwhip.BF16)):
        qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(view), e, xb.ptr, xcode, 0, *plan, y.ptr, dt, 0))
    qwhip.check(lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(view), e, xb.ptr, xcode, 0, *plan, 1, act1.ptr, 0))
    qwhip.check(lib.qwhip_swiglu_fwht(st, y16.ptr, qwhip.F16, act2.ptr, pairs, inter, 1))
    dev.stream.sync()
    w = w16.reshape(e, n, k).astype(np.float64)
    xs = xval.astype(np.float16).astype(np.float64)[g["stok"]]
    want = np.concatenate([xs[g["off"][i]:g["off"][i + 1]] @ w[i].T for i in range(e)])
    size = np.concatenate([np.abs(xs[g["off"][i]:g["off"][i + 1]]) @ np.abs(w[i]).T for i in range(e)])
    got = y32.download(np.float32, (pairs, n))
    assert np.all(np.abs(got - want) <= k * 2.0 ** -24 * size)        # k rounded additions of exact products
    assert np.array_equal(y16.download(np.float16, (pairs, n)), got.astype(np.float16))
    assert np.array_equal(yb.download(np.uint16, (pairs, n)), qo.f32_to_bf16_bits(got))
    assert np.array_equal(act1.download(np.uint16, (pairs, inter)), act2.download(np.uint16, (pairs, inter)))


_FEW_EACH = [1, 16, 17, 0, 32, 33, 64, 65, 3, 2, 5] + [0] * 29     # six rows an expert: the row-tile kernel, one to four passes of 16


@pytest.mark.parametrize("fmt", sorted(f for f in H.FORMATS if f != "aq8_g256"))
@pytest.mark.parametrize("counts,k,inter,xdt,compact", [
    (_FEW_EACH, 640, 96, "f16", True), (_FEW_EACH, 1024, 32, "bf16", False), (_FEW_EACH, 2176, 160, "f16", True),
    (_FEW_EACH, 3968, 32, "f16", False), ([15, 1, 9, 0, 3], 1536, 1024, "bf16", True), ([40, 20, 0, 33, 15], 1536, 96, "f16", True)])
def test_grouped_gemm_of_few_rows_an_expert(dev, fmt, counts, k, inter, xdt, compact):
    """The row-tile kernel's edges: fragments and passes, one step a wave and two, a last half step, one to several bands of row tiles."""
    test_grouped_gemm_spans(dev, fmt, counts, k, inter, xdt, compact)


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq8_g32", "hq6_g32", "hq4_g64"])
@pytest.mark.parametrize("counts,k,inter", [([40, 20, 0, 33, 17], 1536, 1024), ([33, 20, 0, 32, 11], 640, 2048)], ids=["two-steps", "one-step"])
def test_grouped_row_tiles_of_two_fragments(dev, fmt, counts, k, inter):
    """About twenty rows an expert: 32 rows share a row tile, and an expert of one fragment, of part of a second and of a second tile."""
    test_grouped_gemm_spans(dev, fmt, counts, k, inter, "f16", True)


def test_grouped_calls_slow_on_few_experts_leave_the_row_tiles(dev):
    """297 tokens x top-4 of 256 experts, 1280 x 512: with every token on the same experts the row tiles took 1.3 of the direct-operand kernel's
    time, on routes falling as 1 / rank 1.2.  A list of more than 768 places is that kernel's: the same bits say that it has the call."""
    fmt, e, n, k, top = "hq4_g32_m5", 256, 1280, 512, 4
    blocks, _ = H.make_bank(fmt, n, k, seed=3)
    ids = np.tile(np.arange(top), (297, 1)).astype(np.int32)
    pairs, g, x = ids.size, _group(dev, ids, e, top), H.make_x(ids.size, k, 5).astype(np.float16)
    b, bank, xb, y = g["bufs"], dev.put(np.tile(blocks.reshape(-1), e)), dev.put(x), dev.alloc(pairs * n * 4)
    view, got = H.view_of(dev, bank, fmt, e * n, k), []
    assert g["max_tiles"] <= 768
    for capacity in (g["max_tiles"], 769):
        qwhip.check(dev.lib.qwhip_moe_grouped_gemm(dev.stream.handle, C.byref(view), e, xb.ptr, qwhip.F16, 0, None, b["off"].ptr, b["te"].ptr,
                                                   b["tr"].ptr, b["tc"].ptr, capacity, pairs, y.ptr, qwhip.F32, 0))
        dev.stream.sync()
        got.append(y.download(np.float32, (pairs, n)))
    assert np.array_equal(got[0], got[1])


# lists of one entry, of one wave's 64 and one more, of seven waves' with several chunks in the last; one expert with every row
_LISTS = [[5], [1] * 64, [2] * 65, [int(c) for c in np.random.default_rng(1).integers(0, 4, 448)] + [70, 33], [0] * 20 + [96] + [0] * 19]


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq6_g32"])
@pytest.mark.parametrize("counts", _LISTS, ids=["one", "64", "65", "450", "same"])
def test_grouped_row_tiles_find_every_chunk(dev, fmt, counts):
    """The row-tile kernel deals (entry, chunk of rows, band) over its workgroups: each is somebody's, once."""
    test_grouped_gemm_spans(dev, fmt, counts, 384, 96, "f16", True)


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq3_g32"])
def test_grouped_row_tiles_take_any_tile_list(dev, fmt):
    test_grouped_gemm_takes_any_tile_list(dev, fmt, _FEW_EACH, 96)


def test_grouped_row_tiles_capacity_of_the_tile_list(dev):
    """Lists of more places than entries: the entries alone are read.  Up to 768 places the row-tile kernel looks through them, past that the
    direct-operand kernel has the call, whose fp32 sums add in another order."""
    fmt, e, k, inter = "hq4_g32_m5", len(_FEW_EACH), 768, 96
    n = 2 * inter
    blocks, w16 = H.make_bank(fmt, e * n, k, seed=22)
    ids = np.repeat(np.arange(e), _FEW_EACH).astype(np.int32).reshape(-1, 1)
    pairs, g, x = ids.size, _group(dev, ids, e, 1), H.make_x(ids.size, k, 5).astype(np.float16)
    b, bank, xb, y = g["bufs"], dev.put(blocks), dev.put(x), dev.alloc(pairs * n * 4)
    view, got = H.view_of(dev, bank, fmt, e * n, k), []
    for capacity in (g["max_tiles"], 768, 769, 4000):
        qwhip.check(dev.lib.qwhip_moe_grouped_gemm(dev.stream.handle, C.byref(view), e, xb.ptr, qwhip.F16, 0, b["stok"].ptr, b["off"].ptr, b["te"].ptr,
                                                   b["tr"].ptr, b["tc"].ptr, capacity, pairs, y.ptr, qwhip.F32, 0))
        dev.stream.sync()
        got.append(y.download(np.float32, (pairs, n)))
    xs, w = x.astype(np.float64)[g["stok"]], w16.reshape(e, n, k).astype(np.float64)
    rows = [(xs[g["off"][i]:g["off"][i + 1]], w[i].T) for i in range(e)]
    want, size = np.concatenate([a @ c for a, c in rows]), np.concatenate([np.abs(a) @ np.abs(c) for a, c in rows])
    for out in got:
        assert np.all(np.abs(out - want) <= k * 2.0 ** -24 * size)      # k rounded additions of exact products
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[2], got[3]) and not np.array_equal(got[0], got[2])


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq8_g32", "hq4_g64"])
@pytest.mark.parametrize("counts,inter", [(_SPANS_FEW, 96), (_SPANS_MANY, 96), ([2300, 40], 96), (_SPANS_MANY, 6656), ([2300, 40], 4992)])
def test_grouped_gemm_takes_any_tile_list(dev, fmt, counts, inter):
    """A caller's own list of tiles - another order, a part of the sort's - gives the rows of the tiles that are in it, the same bits
    as the whole list, and leaves the other rows alone: spans of 64 rows, and on the wide banks of 128 (96), but for HQ4_G32_M5."""
    e, k = len(counts), 768 if inter == 96 else 128
    n = 2 * inter
    blocks, _ = H.make_bank(fmt, min(e * n, 3001), k, seed=22)
    blocks = blocks[np.random.default_rng(e).integers(0, len(blocks), e * n)]
    ids = np.repeat(np.arange(e), counts).astype(np.int32).reshape(-1, 1)
    pairs = ids.size
    g = _group(dev, ids, e, 1)
    lib, st, b = dev.lib, dev.stream.handle, g["bufs"]
    bank, xb = dev.put(blocks), dev.put(H.make_x(pairs, k, 5).astype(np.float16))
    view = H.view_of(dev, bank, fmt, e * n, k)
    code_rows = np.array([64, 16, 32, 64])
    bm = code_rows[g["tr"] >> 24]
    start = g["off"][g["te"]] + (g["tr"] & 0xFFFFFF) * bm
    stop = np.minimum(start + bm, g["off"][g["te"] + 1])

    def both_doors(te, tr):
        bufs = [dev.put(te.astype(np.int32)), dev.put(tr.astype(np.int32)), dev.put(np.array([te.size], np.int32))]
        y, act = dev.put(np.full((pairs, n), 0x5555, np.uint16)), dev.put(np.full((pairs, inter), 0x5555, np.uint16))
        plan = (b["stok"].ptr, b["off"].ptr, *(t.ptr for t in bufs), g["max_tiles"], pairs)
        qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(view), e, xb.ptr, qwhip.F16, 0, *plan, y.ptr, qwhip.F16, 0))
        qwhip.check(lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(view), e, xb.ptr, qwhip.F16, 0, *plan, 1, act.ptr, 0))
        dev.stream.sync()
        out = np.concatenate([y.download(np.uint16, (pairs, n)), act.download(np.uint16, (pairs, inter))], axis=1)
        for t in (*bufs, y, act):
            t.free()
        return out

    whole = both_doors(g["te"], g["tr"])
    order = np.random.default_rng(3).permutation(g["tc"])
    for pick in (np.arange(g["tc"])[::-1], order, np.arange(0, g["tc"], 2), np.arange(1, g["tc"]), order[: g["tc"] // 2]):
        listed = np.zeros(pairs, bool)
        for t in pick:
            listed[start[t]:stop[t]] = True
        assert np.array_equal(both_doors(g["te"][pick], g["tr"][pick]), np.where(listed[:, None], whole, 0x5555))


def test_fused_gate_up_swiglu_refusals(dev):
    blocks, _ = H.make_bank("hq4_g32_m5", 4 * 2 * 48, 64, 1)
    bank, xb, act = dev.put(blocks), dev.put(np.zeros((4, 64), np.float16)), dev.alloc(4096)
    z = dev.put(np.zeros(64, np.int32))
    lib, st = dev.lib, dev.stream.handle
    v = H.view_of(dev, bank, "hq4_g32_m5", 4 * 2 * 48, 64)
    args = (z.ptr, z.ptr, z.ptr, z.ptr, 4, 4, 1, act.ptr, 0)
    assert lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(v), 4, xb.ptr, qwhip.F16, 0, None, *args) == qwhip.E_BAD_GEOMETRY   # inter = 48
    v2 = H.view_of(dev, bank, "hq4_g32_m5", 4 * 2 * 48, 64)
    assert lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(v2), 3, xb.ptr, qwhip.F32, 0, None, *args) == qwhip.E_BAD_WEIGHTS   # f32 activations
    assert lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(v2), 5, xb.ptr, qwhip.BF16, 0, None, *args) == qwhip.E_BAD_SHAPE    # 384 rows over 5 experts


def test_grouped_gemm_refuses_expert_of_4gib(dev):
    """One expert whose rows span 4 GiB or more is refused by both doors before any launch: the kernels address the rows
    of an expert with 32-bit offsets. The bank is device memory that nothing reads."""
    k, rows = 16384, 419456                      # 419456 rows x 10240 bytes = 4.0002 GiB
    bank = dev.alloc(rows * (k // 32) * 20)
    xb, out, z = dev.put(np.zeros((4, k), np.float16)), dev.alloc(4096), dev.put(np.zeros(64, np.int32))
    lib, st = dev.lib, dev.stream.handle
    v = H.view_of(dev, bank, "hq4_g32_m5", rows, k)
    tiles = (z.ptr, z.ptr, z.ptr, z.ptr, 4, 4)
    assert lib.qwhip_moe_grouped_gemm(st, C.byref(v), 1, xb.ptr, qwhip.F16, 0, None, *tiles, out.ptr, qwhip.F16, 0) == qwhip.E_BAD_GEOMETRY
    assert lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(v), 1, xb.ptr, qwhip.F16, 0, None, *tiles, 1, out.ptr, 0) == qwhip.E_BAD_GEOMETRY


@pytest.mark.parametrize("xdt", ["f32", "f16"])
@pytest.mark.parametrize("t,e,h", [(1, 20, 96), (3, 20, 96), (300, 1040, 96)])
def test_router_gemm_keeps_infinities(dev, t, e, h, xdt):
    """An infinite activation or weight gives the infinity, or the NaN, that the plain sum of the products gives."""
    rng = np.random.default_rng(e)
    x = rng.standard_normal((t, h)).astype(np.float16).astype(np.float32)
    w = qo.round_bf16(rng.standard_normal((e, h)).astype(np.float32))
    x[:, 5] = 1.0                                     # one bf16 term, the others zero
    x[0, 7], x[t - 1, 40] = np.inf, -np.inf
    w[2, 5], w[e - 1, 5], w[4, 7], w[6, 9] = np.inf, -np.inf, 0.0, np.nan
    xb = dev.put(x if xdt == "f32" else x.astype(np.float16))
    wb, lb = dev.put(qo.f32_to_bf16_bits(w)), dev.alloc(t * e * 4)
    qwhip.check(dev.lib.qwhip_router_gemm(dev.stream.handle, xb.ptr, qwhip.F32 if xdt == "f32" else qwhip.F16, wb.ptr, qwhip.BF16, t, e, h, lb.ptr))
    dev.stream.sync()
    got = lb.download(np.float32, (t, e))
    with np.errstate(invalid="ignore"):
        want = np.stack([(w.astype(np.float64) * r).sum(axis=1) for r in x.astype(np.float64)])
    odd = ~np.isfinite(want)
    assert odd.any() and np.array_equal(got[odd], want[odd].astype(np.float32), equal_nan=True)
    assert np.isfinite(got[~odd]).all()
    if (~odd).any():
        assert np.abs(got[~odd] - want[~odd]).max() <= 1e-4
    for b in (xb, wb, lb):
        b.free()


@pytest.mark.parametrize("xdt", ["f32", "f16"])
@pytest.mark.parametrize("t,e", [(2, 33), (17, 33), (1025, 257)])
def test_router_gemm_rows_that_are_not_finite(dev, t, e, xdt):
    """Rows of 2080 columns with a NaN or an infinity, summed again by the whole wavefront: the class the plain sum gives, the rows beside
    them untouched, and the bits of a call of their own."""
    h, rng = 2080, np.random.default_rng(t)
    x = rng.standard_normal((t, h)).astype(np.float16)
    w = qo.round_bf16(rng.standard_normal((e, h)).astype(np.float32) * 0.05)
    clean = x.copy()
    x[0, 2079], x[t - 1, 511], x[t - 1, 512] = np.inf, -np.inf, np.inf
    if t > 2:
        x[1, 1024] = np.nan
    cast = (lambda v: v.astype(np.float32)) if xdt == "f32" else (lambda v: v)
    code = qwhip.F32 if xdt == "f32" else qwhip.F16
    xb, cb, wb, lb = dev.put(cast(x)), dev.put(cast(clean)), dev.put(qo.f32_to_bf16_bits(w)), dev.alloc(t * e * 4)
    door = lambda b, n: qwhip.check(dev.lib.qwhip_router_gemm(dev.stream.handle, b, code, wb.ptr, qwhip.BF16, n, e, h, lb.ptr))  # noqa: E731
    door(cb.ptr, t)
    want = lb.download(np.float32, (t, e))
    door(xb.ptr, t)
    got = lb.download(np.float32, (t, e))
    with np.errstate(invalid="ignore"):
        for r in range(t):
            if np.isfinite(x[r]).all():
                assert np.array_equal(got[r], want[r])
            else:
                plain = (w.astype(np.float64) * x[r].astype(np.float64)).sum(axis=1).astype(np.float32)
                assert np.array_equal(got[r], plain, equal_nan=True), r
    door(xb.ptr, 1)
    assert np.array_equal(lb.download(np.float32, (e,)), got[0], equal_nan=True)
    for b in (xb, cb, wb, lb):
        b.free()


# (format, gate_up kernel override): every container runs the column-stationary kernels, override 2 keeps gate_up on the
# general kernel.
@pytest.mark.parametrize("fmt,gu_flags", [("hq4_g32_m5", 0), ("hq4_g32_m5", 2 << 8), ("hq4_g32", 0), ("hq3_g32", 0), ("hq6_g32", 0)])
@pytest.mark.parametrize("experts,hidden,inter,k", [(16, 512, 192, 4), (8, 1280, 96, 3), (4, 2048, 768, 4)])
@pytest.mark.parametrize("t", [1, 3, 8])
@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_moe_decode_chain_matches_oracle(dev, t, xdt, experts, hidden, inter, k, fmt, gu_flags):
    """Decode / verify path: routed gate_up GEMV (+SwiGLU+FWHT) and routed down GEMV with weighted combine,
    un-rotated activations in, fused rotation; shapes with partial 32-block chunks and ragged row tiles."""
    gu_blocks, gu16, dn_blocks, dn16 = _moe_banks(experts, hidden, inter, seed=21, fmt=fmt)
    rng = np.random.default_rng(6)
    x32 = rng.standard_normal((t, hidden)).astype(np.float32)
    if xdt == "f16":
        xh, code, xv = x32.astype(np.float16), qwhip.F16, x32.astype(np.float16).astype(np.float32)
    else:
        xh, code, xv = qo.f32_to_bf16_bits(x32), qwhip.BF16, qo.round_bf16(x32)
    logits = rng.standard_normal((t, experts)).astype(np.float32)
    idx, wts = _route(dev, logits, k)
    idx[0, k - 1] = -1                                         # an empty route is skipped
    shared = rng.standard_normal((t, hidden)).astype(np.float32)
    gate = rng.random(t).astype(np.float32)
    lib, st = dev.lib, dev.stream.handle
    gub, dnb, xb, ib, wb = dev.put(gu_blocks), dev.put(dn_blocks), dev.put(xh), dev.put(idx), dev.put(wts)
    sb, gb = dev.put(shared), dev.put(gate)
    act, out = dev.alloc(t * k * inter * 2), dev.alloc(t * hidden * 4)
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    vdn = H.view_of(dev, dnb, fmt, experts * hidden, inter)
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(vgu), experts, xb.ptr, code, gu_flags, ib.ptr, t, k, act.ptr))
    qwhip.check(lib.qwhip_moe_down_decode(st, C.byref(vdn), experts, act.ptr, ib.ptr, wb.ptr, t, k, sb.ptr, gb.ptr, out.ptr, qwhip.F32))
    dev.stream.sync()
    got = out.download(np.float32, (t, hidden))
    x_rot = qo.fwht32_ortho(xv).astype(np.float16)
    ref = qo.moe_forward_f64(x_rot, idx, wts, gu16, dn16, act_f16=True, rotate_act=True) + gate[:, None].astype(np.float64) * shared
    assert qo.normalized_error(got, ref) <= TOL
    a = act.download(np.float16, (t, k, inter))
    assert np.all(a[0, k - 1] == 0)


# Group widths of several slices and every code width, at rows that end inside a 32-slice chunk and at one slice row per expert;
# the general kernel's f16 weights and the column form's factored sum differ by the weights' f16 rounding, 2^-11 of a product.
@pytest.mark.parametrize("fmt", ["aq4_g32", "hq4_g128", "hq8_g64", "aq8_g256", "aq2_g64", "aq6_g128", "hq3_g32"])
@pytest.mark.parametrize("t,experts,hidden,inter,k", [(2, 4, 1280, 256, 3), (1, 3, 256, 512, 2), (3, 2, 4352, 256, 1)])
def test_moe_decode_column_form_of_every_container(dev, fmt, t, experts, hidden, inter, k):
    rot = H.FORMATS[fmt][4]
    gu_blocks, gu16, dn_blocks, dn16 = _moe_banks(experts, hidden, inter, seed=33, fmt=fmt)
    rng = np.random.default_rng(34)
    x = rng.standard_normal((t, hidden)).astype(np.float16)
    idx, wts = _route(dev, rng.standard_normal((t, experts)).astype(np.float32), k)
    lib, st = dev.lib, dev.stream.handle
    gub, dnb, xb, ib, wb = dev.put(gu_blocks), dev.put(dn_blocks), dev.put(x), dev.put(idx), dev.put(wts)
    act, act2, out = dev.alloc(t * k * inter * 2), dev.alloc(t * k * inter * 2), dev.alloc(t * hidden * 4)
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    vdn = H.view_of(dev, dnb, fmt, experts * hidden, inter)
    for flags, a in ((0, act), (2 << 8, act2)):
        qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(vgu), experts, xb.ptr, qwhip.F16, flags, ib.ptr, t, k, a.ptr))
    qwhip.check(lib.qwhip_moe_down_decode(st, C.byref(vdn), experts, act.ptr, ib.ptr, wb.ptr, t, k, None, None, out.ptr, qwhip.F32))
    dev.stream.sync()
    col, general = (a.download(np.float16, (t, k, inter)).astype(np.float64) for a in (act, act2))
    assert qo.normalized_error(col, general) <= TOL
    ref = qo.moe_forward_f64(H.x_in_basis(x, fmt), idx, wts, gu16, dn16, act_f16=True, rotate_act=rot)
    assert qo.normalized_error(out.download(np.float32, (t, hidden)), ref) <= TOL


@pytest.mark.parametrize("fmt", ["aq4_g32", "hq4_g128", "hq8_g64", "aq8_g256", "aq2_g64", "aq6_g128", "hq3_g32"])
@pytest.mark.parametrize("pre", [0, qwhip.X_PREROTATED])
def test_routed_projections_keep_infinities(dev, fmt, pre):
    """An infinite activation gives the infinities (or, against a weight of zero or another infinity, the NaN) of its products with the
    f16 weights: gate|up as the general kernel gives them, down as the plain sum; rows without one are left alone."""
    rot = H.FORMATS[fmt][4]
    t, experts, hidden, inter, k = 4, 3, 1280, 256, 2
    gu_blocks, _, dn_blocks, dn16 = _moe_banks(experts, hidden, inter, seed=61, fmt=fmt)
    rng = np.random.default_rng(62)
    x = rng.standard_normal((t, hidden)).astype(np.float16)
    x[0, 5], x[1, 1100], x[2, 40], x[2, 700] = np.inf, -np.inf, np.inf, -np.inf
    idx, wts = np.array([[0, 1], [2, 0], [1, 2], [0, 2]], np.int32), (rng.random((t, k)) + 0.2).astype(np.float32)
    act = rng.standard_normal((t, k, inter)).astype(np.float16)
    act[0, 1, 3], act[1, 0, 255], act[2, 0, 32], act[2, 1, 64], act[2, 1, 70] = np.inf, -np.inf, np.nan, np.inf, np.inf
    lib, st = dev.lib, dev.stream.handle
    gub, dnb, xb, ib, wb, ab = dev.put(gu_blocks), dev.put(dn_blocks), dev.put(x), dev.put(idx), dev.put(wts), dev.put(act)
    outs = [dev.alloc(t * k * inter * 2) for _ in range(2)] + [dev.alloc(t * hidden * 4)]
    vgu, vdn = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden), H.view_of(dev, dnb, fmt, experts * hidden, inter)
    for flags, o in ((pre, outs[0]), (pre | (2 << 8), outs[1])):
        qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(vgu), experts, xb.ptr, qwhip.F16, flags, ib.ptr, t, k, o.ptr))
    qwhip.check(lib.qwhip_moe_down_decode(st, C.byref(vdn), experts, ab.ptr, ib.ptr, wb.ptr, t, k, None, None, outs[2].ptr, qwhip.F32))
    dev.stream.sync()
    col, general = (o.download(np.float16, (t, k, inter)).astype(np.float32) for o in outs[:2])
    odd = ~np.isfinite(general)
    assert odd[:3].any() and not odd[3].any()
    assert np.array_equal(col[odd], general[odd], equal_nan=True)
    assert np.isfinite(col[~odd]).all() and qo.normalized_error(col[~odd].astype(np.float64), general[~odd].astype(np.float64)) <= TOL
    with np.errstate(invalid="ignore"):
        want = np.stack([sum(float(wts[r, j]) * (dn16[idx[r, j]].astype(np.float64) * act[r, j].astype(np.float64)).sum(axis=1)
                             for j in range(k)) for r in range(t)])
    got = outs[2].download(np.float32, (t, hidden))
    assert np.isinf(want[:2]).any() and np.isnan(want[2]).all() and np.isfinite(want[3]).all()
    assert np.array_equal(got[:3], want[:3].astype(np.float32), equal_nan=True)
    assert qo.normalized_error(got[3], want[3]) <= TOL
    for b in (gub, dnb, xb, ib, wb, ab, *outs):
        b.free()


@pytest.mark.parametrize("fmt", ["hq6_g32", "aq6_g128", "hq3_g32", "aq2_g64", "hq8_g64", "aq4_g32"])
@pytest.mark.parametrize("mag,spike", [(1.0, 0.0), (1e-2, 0.0), (1e-4, 0.0), (1e-5, 0.0), (1e-5, 16376.0), (1e-5, 16384.0), (1e-4, 32752.0),
                                       (1e-4, 65504.0)])
def test_routed_down_keeps_every_bit_of_small_activations(dev, fmt, mag, spike):
    """f16 subnormal activations (gated activations have no norm behind them) and, in one group of a row, a value near the largest f16,
    against the un-rounded affine weights: exact products, so fp32 sums and the cancellation of s sum(q x) against b sum(x), at most
    some 30 times the result, are all there is: 2^-24 x 30 x a few."""
    kind, bits, group, is_m5, _ = H.FORMATS[fmt]
    t, e, k, h, inter = 2, 3, 2, 80, 768
    blocks, _ = H.make_bank(fmt, e * h, inter, 51)
    w = qo.weights_affine_f64(blocks, bits, group, is_m5).reshape(e, h, inter)
    rng = np.random.default_rng(52)
    act = (rng.standard_normal((t, k, inter)) * mag).astype(np.float16)
    if spike:
        act[1, 0, 37], act[1, 1, 64 + 30] = spike, -spike
    idx, wts = np.array([[2, 0], [1, 2]], np.int32), (rng.random((t, k)) + 0.2).astype(np.float32)
    ref = np.zeros((t, h))
    for r in range(t):
        for j in range(k):
            ref[r] += float(wts[r, j]) * (w[idx[r, j]] @ act[r, j].astype(np.float64))
    bank, ab, ib, wb, out = dev.put(blocks), dev.put(act), dev.put(idx), dev.put(wts), dev.alloc(t * h * 4)
    v = H.view_of(dev, bank, fmt, e * h, inter)
    qwhip.check(dev.lib.qwhip_moe_down_decode(dev.stream.handle, C.byref(v), e, ab.ptr, ib.ptr, wb.ptr, t, k, None, None, out.ptr, qwhip.F32))
    got = out.download(np.float32, (t, h))
    for r in range(t):   # row by row: the spike's row must not hide the other
        assert qo.normalized_error(got[r], ref[r]) <= 2e-5, r
    for b in (bank, ab, ib, wb, out):
        b.free()


@pytest.mark.parametrize("fmt", ["hq6_g32", "aq6_g128", "hq3_g32"])
@pytest.mark.parametrize("spike", [16376.0, 16392.0, 32752.0, 32768.0, 65504.0])
def test_routed_gate_up_takes_the_largest_activations(dev, fmt, spike):
    """An activation at, and past, the largest one the scaled operands hold: the general kernel's result, up to its weights' f16 rounding."""
    kind, bits, group, is_m5, rot = H.FORMATS[fmt]
    t, e, k, h, inter = 2, 2, 2, 1280, 96
    w = H.make_weights(e * 2 * inter, h, 53, std=2e-4)
    blocks, _ = qo.quant_hq_blocks(w, bits=bits, group=group, is_m5=is_m5, rotate=rot)
    rng = np.random.default_rng(54)
    x = rng.standard_normal((t, h)).astype(np.float16)
    x[0, 7], x[0, 1030], x[1, 31] = spike, -spike, -spike
    idx = np.array([[0, 1], [1, 0]], np.int32)
    bank, xb, ib = dev.put(blocks), dev.put(x), dev.put(idx)
    outs = [dev.alloc(t * k * inter * 2) for _ in range(2)]
    v = H.view_of(dev, bank, fmt, e * 2 * inter, h)
    for flags, o in ((0, outs[0]), (2 << 8, outs[1])):
        qwhip.check(dev.lib.qwhip_moe_gateup_decode(dev.stream.handle, C.byref(v), e, xb.ptr, qwhip.F16, flags | qwhip.X_PREROTATED, ib.ptr, t, k, o.ptr))
    dev.stream.sync()
    col, general = (o.download(np.float16, (t, k * inter)).astype(np.float64) for o in outs)
    assert np.isfinite(general).all() and np.abs(general).max() > 0.1
    for r in range(t):
        assert qo.normalized_error(col[r], general[r]) <= TOL
    for b in (bank, xb, ib, *outs):
        b.free()


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
@pytest.mark.parametrize("hidden,inter", [(256, 96), (2048, 160), (3072, 64), (5120, 40)])
@pytest.mark.parametrize("t,k,experts", [(2, 8, 12), (3, 4, 6), (4, 8, 40), (4, 16, 20), (4, 8, 8)])
def test_gateup_decode_reads_a_shared_expert_once_with_the_same_bits(dev, t, k, experts, hidden, inter, xdt):
    """A verify window of 2..4 tokens whose rows share experts: QWHIP_MOE_REUSE_EXPERTS reads a shared expert once for all
    of its tokens (encodeMoEGateUpF32R1's reuseExpertsAcrossTokens, QWGemmMoE.swift:119-132; QWMoEReuseTests.swift:46-186 compares
    the two modes) and must leave the bits of the launch that keeps every (token, route) pair to itself.  Few experts force
    sharing (with 8 experts and top-8 every token routes to all of them); the list also holds a repeated expert inside one
    token, an absent route, and the route door is run on the same window."""
    fmt = "hq4_g32_m5"
    gu_blocks, _ = H.make_bank(fmt, experts * 2 * inter, hidden, 77)
    rng = np.random.default_rng(1000 * t + k + hidden)
    x32 = rng.standard_normal((t, hidden)).astype(np.float32)
    xh, code = (x32.astype(np.float16), qwhip.F16) if xdt == "f16" else (qo.f32_to_bf16_bits(x32), qwhip.BF16)
    logits = rng.standard_normal((t, experts)).astype(np.float32)
    ref_idx, _ = qo.moe_route(logits, min(k, experts), True, 1.0)
    idx = np.full((t, k), -1, np.int32)
    idx[:, :ref_idx.shape[1]] = ref_idx
    if k > ref_idx.shape[1]:
        idx[:, ref_idx.shape[1]:] = rng.integers(0, experts, (t, k - ref_idx.shape[1]))   # repeats inside a token
    idx[t - 1, 1] = idx[t - 1, 0]                              # a token's second route to one expert
    idx[0, k - 1] = -1                                         # an absent route
    shared_pairs = sum(int(np.isin(idx[r][idx[r] >= 0], idx[:r][idx[:r] >= 0]).sum()) for r in range(1, t))
    assert shared_pairs > 0
    lib, st = dev.lib, dev.stream.handle
    gub, xb, ib = dev.put(gu_blocks), dev.put(xh), dev.put(idx)
    v = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    a1, a2 = dev.put(np.full((t, k, inter), 3, np.float16)), dev.put(np.full((t, k, inter), 5, np.float16))
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(v), experts, xb.ptr, code, qwhip.MOE_REUSE_EXPERTS, ib.ptr, t, k, a1.ptr))
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(v), experts, xb.ptr, code, 0, ib.ptr, t, k, a2.ptr))
    dev.stream.sync()
    one, two = a1.download(np.uint16, (t, k, inter)), a2.download(np.uint16, (t, k, inter))
    assert np.array_equal(one, two)
    assert np.all(one[idx < 0] == 0) and np.any(one != 0)
    if k <= experts:   # the same window through the door that routes inside the launch
        i1, w1, i2, w2 = (dev.alloc(t * k * 4 + 256) for _ in range(4))
        lb = dev.put(logits)
        qwhip.check(lib.qwhip_moe_route_gateup_decode(st, C.byref(v), experts, xb.ptr, code, qwhip.MOE_REUSE_EXPERTS, lb.ptr, t, k, 1, 1.0, i1.ptr, w1.ptr, a1.ptr))
        qwhip.check(lib.qwhip_moe_route_gateup_decode(st, C.byref(v), experts, xb.ptr, code, 0, lb.ptr, t, k, 1, 1.0,
                                                      i2.ptr, w2.ptr, a2.ptr))
        dev.stream.sync()
        assert np.array_equal(i1.download(np.int32, (t, k)), ref_idx) and np.array_equal(i2.download(np.int32, (t, k)), ref_idx)
        assert np.array_equal(w1.download(np.uint32, (t, k)), w2.download(np.uint32, (t, k)))
        assert np.array_equal(a1.download(np.uint16, (t, k, inter)), a2.download(np.uint16, (t, k, inter)))


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64"])
@pytest.mark.parametrize("t", [1, 3])
def test_decode_chain_replays_from_a_hip_graph(dev, fmt, t):
    """The decode doors only enqueue kernels, so a caller bound by launch latency can capture the chain (routing + gate_up,
    down + combine) as a HIP graph.  The graph is replayed several times with eager launches and synchronisations of the
    same doors in between (on other buffers and other inputs), and every replay must leave the eager chain's bits."""
    experts, hidden, inter, k = 16, 512, 192, 4
    gu_blocks, _, dn_blocks, _ = _moe_banks(experts, hidden, inter, seed=31, fmt=fmt)
    rng = np.random.default_rng(12)
    lib, st = dev.lib, dev.stream.handle
    gub, dnb = dev.put(gu_blocks), dev.put(dn_blocks)
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    vdn = H.view_of(dev, dnb, fmt, experts * hidden, inter)

    def buffers():
        return dict(x=dev.alloc(t * hidden * 2), lg=dev.alloc(t * experts * 4), idx=dev.alloc(t * k * 4 + 256), wts=dev.alloc(t * k * 4 + 256),
                    act=dev.alloc(t * k * inter * 2), out=dev.alloc(t * hidden * 4))

    def chain(b):
        qwhip.check(lib.qwhip_moe_route_gateup_decode(st, C.byref(vgu), experts, b["x"].ptr, qwhip.F16, 0, b["lg"].ptr, t, k, 1, 1.0,
                                                      b["idx"].ptr, b["wts"].ptr, b["act"].ptr))
        qwhip.check(lib.qwhip_moe_down_decode(st, C.byref(vdn), experts, b["act"].ptr, b["idx"].ptr, b["wts"].ptr, t, k, None, None,
                                              b["out"].ptr, qwhip.F32))

    def fill(b):
        b["x"].upload(rng.standard_normal((t, hidden)).astype(np.float16))
        b["lg"].upload(rng.standard_normal((t, experts)).astype(np.float32))

    g, e = buffers(), buffers()          # the graph's buffers and the eager chain's
    fill(g)
    chain(g)                             # the kernels are loaded before the capture
    dev.stream.sync()
    graph = qwhip.Graph(dev.stream, lambda: chain(g))
    for replay in range(4):
        fill(g)                                            # new inputs in the captured buffers
        e["x"].upload(g["x"].download(np.float16, (t, hidden)))
        e["lg"].upload(g["lg"].download(np.float32, (t, experts)))
        g["out"].upload(np.full((t, hidden), 7.0, np.float32))
        graph.launch()
        chain(e)                                           # the same doors, eagerly, behind the replay on the stream
        dev.stream.sync()
        assert np.array_equal(g["out"].download(np.uint32, (t, hidden)), e["out"].download(np.uint32, (t, hidden))), replay
        assert np.array_equal(g["idx"].download(np.int32, (t, k)), e["idx"].download(np.int32, (t, k))), replay
    graph.destroy()


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g32"])
@pytest.mark.parametrize("t,experts,hidden,inter,k", [(1, 128, 512, 96, 8), (3, 16, 1280, 192, 4), (8, 200, 256, 64, 3)])
def test_fused_route_gateup_decode_equals_the_two_launches(dev, fmt, t, experts, hidden, inter, k):
    """qwhip_moe_route_gateup_decode leaves the ids, weights and activations of qwhip_moe_route + qwhip_moe_gateup_decode, bit
    for bit (the HQ4_G32_M5 bank routes inside the gate_up kernel, the bit-stream bank runs the two launches)."""
    gu_blocks, _, _, _ = _moe_banks(experts, hidden, inter, seed=23, fmt=fmt)
    rng = np.random.default_rng(8)
    xh = rng.standard_normal((t, hidden)).astype(np.float16)
    logits = rng.standard_normal((t, experts)).astype(np.float32)
    logits[0, 3] = np.inf                                      # a non-finite logit never wins
    logits[t - 1, 5] = logits[t - 1, 9]                        # a tie goes to the lower id
    lib, st = dev.lib, dev.stream.handle
    gub, xb, lb = dev.put(gu_blocks), dev.put(xh), dev.put(logits)
    vgu = H.view_of(dev, gub, fmt, experts * 2 * inter, hidden)
    i2, w2, a2 = dev.alloc(t * k * 4 + 256), dev.alloc(t * k * 4 + 256), dev.alloc(t * k * inter * 2)
    i1, w1, a1 = dev.alloc(t * k * 4 + 256), dev.alloc(t * k * 4 + 256), dev.alloc(t * k * inter * 2)
    qwhip.check(lib.qwhip_moe_route(st, lb.ptr, t, experts, k, 1, 2.5, i2.ptr, w2.ptr))
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(vgu), experts, xb.ptr, qwhip.F16, 0, i2.ptr, t, k, a2.ptr))
    qwhip.check(lib.qwhip_moe_route_gateup_decode(st, C.byref(vgu), experts, xb.ptr, qwhip.F16, 0, lb.ptr, t, k, 1, 2.5, i1.ptr, w1.ptr, a1.ptr))
    dev.stream.sync()
    assert np.array_equal(i1.download(np.int32, (t, k)), i2.download(np.int32, (t, k)))
    assert np.array_equal(w1.download(np.uint32, (t, k)), w2.download(np.uint32, (t, k)))
    assert np.array_equal(a1.download(np.uint16, (t, k, inter)), a2.download(np.uint16, (t, k, inter)))
    ref_idx, ref_w = qo.moe_route(logits, k, True, 2.5)
    assert np.array_equal(i1.download(np.int32, (t, k)), ref_idx)


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g32"])
@pytest.mark.parametrize("t,experts", [(2, 300), (1, 512)])
def test_fused_route_gateup_decode_with_eight_experts_a_lane(dev, fmt, t, experts):
    test_fused_route_gateup_decode_equals_the_two_launches(dev, fmt, t, experts, 256, 64, 3)


def test_online_quantizer_writes_the_packers_bytes(dev):
    """Device HQ4_G32_M5 quantizer vs the oracle's restatement of the packer, byte-identical
    (Tests/QWFlashNextMetalTests/QUANT/FNMetalOnlineQuantTests.swift:243), bf16 and f32 sources, rotate on/off."""
    w = H.make_weights(96, 1024, seed=4)
    w[3, :32] = 0.0
    w[5, 7] = 3.0
    for src_kind in ("f32", "bf16"):
        if src_kind == "bf16":
            host, code, val = qo.f32_to_bf16_bits(w), qwhip.BF16, qo.round_bf16(w)
        else:
            host, code, val = w, qwhip.F32, w
        for rotate in (1, 0):
            sb, ob = dev.put(host), dev.alloc(96 * 32 * 20)
            qwhip.check(dev.lib.qwhip_quantize_hq4_g32(dev.stream.handle, sb.ptr, code, 96, 1024, rotate, ob.ptr))
            got = ob.download(np.uint8, (96, 32, 20))
            assert np.array_equal(got, qo.quant_hq4_blocks(val, rotate=bool(rotate)))


def test_swiglu_fwht_more_rows_than_a_grid_dimension(dev):
    """65,600 rows of one rotation group: the rows past the grid's 65,535 are taken by its second step."""
    rows, inter = 65600, 32
    gu = np.random.default_rng(5).standard_normal((rows, 2 * inter)).astype(np.float32)
    gb, ab = dev.put(gu), dev.alloc(rows * inter * 2)
    qwhip.check(dev.lib.qwhip_swiglu_fwht(dev.stream.handle, gb.ptr, qwhip.F32, ab.ptr, rows, inter, 1))
    want = qo.swiglu_fwht_f16(gu[:, :inter], gu[:, inter:], rotate=True).astype(np.float32)
    assert qo.normalized_error(ab.download(np.float16, (rows, inter)), want) <= 2e-3


@pytest.mark.parametrize("inter", [32, 96, 608, 1024, 1056])
@pytest.mark.parametrize("rows", [7, 1024, 1501])
def test_gated_activation_of_rows_that_share_a_workgroup(dev, rows, inter):
    """From 1024 rows on, rows of up to 1024 channels share workgroups (64 of 32, three of 608, two of 1024): full and part filled last
    workgroups, and a row count and a row length past the lines.  The fp32 door rounds to the f16 door's bits."""
    gu = (np.random.default_rng(inter + rows).standard_normal((rows, 2 * inter)) * 2).astype(np.float32)
    gb, ab, fb = dev.put(gu), dev.alloc(rows * inter * 2), dev.alloc(rows * inter * 4)
    for rotate in (1, 0):
        qwhip.check(dev.lib.qwhip_swiglu_fwht(dev.stream.handle, gb.ptr, qwhip.F32, ab.ptr, rows, inter, rotate))
        got = ab.download(np.float16, (rows, inter))
        want = qo.swiglu_fwht_f16(gu[:, :inter], gu[:, inter:], rotate=bool(rotate)).astype(np.float32)
        assert np.max(np.abs(got.astype(np.float32) - want)) <= 2e-3 * max(1.0, float(np.max(np.abs(want))))
        if rotate:
            qwhip.check(dev.lib.qwhip_silu_mul_f32(dev.stream.handle, gb.ptr, fb.ptr, rows, inter))
            assert np.array_equal(fb.download(np.float32, (rows, inter)).astype(np.float16), got)
    for b in (gb, ab, fb):
        b.free()


def test_swiglu_fwht_matches_oracle(dev):
    rng = np.random.default_rng(2)
    rows, inter = 9, 160
    gu = (rng.standard_normal((rows, 2 * inter)) * 2).astype(np.float16)
    gb, ab = dev.put(gu), dev.alloc(rows * inter * 2)
    for rotate in (1, 0):
        qwhip.check(dev.lib.qwhip_swiglu_fwht(dev.stream.handle, gb.ptr, qwhip.F16, ab.ptr, rows, inter, rotate))
        got = ab.download(np.float16, (rows, inter)).astype(np.float32)
        want = qo.swiglu_fwht_f16(gu[:, :inter].astype(np.float32), gu[:, inter:].astype(np.float32), rotate=bool(rotate)).astype(np.float32)
        assert np.max(np.abs(got - want)) <= 2e-3 * max(1.0, float(np.max(np.abs(want))))


@pytest.mark.parametrize("t", [1, 2048])
def test_moe_full_size_operator(t):
    """C4 at its real shape (128 experts, top-8, hidden 2048, intermediate 768, bf16 hidden rows): device-quantized banks
    byte-checked against the oracle on expert 0, routing identical, EVERY token against the fp64 oracle (prefill: the
    oracle's expert-ordered form, which makes the 155 GFLOP of fp64 products a matter of seconds)."""
    import argparse

    import bench
    out = bench.run_moe(argparse.Namespace(steps=2, warmup=1, no_cpu=True), t, "full-size parity")
    assert out["normalized_error"] <= TOL and out["tokens_checked"] == t and out["config"]["activations"] == "bf16"
    assert out["worst_token_error"] <= TOL


def test_moe_full_size_operator_f16_rows():
    """The same prefill batch on f16 hidden rows (the reference's own activation type), every token."""
    import argparse

    import bench
    out = bench.run_moe(argparse.Namespace(steps=2, warmup=1, no_cpu=True, moe_f16=True), 2048, "full-size parity, f16 rows")
    assert out["normalized_error"] <= TOL and out["tokens_checked"] == 2048 and out["config"]["activations"] == "f16"


@pytest.mark.parametrize("hidden", [256, 1000])
@pytest.mark.parametrize("dtype", ["f32", "f16"])
def test_combine_identity_slots_and_unit_weights(dev, hidden, dtype):
    """The door's invPerm: nil and unweightedSingle forms (encodeMoEDownReduceCombineF32, QWGemmMoE.swift:299-332): without
    a permutation route k of token t is row t * top_k + k, without weights every route counts once; with one route that is
    out = dn + gate * shared (the last step of the latent operator), in place when the types agree."""
    rng = np.random.default_rng(hidden)
    t, k = 5, 3
    dn = rng.standard_normal((t * k, hidden)).astype(np.float32)
    dn_h = dn.astype(np.float16) if dtype == "f16" else dn
    wts = rng.random((t, k)).astype(np.float32)
    shared = rng.standard_normal((t, hidden)).astype(np.float32)
    gate = rng.random(t).astype(np.float32)
    lib, st = dev.lib, dev.stream.handle
    code = qwhip.F16 if dtype == "f16" else qwhip.F32
    d_dn, d_w, d_sh, d_g, d_out = dev.put(dn_h), dev.put(wts), dev.put(shared), dev.put(gate), dev.alloc(t * hidden * 4)
    base = dn_h.astype(np.float64).reshape(t, k, hidden)
    # identity slots with weights
    qwhip.check(lib.qwhip_moe_combine(st, d_dn.ptr, code, None, d_w.ptr, t, k, hidden, None, None, d_out.ptr, qwhip.F32))
    dev.stream.sync()
    want = (base * wts[:, :, None].astype(np.float64)).sum(1)
    assert np.max(np.abs(d_out.download(np.float32, (t, hidden)) - want)) <= 1e-5 * np.abs(want).max()
    # unit weights with the gated shared rows
    qwhip.check(lib.qwhip_moe_combine(st, d_dn.ptr, code, None, None, t, k, hidden, d_sh.ptr, d_g.ptr, d_out.ptr, qwhip.F32))
    dev.stream.sync()
    want = base.sum(1) + gate[:, None].astype(np.float64) * shared
    assert np.max(np.abs(d_out.download(np.float32, (t, hidden)) - want)) <= 1e-5 * np.abs(want).max()
    if dtype == "f32":   # one route, in place: dn += gate * shared
        rows = dev.put(dn[:t])
        qwhip.check(lib.qwhip_moe_combine(st, rows.ptr, qwhip.F32, None, None, t, 1, hidden, d_sh.ptr, d_g.ptr, rows.ptr, qwhip.F32))
        dev.stream.sync()
        want = dn[:t].astype(np.float64) + gate[:, None].astype(np.float64) * shared
        assert np.max(np.abs(rows.download(np.float32, (t, hidden)) - want)) <= 1e-6 * np.abs(want).max()
        rows.free()
    for b in (d_dn, d_w, d_sh, d_g, d_out):
        b.free()


# ---- group-latent MoE: the doors and the whole block -------------------------------------------------------------------
def _latent_routes(rng, t, e, k, ng, hole=True):
    idx = np.stack([rng.permutation(e)[:k] for _ in range(t)]).astype(np.int32)
    if hole and t * k > 1:
        idx[0, k - 1] = -1
    wts = (rng.random((t, k)) + 0.1).astype(np.float32)
    labels = rng.integers(0, ng, e).astype(np.int32)
    return idx, wts, labels


@pytest.mark.parametrize("t,e,k,ng", [(1, 32, 4, 4), (7, 100, 8, 8), (300, 128, 8, 32), (5, 16, 2, 1)])
def test_latent_groups_and_compose_rows(dev, t, e, k, ng):
    """group ids / latent rows of the routes against the oracle's rule, and the composed gather rows of a second sort."""
    rng = np.random.default_rng(t + ng)
    idx, _, labels = _latent_routes(rng, t, e, k, ng)
    lib, st = dev.lib, dev.stream.handle
    ib, lb, gb, rb = dev.put(idx), dev.put(labels), dev.alloc(t * ng * 4), dev.alloc(t * k * 4)
    qwhip.check(lib.qwhip_moe_latent_groups(st, ib.ptr, lb.ptr, t, k, e, ng, gb.ptr, rb.ptr))
    dev.stream.sync()
    gids, rows = qo.moe_latent_groups(idx, labels, ng)
    assert np.array_equal(gb.download(np.int32, (t, ng)), gids)
    assert np.array_equal(rb.download(np.int32, (t, k)), rows)
    pairs = t * k
    sp = rng.permutation(pairs).astype(np.int32)
    slot = rng.permutation(t * ng).astype(np.int32)
    slot[gids.ravel() < 0] = -1                                 # rows of absent groups have no slot
    ob, spb, slb = dev.alloc(pairs * 4), dev.put(sp), dev.put(slot)
    qwhip.check(lib.qwhip_moe_compose_rows(st, spb.ptr, pairs, rb.ptr, t * ng, slb.ptr, ob.ptr))
    dev.stream.sync()
    pr = rows.ravel()[sp]
    want = np.where(pr >= 0, np.maximum(slot[np.maximum(pr, 0)], 0), 0)
    assert np.array_equal(ob.download(np.int32, (pairs,)), want)
    assert lib.qwhip_moe_latent_groups(st, ib.ptr, lb.ptr, t, k, e, 33, gb.ptr, rb.ptr) == qwhip.E_BAD_SHAPE


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq8_g32", "hq4_g64"])
@pytest.mark.parametrize("t,ng,lat,hidden", [(1, 4, 64, 256), (3, 8, 96, 512), (8, 4, 40, 1280)])
def test_routed_gemv_keeps_one_row_per_route(dev, fmt, t, ng, lat, hidden):
    """out[t, r] = wts * W[idx[t, r]] . x: every route its own output row, one activation row per token or per route, unit
    weights when none are given, zeros for an absent route."""
    blocks, w16 = H.make_bank(fmt, ng * lat, hidden, 41)
    w = w16.reshape(ng, lat, hidden).astype(np.float64)
    rng = np.random.default_rng(3)
    ids = np.tile(np.arange(ng, dtype=np.int32), (t, 1))
    ids[rng.random((t, ng)) < 0.3] = -1
    wts = (rng.random((t, ng)) + 0.2).astype(np.float32)
    x_tok = rng.standard_normal((t, hidden)).astype(np.float16)
    x_rt = rng.standard_normal((t, ng, hidden)).astype(np.float16)
    lib, st = dev.lib, dev.stream.handle
    bank, ib, wb = dev.put(blocks), dev.put(ids), dev.put(wts)
    v = H.view_of(dev, bank, fmt, ng * lat, hidden)
    for per_token, x, wbuf, odt in ((1, x_tok, None, qwhip.F16), (0, x_rt, wb, qwhip.F32)):
        out, xb = dev.put(np.full((t, ng, lat), 7, np.float32)), dev.put(x)
        qwhip.check(lib.qwhip_moe_routed_gemv(st, C.byref(v), ng, xb.ptr, per_token, ib.ptr, wbuf.ptr if wbuf else None, t, ng,
                                              out.ptr, odt))
        dev.stream.sync()
        if odt == qwhip.F16:
            got = out.download(np.float16, (2 * t * ng * lat,))[: t * ng * lat]
        else:
            got = out.download(np.float32, (t * ng * lat,))
        got = got.reshape(t, ng, lat).astype(np.float64)
        ref = np.zeros((t, ng, lat))
        for r in range(t):
            for g in range(ng):
                if ids[r, g] >= 0:
                    xv = (x[r] if per_token else x[r, g]).astype(np.float64)
                    ref[r, g] = (wts[r, g] if wbuf else 1.0) * (w[ids[r, g]] @ xv)
        assert qo.normalized_error(got, ref) <= TOL
        assert np.all(got[ids < 0] == 0)


@pytest.mark.parametrize("fmt,gu_flags", [("hq4_g32_m5", 0), ("hq4_g32_m5", 2 << 8), ("hq4_g64", 0)])
@pytest.mark.parametrize("t,e,k,ng,lat,inter", [(1, 16, 4, 4, 64, 64), (4, 32, 4, 4, 256, 96), (8, 8, 3, 2, 1792, 64)])
def test_gateup_decode_rows_reads_the_given_rows(dev, fmt, gu_flags, t, e, k, ng, lat, inter):
    """qwhip_moe_gateup_decode_rows == qwhip_moe_gateup_decode over the gathered rows, bit for bit."""
    gu_blocks, _ = H.make_bank(fmt, e * 2 * inter, lat, 43)
    rng = np.random.default_rng(t)
    idx, _, labels = _latent_routes(rng, t, e, k, ng)
    _, rows = qo.moe_latent_groups(idx, labels, ng)
    xl = rng.standard_normal((t * ng, lat)).astype(np.float16)
    lib, st = dev.lib, dev.stream.handle
    bank, ib = dev.put(gu_blocks), dev.put(idx)
    v = H.view_of(dev, bank, fmt, e * 2 * inter, lat)
    a1, a2 = dev.put(np.full((t * k, inter), 3, np.float16)), dev.put(np.full((t * k, inter), 5, np.float16))
    flags = qwhip.X_PREROTATED | gu_flags
    xlb, rwb, gab = dev.put(xl), dev.put(rows), dev.put(xl[np.maximum(rows.ravel(), 0)])
    qwhip.check(lib.qwhip_moe_gateup_decode_rows(st, C.byref(v), e, xlb.ptr, qwhip.F16, flags, ib.ptr, rwb.ptr, t, k, a1.ptr))
    qwhip.check(lib.qwhip_moe_gateup_decode(st, C.byref(v), e, gab.ptr, qwhip.F16, flags, ib.ptr, t * k, 1, a2.ptr))
    dev.stream.sync()
    one, two = a1.download(np.float16, (t * k, inter)), a2.download(np.float16, (t * k, inter))
    assert np.array_equal(one.view(np.uint16), two.view(np.uint16))
    assert np.any(one != 0) and np.all(one[idx.ravel() < 0] == 0)
    if 2 <= t <= 4:   # a shared expert read once: every pair still reads its own latent row
        a3 = dev.put(np.full((t * k, inter), 7, np.float16))
        qwhip.check(lib.qwhip_moe_gateup_decode_rows(st, C.byref(v), e, xlb.ptr, qwhip.F16, flags | qwhip.MOE_REUSE_EXPERTS, ib.ptr, rwb.ptr, t, k,
                                                     a3.ptr))
        dev.stream.sync()
        assert np.array_equal(a3.download(np.uint16, (t * k, inter)), two.view(np.uint16))


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "hq8_g32"])
@pytest.mark.parametrize("t,e,k,ng,lat,inter", [(1, 16, 4, 4, 64, 64), (4, 32, 8, 8, 160, 128), (8, 8, 3, 2, 1792, 64)])
def test_down_decode_groups_sums_the_routes_of_each_group(dev, fmt, t, e, k, ng, lat, inter):
    dn_blocks, dn16 = H.make_bank(fmt, e * lat, inter, 47)
    w = dn16.reshape(e, lat, inter).astype(np.float64)
    rng = np.random.default_rng(ng + t)
    idx, wts, labels = _latent_routes(rng, t, e, k, ng)
    act = rng.standard_normal((t, k, inter)).astype(np.float16)
    lib, st = dev.lib, dev.stream.handle
    bank = dev.put(dn_blocks)
    v = H.view_of(dev, bank, fmt, e * lat, inter)
    out = dev.put(np.full((t, ng, lat), 9, np.float32))
    ab, ib, wb, lb = dev.put(act), dev.put(idx), dev.put(wts), dev.put(labels)
    qwhip.check(lib.qwhip_moe_down_decode_groups(st, C.byref(v), e, ab.ptr, ib.ptr, wb.ptr, lb.ptr, ng, t, k, out.ptr, qwhip.F32))
    dev.stream.sync()
    got = out.download(np.float32, (t, ng, lat)).astype(np.float64)
    ref = np.zeros((t, ng, lat))
    for r in range(t):
        for j in range(k):
            if idx[r, j] >= 0:
                ref[r, labels[idx[r, j]]] += wts[r, j] * (w[idx[r, j]] @ act[r, j].astype(np.float64))
    assert qo.normalized_error(got, ref) <= TOL
    gids, _ = qo.moe_latent_groups(idx, labels, ng)
    assert np.all(got[gids < 0] == 0)


@pytest.mark.parametrize("t,k,ng,width,ddt,odt,perm", [(5, 4, 4, 64, "f32", "f16", True), (300, 8, 8, 1792, "f16", "f32", True),
                                                       (3, 3, 2, 100, "f32", "f32", False)])
def test_combine_groups(dev, t, k, ng, width, ddt, odt, perm):
    rng = np.random.default_rng(width)
    e = 4 * ng
    idx, wts, labels = _latent_routes(rng, t, e, k, ng)
    pairs = t * k
    dn = rng.standard_normal((pairs, width)).astype(np.float32)
    dnh = dn.astype(np.float16) if ddt == "f16" else dn
    inv = rng.permutation(pairs).astype(np.int32) if perm else None
    if perm:
        inv[idx.ravel() < 0] = -1
    lib, st = dev.lib, dev.stream.handle
    out = dev.alloc(t * ng * width * 4)
    db, pb, wb, ib, lb = dev.put(dnh), (dev.put(inv) if perm else None), dev.put(wts), dev.put(idx), dev.put(labels)
    qwhip.check(lib.qwhip_moe_combine_groups(st, db.ptr, qwhip.F16 if ddt == "f16" else qwhip.F32, pb.ptr if perm else None,
                                             wb.ptr, ib.ptr, lb.ptr, e, t, k, ng, width, out.ptr, qwhip.F16 if odt == "f16" else qwhip.F32))
    dev.stream.sync()
    got = out.download(np.float16 if odt == "f16" else np.float32, (t, ng, width)).astype(np.float64)
    ref = np.zeros((t, ng, width))
    for r in range(t):
        for j in range(k):
            if idx[r, j] < 0:
                continue
            slot = int(inv[r * k + j]) if perm else r * k + j
            ref[r, labels[idx[r, j]]] += float(wts[r, j]) * dnh[slot].astype(np.float64)
    assert qo.normalized_error(got, ref) <= (2e-3 if odt == "f16" else 1e-6)
    # a route whose id is not below the expert count has no label: it counts as absent (nothing past the labels is read)
    idx2 = idx.copy()
    idx2[0, 0] = e + 5
    idx2[t - 1, k - 1] = (7 << 16) | e
    ib2 = dev.put(idx2)
    qwhip.check(lib.qwhip_moe_combine_groups(st, db.ptr, qwhip.F16 if ddt == "f16" else qwhip.F32, pb.ptr if perm else None,
                                             wb.ptr, ib2.ptr, lb.ptr, e, t, k, ng, width, out.ptr, qwhip.F16 if odt == "f16" else qwhip.F32))
    dev.stream.sync()
    got2 = out.download(np.float16 if odt == "f16" else np.float32, (t, ng, width)).astype(np.float64)
    for (r, j) in ((0, 0), (t - 1, k - 1)):
        if idx[r, j] >= 0:
            slot = int(inv[r * k + j]) if perm else r * k + j
            ref[r, labels[idx[r, j]]] -= float(wts[r, j]) * dnh[slot].astype(np.float64)
    assert qo.normalized_error(got2, ref) <= (2e-3 if odt == "f16" else 1e-5)


def _group_latent_block(dev, fmts, t, e, k, ng, hidden, lat, inter, x16, idx, wts, labels, banks):
    """The block from the doors: decode (t <= 8) through the routed GEMVs, prefill through two pair sorts and the grouped GEMMs."""
    lib, st = dev.lib, dev.stream.handle
    f_lat, f_exp = fmts
    bd, bu, bgu, bdn = dev.put(banks["d"]), dev.put(banks["u"]), dev.put(banks["gu"]), dev.put(banks["dn"])
    vd = H.view_of(dev, bd, f_lat, ng * lat, hidden)
    vu = H.view_of(dev, bu, f_lat, ng * hidden, lat)
    vgu = H.view_of(dev, bgu, f_exp, e * 2 * inter, lat)
    vdn = H.view_of(dev, bdn, f_exp, e * lat, inter)
    ones = dev.put(np.ones((t, ng), np.float32))
    xb, ib, wb, lb = dev.put(x16), dev.put(idx), dev.put(wts), dev.put(labels)
    gids, rows = dev.alloc(t * ng * 4), dev.alloc(t * k * 4)
    out = dev.alloc(t * hidden * 4)
    pairs = t * k
    qwhip.check(lib.qwhip_moe_latent_groups(st, ib.ptr, lb.ptr, t, k, e, ng, gids.ptr, rows.ptr))
    act = dev.alloc(pairs * inter * 2)
    z16 = dev.alloc(t * ng * lat * 2)
    if t <= 8:
        xl = dev.alloc(t * ng * lat * 2)
        qwhip.check(lib.qwhip_moe_routed_gemv(st, C.byref(vd), ng, xb.ptr, 1, gids.ptr, None, t, ng, xl.ptr, qwhip.F16))
        qwhip.check(lib.qwhip_moe_gateup_decode_rows(st, C.byref(vgu), e, xl.ptr, qwhip.F16, qwhip.X_PREROTATED, ib.ptr, rows.ptr, t, k, act.ptr))
        qwhip.check(lib.qwhip_moe_down_decode_groups(st, C.byref(vdn), e, act.ptr, ib.ptr, wb.ptr, lb.ptr, ng, t, k, z16.ptr, qwhip.F16))
        qwhip.check(lib.qwhip_moe_down_decode(st, C.byref(vu), ng, z16.ptr, gids.ptr, ones.ptr, t, ng, None, None, out.ptr, qwhip.F32))
    else:
        dev.stream.sync()
        g1 = _group(dev, gids.download(np.int32, (t, ng)), ng, ng)
        b1 = g1["bufs"]
        n1 = t * ng
        xl = dev.alloc(n1 * lat * 2)
        qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vd), ng, xb.ptr, qwhip.F16, 0, b1["stok"].ptr, b1["off"].ptr, b1["te"].ptr, b1["tr"].ptr,
                                               b1["tc"].ptr, g1["max_tiles"], n1, xl.ptr, qwhip.F16, 0))
        g2 = _group(dev, idx, e, k)
        b2 = g2["bufs"]
        rows2 = dev.alloc(pairs * 4)
        qwhip.check(lib.qwhip_moe_compose_rows(st, b2["sp"].ptr, pairs, rows.ptr, n1, b1["inv"].ptr, rows2.ptr))
        qwhip.check(lib.qwhip_moe_grouped_gemm_swiglu(st, C.byref(vgu), e, xl.ptr, qwhip.F16, 0, rows2.ptr, b2["off"].ptr, b2["te"].ptr, b2["tr"].ptr,
                                                      b2["tc"].ptr, g2["max_tiles"], pairs, 1, act.ptr, 0))
        dn = dev.alloc(pairs * lat * 4)
        qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vdn), e, act.ptr, qwhip.F16, 0, None, b2["off"].ptr, b2["te"].ptr, b2["tr"].ptr,
                                               b2["tc"].ptr, g2["max_tiles"], pairs, dn.ptr, qwhip.F32, 0))
        qwhip.check(lib.qwhip_moe_combine_groups(st, dn.ptr, qwhip.F32, b2["inv"].ptr, wb.ptr, ib.ptr, lb.ptr, e, t, k, ng, lat, z16.ptr, qwhip.F16))
        yu = dev.alloc(n1 * hidden * 4)
        qwhip.check(lib.qwhip_moe_grouped_gemm(st, C.byref(vu), ng, z16.ptr, qwhip.F16, 0, b1["sp"].ptr, b1["off"].ptr, b1["te"].ptr, b1["tr"].ptr,
                                               b1["tc"].ptr, g1["max_tiles"], n1, yu.ptr, qwhip.F32, 0))
        qwhip.check(lib.qwhip_moe_combine(st, yu.ptr, qwhip.F32, b1["inv"].ptr, None, t, ng, hidden, None, None, out.ptr, qwhip.F32))
    dev.stream.sync()
    return out.download(np.float32, (t, hidden))


@pytest.mark.parametrize("fmts", [("hq8_g32", "hq4_g64"), ("hq4_g32_m5", "hq4_g32_m5")])
@pytest.mark.parametrize("t,e,k,ng,hidden,lat,inter", [(1, 32, 4, 4, 64, 64, 64), (4, 32, 4, 4, 256, 128, 64), (8, 64, 8, 8, 512, 192, 128),
                                                       (16, 32, 4, 4, 64, 64, 64), (64, 32, 4, 4, 256, 128, 64), (130, 64, 8, 8, 512, 192, 128)])
def test_group_latent_block_matches_oracle(dev, fmts, t, e, k, ng, hidden, lat, inter):
    """latentD -> routed experts in the latent width -> sum by group -> latentU, decode and prefill forms, against
    moe_group_latent_forward_f64 (the sizes of FNLatentMoETests among them: H = L = I = 64, 32 experts, 4 groups, 4 routes)."""
    f_lat, f_exp = fmts
    banks, w = {}, {}
    banks["d"], w["d"] = H.make_bank(f_lat, ng * lat, hidden, 51)
    banks["u"], w["u"] = H.make_bank(f_lat, ng * hidden, lat, 52)
    banks["gu"], w["gu"] = H.make_bank(f_exp, e * 2 * inter, lat, 53)
    banks["dn"], w["dn"] = H.make_bank(f_exp, e * lat, inter, 54)
    rng = np.random.default_rng(t * 7 + ng)
    x16 = qo.rotate_activation_f16(rng.standard_normal((t, hidden)).astype(np.float32))
    logits = rng.standard_normal((t, e)).astype(np.float32)
    idx, wts = _route(dev, logits, k)
    labels = (np.arange(e) % ng).astype(np.int32)
    if t >= 4:
        labels[idx[1]] = labels[idx[1, 0]]                    # one token with all its routes in one group
    got = _group_latent_block(dev, fmts, t, e, k, ng, hidden, lat, inter, x16, idx, wts, labels, banks)
    ref = qo.moe_group_latent_forward_f64(x16, idx, wts, labels, w["d"].reshape(ng, lat, hidden), w["gu"].reshape(e, 2 * inter, lat),
                                          w["dn"].reshape(e, lat, inter), w["u"].reshape(ng, hidden, lat))
    assert qo.normalized_error(got, ref) <= TOL


@pytest.mark.parametrize("m,k,e,budget,norm", [(2, 8, 32, 10, 1), (4, 16, 64, 20, 1), (3, 4, 8, 6, 0), (4, 8, 128, 9, 1), (2, 4, 16, 2, 1), (4, 16, 512, 40, 1)])
def test_route_budget_matches_oracle(dev, m, k, e, budget, norm):
    """The expert budget of a verify window: ids identical to the oracle, weights to 1e-6; duplicates across rows, ties and a
    route already empty included; no-op and refused shapes."""
    rng = np.random.default_rng(m * 100 + k)
    lg = rng.standard_normal((m, e)).astype(np.float32)
    lg[1] = lg[0] + rng.standard_normal(e).astype(np.float32) * 0.05          # row 1 shares most experts with row 0
    idx, wts = _route(dev, lg, k)
    if m > 2:
        idx[2, k - 1], wts[2, k - 1] = -1, 0.0
        wts[2, 0] = wts[m - 1, 1]                                              # a tie between two candidates
    ib, wb = dev.put(idx), dev.put(wts)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_moe_route_budget(st, ib.ptr, wb.ptr, m, k, budget, norm))
    dev.stream.sync()
    gi, gw = ib.download(np.int32, (m, k)), wb.download(np.float32, (m, k))
    ri, rw = qo.moe_route_budget(idx, wts, budget, bool(norm))
    assert np.array_equal(gi, ri)
    np.testing.assert_allclose(gw, rw, rtol=1e-6, atol=0)
    assert np.array_equal(gi[0], idx[0]) and len({int(v) for v in gi.ravel() if v >= 0}) <= max(k, budget)
    qwhip.check(lib.qwhip_moe_route_budget(st, ib.ptr, wb.ptr, m, k, m * k, norm))   # nothing to prune
    dev.stream.sync()
    assert np.array_equal(ib.download(np.int32, (m, k)), gi)
    assert lib.qwhip_moe_route_budget(st, ib.ptr, wb.ptr, 5, 4, 3, 1) == qwhip.E_BAD_SHAPE
    assert lib.qwhip_moe_route_budget(st, ib.ptr, wb.ptr, 1, 4, 3, 1) == qwhip.E_BAD_SHAPE
