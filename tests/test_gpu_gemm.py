"""GPU parity of the prefill GEMM (f16 MFMA, fp32 accumulate) against the fp64 oracle, through the C ABI.
Bar: normalized error <= 2e-3 (bf16 / f16 stores); fp32 stores are held to 2e-5."""
import ctypes as C

import numpy as np
import pytest

from oracle import qworacle as qo
from qwegn_amd import qwhip
from tests import helpers as H

pytestmark = pytest.mark.gpu
TOL = 2e-3
# kernel overrides (flags bits 8..11) with their K ranges (bits 12..15): a form that cannot take the call is refused
DIRECT_64, DIRECT_WIDE, SPLIT_PINGPONG = 6, 7, 8


def form(code, ranges=0):
    return code | ranges << 4


@pytest.fixture(scope="module")
def dev():
    return qwhip.Device(0)


def run_gemm(dev, fmt, m, n, k, *, xdtype="bf16", ydtype="bf16", prerot=True, cfg=0, seed=0, workspace=True, workspace_bytes=None):
    blocks, w16 = H.make_bank(fmt, n, k, seed=seed)
    x32 = H.make_x(m, k, seed + 7)
    rotate = H.FORMATS[fmt][4]
    if xdtype == "bf16":
        x_val, x_host, xcode = qo.round_bf16(x32), qo.f32_to_bf16_bits(x32), qwhip.BF16
    else:
        x_host, xcode = x32.astype(np.float16), qwhip.F16
        x_val = x_host.astype(np.float32)
    if prerot or not rotate:
        # activations arrive in the container's basis; the kernel converts them to f16
        x_basis = x_val.astype(np.float16)
        flags = qwhip.X_PREROTATED
    else:
        x_basis = qo.fwht32_ortho(x_val).astype(np.float16)
        flags = 0
    flags |= (cfg << 8)
    ysize = {"bf16": 2, "f16": 2, "f32": 4}[ydtype]
    ycode = {"bf16": qwhip.BF16, "f16": qwhip.F16, "f32": qwhip.F32}[ydtype]
    bank, xb, yb = dev.put(blocks), dev.put(x_host), dev.alloc(m * n * ysize)
    ws = dev.alloc(workspace_bytes if workspace_bytes else m * k * 2) if workspace else None
    view = H.view_of(dev, bank, fmt, n, k)
    st = dev.lib.qwhip_gemm(dev.stream.handle, C.byref(view), xb.ptr, xcode, m, 0, yb.ptr, ycode, 0, flags,
                            ws.ptr if ws else None, ws.nbytes if ws else 0)
    out = None
    if st == qwhip.OK:
        dev.stream.sync()
        if ydtype == "bf16":
            out = qo.bf16_bits_to_f32(yb.download(np.uint16, (m, n)))
        elif ydtype == "f16":
            out = yb.download(np.float16, (m, n)).astype(np.float32)
        else:
            out = yb.download(np.float32, (m, n))
    for b in (bank, xb, yb, ws):
        if b is not None:
            b.free()
    ref = qo.matmul_ref_f64(x_basis, w16)
    return st, out, ref


@pytest.mark.parametrize("cfg", [1, 2, 3, 4, 5, 14, 15])
def test_gemm_hq4_tile_shapes_f32_out(dev, cfg):
    st, out, ref = run_gemm(dev, "hq4_g32_m5", 512, 640, 1024, ydtype="f32", cfg=cfg)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5


@pytest.mark.parametrize("m,n,k", [(1, 16, 64), (37, 48, 128), (300, 336, 192), (257, 1040, 320)])
def test_gemm_ragged_shapes(dev, m, n, k):
    st, out, ref = run_gemm(dev, "hq4_g32_m5", m, n, k, ydtype="f32")
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5


@pytest.mark.parametrize("fmt", ["aq4_g32", "hq4_g64", "hq8_g32", "hq4_g128", "aq8_g256", "aq2_g64", "hq3_g32", "hq6_g32", "aq6_g128"])
@pytest.mark.parametrize("xdtype,ydtype", [("f16", "f16"), ("bf16", "bf16")])
def test_gemm_block_formats(dev, fmt, xdtype, ydtype):
    st, out, ref = run_gemm(dev, fmt, 192, 256, 768, xdtype=xdtype, ydtype=ydtype, seed=3)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


@pytest.mark.parametrize("fmt", ["aq2_g64", "hq3_g32", "hq6_g32", "aq6_g128"])
@pytest.mark.parametrize("cfg,xdtype,workspace", [(15, "f16", True), (0, "bf16", False), (1, "f16", True), (2, "f16", True), (3, "f16", True)])
def test_gemm_narrow_and_six_bit_streams_on_every_kernel(dev, fmt, cfg, xdtype, workspace):
    """2-, 3- and 6-bit streams (codes cut out of the slice's words, also across word boundaries) on the unpipelined kernel
    (f16, and bf16 converted in the tile) and on the DMA-fed kernel's tile shapes, fp32 out, ragged in both directions."""
    st, out, ref = run_gemm(dev, fmt, 300, 336, 384, xdtype=xdtype, ydtype="f32", cfg=cfg, seed=11, workspace=workspace)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq8_g32", "hq4_g64", "aq2_g64", "hq3_g32", "hq6_g32"])
@pytest.mark.parametrize("cfg", [1, 5])
def test_gemm_pingpong_kernel_ragged_tiles(dev, fmt, cfg):
    """The 8-wave ping-pong kernel (256 x 320 and 128 x 320 tiles; the 8-bit containers run the DMA-fed kernel at these
    shapes) on a shape whose last tile row holds one 64-row block and whose last tile column is ragged, for every weight
    format family."""
    st, out, ref = run_gemm(dev, fmt, 320, 400, 640, xdtype="f16", ydtype="f32", cfg=cfg, seed=5)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5
    st, out, ref = run_gemm(dev, fmt, 64, 320, 64, xdtype="bf16", ydtype="bf16", cfg=cfg, seed=6)   # a single K-step
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq4_g64", "aq2_g64", "hq3_g32", "hq6_g32"])
@pytest.mark.parametrize("m", [1, 37, 100, 257, 333, 575])
@pytest.mark.parametrize("cfg", [1, 5])
def test_gemm_pingpong_kernel_ragged_rows(dev, fmt, m, cfg):
    """Row counts that are not whole 64-row blocks on the ping-pong kernel (256 x 320 and 128 x 320 tiles): threads whose row
    lies past the last one re-read the tile's first row and store nothing (last tile rows of 1 to 77 rows; one tile of
    fewer than 64)."""
    st, out, ref = run_gemm(dev, fmt, m, 400, 320, xdtype="f16", ydtype="f32", cfg=cfg, seed=7)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5
    st, out, ref = run_gemm(dev, fmt, m, 336, 192, xdtype="bf16", ydtype="bf16", cfg=cfg, seed=8)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


def test_gemm_half_height_tile_at_2048_rows(dev):
    """M = 2048 on the benchmark bank: the automatic choice is the ping-pong kernel's 128 x 320 tile (256 tiles)."""
    st, out, ref = run_gemm(dev, "hq4_g32_m5", 2048, 5120, 5120, xdtype="bf16", ydtype="bf16")
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


def test_gemm_ragged_rows_at_the_prefill_shape(dev):
    """M = 4001 on the benchmark bank (automatic dispatch, bf16 in / bf16 out): the last tile row holds 161 rows."""
    st, out, ref = run_gemm(dev, "hq4_g32_m5", 4001, 5120, 5120, xdtype="bf16", ydtype="bf16")
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "aq2_g64", "hq3_g32", "hq6_g32", "hq8_g32"])
@pytest.mark.parametrize("m,n,k,cfg", [(64, 640, 1024, form(SPLIT_PINGPONG, 2)), (200, 400, 2048, form(SPLIT_PINGPONG, 4)),
                                       (37, 336, 1536, form(SPLIT_PINGPONG, 5)), (512, 1280, 5120, form(SPLIT_PINGPONG, 8)), (64, 640, 1088, 0)])
def test_gemm_split_k_with_a_workspace_for_partial_planes(dev, fmt, m, n, k, cfg):
    """The ping-pong tile with the K-steps of a tile dealt over several workgroups and a second launch that sums the planes: even
    ranges, a short last one (24 K-steps over five ranges of 5), behind the rotated copy of un-rotated rows; k = 1088, an odd
    number of K-steps, is the automatic choice's.  Same bar as the one-launch form."""
    big = 64 << 20
    st, out, ref = run_gemm(dev, fmt, m, n, k, xdtype="f16", ydtype="f32", seed=9, workspace_bytes=big, cfg=cfg)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5
    st, out1, _ = run_gemm(dev, fmt, m, n, k, xdtype="f16", ydtype="f32", seed=9, workspace=False, cfg=5)
    assert qo.normalized_error(out, out1) <= 2e-6          # the ranges only change the order of the fp32 sums
    assert not np.array_equal(out, out1)                   # and they do
    st, out, ref = run_gemm(dev, fmt, m, n, k, xdtype="bf16", ydtype="bf16", seed=10, workspace_bytes=big, cfg=cfg)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL
    st, out, ref = run_gemm(dev, fmt, m, n, k, xdtype="f16", ydtype="f16", prerot=False, seed=11, workspace_bytes=big, cfg=cfg)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


@pytest.mark.parametrize("k,cfg,ws_mb", [(1088, form(DIRECT_64), 1), (1088, form(DIRECT_WIDE), 1), (1024, form(DIRECT_64, 2), 0),
                                         (1024, form(SPLIT_PINGPONG, 2), 0), (1024, form(SPLIT_PINGPONG), 1), (1024, form(SPLIT_PINGPONG, 7), 1)])
def test_gemm_named_forms_refuse_what_they_cannot_take(dev, k, cfg, ws_mb):
    """K of an odd number of K-steps on the direct-operand kernel, K ranges without room for their planes, ranges of which one would
    be empty (16 K-steps over 7), one range of the split form: refused, on both dense doors."""
    m, n = 33, 64
    bank, xb, y = dev.put(H.make_bank("hq4_g32_m5", n, k, 1)[0]), dev.put(np.zeros((m, k), np.float16)), dev.alloc(m * n * 2)
    ws = dev.alloc(max(16, ws_mb << 20))
    view = H.view_of(dev, bank, "hq4_g32_m5", n, k)
    lib, st, flags, wsp = dev.lib, dev.stream.handle, qwhip.X_PREROTATED | cfg << 8, (ws.ptr, ws_mb << 20) if ws_mb else (None, 0)
    assert lib.qwhip_gemm(st, C.byref(view), xb.ptr, qwhip.F16, m, 0, y.ptr, qwhip.F16, 0, flags, *wsp) == qwhip.E_BAD_SHAPE
    assert lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, qwhip.F16, m, 0, 1, y.ptr, 0, flags, *wsp) == qwhip.E_BAD_SHAPE


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "hq8_g32"])
@pytest.mark.parametrize("m,ws_mb,cfg", [(333, 0, 1), (333, 0, 5), (333, 64, form(SPLIT_PINGPONG, 3)), (2100, 0, 0), (333, 0, form(DIRECT_64)),
                                         (333, 0, form(DIRECT_WIDE)), (333, 64, form(DIRECT_WIDE, 3))])
def test_gemm_strided_rows_on_every_form(dev, fmt, m, ws_mb, cfg):
    """Activation rows ldx > k apart and output rows ldy > n apart (both in elements) through the one-launch forms of the ping-pong
    kernel (256 x 320 and 128 x 320 tiles, ragged row counts), its split-K form and the direct-operand kernel's: padding columns of
    the output stay untouched."""
    n, k, ldx, ldy = 656, 1024, 1024 + 64, 656 + 8
    blocks, w16 = H.make_bank(fmt, n, k, seed=13)
    x32 = H.make_x(m, k, 17)
    xp = np.zeros((m, ldx), np.float16)
    xp[:, :k] = x32.astype(np.float16)
    xp[:, k:] = np.float16(777.0)                      # never read
    bank, xb = dev.put(blocks), dev.put(xp)
    yb = dev.put(np.full((m, ldy), 0x7FC0, np.uint16))  # bf16 NaN pattern in the padding
    ws = dev.alloc(ws_mb << 20) if ws_mb else None
    view = H.view_of(dev, bank, fmt, n, k)
    st = dev.lib.qwhip_gemm(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, ldx, yb.ptr, qwhip.BF16, ldy,
                            qwhip.X_PREROTATED | cfg << 8, ws.ptr if ws else None, ws.nbytes if ws else 0)
    assert st == qwhip.OK
    dev.stream.sync()
    raw = yb.download(np.uint16, (m, ldy))
    for b in (bank, xb, yb, ws):
        if b is not None:
            b.free()
    assert np.all(raw[:, n:] == 0x7FC0)
    ref = qo.matmul_ref_f64(xp[:, :k], w16)
    assert qo.normalized_error(qo.bf16_bits_to_f32(raw[:, :n]), ref) <= TOL


def test_gemm_rotation_prepass_with_workspace(dev):
    st, out, ref = run_gemm(dev, "hq4_g32_m5", 130, 256, 512, prerot=False, ydtype="f32")
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5
    st, _, _ = run_gemm(dev, "hq4_g32_m5", 130, 256, 512, prerot=False, workspace=False)
    assert st == qwhip.E_BASIS


def test_gemm_geometry_errors(dev):
    st, _, _ = run_gemm(dev, "hq4_g32_m5", 8, 24, 64)      # n % 16 != 0
    assert st == qwhip.E_BAD_GEOMETRY
    st, _, _ = run_gemm(dev, "hq4_g32_m5", 8, 32, 96)      # k % 64 != 0
    assert st == qwhip.E_BAD_GEOMETRY


def test_gemm_matches_per_row_gemv(dev):
    """Kernel-vs-kernel: batched GEMM against the per-row GEMV, max |diff| in f16 < 0.05
    (Tests/QWGEMMTests/QWBatchedGemmTests.swift:130-139)."""
    fmt, m, n, k = "hq4_g32_m5", 16, 512, 1024
    blocks, _ = H.make_bank(fmt, n, k, seed=9)
    x16 = H.make_x(m, k, 10).astype(np.float16)
    bank, xb = dev.put(blocks), dev.put(x16)
    yg, yv = dev.alloc(m * n * 2), dev.alloc(m * n * 2)
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, qwhip.F16, m, 0, yg.ptr, qwhip.F16, 0, qwhip.X_PREROTATED, None, 0))
    qwhip.check(lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, m, qwhip.X_PREROTATED, yv.ptr, None))
    a = yg.download(np.float16, (m, n)).astype(np.float32)
    b = yv.download(np.float16, (m, n)).astype(np.float32)
    assert np.max(np.abs(a - b)) < 0.05


def test_gemm_full_size_prefill_config(dev):
    """HQ4_G32 prefill GEMM at its benchmark shape: M = 4096, K = 5120, N = 5120, bf16 in / bf16 out."""
    st, out, ref = run_gemm(dev, "hq4_g32_m5", 4096, 5120, 5120, xdtype="bf16", ydtype="bf16")
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= TOL


@pytest.mark.parametrize("fmt,xdtype,prerot", [("hq4_g32_m5", "f16", True), ("hq4_g32_m5", "bf16", True), ("hq4_g64", "f16", False),
                                               ("hq3_g32", "f16", True), ("aq2_g64", "f16", True),
                                               ("aq4_g32", "f16", True)])
@pytest.mark.parametrize("m,inter,k,rot", [(64, 160, 128, 1), (256, 352, 256, 1), (320, 1024, 192, 0), (576, 96, 64, 1), (37, 160, 128, 1),
                                           (333, 352, 256, 0)])
def test_gemm_swiglu_equals_gemm_then_swiglu(dev, fmt, xdtype, prerot, m, inter, k, rot):
    """qwhip_gemm_swiglu == qwhip_gemm (f16 out) + qwhip_swiglu_fwht, bit for bit (column tiles of 160 outputs with a partial
    last one, several row tiles, bf16 and un-rotated activations through the workspace), and within the bar of the oracle."""
    n = 2 * inter
    blocks, w16 = H.make_bank(fmt, n, k, seed=5)
    x32 = H.make_x(m, k, 12)
    rotate = H.FORMATS[fmt][4]
    if xdtype == "bf16":
        x_val, x_host, xcode = qo.round_bf16(x32), qo.f32_to_bf16_bits(x32), qwhip.BF16
    else:
        x_host, xcode = x32.astype(np.float16), qwhip.F16
        x_val = x_host.astype(np.float32)
    flags = qwhip.X_PREROTATED if (prerot or not rotate) else 0
    x_basis = x_val.astype(np.float16) if flags else qo.fwht32_ortho(x_val).astype(np.float16)
    bank, xb = dev.put(blocks), dev.put(x_host)
    gu, act2, act1 = dev.alloc(m * n * 2), dev.put(np.zeros((m, inter), np.float16)), dev.put(np.zeros((m, inter), np.float16))
    ws = dev.alloc(m * k * 2)
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, 0, gu.ptr, qwhip.F16, 0, flags, ws.ptr, ws.nbytes))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F16, act2.ptr, m, inter, rot))
    qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, rot, act1.ptr, 0, flags, ws.ptr, ws.nbytes))
    dev.stream.sync()
    one, two = act1.download(np.float16, (m, inter)), act2.download(np.float16, (m, inter))
    assert np.array_equal(one.view(np.uint16), two.view(np.uint16))
    g = qo.matmul_ref_f64(x_basis, w16).astype(np.float16).astype(np.float32)
    want = qo.swiglu_fwht_f16(g[:, :inter], g[:, inter:], rotate=bool(rot)).astype(np.float32)
    assert qo.normalized_error(one.astype(np.float32), want) <= TOL


@pytest.mark.parametrize("fmt,m", [("hq8_g32", 128), ("hq3_g32", 64), ("hq6_g32", 128), ("aq6_g128", 75), ("hq4_g32_m5", 37), ("aq2_g64", 200)])
@pytest.mark.parametrize("xdtype,prerot", [("f16", True), ("bf16", False)])
def test_gemm_swiglu_every_container_and_row_count_in_one_launch(dev, fmt, m, xdtype, prerot):
    """The 6- and 8-bit containers and ragged row counts on the fused door (once two launches through the workspace): the same
    bits as the two doors called one after the other, whatever workspace beyond the activation copy is handed over (K = 384 is
    too short for K ranges, which a roomy workspace would otherwise bring)."""
    inter, k = 224, 384
    n = 2 * inter
    rotate = H.FORMATS[fmt][4]
    blocks, _ = H.make_bank(fmt, n, k, seed=4)
    x32 = H.make_x(m, k, 13)
    if xdtype == "bf16":
        x_host, xcode = qo.f32_to_bf16_bits(x32), qwhip.BF16
    else:
        x_host, xcode = x32.astype(np.float16), qwhip.F16
    flags = qwhip.X_PREROTATED if (prerot or not rotate) else 0
    bank, xb = dev.put(blocks), dev.put(x_host)
    gu, act2, act1 = dev.alloc(m * n * 2), dev.put(np.zeros((m, inter), np.float16)), dev.put(np.zeros((m, inter), np.float16))
    ws1, ws2 = dev.alloc(m * k * 2), dev.alloc(m * n * 2 + m * k * 2)
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, 0, gu.ptr, qwhip.F16, 0, flags, ws1.ptr, ws1.nbytes))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F16, act2.ptr, m, inter, 1))
    qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, act1.ptr, 0, flags, ws2.ptr, ws2.nbytes))
    dev.stream.sync()
    one, two = act1.download(np.float16, (m, inter)), act2.download(np.float16, (m, inter))
    assert np.array_equal(one.view(np.uint16), two.view(np.uint16))
    assert np.any(one != 0)
    # a workspace that holds only the activation copy is enough: the door is one launch for every container and row count
    assert lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, act1.ptr, 0, flags, ws1.ptr, ws1.nbytes) == qwhip.OK
    dev.stream.sync()


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "hq8_g32", "hq3_g32"])
@pytest.mark.parametrize("m,inter,k,xdtype,prerot,cfg", [
    (64, 320, 2048, "f16", True, form(SPLIT_PINGPONG, 4)), (100, 480, 1536, "bf16", True, form(SPLIT_PINGPONG, 5)),
    (37, 160, 1024, "f16", False, form(DIRECT_64, 3)), (128, 800, 5120, "bf16", False, form(DIRECT_WIDE, 7)),
    (64, 320, 2048, "f16", True, 0), (100, 480, 1536, "bf16", True, 0), (37, 160, 1088, "f16", False, 0)])
def test_gemm_swiglu_split_k_with_a_roomy_workspace(dev, fmt, m, inter, k, xdtype, prerot, cfg):
    """Few tiles, a long K and a workspace with room for planes: the fused door deals the K-steps over several workgroups (the
    ping-pong tile and both spans of the direct-operand kernel, short last ranges among them, and what it takes by itself), sums the
    planes and runs the SwiGLU pass - the same bits as qwhip_gemm followed by qwhip_swiglu_fwht, within the bar of the oracle, and
    within rounding of its own one-launch form (flags bits 8..11 = 1 keep that)."""
    n = 2 * inter
    blocks, w16 = H.make_bank(fmt, n, k, seed=6)
    x32 = H.make_x(m, k, 14)
    rotate = H.FORMATS[fmt][4]
    if xdtype == "bf16":
        x_val, x_host, xcode = qo.round_bf16(x32), qo.f32_to_bf16_bits(x32), qwhip.BF16
    else:
        x_host, xcode = x32.astype(np.float16), qwhip.F16
        x_val = x_host.astype(np.float32)
    flags = qwhip.X_PREROTATED if (prerot or not rotate) else 0
    x_basis = x_val.astype(np.float16) if flags else qo.fwht32_ortho(x_val).astype(np.float16)
    named = flags | cfg << 8
    bank, xb = dev.put(blocks), dev.put(x_host)
    gu = dev.alloc(m * n * 2)
    acts = [dev.put(np.zeros((m, inter), np.float16)) for _ in range(3)]
    ws = dev.alloc(64 << 20)
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st = dev.lib, dev.stream.handle
    # bf16 rows go through the separate conversion pass in both doors (flags bit 16 asks qwhip_gemm for it), so both split alike
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, 0, gu.ptr, qwhip.F16, 0, named | (1 << 16), ws.ptr, ws.nbytes))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F16, acts[0].ptr, m, inter, 1))
    qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, acts[1].ptr, 0, named, ws.ptr, ws.nbytes))
    qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, acts[2].ptr, 0, flags | (1 << 8), ws.ptr, ws.nbytes))
    dev.stream.sync()
    two, split, one = (a.download(np.float16, (m, inter)) for a in acts)
    for b in (bank, xb, gu, ws, *acts):
        b.free()
    assert np.array_equal(split.view(np.uint16), two.view(np.uint16))
    g = qo.matmul_ref_f64(x_basis, w16).astype(np.float16).astype(np.float32)
    want = qo.swiglu_fwht_f16(g[:, :inter], g[:, inter:], rotate=True).astype(np.float32)
    assert qo.normalized_error(split.astype(np.float32), want) <= TOL
    assert qo.normalized_error(one.astype(np.float32), want) <= TOL
    assert qo.normalized_error(split.astype(np.float32), one.astype(np.float32)) <= TOL


@pytest.mark.parametrize("fmt,m,inter,k,xdtype,prerot,ldpad", [
    ("hq4_g32_m5", 64, 320, 2048, "f16", True, 0), ("hq4_g32_m5", 64, 320, 2048, "bf16", True, 8), ("hq4_g64", 200, 2048, 2048, "f16", True, 0),
    ("hq6_g32", 33, 352, 1920, "bf16", True, 0), ("aq4_g32", 100, 480, 1088, "f16", True, 16), ("hq3_g32", 37, 160, 2048, "bf16", False, 8)])
@pytest.mark.parametrize("planes", [0, 1, 2, 3, 4, 9])
def test_gemm_swiglu_takes_the_k_ranges_of_the_plain_door(dev, fmt, m, inter, k, xdtype, prerot, ldpad, planes):
    """A workspace that holds exactly `planes` fp32 planes behind the copy of the rows (made by both doors or by neither; where neither
    makes one, the first plane lies where a bf16 copy would): the fused door gives the bits of the two doors on that workspace, with act
    rows ldpad elements apart from their neighbours too, whose padding stays as it was."""
    n = 2 * inter
    blocks, _ = H.make_bank(fmt, n, k, seed=8)
    x32 = H.make_x(m, k, 15) * 2
    x_host, xcode = (qo.f32_to_bf16_bits(x32), qwhip.BF16) if xdtype == "bf16" else (x32.astype(np.float16), qwhip.F16)
    flags = qwhip.X_PREROTATED if prerot else 0
    copy = 0 if prerot else (m * k * 2 + 255) // 256 * 256
    size = max(m * k * 2, copy + planes * m * n * 4)           # the fused door wants room for a copy of bf16 rows in any case
    bank, xb, ws = dev.put(blocks), dev.put(x_host), dev.alloc(size)
    gu, act2 = dev.alloc(m * n * 2), dev.alloc(m * inter * 2)
    ld = inter + ldpad
    act1 = dev.put(np.full((m, ld), 0x7E01, np.uint16))
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st = dev.lib, dev.stream.handle
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, 0, gu.ptr, qwhip.F16, 0, flags, ws.ptr, size))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F16, act2.ptr, m, inter, 1))
    qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, act1.ptr, ld, flags, ws.ptr, size))
    dev.stream.sync()
    one, two = act1.download(np.uint16, (m, ld)), act2.download(np.uint16, (m, inter))
    for b in (bank, xb, ws, gu, act1, act2):
        b.free()
    assert np.array_equal(one[:, :inter], two)
    assert np.all(one[:, inter:] == 0x7E01)


@pytest.mark.parametrize("fmt", sorted(f for f in H.FORMATS if f != "aq8_g256"))
@pytest.mark.parametrize("m,n,k,xdtype,cfg", [
    (17, 272, 1920, "f16", form(DIRECT_64, 4)), (65, 272, 2048, "bf16", form(DIRECT_64, 6)), (33, 4112, 2048, "f16", form(DIRECT_64)),
    (40, 1088, 1024, "f16", form(DIRECT_64)), (97, 4112, 2048, "bf16", form(DIRECT_WIDE)), (150, 272, 1920, "bf16", form(DIRECT_WIDE, 4)),
    (333, 1040, 2048, "f16", form(DIRECT_WIDE, 3)), (129, 1088, 1024, "f16", form(DIRECT_WIDE)), (1, 64, 128, "f16", form(DIRECT_WIDE))])
def test_gemm_direct_operand_kernel(dev, fmt, m, n, k, xdtype, cfg):
    """The direct-operand kernel: spans of 64 and of 128 rows (96 on the 6- and 8-bit containers), in one launch and over K ranges with
    a short last one, f16 and bf16 rows, ragged rows, partial column tiles, one pair of K-steps.  fp32 sums of k exact products against
    fp64; the 2-byte outputs are their roundings, and the gate|up door (partial tiles of 128 outputs) gives the two doors' bits."""
    ws_mb = 64 if cfg >> 4 else 0
    blocks, w16 = H.make_bank(fmt, n, k, seed=31)
    x32 = H.make_x(m, k, 7)
    x_host, xcode = (qo.f32_to_bf16_bits(x32), qwhip.BF16) if xdtype == "bf16" else (x32.astype(np.float16), qwhip.F16)
    xs = (qo.round_bf16(x32) if xdtype == "bf16" else x32).astype(np.float16).astype(np.float64)
    bank, xb, ws = dev.put(blocks), dev.put(x_host), dev.alloc(max(1, ws_mb << 20))
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st, flags = dev.lib, dev.stream.handle, qwhip.X_PREROTATED | cfg << 8
    wsp = (ws.ptr, ws_mb << 20) if ws_mb else (None, 0)
    y32, y16, yb = dev.alloc(m * n * 4), dev.alloc(m * n * 2), dev.alloc(m * n * 2)
    for y, dt in ((y32, qwhip.F32), (y16, qwhip.F16), (yb, qwhip.BF16)):
        qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, 0, y.ptr, dt, 0, flags, *wsp))
    dev.stream.sync()
    got = y32.download(np.float32, (m, n))
    w = w16.astype(np.float64)
    assert np.all(np.abs(got - xs @ w.T) <= k * 2.0 ** -24 * (np.abs(xs) @ np.abs(w).T))      # k rounded additions of exact products
    assert np.array_equal(y16.download(np.float16, (m, n)), got.astype(np.float16))
    assert np.array_equal(yb.download(np.uint16, (m, n)), qo.f32_to_bf16_bits(got))
    if xdtype == "f16" and n % 64 == 0:
        act1, act2 = dev.alloc(m * n), dev.alloc(m * n)   # [m, n / 2] f16
        qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xb.ptr, xcode, m, 0, 1, act1.ptr, 0, flags, *wsp))
        qwhip.check(lib.qwhip_swiglu_fwht(st, y16.ptr, qwhip.F16, act2.ptr, m, n // 2, 1))
        dev.stream.sync()
        assert np.array_equal(act1.download(np.uint16, (m, n // 2)), act2.download(np.uint16, (m, n // 2)))
        act1.free(), act2.free()
    for b in (bank, xb, ws, y32, y16, yb):
        b.free()


@pytest.mark.parametrize("fmt", sorted(H.FORMATS))
@pytest.mark.parametrize("m,n,k,xdtype,ranges", [
    (17, 272, 1920, "f16", 1), (32, 64, 64, "bf16", 1), (1, 1040, 192, "f16", 1), (33, 4160, 1088, "bf16", 2), (48, 320, 2048, "f16", 1),
    (64, 8384, 1280, "f16", 1), (49, 4112, 2112, "bf16", 3), (64, 128, 4096, "f16", 4), (31, 16448, 4096, "f16", 1)])
def test_gemm_row_tile_kernel(dev, fmt, m, n, k, xdtype, ranges):
    """The row-tile kernel: two, three and four fragments of rows, half a step to the most steps a wave, one workgroup to several tiles
    each, one launch and K ranges, strided rows.  fp32 sums of k exact products against fp64; the 2-byte outputs are their roundings; the
    gate|up door gives the two doors' bits in one launch (no workspace) and over one plane."""
    group = max(64, H.FORMATS[fmt][2])
    k = -(-k // group) * group
    cfg, ldx, ldy = form(9, ranges), k + 24, n + 8
    blocks, w16 = H.make_bank(fmt, n, k, seed=33)
    x32 = H.make_x(m, k, 8)
    x_host, xcode = (qo.f32_to_bf16_bits(x32), qwhip.BF16) if xdtype == "bf16" else (x32.astype(np.float16), qwhip.F16)
    xs = (qo.round_bf16(x32) if xdtype == "bf16" else x32).astype(np.float16).astype(np.float64)
    strided = np.zeros((m, ldx), x_host.dtype)
    strided[:, :k] = x_host
    strided[:, k:] = 0x7E00 if xdtype == "bf16" else np.nan    # not read
    bank, xb, xp, ws = dev.put(blocks), dev.put(strided), dev.put(x_host), dev.alloc(64 << 20)
    view = H.view_of(dev, bank, fmt, n, k)
    lib, st, flags = dev.lib, dev.stream.handle, qwhip.X_PREROTATED | cfg << 8
    y32, y16, yb = dev.alloc(m * ldy * 4), dev.alloc(m * ldy * 2), dev.alloc(m * ldy * 2)
    for y, dt in ((y32, qwhip.F32), (y16, qwhip.F16), (yb, qwhip.BF16)):
        qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, ldx, y.ptr, dt, ldy, flags, ws.ptr, 64 << 20))
    dev.stream.sync()
    got = y32.download(np.float32, (m, ldy))[:, :n]
    w = w16.astype(np.float64)
    y32b = dev.alloc(m * ldy * 4)
    qwhip.check(lib.qwhip_gemm(st, C.byref(view), xb.ptr, xcode, m, ldx, y32b.ptr, qwhip.F32, ldy, qwhip.X_PREROTATED | 5 << 8, None, 0))
    dev.stream.sync()
    assert not np.array_equal(got, y32b.download(np.float32, (m, ldy))[:, :n])               # not the tiles, which add in another order
    y32b.free()
    assert np.all(np.abs(got - xs @ w.T) <= k * 2.0 ** -24 * (np.abs(xs) @ np.abs(w).T))      # k rounded additions of exact products
    assert np.array_equal(y16.download(np.float16, (m, ldy))[:, :n], got.astype(np.float16))
    assert np.array_equal(yb.download(np.uint16, (m, ldy))[:, :n], qo.f32_to_bf16_bits(got))
    if n % 64 == 0:
        act1, act2 = dev.alloc(m * n), dev.alloc(m * n)   # [m, n / 2] f16
        flat = dev.put(got.astype(np.float16))
        rooms = [64 << 20, m * k * 2] if xdtype == "bf16" or ranges > 1 else [64 << 20, 0]
        for rot in (0, 1):
            qwhip.check(lib.qwhip_swiglu_fwht(st, flat.ptr, qwhip.F16, act2.ptr, m, n // 2, rot))
            for room in rooms if ranges == 1 else rooms[:1]:
                qwhip.check(lib.qwhip_gemm_swiglu(st, C.byref(view), xp.ptr, xcode, m, 0, rot, act1.ptr, 0, flags, ws.ptr if room else None, room))
                dev.stream.sync()
                assert np.array_equal(act1.download(np.uint16, (m, n // 2)), act2.download(np.uint16, (m, n // 2))), (rot, room)
        act1.free(), act2.free(), flat.free()
    for b in (bank, xb, xp, ws, y32, y16, yb):
        b.free()


def test_gemm_ranges_fit_an_xcd(dev):
    """An eighth of the tiles, rounded up, over the ranges is what an XCD's 32 units hold: 50 tiles over five ranges are 35 workgroups on
    an XCD although they are 250 on the chip.  The automatic choice is another form (other fp32 sums)."""
    fmt, m, n, k = "hq4_g64", 640, 2560, 9728
    st, out, ref = run_gemm(dev, fmt, m, n, k, xdtype="f16", ydtype="f32", seed=9, workspace_bytes=96 << 20)
    assert st == qwhip.OK
    assert qo.normalized_error(out, ref) <= 2e-5
    st, other, _ = run_gemm(dev, fmt, m, n, k, xdtype="f16", ydtype="f32", seed=9, workspace_bytes=96 << 20, cfg=form(DIRECT_WIDE, 5))
    assert st == qwhip.OK
    assert qo.normalized_error(out, other) <= 4e-5         # each within 2e-5 of the exact sums
    assert not np.array_equal(out, other)


def test_gemm_swiglu_refusals(dev):
    blocks, _ = H.make_bank("hq8_g32", 128, 64, seed=1)
    bank, xb, act = dev.put(blocks), dev.put(np.zeros((64, 64), np.float16)), dev.alloc(64 * 64 * 2)
    v8 = H.view_of(dev, bank, "hq8_g32", 128, 64)
    lib, st = dev.lib, dev.stream.handle
    assert lib.qwhip_gemm_swiglu(st, C.byref(v8), xb.ptr, qwhip.F16, 64, 0, 1, act.ptr, 0, qwhip.X_PREROTATED, None, 0) == qwhip.OK   # every container
    blocks4, _ = H.make_bank("hq4_g32_m5", 128, 64, seed=1)
    bank4 = dev.put(blocks4)
    v4 = H.view_of(dev, bank4, "hq4_g32_m5", 128, 64)
    assert lib.qwhip_gemm_swiglu(st, C.byref(v4), xb.ptr, qwhip.F16, 37, 0, 1, act.ptr, 0, qwhip.X_PREROTATED, None, 0) == qwhip.OK   # any row count
    assert lib.qwhip_gemm_swiglu(st, C.byref(v4), xb.ptr, qwhip.F16, 64, 0, 1, act.ptr, 0, 0, None, 0) == qwhip.E_BASIS   # rotation needs the workspace
    assert lib.qwhip_gemm_swiglu(st, C.byref(v4), xb.ptr, qwhip.BF16, 64, 0, 1, act.ptr, 0, qwhip.X_PREROTATED, None, 0) == qwhip.E_BAD_GEOMETRY
