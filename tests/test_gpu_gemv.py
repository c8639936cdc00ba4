"""GPU parity of the elementwise seams, the dequant side output and the decode / verify GEMV
(through the C ABI) against the CPU oracle.  Bars: bit-exact for rotated activations and
dequantized f16 weights; normalized error <= 2e-3 against the fp64 evaluation of
dequant + matmul for outputs."""
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


def _bf16(x32):
    return qo.f32_to_bf16_bits(x32)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
def test_fwht32_bit_exact(dev, dtype):
    x = H.make_x(7, 640, 1)
    if dtype == "f16":
        host, code, ref_in = x.astype(np.float16), qwhip.F16, x.astype(np.float16).astype(np.float32)
    elif dtype == "bf16":
        host, code, ref_in = _bf16(x), qwhip.BF16, qo.round_bf16(x)
    else:
        host, code, ref_in = x, qwhip.F32, x
    src = dev.put(host)
    dst = dev.alloc(x.size * 2)
    qwhip.check(dev.lib.qwhip_fwht32(dev.stream.handle, src.ptr, code, dst.ptr, x.size))
    got = dst.download(np.float16, x.shape)
    want = qo.fwht32_ortho(ref_in).astype(np.float16)
    assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("fmt", list(H.FORMATS))
def test_dequant_f16_bit_exact(dev, fmt):
    n, k = 24, 512
    blocks, w16 = H.make_bank(fmt, n, k, seed=3)
    bank = dev.put(blocks)
    out = dev.alloc(n * k * 2)
    view = H.view_of(dev, bank, fmt, n, k)
    qwhip.check(dev.lib.qwhip_dequant_f16(dev.stream.handle, C.byref(view), out.ptr))
    got = out.download(np.float16, (n, k))
    assert np.array_equal(got.view(np.uint16), w16.view(np.uint16))


def _run_gemv(dev, fmt, n, k, m, *, prerot, xdtype="f16", variant=0, rt=0, seed=0, outliers=False):
    blocks, w16 = H.make_bank(fmt, n, k, seed=seed)
    x32 = H.make_x(m, k, seed + 100, outliers=outliers)
    if xdtype == "f16":
        x_host, code = x32.astype(np.float16), qwhip.F16
        x_val = x_host.astype(np.float32)
    else:
        x_host, code = _bf16(x32), qwhip.BF16
        x_val = qo.round_bf16(x32)
    rotate = H.FORMATS[fmt][4]
    x_basis = (qo.fwht32_ortho(x_val) if rotate else x_val).astype(np.float16)   # what the kernel contracts
    if prerot:
        x_dev_host, code = x_basis, qwhip.F16
    else:
        x_dev_host = x_host
    bank = dev.put(blocks)
    xb = dev.put(x_dev_host)
    y16 = dev.alloc(m * n * 2)
    y32 = dev.alloc(m * n * 4)
    view = H.view_of(dev, bank, fmt, n, k)
    flags = (qwhip.X_PREROTATED if prerot else 0) | (variant << 8) | (rt << 12)
    qwhip.check(dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, code, m, flags, y16.ptr, y32.ptr))
    dev.stream.sync()
    g16 = y16.download(np.float16, (m, n))
    g32 = y32.download(np.float32, (m, n))
    ref = qo.matmul_ref_f64(x_basis, w16)
    for b in (bank, xb, y16, y32):
        b.free()
    return g16, g32, ref


@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("prerot", [False, True])
@pytest.mark.parametrize("n,k", [(256, 5120), (1000, 1024), (37, 96), (64, 32)])
def test_gemv_hq4_m1(dev, variant, prerot, n, k):
    g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", n, k, 1, prerot=prerot, variant=variant, outliers=True)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("kw", [0, 2, 4])
@pytest.mark.parametrize("prerot,xdtype", [(False, "f16"), (False, "bf16"), (True, "f16")])
@pytest.mark.parametrize("n,k,m", [(256, 5120, 1), (1000, 1024, 1), (72, 128, 2), (300, 2048, 5)])
def test_gemv_hq4_dma_streamer(dev, kw, prerot, xdtype, n, k, m):
    """The DMA streamer on HQ4_G32_M5: K-splits, fused rotation, ragged N, a ragged last step (k = 128 is half a step)."""
    g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", n, k, m, prerot=prerot, xdtype=xdtype, variant=3, rt=kw, outliers=True, seed=n)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["aq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64"])
@pytest.mark.parametrize("m", [1, 4, 16])
def test_gemv_blocks_dma_streamer_staged_activations(dev, fmt, m):
    """Pre-rotated f16 activations, m up to 16: per-step activation panels staged once per workgroup; few workgroups
    (deep prefetch ring) and many workgroups."""
    for n, k in [(200, 2048), (4096, 512)]:
        g16, g32, ref = _run_gemv(dev, fmt, n, k, m, prerot=True, variant=3, seed=m)
        assert qo.normalized_error(g32, ref) <= 2e-5
        assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("rt", [1, 2, 4])
@pytest.mark.parametrize("xdtype", ["f16", "bf16"])
def test_gemv_hq4_mfma_row_tiles_and_dtypes(dev, rt, xdtype):
    g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", 200, 2048, 1, prerot=False, xdtype=xdtype, variant=2, rt=rt)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["aq4_g32", "hq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64", "aq8_g256"])
@pytest.mark.parametrize("m", [1, 2, 3, 8, 16])
def test_gemv_blocks_small_m(dev, fmt, m):
    """The kernels that contract exact f16 weights on the matrix cores (override 2), fused rotation where the
    container is rotated."""
    g16, g32, ref = _run_gemv(dev, fmt, 272, 1536, m, prerot=False, seed=5, variant=2)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


def _affine_ref(fmt, n, k, m, seed, xdtype="f16"):
    """fp64 x . W^T with the un-rounded affine weights: what the factorised kernels compute."""
    kind, bits, group, is_m5, rotate = H.FORMATS[fmt]
    blocks, _ = H.make_bank(fmt, n, k, seed=seed)
    x32 = H.make_x(m, k, seed + 100)
    xv = x32.astype(np.float16).astype(np.float32) if xdtype == "f16" else qo.round_bf16(x32)
    xb = (qo.fwht32_ortho(xv) if rotate else xv).astype(np.float16).astype(np.float64)
    return xb @ qo.weights_affine_f64(blocks, bits, group, is_m5).T


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64", "aq8_g256"])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8])
def test_gemv_column_stationary_small_m(dev, fmt, m):
    """Column-stationary small-M kernel (override 6), activations handed over in the basis: tight against the
    factorised form it computes (scale * sum(code x) + bias * sum(x) per slice), and inside the judged bar against the
    f16-weight reference.  k = 1536 leaves the second 32-slice chunk half empty; n = 272 leaves ragged row sets."""
    g16, g32, ref = _run_gemv(dev, fmt, 272, 1536, m, prerot=True, seed=5, variant=6)
    assert qo.normalized_error(g32, _affine_ref(fmt, 272, 1536, m, 5)) <= 2e-5
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt,m,xdtype", [("aq4_g32", 1, "bf16"), ("aq8_g256", 4, "bf16"), ("aq4_g32", 3, "bf16"), ("aq4_g32", 2, "f16")])
def test_gemv_column_stationary_is_the_automatic_choice_for_unrotated_containers(dev, fmt, m, xdtype):
    """Standard-basis containers need no rotation: the automatic dispatch takes the column-stationary kernel, bf16 and
    f16 activations."""
    g16, g32, ref = _run_gemv(dev, fmt, 300, 2048, m, prerot=False, xdtype=xdtype, seed=9)
    assert qo.normalized_error(g32, _affine_ref(fmt, 300, 2048, m, 9, xdtype)) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g32", "hq4_g64", "hq8_g32", "hq8_g64"])
@pytest.mark.parametrize("xdtype", ["f16", "bf16"])
@pytest.mark.parametrize("n,k", [(272, 1536), (96, 17408), (40, 64)])
def test_gemv_column_stationary_fused_rotation(dev, fmt, xdtype, n, k):
    """One un-rotated activation row: the kernel rotates it on the matrix cores in its prologue (override 6)."""
    g16, g32, ref = _run_gemv(dev, fmt, n, k, 1, prerot=False, xdtype=xdtype, seed=7, variant=6)
    assert qo.normalized_error(g32, _affine_ref(fmt, n, k, 1, 7, xdtype)) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64", "aq8_g256"])
@pytest.mark.parametrize("m", [1, 3, 5, 8, 13, 16])
def test_gemv_block_mfma_kernel(dev, fmt, m):
    """4x4x4-block MFMA kernel (override 7), activations handed over in the basis: tight against the factorised form,
    inside the judged bar against the f16-weight reference.  n = 270 ends in a partial row quad, k = 1536 = 3 chunks
    of 16 slices."""
    g16, g32, ref = _run_gemv(dev, fmt, 270, 1536, m, prerot=True, seed=5, variant=7)
    assert qo.normalized_error(g32, _affine_ref(fmt, 270, 1536, m, 5)) <= 2e-5
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt,n,k,m,xdtype", [("hq4_g64", 96, 17408, 8, "f16"), ("hq4_g64", 50, 17408, 16, "f16"),
                                              ("aq4_g32", 300, 2080, 6, "bf16"), ("aq8_g256", 64, 5120, 16, "bf16"),
                                              ("hq8_g32", 5, 64, 2, "f16")])
def test_gemv_block_mfma_kernel_k_ranges_and_dtypes(dev, fmt, n, k, m, xdtype):
    """Long rows take several K ranges (k = 17408: three ranges of 12 chunks, partials accumulate in LDS); k = 2080 ends
    in a partial chunk; bf16 activations on the standard-basis containers; a bank smaller than one row quad per set."""
    prerot = H.FORMATS[fmt][4]
    g16, g32, ref = _run_gemv(dev, fmt, n, k, m, prerot=prerot, xdtype=xdtype, seed=8, variant=7)
    assert qo.normalized_error(g32, _affine_ref(fmt, n, k, m, 8, "f16" if prerot else xdtype)) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64", "aq8_g256"])
@pytest.mark.parametrize("m", [1, 5, 16])
def test_gemv_transposing_mfma_kernel(dev, fmt, m):
    """Transposing MFMA kernel (override 8): coalesced loads parked in LDS, exact f16 weights on the matrix cores.
    n = 270 ends in a partial 16-row tile, k = 1536 = 3 chunks of 16 slices."""
    g16, g32, ref = _run_gemv(dev, fmt, 270, 1536, m, prerot=True, seed=5, variant=8)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt,n,k,m,xdtype", [("hq4_g64", 96, 17408, 16, "f16"), ("aq4_g32", 300, 2080, 6, "bf16"),
                                              ("aq8_g256", 64, 5120, 16, "bf16"), ("hq8_g32", 5, 64, 2, "f16"),
                                              ("hq8_g32", 1000, 5120, 13, "f16")])
def test_gemv_transposing_mfma_kernel_k_ranges_and_dtypes(dev, fmt, n, k, m, xdtype):
    """Long rows take several K ranges (partial tiles accumulate in LDS), a partial last chunk, bf16 activations, a bank
    smaller than one tile, several tile slots per workgroup."""
    prerot = H.FORMATS[fmt][4]
    g16, g32, ref = _run_gemv(dev, fmt, n, k, m, prerot=prerot, xdtype=xdtype, seed=8, variant=8)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "aq4_g32", "hq4_g32", "hq4_g64", "hq4_g128", "hq8_g32", "hq8_g64", "aq8_g256"])
@pytest.mark.parametrize("m", [2, 5, 8, 9, 16])
def test_gemv_split_k_mfma_kernel(dev, fmt, m):
    """Split-K MFMA kernel (override 9): slices land in LDS straight from the bank, exact f16 weights on the matrix cores.
    n = 270 ends in a partial 16-row tile; k = 1536 is one K range (outputs stored by the kernel itself)."""
    g16, g32, ref = _run_gemv(dev, fmt, 270, 1536, m, prerot=True, seed=5, variant=9)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt,n,k,m,xdtype,tune", [
    ("hq4_g64", 96, 17408, 16, "f16", 0),        # six K ranges, partial sums through the stream's scratch
    ("hq4_g64", 5120, 17408, 8, "f16", 0),       # the verify down projection: every compute unit busy
    ("aq4_g32", 300, 2176, 6, "bf16", 0x08),     # 32 KiB image: two ranges, the last one short and not whole windows
    ("aq8_g256", 64, 5120, 16, "bf16", 0),       # 8-bit stream, sixteen activation rows, four ranges
    ("hq8_g32", 5, 128, 2, "f16", 0),            # a bank smaller than a tile, a row shorter than one window
    ("hq4_g32_m5", 1000, 5120, 13, "f16", 3),    # three groups in flight
    ("hq4_g32_m5", 1000, 5120, 3, "f16", 0x24),  # four groups in flight, four waves per workgroup
    ("hq4_g128", 333, 4096, 7, "f16", 0x46),     # six groups in flight, two waves per workgroup
    ("hq8_g64", 700, 8192, 12, "f16", 0x18),     # 128 KiB image
])
def test_gemv_split_k_mfma_kernel_k_ranges_and_tunings(dev, fmt, n, k, m, xdtype, tune):
    prerot = H.FORMATS[fmt][4]
    g16, g32, ref = _run_gemv(dev, fmt, n, k, m, prerot=prerot, xdtype=xdtype, seed=8, variant=9, rt=tune)
    assert qo.normalized_error(g32, ref) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


def test_gemv_split_k_mfma_kernel_refusals_and_stream_order(dev):
    """Outside its envelope the override is refused before any launch; two calls in a row on one stream share the scratch of
    partial sums in stream order (the second, smaller call must not see the first one's sums)."""
    lib, st = dev.lib, dev.stream.handle
    blocks, _ = H.make_bank("hq4_g32_m5", 32, 160, 0)
    bank, xb, y = dev.put(blocks), dev.put(np.zeros((2, 160), np.float16)), dev.alloc(2 * 32 * 2)
    v = dev.view(bank, 32, 160, qwhip.KIND_HQ4_G32_M5)
    flags = qwhip.X_PREROTATED | (9 << 8)
    assert lib.qwhip_gemv(st, C.byref(v), xb.ptr, qwhip.F16, 2, flags, y.ptr, None) == qwhip.E_BAD_GEOMETRY      # k % 128
    v128 = dev.view(bank, 32, 128, qwhip.KIND_HQ4_G32_M5, nbytes=32 * 4 * 20)
    assert lib.qwhip_gemv(st, C.byref(v128), xb.ptr, qwhip.F16, 1, flags, y.ptr, None) == qwhip.E_BAD_GEOMETRY   # m = 1
    assert lib.qwhip_gemv(st, C.byref(v128), xb.ptr, qwhip.F16, 2, 9 << 8, y.ptr, None) == qwhip.E_BAD_GEOMETRY  # not in the basis
    for b in (bank, xb, y):
        b.free()
    for variant in (0, 9, 10):      # the automatic choice is the row-tile kernel's ranges
        for n, k, m in ((640, 17408, 16), (96, 8192, 6)):
            g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", n, k, m, prerot=True, seed=n, variant=variant)
            assert qo.normalized_error(g32, ref) <= 2e-5

_ROWS_FORMATS = ["hq4_g32_m5", "aq4_g32", "hq4_g128", "hq8_g32", "aq8_g256", "aq2_g64", "hq3_g32", "aq6_g128"]


@pytest.mark.parametrize("fmt", _ROWS_FORMATS)
@pytest.mark.parametrize("n,k,m,xdtype", [
    (270, 1536, 2, "f16"),       # one step a wave, a partial row tile
    (5, 256, 7, "bf16"),         # a bank smaller than a tile, two waves
    (37, 1792, 16, "f16"),       # every activation row there
    (1000, 2304, 12, "bf16"),    # two steps a wave, the last wave half empty
    (16 * 300 + 3, 512, 13, "f16"),   # several tiles a workgroup, the last sum short
    (300, 4352, 5, "f16"),       # four steps a wave
    (96, 6400, 9, "f16"),        # two K ranges, partial sums through the stream's scratch
    (50, 17408, 3, "bf16"),      # three K ranges
])
def test_gemv_row_tile_kernel(dev, fmt, n, k, m, xdtype):
    """Row-tile kernel (override 10): tight against what it computes - the codes' own weights up to 12 rows, the exact f16 weights on
    13 and more (4- and 8-bit banks) and on six and more long 4-bit rows.  fp32 sums: K products of two exact f16, one rounding a
    slice and product of 32; 2e-6 is about three times the largest error measured against 64 bits (7.5e-7)."""
    g16, g32, ref = _run_gemv(dev, fmt, n, k, m, prerot=True, xdtype=xdtype, seed=5, variant=10)
    four = fmt in ("hq4_g32_m5", "aq4_g32", "hq4_g128")
    exact_f16 = (four or "8_" in fmt) and (m >= 13 or (four and m >= 6 and k >= 8192))
    assert qo.normalized_error(g32, ref if exact_f16 else _affine_ref(fmt, n, k, m, 5, xdtype)) <= 2e-6
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("tune", range(1, 8))
@pytest.mark.parametrize("k", [640, 2560, 5120])
def test_gemv_row_tile_kernel_steps_codes(dev, k, tune):
    """Any code for the steps a wave contracts every column (5 steps, 20 and 40 of 128 columns)."""
    _, g32, _ = _run_gemv(dev, "hq4_g32_m5", 100, k, 8, prerot=True, seed=5, variant=10, rt=tune)
    assert qo.normalized_error(g32, _affine_ref("hq4_g32_m5", 100, k, 8, 5, "f16")) <= 2e-6


@pytest.mark.parametrize("tune", [0x08, 0x10, 0x18])
def test_gemv_row_tile_kernel_workgroups_code(dev, tune):
    """The code for the workgroups a unit: the grid alone changes, also where LDS holds fewer (twelve waves, several tiles each)."""
    n, k, m = 64 * 577, 6144, 5
    bank = dev.put(np.tile(H.make_bank("hq4_g32_m5", 64, k, 3)[0].reshape(-1), 577))
    xb, y = dev.put(H.make_x(m, k, 4).astype(np.float16)), dev.alloc(m * n * 4)
    view, outs = H.view_of(dev, bank, "hq4_g32_m5", n, k), []
    for code in (0, tune):
        qwhip.check(dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, qwhip.X_PREROTATED | (10 << 8) | (code << 12), None, y.ptr))
        dev.stream.sync()
        outs.append(y.download(np.uint32, (m, n)))
    for b in (bank, xb, y):
        b.free()
    assert np.array_equal(*outs) and np.array_equal(outs[0][:, :64], outs[0][:, -64:])


def test_gemv_row_tile_kernel_reads_its_code_where_it_is_named(dev):
    """Tuning bits without an override leave the automatic choice's sums alone; with the override another split of the columns over the
    waves adds in another order."""
    runs = [_run_gemv(dev, "hq4_g32_m5", 64, 1024, 8, prerot=True, seed=5, variant=v, rt=rt)[1] for v, rt in ((0, 0), (0, 2), (0, 4), (10, 0), (10, 4))]
    assert all(np.array_equal(runs[0], r) for r in runs[1:4]) and not np.array_equal(runs[0], runs[4])


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq8_g64", "hq3_g32", "aq6_g128"])
@pytest.mark.parametrize("m", [5, 16])
def test_gemv_row_tile_kernel_keeps_an_infinity_in_its_row(dev, fmt, m):
    """The m activation rows share the instructions: a row that is not finite leaves the others' bits alone."""
    n, k = 48, 1536
    blocks, _ = H.make_bank(fmt, n, k, 3)
    x16 = H.make_x(m, k, 4).astype(np.float16)
    bad = x16.copy()
    bad[2, 700] = np.inf
    bank, outs = dev.put(blocks), []
    view = H.view_of(dev, bank, fmt, n, k)
    for x in (x16, bad):
        xb, y = dev.put(x), dev.alloc(m * n * 4)
        qwhip.check(dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, qwhip.X_PREROTATED | (10 << 8), None, y.ptr))
        dev.stream.sync()
        outs.append(y.download(np.float32, (m, n)))
        xb.free()
        y.free()
    bank.free()
    rest = [i for i in range(m) if i != 2]
    assert np.array_equal(outs[0][rest].view(np.uint32), outs[1][rest].view(np.uint32))
    assert not np.isfinite(outs[1][2]).any()


@pytest.mark.parametrize("m", [8, 12])
def test_gemv_row_tile_kernel_weights_follow_the_shape(dev, m):
    """The plain door, whose planes have all of the partial-sum area, and the gate|up door, whose image takes a part of it, contract the
    same weights: the bits of one are those of the other and the activation pass."""
    reps, k = 8 * 1094 // m, 8192
    n = 64 * reps
    bank = dev.put(np.tile(H.make_bank("hq4_g32_m5", 64, k, 3)[0].reshape(-1), reps))
    xb, gu, a1, a2 = dev.put(H.make_x(m, k, 4).astype(np.float16)), dev.alloc(m * n * 4), dev.alloc(m * n), dev.alloc(m * n)
    view, lib, st, fl = H.view_of(dev, bank, "hq4_g32_m5", n, k), dev.lib, dev.stream.handle, qwhip.X_PREROTATED
    qwhip.check(lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, m, fl, None, gu.ptr))
    qwhip.check(lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F32, a2.ptr, m, n // 2, 0))
    qwhip.check(lib.qwhip_gemv_silu_pair(st, C.byref(view), xb.ptr, qwhip.F16, m, fl, 0, a1.ptr))
    dev.stream.sync()
    one, two = a1.download(np.uint16, (m, n // 2)), a2.download(np.uint16, (m, n // 2))
    for b in (bank, xb, gu, a1, a2):
        b.free()
    assert np.array_equal(one, two)


def test_gemv_row_tile_kernel_longest_rows(dev):
    """256 ranges of 6144 columns; one step more, and rows of 25 million columns, are refused on the host: more ranges than compute units
    would divide by zero."""
    k = 256 * 6144
    g32, ref = _run_gemv(dev, "hq4_g32_m5", 16, k, 2, prerot=True, seed=5, variant=10)[1:]
    assert qo.normalized_error(g32, ref) <= TOL      # the codes against their f16 weights
    bank, xb, y = dev.alloc(16 * (k + 128) // 32 * 20), dev.alloc(2 * (k + 128) * 2), dev.alloc(2 * 16 * 4)
    v = dev.view(bank, 16, k + 128, qwhip.KIND_HQ4_G32_M5)
    assert dev.lib.qwhip_gemv(dev.stream.handle, C.byref(v), xb.ptr, qwhip.F16, 2, qwhip.X_PREROTATED | (10 << 8), None, y.ptr) == qwhip.E_BAD_GEOMETRY
    v = dev.view(bank, 1, 16 * (k + 128), qwhip.KIND_HQ4_G32_M5)
    assert dev.lib.qwhip_gemv(dev.stream.handle, C.byref(v), xb.ptr, qwhip.F16, 2, qwhip.X_PREROTATED | (10 << 8), None, y.ptr) == qwhip.E_BAD_GEOMETRY
    for b in (bank, xb, y):
        b.free()


def test_gemv_row_tile_kernel_refuses_what_was_refused(dev):
    """Rows in the basis only, two to sixteen; 2-, 3- and 6-bit rows too long for the dot2 kernel are refused by the automatic choice."""
    lib, st = dev.lib, dev.stream.handle
    blocks, _ = H.make_bank("hq6_g32", 32, 17408, 0)
    bank, xb, y = dev.put(blocks), dev.put(np.zeros((7, 17408), np.float16)), dev.alloc(7 * 32 * 4)
    v = H.view_of(dev, bank, "hq6_g32", 32, 17408)
    assert lib.qwhip_gemv(st, C.byref(v), xb.ptr, qwhip.F16, 7, qwhip.X_PREROTATED, None, y.ptr) == qwhip.E_BAD_GEOMETRY
    assert lib.qwhip_gemv(st, C.byref(v), xb.ptr, qwhip.F16, 7, 10 << 8, None, y.ptr) == qwhip.E_BAD_GEOMETRY
    assert lib.qwhip_gemv(st, C.byref(v), xb.ptr, qwhip.F16, 1, qwhip.X_PREROTATED | (10 << 8), None, y.ptr) == qwhip.E_BAD_GEOMETRY
    for b in (bank, xb, y):
        b.free()


@pytest.mark.parametrize("fmt", _ROWS_FORMATS)
@pytest.mark.parametrize("inter,k,m,rot_out", [(32, 512, 2, 1), (160, 1536, 6, 1), (176, 2560, 13, 0), (48, 5120, 16, 0), (4128, 1024, 3, 1)])
def test_gemv_silu_pair_row_tiles(dev, fmt, inter, k, m, rot_out):
    """The gated form (16 or, rotated, 32 channels a unit; 4128 channels leave workgroups a second one): bit for bit the plain row-tile
    GEMV, the gated activation and the rotation one after the other, whose sums and roundings are the same."""
    blocks, _ = H.make_bank(fmt, 2 * inter, k, seed=inter)
    x16 = H.make_x(m, k, 9).astype(np.float16)
    xb, bank = dev.put(x16), dev.put(blocks)
    a1, a2, gu = dev.alloc(m * inter * 2), dev.alloc(m * inter * 2), dev.alloc(m * 2 * inter * 4)
    view = H.view_of(dev, bank, fmt, 2 * inter, k)
    st, fl = dev.stream.handle, qwhip.X_PREROTATED
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(st, C.byref(view), xb.ptr, qwhip.F16, m, fl, rot_out, a1.ptr))
    qwhip.check(dev.lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, m, fl | (10 << 8), None, gu.ptr))
    qwhip.check(dev.lib.qwhip_swiglu_fwht(st, gu.ptr, qwhip.F32, a2.ptr, m, inter, rot_out))
    dev.stream.sync()
    one, two = a1.download(np.uint16, (m, inter)), a2.download(np.uint16, (m, inter))
    for b in (bank, xb, a1, a2, gu):
        b.free()
    assert np.array_equal(one, two)


@pytest.mark.parametrize("fmt", ["aq2_g64", "hq3_g32", "hq6_g32", "aq6_g128"])
@pytest.mark.parametrize("m", [1, 3, 8, 12])
def test_gemv_narrow_and_six_bit_streams(dev, fmt, m):
    """2-, 3- and 6-bit containers (QWAQBlock.supported, QWAQBlock.swift:17-23) on the column-stationary dot2 kernel:
    rows already in the basis, eight per launch; tight against the factorised form, inside the judged bar against the
    f16-weight reference."""
    g16, g32, ref = _run_gemv(dev, fmt, 272, 1536, m, prerot=True, seed=5)
    assert qo.normalized_error(g32, _affine_ref(fmt, 272, 1536, m, 5)) <= 2e-5
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("fmt", ["hq3_g32", "hq6_g32"])
@pytest.mark.parametrize("xdtype", ["f16", "bf16"])
def test_gemv_narrow_streams_fused_rotation_and_basis_errors(dev, fmt, xdtype):
    """One un-rotated row is rotated in the prologue; several un-rotated rows are rotated once into the stream's scratch
    and then run as rows in the basis; under a kernel override there is no such pass and the rows are refused
    (QWHIP_E_BASIS) before any launch."""
    g16, g32, ref = _run_gemv(dev, fmt, 100, 2048, 1, prerot=False, xdtype=xdtype, seed=7)
    assert qo.normalized_error(g32, _affine_ref(fmt, 100, 2048, 1, 7, xdtype)) <= 2e-5
    g16, g32, ref = _run_gemv(dev, fmt, 100, 2048, 11, prerot=False, xdtype=xdtype, seed=8)
    assert qo.normalized_error(g32, _affine_ref(fmt, 100, 2048, 11, 8, xdtype)) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL
    blocks, _ = H.make_bank(fmt, 64, 256, seed=1)
    bank, xb, yb = dev.put(blocks), dev.put(np.zeros((4, 256), np.float16)), dev.alloc(4 * 64 * 4)
    view = H.view_of(dev, bank, fmt, 64, 256)
    st = dev.stream.handle
    assert dev.lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, 4, 6 << 8, None, yb.ptr) == qwhip.E_BASIS


@pytest.mark.parametrize("fmt,n,k", [("hq4_g32_m5", 300, 5120), ("hq8_g32", 272, 1536), ("hq4_g64", 96, 17408), ("hq6_g32", 130, 2048)])
@pytest.mark.parametrize("m", [2, 5, 16])
@pytest.mark.parametrize("xdtype", ["f16", "bf16"])
def test_gemv_several_unrotated_rows_equal_the_rows_rotated_first(dev, fmt, n, k, m, xdtype):
    """A rotated container given m > 1 un-rotated rows: the launcher's rotation pass + the kernels for rows in the basis.
    Bit-identical to qwhip_fwht32 followed by the pre-rotated call (the same two steps done by the caller), except where
    two rows stay on a streamer kernel."""
    blocks, w16 = H.make_bank(fmt, n, k, seed=21)
    x32 = H.make_x(m, k, 121)
    if xdtype == "f16":
        x_host, code = x32.astype(np.float16), qwhip.F16
    else:
        x_host, code = _bf16(x32), qwhip.BF16
    bank, xb = dev.put(blocks), dev.put(x_host)
    xr, ya, yb_ = dev.alloc(m * k * 2), dev.alloc(m * n * 4), dev.alloc(m * n * 4)
    view = H.view_of(dev, bank, fmt, n, k)
    st = dev.stream.handle
    qwhip.check(dev.lib.qwhip_gemv(st, C.byref(view), xb.ptr, code, m, 0, None, ya.ptr))
    qwhip.check(dev.lib.qwhip_fwht32(st, xb.ptr, code, xr.ptr, m * k))
    qwhip.check(dev.lib.qwhip_gemv(st, C.byref(view), xr.ptr, qwhip.F16, m, qwhip.X_PREROTATED, None, yb_.ptr))
    dev.stream.sync()
    a, b = ya.download(np.float32, (m, n)), yb_.download(np.float32, (m, n))
    x_basis = xr.download(np.float16, (m, k))
    for buf in (bank, xb, xr, ya, yb_):
        buf.free()
    if m == 2 and k <= 8192:   # two rows on a small bank stay on a streamer (rotation in its prologue, exact f16 weights)
        assert qo.normalized_error(a, b) <= 1e-3
    else:
        assert np.array_equal(a, b)
    assert qo.normalized_error(a, qo.matmul_ref_f64(x_basis, w16)) <= TOL


@pytest.mark.parametrize("m", [1, 4])
def test_gemv_column_stationary_long_rows(dev, m):
    """k = 17408: 17 half-waves per row, one row set per workgroup."""
    g16, g32, ref = _run_gemv(dev, "hq4_g64", 96, 17408, m, prerot=True, seed=6, variant=6)
    assert qo.normalized_error(g32, _affine_ref("hq4_g64", 96, 17408, m, 6)) <= 2e-5
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("m", [2, 16])
def test_gemv_rotation_per_lane_path(dev, m):
    """m*k too large for the LDS staging: on the MFMA streamer (kernel override 2) the rotation runs per lane from global
    memory."""
    g16, g32, ref = _run_gemv(dev, "hq4_g64", 96, 17408, m, prerot=False, seed=6, variant=2)
    assert qo.normalized_error(g32, ref) <= 2e-5


@pytest.mark.parametrize("fmt,flags", [("hq4_g32_m5", 0), ("hq4_g32_m5", 2 << 8), ("hq4_g64", 0), ("aq8_g256", 0), ("aq2_g64", 0), ("hq3_g32", 0),
                                       ("hq6_g32", 0), ("aq6_g128", 0)])
@pytest.mark.parametrize("m", [1, 3])
@pytest.mark.parametrize("prerot,rot_out", [(False, 1), (True, 1), (True, 0)])
def test_gemv_silu_pair_matches_oracle(dev, fmt, flags, m, prerot, rot_out):
    """gate|up GEMV with the SwiGLU epilogue (EncodeKernels.swift:298-326): act = f16(FWHT32(silu(Wg.x) * (Wu.x))) on
    fp32 accumulators; HQ4_G32_M5 on the column-stationary kernel and (override 2) on the general one."""
    inter, k = 160, 1536
    kind, bits, group, is_m5, rotate = H.FORMATS[fmt]
    blocks, w16 = H.make_bank(fmt, 2 * inter, k, seed=12)
    x16 = H.make_x(m, k, 112).astype(np.float16)
    x_basis = H.x_in_basis(x16, fmt)
    xb = dev.put(x_basis if prerot else x16)
    bank, act = dev.put(blocks), dev.alloc(m * inter * 2)
    view = H.view_of(dev, bank, fmt, 2 * inter, k)
    fl = (qwhip.X_PREROTATED if prerot else 0) | flags
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, fl, rot_out, act.ptr))
    dev.stream.sync()
    got = act.download(np.float16, (m, inter)).astype(np.float32)
    gu = qo.matmul_ref_f64(x_basis, w16)
    want = qo.swiglu_fwht_f16(gu[:, :inter].astype(np.float32), gu[:, inter:].astype(np.float32), rotate=bool(rot_out)).astype(np.float32)
    assert qo.normalized_error(got, want) <= TOL
    for b in (bank, xb, act):
        b.free()


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "hq8_g32", "aq2_g64", "hq3_g32", "aq6_g128"])
@pytest.mark.parametrize("inter,k", [(160, 1536), (100, 5120), (777, 4096), (64, 12288), (2080, 2048)])
@pytest.mark.parametrize("prerot,rot_out", [(False, 0), (True, 0), (True, 1)])
def test_gemv_silu_pair_one_row_forms(dev, fmt, inter, k, prerot, rot_out, xdt):
    """One activation row: the gate|up forms of the one-row GEMV kernels (gate and up rows of a channel in neighbouring row
    slots of one workgroup, the bank walked as two bands; with the output rotation a rotation pass over the fp32 gated values
    behind the launch).  Against the oracle, and against the kernel the door used before on the same call (flags bits 8..11:
    3 = the MoE decode kernel for HQ4_G32_M5, 2 = the general kernel), which sums in another order: both within the bar of the
    reference and within 1e-3 of each other.  Odd channel counts, channel counts below and above a workgroup's share, rows of
    48 to 384 blocks, the input rotation fused or the row handed over rotated, f16 and bf16 rows."""
    kind, bits, group, is_m5, rotated = H.FORMATS[fmt]
    blocks, w16 = H.make_bank(fmt, 2 * inter, k, seed=inter + k)
    x32 = H.make_x(1, k, 7)
    if xdt == "f16":
        code, x16 = qwhip.F16, x32.astype(np.float16)
        x_basis = H.x_in_basis(x16, fmt)                        # f16: what the fused rotation leaves, or what is handed over
        xin = x_basis if prerot else x16
    else:
        code = qwhip.BF16
        if prerot and rotated:                                  # the producer's rotation in fp32, one bf16 rounding
            xin = qo.f32_to_bf16_bits(qo.fwht32_ortho(x32))
            x_basis = qo.bf16_bits_to_f32(xin)
        else:
            xin = qo.f32_to_bf16_bits(x32)
            x_basis = H.x_in_basis(qo.round_bf16(x32), fmt)
    xb, bank = dev.put(xin), dev.put(blocks)
    a1, a2 = dev.put(np.full(inter, 3, np.float16)), dev.put(np.full(inter, 5, np.float16))
    view = H.view_of(dev, bank, fmt, 2 * inter, k)
    fl = qwhip.X_PREROTATED if prerot else 0
    before = (3 << 8) if is_m5 else (2 << 8)
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(dev.stream.handle, C.byref(view), xb.ptr, code, 1, fl, rot_out, a1.ptr))
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(dev.stream.handle, C.byref(view), xb.ptr, code, 1, fl | before, rot_out, a2.ptr))
    dev.stream.sync()
    one = a1.download(np.float16, (1, inter)).astype(np.float32)
    two = a2.download(np.float16, (1, inter)).astype(np.float32)
    gu = qo.matmul_ref_f64(np.asarray(x_basis, np.float32).reshape(1, k), w16)
    want = qo.swiglu_fwht_f16(gu[:, :inter].astype(np.float32), gu[:, inter:].astype(np.float32),
                              rotate=bool(rot_out) and inter % 32 == 0).astype(np.float32)
    assert qo.normalized_error(one, want) <= TOL and qo.normalized_error(two, want) <= TOL
    assert qo.normalized_error(one, two) <= 1e-3
    for b in (bank, xb, a1, a2):
        b.free()


@pytest.mark.parametrize("fmt", ["hq4_g32_m5", "hq4_g64", "hq8_g32", "aq2_g64"])
@pytest.mark.parametrize("m", [2, 5, 8, 16])
@pytest.mark.parametrize("inter,k,prerot,rot_out", [(160, 1536, True, 1), (96, 17408, True, 1), (777, 4096, True, 0), (160, 1536, False, 1)])
def test_gemv_silu_pair_several_rows_read_the_bank_once(dev, fmt, m, inter, k, prerot, rot_out):
    """Two to sixteen rows: the verify GEMV over the whole gate|up bank into an fp32 image in the stream's scratch, then the
    gated activation (+ rotation) pass.  Against the oracle and against the kernel the door used before (flags bits 8..11: 3 /
    2).  K = 17408 sends the 4-bit banks through the split-K GEMV, whose partial sums share the scratch with the image."""
    kind, bits, group, is_m5, rotated = H.FORMATS[fmt]
    if not prerot and not rotated:
        pytest.skip("plain container: nothing to rotate")
    blocks, w16 = H.make_bank(fmt, 2 * inter, k, seed=inter + k + m)
    x16 = H.make_x(m, k, 9).astype(np.float16)
    x_basis = H.x_in_basis(x16, fmt)
    xb, bank = dev.put(x_basis if prerot else x16), dev.put(blocks)
    a1, a2 = dev.put(np.full((m, inter), 3, np.float16)), dev.put(np.full((m, inter), 5, np.float16))
    view = H.view_of(dev, bank, fmt, 2 * inter, k)
    fl = qwhip.X_PREROTATED if prerot else 0
    before = (3 << 8) if is_m5 else (2 << 8)
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, fl, rot_out, a1.ptr))
    qwhip.check(dev.lib.qwhip_gemv_silu_pair(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, fl | before, rot_out, a2.ptr))
    dev.stream.sync()
    one = a1.download(np.float16, (m, inter)).astype(np.float32)
    two = a2.download(np.float16, (m, inter)).astype(np.float32)
    gu = qo.matmul_ref_f64(x_basis, w16)
    want = qo.swiglu_fwht_f16(gu[:, :inter].astype(np.float32), gu[:, inter:].astype(np.float32),
                              rotate=bool(rot_out) and inter % 32 == 0).astype(np.float32)
    assert qo.normalized_error(one, want) <= TOL and qo.normalized_error(two, want) <= TOL
    assert qo.normalized_error(one, two) <= 1e-3
    for b in (bank, xb, a1, a2):
        b.free()


def test_gemv_affine_known_answer(dev):
    """Code 1, scale 1.0, bias 0.25, x = one-hot: every output is exactly 1.25 - the -1024 must be
    stripped before the FMA, not folded into an f16 bias
    (Tests/QWGEMMTests/QWAQBatchedGemmTests.swift:194-205)."""
    n, k = 64, 128
    blocks = np.zeros((n, k // 32, 20), dtype=np.uint8)
    blocks[..., 0:2] = np.array([1.0], dtype=np.float16).view(np.uint8)
    blocks[..., 2:4] = np.array([0.25], dtype=np.float16).view(np.uint8)
    blocks[..., 4:] = 0x11
    x = np.zeros((1, k), dtype=np.float16)
    x[0, 5] = 1.0
    bank, xb, y32 = dev.put(blocks), dev.put(x), dev.alloc(n * 4)
    view = dev.view(bank, n, k, qwhip.KIND_NATIVE_AFFINE, 4, 32)
    qwhip.check(dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, 1, 0, None, y32.ptr))
    got = y32.download(np.float32, (n,))
    assert np.all(got == np.float32(1.25))


_FULL = {}


def _full_bank(dev, fmt, n, k):
    """One bank per BASELINE shape, quantized once per session and kept on the device."""
    key = (fmt, n, k)
    if key not in _FULL:
        blocks, w16 = H.make_bank(fmt, n, k, seed=0)
        _FULL[key] = (dev.put(blocks), w16)
    return _FULL[key]


def _run_full(dev, fmt, n, k, m, *, prerot, variant=0, outliers=False, seed=0):
    bank, w16 = _full_bank(dev, fmt, n, k)
    x16 = H.make_x(m, k, seed + 100, outliers=outliers).astype(np.float16)
    x_basis = H.x_in_basis(x16, fmt)
    xb = dev.put(x_basis if prerot else x16)
    y16, y32 = dev.alloc(m * n * 2), dev.alloc(m * n * 4)
    view = H.view_of(dev, bank, fmt, n, k)
    flags = (qwhip.X_PREROTATED if prerot else 0) | (variant << 8)
    qwhip.check(dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, m, flags, y16.ptr, y32.ptr))
    dev.stream.sync()
    g16, g32 = y16.download(np.float16, (m, n)), y32.download(np.float32, (m, n))
    for b in (xb, y16, y32):
        b.free()
    return g16, g32, qo.matmul_ref_f64(x_basis, w16)


@pytest.mark.parametrize("variant", [0, 4, 1, 2, 3])
def test_gemv_full_size_decode_config(dev, variant):
    """HQ4_G32 decode GEMV at its benchmark shape (K = 5120, N = 17408, outliers, fused rotation): the automatic
    dispatch (0) and the column-stationary kernel it picks (4), then the other kernels that take the shape."""
    g16, g32, ref = _run_full(dev, "hq4_g32_m5", 17408, 5120, 1, prerot=False, variant=variant, outliers=True)
    assert qo.normalized_error(g32, ref) <= (3e-4 if variant in (0, 4) else 2e-5)   # 0 / 4 skip the f16 rounding of each weight
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("variant", [0, 4])
@pytest.mark.parametrize("prerot", [False, True])
@pytest.mark.parametrize("k", [1024, 3072, 3104, 4096, 5120, 12288, 13312, 17408, 22528, 24576])
def test_gemv_hq4_column_stationary_row_lengths(dev, variant, prerot, k):
    """The automatic m = 1 HQ4_G32_M5 kernel across its launch forms: 4, 2 and 1 row sets per workgroup (k <= 3072,
    <= 12288, above), an odd number of 32-block chunks per row with one row set (k = 13312, 17408: the workgroup ends in
    a half wave), a last chunk that is not full (k = 3104), a long row it takes (22528) and one whose activation image no longer fits its
    LDS budget (24576: the automatic dispatch falls back to the half-wave kernel, the override refuses); n = 300 leaves ragged
    row slots.  Tight against the factorised form it computes, inside the judged bar against the f16-weight reference."""
    if k == 24576 and variant == 4:
        blocks, _ = H.make_bank("hq4_g32_m5", 8, k, seed=1)
        bank, xb, yb = dev.put(blocks), dev.put(np.zeros((1, k), np.float16)), dev.alloc(8 * 4)
        view = H.view_of(dev, bank, "hq4_g32_m5", 8, k)
        assert dev.lib.qwhip_gemv(dev.stream.handle, C.byref(view), xb.ptr, qwhip.F16, 1, 4 << 8, None, yb.ptr) == qwhip.E_BAD_GEOMETRY
        return
    g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", 300, k, 1, prerot=prerot, variant=variant, outliers=True, seed=11)
    blocks, _ = H.make_bank("hq4_g32_m5", 300, k, seed=11)
    x16 = H.make_x(1, k, 111, outliers=True).astype(np.float16)
    xb = qo.rotate_activation_f16(x16).astype(np.float64)
    if k < 24576:
        assert qo.normalized_error(g32, xb @ qo.weights_affine_f64(blocks, 4, 32, True).T) <= 2e-5
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("tune", [0, 1, 2, 3, 4, 5, 0 | (1 << 3), 0 | (2 << 3), 4 | (3 << 3), 0 | (1 << 5), 5 | (1 << 5) | (2 << 3)])
@pytest.mark.parametrize("n,k,xdtype", [(17408, 5120, "f16"), (300, 5120, "bf16"), (1031, 4096, "f16"), (45, 8192, "f16"), (7, 1024, "f16"),
                                        (513, 17408, "f16"), (2050, 3104, "bf16")])
def test_gemv_hq4_column_stationary_windows(dev, tune, n, k, xdtype):
    """Every form of the m = 1 HQ4_G32_M5 column-stationary kernel (override 4, tuning codes: the hand-issued windows of
    (3, 2), (2, 2), (3, 3), (4, 2), (6, 3) rows, the compiled window, half / double / one-and-a-half grids, four row sets)
    on row counts that leave ragged row slots, short sets (a set one row short re-reads), fewer rows than a window, a
    partly filled last chunk (k = 3104) and a workgroup that ends in a half wave (k = 17408).  The hand-issued forms sum a
    row's blocks in the same order with the same roundings: equal bits, whatever the window and the grid (the compiled
    window keeps four partial sums per block where they keep two, so it agrees to rounding only)."""
    g16, g32, ref = _run_gemv(dev, "hq4_g32_m5", n, k, 1, prerot=False, xdtype=xdtype, variant=4, rt=tune, outliers=True, seed=5)
    assert qo.normalized_error(g32, ref) <= TOL and qo.normalized_error(g16, ref) <= TOL
    if tune & 7 != 1:
        b16, b32, _ = _run_gemv(dev, "hq4_g32_m5", n, k, 1, prerot=False, xdtype=xdtype, variant=4, rt=0, outliers=True, seed=5)
        assert np.array_equal(g32.view(np.uint32), b32.view(np.uint32)) and np.array_equal(g16.view(np.uint16), b16.view(np.uint16))


@pytest.mark.parametrize("fmt,n,k", [("hq8_g32", 7168, 5120), ("hq4_g64", 5120, 17408), ("hq4_g32_m5", 1000, 5120), ("aq4_g32", 512, 4096),
                                     ("hq4_g32", 300, 2048), ("hq8_g64", 256, 1024), ("aq2_g64", 256, 2048), ("hq3_g32", 200, 3072),
                                     ("hq6_g32", 256, 5120), ("hq4_g128", 384, 8192), ("aq8_g256", 128, 16384), ("hq4_g32_m5", 96, 17408)])
@pytest.mark.parametrize("prerot", [True, False])
def test_gemv_row_invariant_mode_rows_together_equal_rows_alone(dev, fmt, n, k, prerot):
    """QWHIP_GEMV_ROW_INVARIANT: for m in {2, 4, 8, 16} every row of the batched call carries the bits of the same row in a
    call of its own (the reference's 1-row vs 2-row check, Tests/QWGEMMTests/QWGemmAQDecodeTests.swift:150-173, made
    exact and taken to 16 rows) - on the two verify banks at their real shapes (q/k/v HQ8_G32 7168 x 5120, down HQ4_G64
    5120 x 17408) and on every container class, rows in the basis and rows the call rotates itself; the results stay
    inside the judged bar against the f16-weight reference."""
    rotated = H.FORMATS[fmt][4]
    if not rotated and not prerot:
        pytest.skip("a standard-basis container has no rotation to fuse")
    bank, w16 = _full_bank(dev, fmt, n, k)
    view = H.view_of(dev, bank, fmt, n, k)
    x16 = H.make_x(16, k, 77, outliers=True).astype(np.float16)
    x_basis = H.x_in_basis(x16, fmt)
    xb = dev.put(x_basis if prerot else x16)
    flags = qwhip.GEMV_ROW_INVARIANT | (qwhip.X_PREROTATED if prerot else 0)
    lib, st = dev.lib, dev.stream.handle
    y_one16, y_one32 = dev.alloc(16 * n * 2), dev.alloc(16 * n * 4)
    for r in range(16):                                   # every row alone
        qwhip.check(lib.qwhip_gemv(st, C.byref(view), xb.ptr + r * k * 2, qwhip.F16, 1, flags, y_one16.ptr + r * n * 2, y_one32.ptr + r * n * 4))
    dev.stream.sync()
    one16, one32 = y_one16.download(np.uint16, (16, n)), y_one32.download(np.uint32, (16, n))
    ref = qo.matmul_ref_f64(x_basis, w16)
    assert qo.normalized_error(one32.view(np.float32), ref) <= TOL
    y16, y32 = dev.alloc(16 * n * 2), dev.alloc(16 * n * 4)
    if prerot:      # a plain decode call (no flag) on a row in the basis gives those bits too: decode runs at full speed
        for r in (0, 5):
            qwhip.check(lib.qwhip_gemv(st, C.byref(view), xb.ptr + r * k * 2, qwhip.F16, 1, qwhip.X_PREROTATED, y16.ptr, y32.ptr))
            dev.stream.sync()
            assert np.array_equal(y32.download(np.uint32, (16, n))[0], one32[r]) and np.array_equal(y16.download(np.uint16, (16, n))[0], one16[r])
    for m in (2, 4, 8, 16, 3, 13):
        qwhip.check(lib.qwhip_fill_u32(st, y32.ptr, 0xFFFFFFFF, 16 * n))
        qwhip.check(lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, m, flags, y16.ptr, y32.ptr))
        dev.stream.sync()
        assert np.array_equal(y32.download(np.uint32, (16, n))[:m], one32[:m]), f"m={m}: fp32 rows differ from the rows alone"
        assert np.array_equal(y16.download(np.uint16, (16, n))[:m], one16[:m]), f"m={m}: f16 rows differ from the rows alone"
    assert lib.qwhip_gemv(st, C.byref(view), xb.ptr, qwhip.F16, 2, flags | (7 << 8), y16.ptr, y32.ptr) == qwhip.E_BAD_SHAPE   # no override in this mode
    for b in (xb, y_one16, y_one32, y16, y32):
        b.free()


def test_gemv_full_size_affine_config(dev):
    """C1: AQ4_G32 decode GEMV, N = 4096, K = 4096, automatic dispatch, standard basis."""
    g16, g32, ref = _run_full(dev, "aq4_g32", 4096, 4096, 1, prerot=False)
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


@pytest.mark.parametrize("m", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("fmt,n,k", [("hq8_g32", 7168, 5120), ("hq4_g64", 5120, 17408)])
def test_gemv_full_size_verify_configs(dev, fmt, n, k, m):
    """C5: the speculative-verify layer pair at its benchmark shapes (q/k/v HQ8_G32 7168 x 5120, down HQ4_G64
    5120 x 17408), automatic dispatch, m draft rows already in the weight basis (the producers' contract); m = 1 is the
    decode row, handed over un-rotated (rotation fused)."""
    g16, g32, ref = _run_full(dev, fmt, n, k, m, prerot=(m > 1), seed=m)
    assert qo.normalized_error(g32, ref) <= TOL
    assert qo.normalized_error(g16, ref) <= TOL


def test_gemv_full_size_down_projection_hq4_m5(dev):
    """The dense down projection of the benchmark model as an HQ4_G32_M5 bank (N = 5120, K = 17408), one un-rotated
    row: 17 chunks of 32 blocks per row, one row set per workgroup."""
    for variant in (0, 1):
        g16, g32, ref = _run_full(dev, "hq4_g32_m5", 5120, 17408, 1, prerot=False, variant=variant, outliers=True)
        assert qo.normalized_error(g32, ref) <= TOL
        assert qo.normalized_error(g16, ref) <= TOL


def test_gemv_rejects_bad_inputs_before_launch(dev):
    blocks, _ = H.make_bank("hq4_g32_m5", 8, 64, 0)
    bank, xb, y = dev.put(blocks), dev.put(np.zeros(64, np.float16)), dev.alloc(64)
    lib, st = dev.lib, dev.stream.handle
    short = dev.view(bank, 8, 64, qwhip.KIND_HQ4_G32_M5, nbytes=8 * 2 * 20 - 1)
    assert lib.qwhip_gemv(st, C.byref(short), xb.ptr, qwhip.F16, 1, 0, y.ptr, None) == qwhip.E_BAD_WEIGHTS
    badk = dev.view(bank, 8, 48, qwhip.KIND_HQ4_G32_M5)
    assert lib.qwhip_gemv(st, C.byref(badk), xb.ptr, qwhip.F16, 1, 0, y.ptr, None) == qwhip.E_BAD_WEIGHTS
    good = dev.view(bank, 8, 64, qwhip.KIND_HQ4_G32_M5)
    assert lib.qwhip_gemv(st, C.byref(good), xb.ptr, qwhip.F32, 1, 0, y.ptr, None) == qwhip.E_BAD_WEIGHTS
    assert lib.qwhip_gemv(st, C.byref(good), xb.ptr, qwhip.F16, 17, 0, y.ptr, None) == qwhip.E_BAD_SHAPE
    assert lib.qwhip_gemv(st, C.byref(good), xb.ptr, qwhip.F16, 1, 0, None, None) == qwhip.E_NULL
    assert lib.qwhip_gemv(st, C.byref(good), xb.ptr, qwhip.F16, 1, 0, y.ptr, None) == qwhip.OK
    dev.stream.sync()
