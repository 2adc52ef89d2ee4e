"""Op-level parity of the HIP kernels with the oracle, through the C-ABI.

Every op of gten::ops (src/gten/ops.h:10-40) runs on the device and in the
oracle on the same seeded inputs (reference byte layouts); results must be
byte-identical: activation rows (Q8 codes + fp16 deltas, fp16 values) and
raw fp32 dot products alike.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as OL
from devutil import DevAct, DevWeight, dev_array, ptr, sync

pytestmark = pytest.mark.gpu

Q8, Q4, F16, F32 = OL.Q8, OL.Q4, OL.F16, OL.F32


def rand_act(oracle, rng, dtype, rows, cols, scale=1.0):
    x = (rng.standard_normal((rows, cols)) * scale).astype(np.float32)
    if dtype == F32:
        return x
    if dtype == F16:
        return x.astype(np.float16).view(np.uint16)
    out = np.zeros((rows, OL.row_bytes(Q8, cols)), np.uint8)
    for r in range(rows):
        oracle.q8_quantize_row(OL.ptr(x[r]), OL.ptr(out[r]), cols)
    return out


def rand_weight(oracle, rng, dtype, rows, cols, scale=0.02):
    w = (rng.standard_normal((rows, cols)) * scale).astype(np.float32)
    if dtype == F16:
        return w.astype(np.float16).view(np.uint16)
    out = np.zeros((rows, OL.row_bytes(dtype, cols)), np.uint8)
    fn = oracle.q8_quantize_weights if dtype == Q8 else oracle.q4_quantize_weights
    fn(OL.ptr(w), rows * cols // 32, OL.ptr(out))
    return out


def assert_same(got, want, what):
    got = np.ascontiguousarray(got).view(np.uint8).reshape(-1)
    want = np.ascontiguousarray(want).view(np.uint8).reshape(-1)
    assert got.shape == want.shape, (what, got.shape, want.shape)
    bad = np.nonzero(got != want)[0]
    assert bad.size == 0, f"{what}: {bad.size} of {got.size} bytes differ, first at {bad[:8]}"


MATMUL_CASES = [
    # (x dtype, w dtype, K, N, rows, start)
    (Q8, Q4, 2048, 2048, 1, 0),
    (Q8, Q4, 5632, 2048, 1, 0),
    (Q8, Q4, 2048, 11264, 1, 0),
    (Q8, Q4, 2304, 250, 3, 1),
    (Q8, Q8, 2048, 2560, 1, 0),
    (Q8, Q8, 8192, 2048, 1, 0),
    (Q8, Q8, 64, 40, 5, 2),
    (Q8, Q4, 1024, 96, 9, 0),
    # prompt rows: short, medium and long prompts, tall weights, columns past a
    # 16-multiple on the fp16 matrix cores, and rows of K % 128 != 0 on the
    # integer ones (their shapes by name: WIDE_ROUTES, INTEGER_CASES)
    (Q8, Q4, 2048, 2560, 64, 0),
    (Q8, Q4, 2048, 2048, 40, 3),
    (Q8, Q4, 5632, 2048, 16, 0),
    (Q8, Q8, 2048, 9000, 24, 0),
    (Q8, Q8, 2304, 300, 100, 7),
    (Q8, Q4, 5760, 1000, 50, 0),
    (Q8, Q4, 1152, 3000, 60, 0),
    (Q8, Q4, 2048, 8192, 260, 0),
    (Q8, Q4, 2048, 700, 300, 0),
    (Q8, Q8, 192, 100, 12, 0),
    (F16, F16, 2048, 2048, 1, 0),
    (F16, F16, 5632, 2048, 1, 0),
    (F16, F16, 128, 44, 4, 1),
    (F16, F16, 2304, 250, 1, 0),
    (F16, F16, 5760, 2304, 1, 0),
    (F16, F16, 2048, 100, 1, 0),
    (F16, F16, 1280, 96, 1, 0),
    (F16, F16, 2048, 2048, 64, 0),
    (F16, F16, 5632, 2048, 16, 3),
    (F16, F16, 2048, 300, 13, 0),
    (F16, F16, 256, 768, 9, 1),
]


@pytest.mark.parametrize("xdt,wdt,K,N,rows,start", MATMUL_CASES)
def test_matmul_fp32_out(gpu, oracle, xdt, wdt, K, N, rows, start):
    rng = np.random.default_rng(K * 7 + N)
    x = rand_act(oracle, rng, xdt, rows, K)
    w = rand_weight(oracle, rng, wdt, N, K)
    want = np.zeros((rows, N), np.float32)
    oracle.matmul(OL.ptr(x), xdt, OL.ptr(w), wdt, OL.ptr(want), F32, K, N, start, rows, None)
    dx, dw = DevAct(x, xdt, rows, K), DevWeight(w, wdt, N, K)
    out = DevAct.empty(F32, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), start, rows, None), "matmul")
    got = out.ref().view(np.float32)
    assert_same(got[start:], want[start:], f"matmul {xdt}x{wdt} K={K} N={N}")


@pytest.mark.parametrize("xdt,wdt,K,N", [(Q8, Q4, 2048, 256), (Q8, Q8, 2048, 512), (F16, F16, 2048, 320)])
def test_matmul_act_out(gpu, oracle, xdt, wdt, K, N):
    rng = np.random.default_rng(N)
    rows = 3
    x = rand_act(oracle, rng, xdt, rows, K)
    w = rand_weight(oracle, rng, wdt, N, K)
    want = np.zeros((rows, OL.row_bytes(xdt, N)), np.uint8)
    oracle.matmul(OL.ptr(x), xdt, OL.ptr(w), wdt, OL.ptr(want), xdt, K, N, 0, rows, None)
    dx, dw, out = DevAct(x, xdt, rows, K), DevWeight(w, wdt, N, K), DevAct.empty(xdt, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), 0, rows, None), "matmul")
    assert_same(out.ref(), want, "matmul act out")


WIDE_CASES = [
    # (w dtype, K, N, rows, start): products of 8 rows and more: one, an odd
    # and an even number of chunks, rows and columns past a tile, a partial
    # last block, Q8 rows stored by the launch and by a pass
    (Q4, 128, 1010, 903, 3),
    (Q4, 384, 4100, 225, 0),
    (Q8, 640, 2050, 310, 0),
    (Q4, 256, 1010, 420, 0),
    (Q8, 384, 3000, 137, 0),
    (Q4, 256, 1010, 21, 1),
    (Q8, 768, 70, 9, 0),
    (Q4, 640, 129, 33, 0),
    (Q8, 128, 40, 8, 0),
]


@pytest.mark.parametrize("wdt,K,N,rows,start", WIDE_CASES)
@pytest.mark.parametrize("odt", [F32, Q8])
def test_matmul_wide(gpu, oracle, wdt, K, N, rows, start, odt):
    rng = np.random.default_rng(K + N)
    x = rand_act(oracle, rng, Q8, rows, K)
    w = rand_weight(oracle, rng, wdt, N, K)
    want = np.zeros((rows, N), np.float32) if odt == F32 else np.zeros((rows, OL.row_bytes(Q8, N)), np.uint8)
    oracle.matmul(OL.ptr(x), Q8, OL.ptr(w), wdt, OL.ptr(want), odt, K, N, start, rows, None)
    dx, dw, out = DevAct(x, Q8, rows, K), DevWeight(w, wdt, N, K), DevAct.empty(odt, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), start, rows, None), "matmul")
    got = out.ref() if odt == Q8 else out.ref().view(np.float32)
    assert_same(got[start:], want[start:], f"matmul Q{8 if wdt == Q8 else 4} K={K} N={N} out {odt}")


WIDE_ROUTES = [
    # (w dtype, K, N, rows, out dtype, route): every shape of the prefill matmul
    # over the weight's own layout, at its lines' edges
    (Q8, 512, 1530, 32, F32, "k_gemm_qw 8x32"),
    (Q8, 512, 1537, 32, F32, "k_gemm_qw 8x64"),
    (Q8, 384, 70, 9, F32, "k_gemm_qw 8x64"),
    (Q4, 256, 70, 9, F32, "k_gemm_qw 8x64"),
    (Q4, 256, 2050, 150, F32, "k_gemm_qw 8x64"),
    (Q8, 256, 3070, 128, Q8, "k_gemm_qw 8x64 + k_write_rows"),
    (Q4, 384, 3073, 128, F32, "k_gemm_qw 16x64"),
    (Q8, 640, 3075, 121, F32, "k_gemm_qw 16x64"),
    (Q8, 128, 3075, 121, Q8, "k_gemm_qw 16x64 + k_write_rows"),
    (Q4, 2304, 3080, 123, Q8, "k_gemm_qw 8x128, rows"),
    (Q4, 2432, 3080, 121, Q8, "k_gemm_qw 16x64 + k_write_rows"),
    (Q4, 128, 4097, 195, F32, "k_gemm_qw 16x128"),
    (Q8, 256, 4100, 195, F32, "k_gemm_qw 16x128"),
    (Q8, 384, 4100, 195, Q8, "k_gemm_qw 16x128, rows"),
]


@pytest.mark.parametrize("wdt,K,N,rows,odt,route", WIDE_ROUTES)
def test_matmul_wide_routes(gpu, oracle, wdt, K, N, rows, odt, route):
    assert gpu.lib().nc_debug_matmul_route(Q8, wdt, odt, rows, N, K).decode() == route
    test_matmul_wide(gpu, oracle, wdt, K, N, rows, 0, odt)


INTEGER_CASES = [
    # (K, N, rows): the integer matrix-core kernel's three shapes (K no multiple
    # of 128): 256 rows and more of 8192 columns and more; 256 rows of fewer, and
    # 32 rows of tall weights; the rest.  One, an odd and an even number of
    # chunks of four blocks, the last one partial
    (96, 8200, 260),
    (160, 8192, 257),
    (160, 300, 259),
    (96, 8193, 33),
    (288, 8192, 250),
    (2080, 70, 30),
    (224, 8300, 9),
]


@pytest.mark.parametrize("wdt", [Q4, Q8])
@pytest.mark.parametrize("K,N,rows", INTEGER_CASES)
def test_matmul_integer_shapes(gpu, oracle, wdt, K, N, rows):
    assert gpu.lib().nc_debug_matmul_route(Q8, wdt, F32, rows, N, K).decode() == "k_gemm_q"
    test_matmul_wide(gpu, oracle, wdt, K, N, rows, 0, F32)


@pytest.mark.parametrize("wdt", [Q4, Q8])
def test_matmul_deltas_off_a_dword(gpu, oracle, wdt):
    """Weight deltas two bytes off a dword: the kernels that load whole dwords do
    not take them."""
    K, N, rows = 256, 300, 40
    rng = np.random.default_rng(wdt)
    x, w = rand_act(oracle, rng, Q8, rows, K), rand_weight(oracle, rng, wdt, N, K)
    want = np.zeros((rows, N), np.float32)
    oracle.matmul(OL.ptr(x), Q8, OL.ptr(w), wdt, OL.ptr(want), F32, K, N, 0, rows, None)
    dx, dw, out = DevAct(x, Q8, rows, K), DevWeight(w, wdt, N, K), DevAct.empty(F32, rows, N)
    deltas = np.zeros(N * K // 32, np.uint16)
    dw.dbuf.download(deltas)
    moved = dev_array(np.concatenate([np.zeros(1, np.uint16), deltas, np.zeros(1, np.uint16)]))
    dw.t.deltas = moved.ptr + 2
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), 0, rows, None), "matmul")
    assert_same(out.ref().view(np.float32), want, "matmul, deltas off a dword")


F16_CASES = [
    # (K, N, rows, start): fp16 products of several rows on the matrix cores:
    # one group, groups past a staged chunk, rows and columns past a tile, and
    # the three launch shapes (up to 384 workgroups of 16 rows, more, and from
    # 640 of 32 rows)
    (64, 70, 2, 0),
    (320, 129, 18, 1),
    (128, 8, 7, 0),
    (192, 1300, 300, 0),
    (64, 1000, 1281, 0),
    # two rows through the one-row kernel, built for the width and not, and
    # where they go to the matrix cores (columns past 4096, K past 8192)
    (2048, 100, 3, 1),
    (1280, 4096, 2, 0),
    (64, 4097, 2, 0),
    (8256, 40, 2, 0),
]


@pytest.mark.parametrize("K,N,rows,start", F16_CASES)
@pytest.mark.parametrize("odt", [F32, F16])
def test_matmul_f16_rows(gpu, oracle, K, N, rows, start, odt):
    rng = np.random.default_rng(K + N)
    x = rand_act(oracle, rng, F16, rows, K, 30.0)
    w = rand_weight(oracle, rng, F16, N, K, 4.0)
    want = np.zeros((rows, N), np.float32) if odt == F32 else np.zeros((rows, OL.row_bytes(F16, N)), np.uint8)
    oracle.matmul(OL.ptr(x), F16, OL.ptr(w), F16, OL.ptr(want), odt, K, N, start, rows, None)
    dx, dw, out = DevAct(x, F16, rows, K), DevWeight(w, F16, N, K), DevAct.empty(odt, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), start, rows, None), "matmul")
    got = out.ref() if odt == F16 else out.ref().view(np.float32)
    assert_same(got[start:], want[start:], f"matmul f16 K={K} N={N} rows={rows} out {odt}")


FEW_CASES = [
    # (w dtype, K, N, rows, start): one to seven rows to Q8 rows, on either
    # side of the lines between k_matvec_qa and the staged route: one block, a
    # part of a thread's last item, a partial last output block, every K on the
    # staged route too
    (Q4, 32, 40, 1, 0),
    (Q4, 2304, 2304, 1, 2),
    (Q8, 5760, 70, 1, 0),
    (Q4, 8192, 96, 1, 0),
    (Q8, 64, 33, 7, 0),
    (Q8, 2304, 100, 5, 1),
    (Q4, 5632, 64, 2, 0),
    (Q8, 3072, 70, 2, 0),
    (Q8, 3104, 70, 2, 0),
    (Q4, 5792, 40, 7, 0),
    (Q8, 5760, 33, 7, 0),
    (Q8, 7168, 48, 3, 0),
    (Q4, 7200, 48, 3, 0),
]


FEW_ROUTES = [
    # (w dtype, K, N, rows, route): every workgroup of k_matvec_qa, one row and
    # several, at the first N its line takes; the last K that several rows'
    # shared memory holds (240 blocks) and the next, the last Q8 K (180 blocks)
    # and the next
    (Q4, 1024, 300, 2, "k_matvec_qa 512x1, rows"),
    (Q4, 1280, 260, 1, "k_matvec_qa 512x2, rows"),
    (Q4, 3072, 260, 2, "k_matvec_qa 512x3, rows"),
    (Q4, 4096, 97, 1, "k_matvec_qa 512x4, rows"),
    (Q4, 4096, 581, 2, "k_matvec_qa 512x4, rows"),
    (Q4, 4096, 580, 2, "k_matvec_q + k_write_rows"),
    (Q4, 5120, 260, 1, "k_matvec_qa 512x5, rows"),
    (Q4, 5120, 1420, 2, "k_matvec_qa 512x5, rows"),
    (Q4, 5760, 570, 1, "k_matvec_qa 960x3, rows"),
    (Q4, 5632, 4097, 7, "k_matvec_qa 960x3, rows"),
    (Q4, 7680, 4097, 1, "k_matvec_qa 960x4, rows"),
    (Q4, 7680, 4097, 2, "k_matvec_qa 960x4, rows"),
    (Q4, 7712, 4097, 2, "k_matvec_q + k_write_rows"),
    (Q4, 8192, 4097, 1, "k_matvec_qa 960x5, rows"),
    (Q4, 8192, 100, 3, "k_matvec_q + k_write_rows"),
    (Q8, 1024, 300, 1, "k_matvec_qa 512x1, rows"),
    (Q8, 2048, 786, 3, "k_matvec_qa 512x2, rows"),
    (Q8, 2048, 785, 3, "k_matvec_q + k_write_rows"),
    (Q8, 2304, 1724, 1, "k_matvec_qa 512x3, rows"),
    (Q8, 2304, 2048, 2, "k_matvec_qa 512x3, rows"),
    (Q8, 2304, 2047, 2, "k_matvec_q + k_write_rows"),
    (Q8, 3104, 4096, 1, "k_matvec_q + k_write_rows"),
    (Q8, 3104, 4097, 1, "k_matvec_qa 512x4, rows"),
    (Q8, 4096, 4097, 3, "k_matvec_qa 512x4, rows"),
    (Q8, 5120, 4100, 1, "k_matvec_qa 512x5, rows"),
    (Q8, 5120, 4100, 2, "k_matvec_qa 512x5, rows"),
    (Q8, 5760, 4100, 1, "k_matvec_qa 960x3, rows"),
    (Q8, 5760, 4100, 7, "k_matvec_qa 960x3, rows"),
    (Q8, 5792, 4100, 2, "k_matvec_q + k_write_rows"),
]


@pytest.mark.parametrize("wdt,K,N,rows,route", FEW_ROUTES)
def test_matmul_few_rows_routes(gpu, oracle, wdt, K, N, rows, route):
    assert gpu.lib().nc_debug_matmul_route(Q8, wdt, Q8, rows, N, K).decode() == route
    test_matmul_few_rows(gpu, oracle, wdt, K, N, rows, 0)


@pytest.mark.parametrize("wdt,K,N,rows,start", FEW_CASES)
def test_matmul_few_rows(gpu, oracle, wdt, K, N, rows, start):
    rng = np.random.default_rng(K + N)
    rows += start
    x = rand_act(oracle, rng, Q8, rows, K)
    w = rand_weight(oracle, rng, wdt, N, K)
    want = np.zeros((rows, OL.row_bytes(Q8, N)), np.uint8)
    oracle.matmul(OL.ptr(x), Q8, OL.ptr(w), wdt, OL.ptr(want), Q8, K, N, start, rows, None)
    dx, dw, out = DevAct(x, Q8, rows, K), DevWeight(w, wdt, N, K), DevAct.empty(Q8, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), start, rows, None), "matmul")
    assert_same(out.ref()[start:], want[start:], f"matmul K={K} N={N} rows={rows}")


@pytest.mark.parametrize("K,N", [(2048, 300), (1280, 44)])
def test_matmul_f16_row(gpu, oracle, K, N):
    rng = np.random.default_rng(K)
    x = rand_act(oracle, rng, F16, 1, K)
    w = rand_weight(oracle, rng, F16, N, K)
    want = np.zeros((1, OL.row_bytes(F16, N)), np.uint8)
    oracle.matmul(OL.ptr(x), F16, OL.ptr(w), F16, OL.ptr(want), F16, K, N, 0, 1, None)
    dx, dw, out = DevAct(x, F16, 1, K), DevWeight(w, F16, N, K), DevAct.empty(F16, 1, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), 0, 1, None), "matmul")
    assert_same(out.ref(), want, "matmul f16 row")


def test_matmul_in_place(gpu, oracle):
    """Output rows over the input rows: the product is read whole first."""
    rng = np.random.default_rng(17)
    d, rows = 1024, 900
    x = rand_act(oracle, rng, Q8, rows, d)
    w = rand_weight(oracle, rng, Q4, d, d)
    want = np.zeros((rows, OL.row_bytes(Q8, d)), np.uint8)
    oracle.matmul(OL.ptr(x), Q8, OL.ptr(w), Q4, OL.ptr(want), Q8, d, d, 0, rows, None)
    dx, dw = DevAct(x, Q8, rows, d), DevWeight(w, Q4, d, d)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(dx.t), 0, rows, None), "matmul")
    assert_same(dx.ref(), want, "matmul in place")


@pytest.mark.parametrize("dt", [Q8, F16])
@pytest.mark.parametrize("d,scale", [(2048, 1.0), (2304, 30.0), (256, 0.01)])
def test_rms_norm(gpu, oracle, dt, d, scale):
    rng = np.random.default_rng(d)
    rows, start = 4, 1
    x = rand_act(oracle, rng, dt, rows, d, scale)
    w = (1 + 0.2 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    oracle.rms_norm(OL.ptr(x), dt, OL.ptr(w), OL.ptr(want), d, start, rows)
    dx, out, dwt = DevAct(x, dt, rows, d), DevAct.empty(dt, rows, d), dev_array(w)
    gpu.check(gpu.lib().nc_rms_norm(C.byref(dx.t), C.c_void_p(dwt.ptr), C.byref(out.t), d, start, rows, None), "rms")
    assert_same(out.ref()[start:], want[start:], "rms_norm")


@pytest.mark.parametrize("dt", [Q8, F16])
@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("d,shift", [(256, 0), (1024, 0), (1280, 0), (1536, 0), (2304, 0), (3072, 0), (4096, 0),
                                     (2048, 2), (320, 0)])
def test_norm_widths(gpu, oracle, dt, kind, d, shift):
    """Widths of one and two slots per thread, means from the exact grid sum and
    from the loop, widths the eight-value norm leaves to the other kernel (256,
    320), and gains at an address it does not take (shift bytes)."""
    rng = np.random.default_rng(d + shift)
    rows, start = 3, 1
    x = rand_act(oracle, rng, dt, rows, d, 3.0)
    w = (1 + 0.2 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    b = (0.1 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    dx, out = DevAct(x, dt, rows, d), DevAct.empty(dt, rows, d)
    pad = np.zeros(shift // 2, np.uint16)
    dw_, db_ = dev_array(np.concatenate([pad, w])), dev_array(b)
    L = gpu.lib()
    if kind == "rms":
        oracle.rms_norm(OL.ptr(x), dt, OL.ptr(w), OL.ptr(want), d, start, rows)
        st = L.nc_rms_norm(C.byref(dx.t), C.c_void_p(dw_.ptr + shift), C.byref(out.t), d, start, rows, None)
    else:
        oracle.layer_norm(OL.ptr(x), dt, OL.ptr(w), OL.ptr(b), OL.ptr(want), d, start, rows)
        st = L.nc_layer_norm(C.byref(dx.t), C.c_void_p(dw_.ptr + shift), C.c_void_p(db_.ptr), C.byref(out.t), start,
                             rows, None)
    gpu.check(st, "norm")
    assert_same(out.ref()[start:], want[start:], f"{kind} norm of {d}")


def hard_rows(rng, dt, d):
    """Rows whose mean rounds at many steps, at few, or at none, and rows whose
    sums hit the largest values: blocks of unequal scales (Q8) or values of
    unequal exponents (fp16)."""
    b = np.repeat(2.0 ** rng.integers(-12, 9, (12, d // 32)), 32, axis=1)
    x = [rng.standard_normal((12, d)) * b]
    if dt == F16:
        x.append(rng.standard_normal((12, d)) * 2.0 ** rng.integers(-14, 8, (12, d)))
    x.append(np.abs(rng.standard_normal((4, d))))  # the running sum only grows
    absorb = rng.integers(-3, 4, (4, d)).astype(np.float64)
    absorb[:, 0] = 1024.0
    absorb[:, 1:11] = 2.0**-14
    big = np.where(rng.random((4, d)) < 0.1, 60000.0, 0.0) * np.where(rng.random((4, d)) < 0.5, 1, -1)
    x += [absorb, big, np.zeros((1, d)), np.full((1, d), 0.5)]
    return np.concatenate(x).astype(np.float32)


@pytest.mark.parametrize("dt,d,each", [(Q8, 1024, 0), (Q8, 1280, 0), (Q8, 1536, 0), (Q8, 2048, 0), (Q8, 2304, 4),
                                       (F16, 2048, 1), (F16, 1280, 1), (F16, 2048, 0), (Q8, 2304, 0), (F16, 2304, 0),
                                       (Q8, 2816, 0)])
def test_layer_norm_hard_rows(gpu, oracle, dt, d, each):
    """Rows that round often, fall back or have no rounding step, in one call or
    `each` rows per call: few enough for every instantiation of the exact grid
    sum that the eight-value norm uses, and many, for the loop."""
    rng = np.random.default_rng(d)
    v = hard_rows(rng, dt, d)
    rows = len(v)
    if dt == F16:
        x = v.astype(np.float16).view(np.uint16)
    else:
        x = np.zeros((rows, OL.row_bytes(Q8, d)), np.uint8)
        for r in range(rows):
            oracle.q8_quantize_row(OL.ptr(v[r]), OL.ptr(x[r]), d)
    w = (1 + 0.2 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    b = (0.1 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    oracle.layer_norm(OL.ptr(x), dt, OL.ptr(w), OL.ptr(b), OL.ptr(want), d, 0, rows)
    grid = each or (dt == Q8 and d <= 2048)
    L = gpu.lib()
    route = L.nc_debug_norm_route(1, dt, d, each or rows).decode()
    assert route == ("k_norm8, grid mean" if grid else "k_norm8, loop mean")
    dx, out = DevAct(x, dt, rows, d), DevAct.empty(dt, rows, d)
    dw_, db_ = dev_array(w), dev_array(b)
    for start in range(0, rows, each or rows):
        end = min(rows, start + (each or rows))
        gpu.check(L.nc_layer_norm(C.byref(dx.t), C.c_void_p(dw_.ptr), C.c_void_p(db_.ptr), C.byref(out.t), start, end,
                                  None), "layer_norm")
    assert_same(out.ref(), want, f"layer norm of {d}")


@pytest.mark.parametrize("dt", [Q8, F16])
@pytest.mark.parametrize("op", ["silu", "mul", "add", "rope"])
@pytest.mark.parametrize("d,rows", [(2048, 515), (2112, 510)])
def test_elementwise_many_rows(gpu, oracle, dt, op, d, rows):
    """Enough values for eight per thread, a last workgroup that is not full."""
    rng = np.random.default_rng(d + rows)
    a, b = rand_act(oracle, rng, dt, rows, d, 4.0), rand_act(oracle, rng, dt, rows, d, 1.0)
    want = a.copy()
    da, db_, out = DevAct(a, dt, rows, d), DevAct(b, dt, rows, d), DevAct.empty(dt, rows, d)
    L = gpu.lib()
    if op == "silu":
        oracle.silu(OL.ptr(a), OL.ptr(want), dt, d, 0, rows)
        st = L.nc_silu(C.byref(da.t), C.byref(out.t), 0, rows, None)
    elif op == "rope":
        tab = np.zeros((rows, 8, 2), np.float32)
        gpu.check(L.nc_rope_table(rows, 64, 0.25, ptr(tab)), "rope_table")
        dtab = dev_array(tab)
        oracle.rotary_emb(OL.ptr(a), OL.ptr(want), dt, d, 64, 0.25, 0, rows)
        st = L.nc_rotary_emb(C.byref(da.t), C.byref(out.t), 64, 0.25, C.c_void_p(dtab.ptr), 0, rows, None)
    else:
        (oracle.multiply if op == "mul" else oracle.add)(OL.ptr(a), OL.ptr(b), OL.ptr(want), dt, d, 0, rows)
        st = (L.nc_multiply if op == "mul" else L.nc_add)(C.byref(da.t), C.byref(db_.t), C.byref(out.t), 0, rows, None)
    gpu.check(st, op)
    assert_same(out.ref(), want, op)


EIGHT_ROWS = {"silu": {Q8: 515, F16: 1283, F32: 1541}}  # past each type's line at 2048 columns


@pytest.mark.parametrize("dt", [Q8, F16, F32])
@pytest.mark.parametrize("op", ["silu", "mul", "add", "scale", "bias"])
def test_eight_value_operators_in_place(gpu, oracle, dt, op):
    """Every operator of eight values per thread with the output over its input,
    rows from a position on, a last workgroup that is not full."""
    d, start = 2048, 2
    n = start + EIGHT_ROWS.get(op, {}).get(dt, 131)
    assert gpu.lib().nc_debug_ew_route(op == "silu", dt, n - start, d).decode() == "k_ew8"
    rng = np.random.default_rng(n + dt)
    a, b = rand_act(oracle, rng, dt, n, d, 4.0), rand_act(oracle, rng, dt, n, d, 1.0)
    bias = (0.1 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want, scale = a.copy(), 0.3
    da, db_, dbias = DevAct(a, dt, n, d), DevAct(b, dt, n, d), dev_array(bias)
    L, A = gpu.lib(), C.byref(da.t)
    if op == "silu":
        oracle.silu(OL.ptr(want), OL.ptr(want), dt, d, start, n)
        st = L.nc_silu(A, A, start, n, None)
    elif op == "scale":
        oracle.scale(OL.ptr(want), dt, scale, d, start, n)
        st = L.nc_scale(A, scale, start, n, None)
    elif op == "bias":
        oracle.bias_add(OL.ptr(want), dt, OL.ptr(bias), d, start, n)
        st = L.nc_bias_add(A, C.c_void_p(dbias.ptr), start, n, None)
    else:
        (oracle.multiply if op == "mul" else oracle.add)(OL.ptr(want), OL.ptr(b), OL.ptr(want), dt, d, start, n)
        st = (L.nc_multiply if op == "mul" else L.nc_add)(A, C.byref(db_.t), A, start, n, None)
    gpu.check(st, op)
    assert_same(da.ref(), want, op)


@pytest.mark.parametrize("dt", [Q8, F16])
def test_rope_many_rows_from_a_position(gpu, oracle, dt):
    """The eight-value rotary embedding of whole heads (every lane rotated), its
    table from a later position on."""
    d, start, n = 2304, 7, 150
    rng = np.random.default_rng(dt)
    a = rand_act(oracle, rng, dt, n, d, 2.0)
    tab = np.zeros((n, 32, 2), np.float32)
    gpu.check(gpu.lib().nc_rope_table(n, 64, 1.0, ptr(tab)), "rope_table")
    dtab, da, out = dev_array(tab), DevAct(a, dt, n, d), DevAct.empty(dt, n, d)
    want = a.copy()
    oracle.rotary_emb(OL.ptr(a), OL.ptr(want), dt, d, 64, 1.0, start, n)
    gpu.check(gpu.lib().nc_rotary_emb(C.byref(da.t), C.byref(out.t), 64, 1.0, C.c_void_p(dtab.ptr), start, n, None),
              "rope")
    assert_same(out.ref()[start:], want[start:], "rope")


def assert_same_f16(got, want, what):
    """Equal bits, any NaN for a NaN."""
    g = np.ascontiguousarray(got).view(np.uint8).reshape(-1).view(np.float16)
    w = np.ascontiguousarray(want).view(np.uint8).reshape(-1).view(np.float16)
    nan = np.isnan(w)
    assert np.array_equal(np.isnan(g), nan), f"{what}: NaN at other places"
    assert nan.any() and not nan.all(), what
    assert_same(g[~nan], w[~nan], what)


def with_specials(rng, a, share=0.002):
    a = a.copy().view(np.float16)
    at = rng.random(a.shape) < share
    a[at] = rng.choice(np.array([np.inf, -np.inf, np.nan, 65504.0, -65504.0], np.float16), int(at.sum()))
    return a.view(np.uint16)


@pytest.mark.parametrize("K,N,rows", [(192, 130, 18), (128, 70, 5)])
def test_matmul_f16_non_finite(gpu, oracle, K, N, rows):
    """Infinities and NaN of one row or column reach no other one on the matrix
    cores."""
    rng = np.random.default_rng(K)
    x, w = rand_act(oracle, rng, F16, rows, K), rand_weight(oracle, rng, F16, N, K)
    x[rows // 2 :] = with_specials(rng, x[rows // 2 :], 0.01)
    w[: N // 2] = with_specials(rng, w[: N // 2], 0.002)
    want = np.zeros((rows, OL.row_bytes(F16, N)), np.uint8)
    oracle.matmul(OL.ptr(x), F16, OL.ptr(w), F16, OL.ptr(want), F16, K, N, 0, rows, None)
    assert gpu.lib().nc_debug_matmul_route(F16, F16, F16, rows, N, K).decode() == "k_mfma_f16, rows"
    dx, dw, out = DevAct(x, F16, rows, K), DevWeight(w, F16, N, K), DevAct.empty(F16, rows, N)
    gpu.check(gpu.lib().nc_matmul_2d(C.byref(dx.t), C.byref(dw.t), C.byref(out.t), 0, rows, None), "matmul")
    assert_same_f16(out.ref(), want, "matmul of non-finite values")


@pytest.mark.parametrize("where", ["k", "v"])
def test_qkv_attn_f16_non_finite_later_rows(gpu, oracle, where):
    """Infinities and NaN in K or V rows reach only the query rows that attend
    them, also within one tile of sixteen: rows before them are those of finite
    values, the last row is the oracle's."""
    hq, hkv, n, start, first = 3, 1, 660, 625, 641
    rng = np.random.default_rng(ord(where))
    q, k, v = (rand_act(oracle, rng, F16, n, h * 64) for h in (hq, hkv, hkv))

    def attn(k, v):
        want = np.zeros((n, OL.row_bytes(F16, hq * 64)), np.uint8)
        oracle.qkv_attn(OL.ptr(q), OL.ptr(k), OL.ptr(v), OL.ptr(want), F16, hq, hkv, 64, start, n)
        return want

    finite = attn(k, v)
    if where == "k":
        k[first:] = with_specials(rng, k[first:], 0.05)
    else:
        v[first:] = with_specials(rng, v[first:], 0.05)
    want = attn(k, v)
    assert gpu.lib().nc_debug_attn_route(F16, hq, n - start, n).decode() == "k_attn_f16"
    dq, dk, dv = DevAct(q, F16, n, hq * 64), DevAct(k, F16, n, hkv * 64), DevAct(v, F16, n, hkv * 64)
    out = DevAct.empty(F16, n, hq * 64)
    gpu.check(gpu.lib().nc_qkv_attn(C.byref(dq.t), C.byref(dk.t), C.byref(dv.t), C.byref(out.t), hq, hkv, 64, start,
                                    n, None), "qkv_attn")
    got = out.ref()
    assert_same(got[start:first], finite[start:first], "rows before the non-finite ones")
    last, ref = (a[n - 1].view(np.float16) for a in (got, want))
    assert np.isnan(ref).any() and np.array_equal(np.isnan(last), np.isnan(ref))
    assert_same(last[~np.isnan(ref)], ref[~np.isnan(ref)], "the last row")


@pytest.mark.parametrize("kind", ["rms", "layer"])
@pytest.mark.parametrize("d", [2048, 2304])
def test_norm_non_finite(gpu, oracle, kind, d):
    rng = np.random.default_rng(d)
    rows = 9
    x = rand_act(oracle, rng, F16, rows, d)
    x[1::2] = with_specials(rng, x[1::2], 0.001)
    w = (1 + 0.2 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    b = (0.1 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    dx, out, dw_, db_ = DevAct(x, F16, rows, d), DevAct.empty(F16, rows, d), dev_array(w), dev_array(b)
    L = gpu.lib()
    if kind == "rms":
        oracle.rms_norm(OL.ptr(x), F16, OL.ptr(w), OL.ptr(want), d, 0, rows)
        st = L.nc_rms_norm(C.byref(dx.t), C.c_void_p(dw_.ptr), C.byref(out.t), d, 0, rows, None)
    else:
        oracle.layer_norm(OL.ptr(x), F16, OL.ptr(w), OL.ptr(b), OL.ptr(want), d, 0, rows)
        st = L.nc_layer_norm(C.byref(dx.t), C.c_void_p(dw_.ptr), C.c_void_p(db_.ptr), C.byref(out.t), 0, rows, None)
    gpu.check(st, "norm")
    assert_same_f16(out.ref(), want, f"{kind} norm of non-finite values")


@pytest.mark.parametrize("dt", [Q8, F16])
def test_rms_norm_per_head(gpu, oracle, dt):
    rng = np.random.default_rng(5)
    rows, heads = 3, 20
    d = heads * 64
    x = rand_act(oracle, rng, dt, rows, d)
    w = (1 + 0.2 * rng.standard_normal(64)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    oracle.rms_norm_heads(OL.ptr(x), dt, OL.ptr(w), OL.ptr(want), heads, 64, 0, rows)
    dx, out, dwt = DevAct(x, dt, rows, d), DevAct.empty(dt, rows, d), dev_array(w)
    gpu.check(gpu.lib().nc_rms_norm(C.byref(dx.t), C.c_void_p(dwt.ptr), C.byref(out.t), 64, 0, rows, None), "rms3d")
    assert_same(out.ref(), want, "rms_norm per head")


@pytest.mark.parametrize("dt", [Q8, F16])
def test_layer_norm(gpu, oracle, dt):
    rng = np.random.default_rng(11)
    rows, d = 3, 2048
    x = rand_act(oracle, rng, dt, rows, d, 2.0)
    x_f = rng.standard_normal(d)
    w = (1 + 0.2 * x_f).astype(np.float16).view(np.uint16)
    b = (0.1 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = np.zeros_like(x)
    oracle.layer_norm(OL.ptr(x), dt, OL.ptr(w), OL.ptr(b), OL.ptr(want), d, 0, rows)
    dx, out, dw_, db_ = DevAct(x, dt, rows, d), DevAct.empty(dt, rows, d), dev_array(w), dev_array(b)
    gpu.check(gpu.lib().nc_layer_norm(C.byref(dx.t), C.c_void_p(dw_.ptr), C.c_void_p(db_.ptr), C.byref(out.t), 0,
                                      rows, None), "layer_norm")
    assert_same(out.ref(), want, "layer_norm")


@pytest.mark.parametrize("dt", [Q8, F16])
@pytest.mark.parametrize("pct,start", [(1.0, 0), (0.25, 5), (1.0, 300)])
def test_rotary_emb(gpu, oracle, dt, pct, start):
    rng = np.random.default_rng(int(pct * 100) + start)
    rows, d = start + 4, 2048
    x = rand_act(oracle, rng, dt, rows, d, 3.0)
    want = x.copy()
    oracle.rotary_emb(OL.ptr(x), OL.ptr(want), dt, d, 64, pct, start, rows)
    d_half = int(64 * pct) // 2
    tab = np.zeros((rows, max(d_half, 1), 2), np.float32)
    gpu.check(gpu.lib().nc_rope_table(rows, 64, pct, ptr(tab)), "rope_table")
    dtab = dev_array(tab)
    dx = DevAct(x, dt, rows, d)
    out = DevAct(x, dt, rows, d)
    gpu.check(gpu.lib().nc_rotary_emb(C.byref(dx.t), C.byref(out.t), 64, pct, C.c_void_p(dtab.ptr), start, rows, None),
              "rope")
    assert_same(out.ref()[start:], want[start:], "rotary_emb")


SCALE = float(np.float32(1.4 / 40 ** 0.5))


@pytest.mark.parametrize("dt", [Q8, F16])
@pytest.mark.parametrize("op", ["silu", "mul", "add", "scale", "bias"])
def test_elementwise(gpu, oracle, dt, op):
    rng = np.random.default_rng(["silu", "mul", "add", "scale", "bias"].index(op))
    rows, d = 3, 5632
    a = rand_act(oracle, rng, dt, rows, d, 4.0)
    b = rand_act(oracle, rng, dt, rows, d, 1.0)
    bias = (0.3 * rng.standard_normal(d)).astype(np.float16).view(np.uint16)
    want = a.copy()
    if op == "silu":
        oracle.silu(OL.ptr(a), OL.ptr(want), dt, d, 0, rows)
    elif op == "mul":
        oracle.multiply(OL.ptr(a), OL.ptr(b), OL.ptr(want), dt, d, 0, rows)
    elif op == "add":
        oracle.add(OL.ptr(a), OL.ptr(b), OL.ptr(want), dt, d, 0, rows)
    elif op == "scale":
        oracle.scale(OL.ptr(want), dt, SCALE, d, 0, rows)
    else:
        oracle.bias_add(OL.ptr(want), dt, OL.ptr(bias), d, 0, rows)
    da, db_, out, dbias = DevAct(a, dt, rows, d), DevAct(b, dt, rows, d), DevAct.empty(dt, rows, d), dev_array(bias)
    L = gpu.lib()
    if op == "silu":
        st = L.nc_silu(C.byref(da.t), C.byref(out.t), 0, rows, None)
    elif op == "mul":
        st = L.nc_multiply(C.byref(da.t), C.byref(db_.t), C.byref(out.t), 0, rows, None)
    elif op == "add":
        st = L.nc_add(C.byref(da.t), C.byref(db_.t), C.byref(out.t), 0, rows, None)
    elif op == "scale":
        st = L.nc_scale(C.byref(da.t), SCALE, 0, rows, None)
        out = da
    else:
        st = L.nc_bias_add(C.byref(da.t), C.c_void_p(dbias.ptr), 0, rows, None)
        out = da
    gpu.check(st, op)
    assert_same(out.ref(), want, op)


ATTN_CASES = [
    # (dtype, n_heads, n_kv_heads, n_ctx, start)
    (Q8, 32, 4, 320, 319),
    (Q8, 32, 4, 1, 0),
    (Q8, 36, 36, 640, 639),
    (Q8, 20, 5, 77, 76),
    (Q8, 8, 2, 64, 0),
    (Q8, 4, 1, 100, 37),
    (F16, 32, 32, 256, 255),
    (F16, 4, 4, 128, 0),
    (F16, 8, 2, 45, 20),
    # contexts of the reference's models: 1024 (its default), 2048, 4096; the
    # single-row softmax sum changes from one wavefront's loop to the exact
    # workgroup sum above 1024 positions; n mod 8 / mod 32 edges; the prefill
    # kernel's 8, 4 and 2 rows per workgroup (m <= 1024, <= 2048, beyond)
    (Q8, 32, 4, 1024, 1023),
    (Q8, 32, 4, 1025, 1024),
    (Q8, 32, 4, 1031, 1030),
    (Q8, 36, 36, 2048, 2047),
    (Q8, 16, 4, 2053, 2040),
    (Q8, 32, 4, 4096, 4095),
    (Q8, 4, 1, 4093, 4080),
    (Q8, 8, 2, 1100, 0),
    (Q8, 4, 1, 3000, 0),
    (F16, 32, 32, 1024, 1023),
    (F16, 32, 32, 2049, 2048),
    (F16, 32, 32, 4096, 4095),
    (F16, 4, 4, 4090, 4081),
    (F16, 4, 2, 1500, 0),
    # one row with its V slice in shared memory (256 to 1024 positions), n mod 8
    # and mod 32 edges, both numbers of K rows per thread
    (Q8, 2, 1, 256, 255),
    (Q8, 2, 2, 511, 510),
    (Q8, 3, 1, 517, 516),
    (F16, 2, 1, 255, 254),
    (F16, 2, 2, 513, 512),
    (F16, 3, 3, 1023, 1022),
    # several fp16 rows of few heads and at most 600 positions, which keep
    # k_attn_rows; the longest context that k_attn_f16 takes and the next
    (F16, 2, 1, 2, 0),
    (F16, 2, 2, 129, 112),
    (F16, 4, 2, 143, 5),
    (F16, 2, 1, 257, 240),
    (F16, 3, 1, 383, 350),
    (F16, 2, 2, 2176, 2170),
    (F16, 2, 2, 2177, 2170),
]


@pytest.mark.parametrize("dt,hq,hkv,n,start", ATTN_CASES)
def test_qkv_attn(gpu, oracle, dt, hq, hkv, n, start):
    rng = np.random.default_rng(hq * 1000 + n)
    q = rand_act(oracle, rng, dt, n, hq * 64, 2.0)
    k = rand_act(oracle, rng, dt, n, hkv * 64, 2.0)
    v = rand_act(oracle, rng, dt, n, hkv * 64, 1.0)
    want = np.zeros((n, OL.row_bytes(dt, hq * 64)), np.uint8)
    oracle.qkv_attn(OL.ptr(q), OL.ptr(k), OL.ptr(v), OL.ptr(want), dt, hq, hkv, 64, start, n)
    dq, dk, dv = DevAct(q, dt, n, hq * 64), DevAct(k, dt, n, hkv * 64), DevAct(v, dt, n, hkv * 64)
    out = DevAct.empty(dt, n, hq * 64)
    gpu.check(gpu.lib().nc_qkv_attn(C.byref(dq.t), C.byref(dk.t), C.byref(dv.t), C.byref(out.t), hq, hkv, 64, start,
                                    n, None), "qkv_attn")
    assert_same(out.ref()[start:], want[start:], "qkv_attn")


F16_TILE_CASES = [
    # (n_heads, n_kv_heads, n_ctx, start) that k_attn_f16 takes: a tile from its
    # first row, parts of a tile, rows across a tile's edge, contexts at a staged
    # chunk's edges (128 positions), every n mod 8, prompts from position 0
    (64, 8, 128, 80),
    (64, 64, 129, 75),
    (36, 36, 143, 5),
    (64, 8, 131, 0),
    (2, 1, 256, 254),
    (2, 2, 261, 256),
    (2, 1, 406, 398),
    (4, 2, 607, 590),
    (3, 1, 639, 606),
    (2, 1, 640, 624),
    (2, 2, 641, 625),
    (2, 1, 644, 627),
    (2, 2, 2176, 2159),
]


@pytest.mark.parametrize("hq,hkv,n,start", F16_TILE_CASES)
def test_qkv_attn_f16_tiles(gpu, oracle, hq, hkv, n, start):
    assert gpu.lib().nc_debug_attn_route(F16, hq, n - start, n).decode() == "k_attn_f16"
    test_qkv_attn(gpu, oracle, F16, hq, hkv, n, start)


@pytest.mark.parametrize("wdt", [Q4, Q8, F16])
def test_token_embed(gpu, oracle, wdt):
    rng = np.random.default_rng(wdt)
    vocab, d, rows = 1000, 2048, 6
    table = rand_weight(oracle, rng, wdt, vocab, d, 0.5)
    adt = F16 if wdt == F16 else Q8
    toks = np.array([0, 999, 5, 5, 123, 640], np.int32)
    want = np.zeros((rows, OL.row_bytes(adt, d)), np.uint8)
    oracle.token_embed(OL.ptr(table), wdt, OL.ptr(toks), OL.ptr(want), adt, d, vocab, 0, rows)
    dtab, dtok, out = DevWeight(table, wdt, vocab, d), dev_array(toks), DevAct.empty(adt, rows, d)
    gpu.check(gpu.lib().nc_token_embed(C.byref(dtab.t), C.c_void_p(dtok.ptr), C.byref(out.t), 0, rows, None), "embed")
    assert_same(out.ref(), want, "token_embed")


@pytest.mark.parametrize("n,offset", [(1, 3), (2, 1), (4099, 2), (32771, 3), (40000, 1)])
@pytest.mark.parametrize("kind", ["ties", "all -inf", "nan"])
def test_argmax_edges(gpu, oracle, n, offset, kind):
    """Vectors at any 4-byte alignment, values before and after the vector
    part, nothing above -inf, NaN never taken."""
    rng = np.random.default_rng(n + offset)
    x = rng.integers(-3, 4, n + offset).astype(np.float32)
    if kind == "all -inf":
        x[:] = -np.inf
    if kind == "nan":
        x[rng.integers(0, n + offset, max(1, n // 3))] = np.nan
    dx, out = dev_array(x), np.zeros(1, np.int32)
    dout = dev_array(out)
    gpu.check(gpu.lib().nc_argmax(C.c_void_p(dx.ptr + 4 * offset), n, C.c_void_p(dout.ptr), None), "argmax")
    dout.download(out)
    assert out[0] == oracle.argmax(OL.ptr(np.ascontiguousarray(x[offset:])), n)


@pytest.mark.parametrize("n", [1, 1000, 32000, 122753])
def test_argmax_first_max(gpu, oracle, n):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    if n > 10:
        x[n // 3] = x[n // 2] = x[n - 1] = 9.0  # ties: the first index wins
    dx = dev_array(x)
    out = np.zeros(1, np.int32)
    dout = dev_array(out)
    gpu.check(gpu.lib().nc_argmax(C.c_void_p(dx.ptr), n, C.c_void_p(dout.ptr), None), "argmax")
    dout.download(out)
    assert out[0] == oracle.argmax(OL.ptr(x), n)


def test_weight_generation_and_quantization(gpu, oracle):
    """Device generator + quantizer equal the oracle's bit for bit."""
    L = gpu.lib()
    n = 2048 * 512
    want_f = np.zeros(n, np.float32)
    oracle.gen_normal(77, 13, 0.02, n, OL.ptr(want_f))
    dbuf = gpu.DeviceBuffer(n * 4)
    gpu.check(L.nc_gen_normal(77, 13, 0.02, n, C.c_void_p(dbuf.ptr), None), "gen_normal")
    got_f = np.zeros(n, np.float32)
    sync()
    dbuf.download(got_f)
    assert_same(got_f, want_f, "gen_normal")
    for dt in (Q8, Q4, F16):
        rows, cols = 512, 2048
        want = np.zeros(rows * OL.row_bytes(dt, cols), np.uint8)
        if dt == F16:
            want = want_f.astype(np.float16).view(np.uint8)
        else:
            (oracle.q8_quantize_weights if dt == Q8 else oracle.q4_quantize_weights)(OL.ptr(want_f), n // 32,
                                                                                    OL.ptr(want))
        w = DevWeight(np.zeros_like(want), dt, rows, cols)
        gpu.check(L.nc_weight_quantize(C.c_void_p(dbuf.ptr), C.byref(w.t), None), "weight_quantize")
        sync()
        cb = np.zeros(w.cbuf.nbytes, np.uint8)
        w.cbuf.download(cb)
        want_codes = np.zeros_like(cb)
        want_deltas = np.zeros(w.dbuf.nbytes, np.uint8)
        gpu.check(L.nc_weight_from_reference(ptr(want), dt, rows, cols, ptr(want_codes), ptr(want_deltas)), "repack")
        assert_same(cb, want_codes, f"codes dtype {dt}")
        if dt != F16:
            db_ = np.zeros(w.dbuf.nbytes, np.uint8)
            w.dbuf.download(db_)
            assert_same(db_, want_deltas, f"deltas dtype {dt}")


def test_expf_exhaustive(gpu, oracle):
    """Device std::exp(float) equals the host glibc expf on all 2^32 inputs."""
    L = gpu.lib()
    chunk = 1 << 27
    dx, dy = gpu.DeviceBuffer(chunk * 4), gpu.DeviceBuffer(chunk * 4)
    y = np.zeros(chunk, np.float32)
    f = oracle.lib.or_expf_mismatches
    f.restype, f.argtypes = C.c_int64, [C.c_void_p, C.c_void_p, C.c_int64, C.POINTER(C.c_int64)]
    total = 0
    first = []
    for start in range(0, 1 << 32, chunk):
        x = np.arange(start, start + chunk, dtype=np.uint64).astype(np.uint32).view(np.float32)
        dx.upload(x)
        gpu.check(L.nc_expf(C.c_void_p(dx.ptr), C.c_void_p(dy.ptr), chunk, None), "expf")
        sync()
        dy.download(y)
        fi = C.c_int64()
        cnt = f(OL.ptr(x), OL.ptr(y), chunk, C.byref(fi))
        total += cnt
        if cnt and len(first) < 8:
            first.append((hex(int(x.view(np.uint32)[fi.value])), float(y[fi.value])))
    assert total == 0, f"{total} inputs differ from glibc expf, e.g. {first}"
