"""The dispatch rules at sizes where both sides were measured, on the CPU.

Each case is a call, the kernel its rule must take, and the times on one MI355X
(us: the kernel the rule takes, the one it passes over).
"""
import pytest

import oracle_lib as OL

Q8, Q4, F16, F32 = OL.Q8, OL.Q4, OL.F16, OL.F32

MATMUL = [
    # (w dtype, rows, N, K, route): Q8 rows in and out
    (Q4, 1, 2048, 2048, "k_matvec_qa 512x2, rows"),  # 4.1, staged 6.1
    (Q4, 1, 256, 2048, "k_matvec_qa 512x2, rows"),  # 3.7, staged 4.5
    (Q4, 1, 2048, 4096, "k_matvec_qa 512x4, rows"),  # 5.5, 960 threads 6.0, staged 6.8
    (Q4, 5, 2048, 4096, "k_matvec_q + k_write_rows"),  # 12.7, direct 13.1
    (Q4, 1, 2048, 5632, "k_matvec_qa 960x3, rows"),  # 6.9, 512 threads 7.6, staged 7.4
    (Q4, 7, 2048, 5632, "k_matvec_q + k_write_rows"),  # 18.9, direct 23.0
    (Q4, 7, 5632, 5632, "k_matvec_qa 960x3, rows"),  # 24.0, staged 32.3
    (Q4, 7, 2048, 7680, "k_matvec_q + k_write_rows"),  # 22.5, direct 29.1
    (Q4, 5, 320, 1280, "k_matvec_qa 512x2, rows"),  # 8.2, staged 8.7
    (Q4, 1, 2048, 7680, "k_matvec_q + k_write_rows"),  # 8.0, direct 8.3
    (Q8, 1, 256, 2048, "k_matvec_qa 512x2, rows"),  # 5.0, staged 7.3 (launch included)
    (Q8, 1, 1024, 2304, "k_matvec_q + k_write_rows"),  # 5.9, direct 6.2
    (Q8, 2, 5632, 2048, "k_matvec_qa 512x2, rows"),  # 7.0, staged 10.6
    (Q8, 7, 2048, 2304, "k_matvec_q + k_write_rows"),  # 13.7, direct 15.0
    (Q8, 1, 2048, 4096, "k_matvec_q + k_write_rows"),  # 7.2, direct 8.1
    (Q8, 1, 2048, 5632, "k_matvec_q + k_write_rows"),  # 7.9, direct 10.4
    (Q8, 5, 2304, 5760, "k_matvec_q + k_write_rows"),  # 17.3, direct 22.5
    (Q8, 5, 5632, 5632, "k_matvec_qa 960x3, rows"),  # 22.7, staged 26.4
    (Q8, 2, 2048, 7680, "k_matvec_q + k_write_rows"),  # 11.3, direct 21.4
    (Q8, 1, 8192, 8192, "k_matvec_q + k_write_rows"),  # 19.1, direct 22.1
]


@pytest.mark.parametrize("wdt,rows,N,K,route", MATMUL)
def test_few_row_products_take_the_faster_route(nc, wdt, rows, N, K, route):
    assert nc.lib().nc_debug_matmul_route(Q8, wdt, Q8, rows, N, K).decode() == route


WIDE = [
    # (w dtype, out dtype, rows, N, K, route)
    (Q8, F32, 16, 2048, 2048, "k_gemm_qw 8x32"),  # 13.9, 8x64 15.0
    (Q4, F32, 64, 2560, 2048, "k_gemm_qw 8x64"),  # 17.5, 16x64 18.9
    (Q4, F32, 128, 2048, 5632, "k_gemm_qw 8x64"),  # 37.2, 16x64 44.8, 16x128 61.8
    (Q8, F32, 201, 2048, 2048, "k_gemm_qw 16x64"),  # 26.0, 8x64 37.8, 8x128 33.4, 16x128 30.8
    (Q8, F32, 256, 2048, 2048, "k_gemm_qw 16x64"),  # 26.6, 8x64 36.7, 8x128 35.1, 16x128 31.3
    (Q8, F32, 16, 32000, 2048, "k_gemm_qw 16x64"),  # 34.4, 8x128 42.6, 16x128 37.4
    (Q4, F32, 128, 6144, 2048, "k_gemm_qw 16x64"),  # 32.5, 16x128 36.3
    (Q4, F32, 512, 6912, 2304, "k_gemm_qw 16x128"),  # 109, 16x64 118
    (Q4, Q8, 256, 2048, 1024, "k_gemm_qw 8x128, rows"),  # 13.6, 16x64 and the pass 15.4
    (Q8, Q8, 201, 2048, 2048, "k_gemm_qw 16x64 + k_write_rows"),  # 25.5, 8x128 30.8
]


@pytest.mark.parametrize("wdt,odt,rows,N,K,route", WIDE)
def test_prefill_products_take_the_faster_shape(nc, wdt, odt, rows, N, K, route):
    assert nc.lib().nc_debug_matmul_route(Q8, wdt, odt, rows, N, K).decode() == route


FP16 = [
    # (out dtype, rows, N, K, route)
    (F32, 1, 2048, 2048, "one fp16 row"),
    (F32, 2, 1280, 1280, "one fp16 row"),  # 8.4, k_mfma_f16 10.0
    (F16, 2, 2304, 5760, "one fp16 row, rows"),  # 14.7, k_mfma_f16 37.5
    (F32, 2, 5632, 2048, "k_mfma_f16"),
    (F16, 3, 1280, 1280, "k_mfma_f16, rows"),
]


@pytest.mark.parametrize("odt,rows,N,K,route", FP16)
def test_two_fp16_rows_take_the_faster_route(nc, odt, rows, N, K, route):
    assert nc.lib().nc_debug_matmul_route(F16, F16, odt, rows, N, K).decode() == route


ATTN = [
    # (dtype, heads, rows, n_ctx, kernel)
    (F16, 32, 16, 128, "k_attn_rows"),  # 10.0, k_attn_f16 12.9
    (F16, 12, 64, 200, "k_attn_rows"),  # 12.5, k_attn_f16 15.8
    (F16, 20, 128, 200, "k_attn_rows"),  # 15.4, k_attn_f16 16.2
    (F16, 32, 8, 300, "k_attn_rows"),  # 15.9, k_attn_f16 16.8
    (F16, 32, 16, 512, "k_attn_rows"),  # 23.1, k_attn_f16 23.6
    (F16, 32, 100, 128, "k_attn_f16"),  # 13.9, k_attn_rows 14.8
    (F16, 32, 2, 256, "k_attn_f16"),  # 12.8, k_attn_rows 13.3
    (F16, 32, 64, 400, "k_attn_f16"),  # 21.4, k_attn_rows 22.6
    (F16, 32, 24, 1000, "k_attn_f16"),  # 36.8, k_attn_rows 40.3
    (F16, 32, 1500, 1500, "k_attn_f16"),  # 344, k_attn_rows 752
    (F16, 32, 8, 2177, "k_attn_rows"),  # its scores do not fit shared memory
    (Q8, 32, 512, 512, "k_attn_rows"),
    (F16, 32, 1, 512, "k_attn1"),  # 8.1, k_attn 9.6
    (Q8, 32, 1, 255, "k_attn"),
]


@pytest.mark.parametrize("dtype,heads,rows,n_ctx,route", ATTN)
def test_attention_takes_the_faster_route(nc, dtype, heads, rows, n_ctx, route):
    assert nc.lib().nc_debug_attn_route(dtype, heads, rows, n_ctx).decode() == route


NORM = [
    # (layer, dtype, width, rows, kernel)
    (0, Q8, 256, 64, "k_norm"),  # 5.5, k_norm8 5.9
    (1, F16, 256, 1500, "k_norm"),  # 12.7, k_norm8 13.4
    (0, Q8, 2048, 512, "k_norm8"),
    (1, F16, 2048, 1500, "k_norm8, loop mean"),  # 26.9, grid 29.7, k_norm 92
    (1, F16, 2048, 16, "k_norm8, loop mean"),  # 11.6, grid 15
    (1, F16, 2048, 1, "k_norm8, grid mean"),  # 10.7, loop 12
    (1, Q8, 2048, 64, "k_norm8, grid mean"),  # 10.8 in the mean, loop 12.6, k_norm 14.2
    (1, Q8, 2048, 128, "k_norm8, loop mean"),  # 13.6, grid 16 in the mean, k_norm 22
    (1, Q8, 1024, 1500, "k_norm8, grid mean"),  # 16.1, loop 19.4
    (1, Q8, 2304, 4, "k_norm8, grid mean"),  # 8.2, loop 13.4
    (1, Q8, 2304, 48, "k_norm8, loop mean"),  # 13.6, grid 8-22
    (1, Q8, 1536, 64, "k_norm8, grid mean"),  # 8.5, loop 11.6
    (1, Q8, 1536, 256, "k_norm8, loop mean"),  # 11.7, grid 16 in the mean
    (1, F16, 2304, 256, "k_norm8, loop mean"),  # 13.5, grid 20.8, k_norm 13.9
    (1, F16, 1280, 1, "k_norm8, grid mean"),  # 8.7, loop 9.6
    (1, F16, 1024, 256, "k_norm8, loop mean"),  # 9.2, grid 12.0, k_norm 10.1
    (1, F16, 3072, 4, "k_norm8, loop mean"),
]


@pytest.mark.parametrize("layer,dtype,d,rows,route", NORM)
def test_norms_take_the_faster_sums(nc, layer, dtype, d, rows, route):
    assert nc.lib().nc_debug_norm_route(layer, dtype, d, rows).decode() == route


EW = [
    # (silu, dtype, rows, cols, kernel)
    (1, Q8, 256, 5632, "k_ew8"),  # 5.4, k_ew 6.2
    (1, F16, 187, 5632, "k_ew"),  # 4.0, k_ew8 4.6
    (1, F16, 400, 2304, "k_ew"),  # 3.9, k_ew8 4.7
    (1, F16, 512, 5632, "k_ew8"),  # 7.0, k_ew 7.1
    (1, F32, 512, 5632, "k_ew"),  # 8.2, k_ew8 8.7
    (1, F32, 1500, 5632, "k_ew8"),  # 18.1, k_ew 20.6
    (0, F32, 400, 2304, "k_ew8"),  # 3.4, k_ew 3.7
    (0, Q8, 16, 2048, "k_ew"),
]


@pytest.mark.parametrize("silu,dtype,rows,cols,route", EW)
def test_elementwise_operators_take_the_faster_kernel(nc, silu, dtype, rows, cols, route):
    assert nc.lib().nc_debug_ew_route(silu, dtype, rows, cols).decode() == route
