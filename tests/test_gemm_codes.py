"""The code operands and accumulator starts of the prefill matmul, on the CPU.

k_gemm_qw hands the fp16 matrix cores raw codes and takes what that adds off
the accumulator's start (the reference's lane sums: gten/ops.cpp:387-490):
Q8 weights as 1024 + (w + 128) with the start -1152 sum x; Q4 low nibbles as
1024 + n against x with -1031 sum x, high nibbles in place as 1024 + 16 n
against x / 16 with -71 sum x.  Each must equal the integer lane sum, with
every operand exact in fp16 and every value on the way an integer below 2^22,
exact in fp32 in any order.
"""
import numpy as np
import pytest

rng = np.random.default_rng(20261204)


def _h1024(byte):
    return (0x6400 | np.asarray(byte, np.uint16)).astype(np.uint16).view(np.float16)


def _codes(lo, hi):
    cases = [(rng.integers(-127, 128, 8), rng.integers(lo, hi + 1, 8)) for _ in range(2000)]
    cases += [(np.full(8, x), np.full(8, w)) for x in (127, -127, 0, 1) for w in (lo, hi, 0 if lo < 0 else 7)]
    cases.append((np.array([127, -127] * 4), np.array([hi, lo] * 4)))
    return cases


def _sum(start, xs, ws, order):
    acc = np.float32(start)
    for i in order:
        p = np.float32(xs[i]) * np.float32(ws[i])
        acc = np.float32(acc + p)
        assert abs(float(p)) < 2**22 and abs(float(acc)) < 2**22
    return acc


@pytest.mark.parametrize("kind", ["q8", "q4-low", "q4-high"])
def test_code_operands_give_the_lane_sum(kind):
    for x, w in _codes(-127, 127) if kind == "q8" else _codes(0, 15):
        sx = int(x.sum())
        if kind == "q8":
            xs, ws, start, want = x.astype(np.float16), _h1024((w + 128) & 255), -1152 * sx, int((x * w).sum())
        elif kind == "q4-low":
            xs, ws, start, want = x.astype(np.float16), _h1024(w), -1031 * sx, int((x * (w - 7)).sum())
        else:
            xs, ws = (x.astype(np.float32) / 16).astype(np.float16), _h1024(w << 4)
            start, want = -71 * sx, int((x * (w - 7)).sum())
            # (1024 + c + 128) / 16 - 72, rounded once, is c / 16
            one = (_h1024((x + 128) & 255).astype(np.float32) / 16 - 72).astype(np.float16)
            assert np.array_equal(one, xs) and np.array_equal(xs.astype(np.float32) * 16, x)
        for order in (range(8), range(7, -1, -1), (0, 4, 1, 5, 2, 6, 3, 7)):
            assert _sum(start, xs, ws, order) == want
