"""The products of few rows, whose K is split over a workgroup's waves, carry
the bits of the same rows in a larger product (tiles of k_gemm) and, up to 16
rows, of the GEMV: at the edges of its 32-row tiles, with a ragged last tile
in n, with chunk counts that do not fill its rounds of eight, for the EXACT
and the int8-activation forms, and with the FFN's prepared hand-off.

The bits are compared, so there is no tolerance; the larger product is checked
against the oracle by the parity tests."""
import sys

import numpy as np
import pytest

import mynah_hip as M

pytestmark = pytest.mark.gpu

ROWS = [16, 17, 31, 32, 33, 63, 64, 65, 128, 129, 250]
FMTS = [M.F32, M.INT8, M.INT4, M.Q4_0, M.Q8_0, M.Q2_K, M.Q3_K, M.Q4_K, M.Q5_K, M.Q6_K]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


def _check(gpu, qt, n, k, big, rows, act=0):
    import torch
    dw = M.DeviceWeight(gpu, M.Weight.make(gpu, qt, gpu.randn(3, 0.02, (n, k))))
    x = torch.from_numpy(gpu.randn(4, 1.0, (big, k))).cuda()
    torch.cuda.synchronize()

    def product(m):
        y = torch.full((m, n), float("nan"), device="cuda")
        torch.cuda.synchronize()
        dw.gemm(x.data_ptr(), y.data_ptr(), m, act)
        torch.cuda.synchronize()
        return y

    try:
        ref = _bits(product(big))
        assert np.isfinite(ref.view(np.float32)).all()
        for m in rows:
            assert np.array_equal(_bits(product(m)), ref[:m]), f"M={m}"
    finally:
        dw.close()


@pytest.mark.parametrize("qt", FMTS, ids=lambda q: M.NAMES[q])
def test_rows_carry_the_larger_products_bits(gpu, qt):
    say("few rows", M.NAMES[qt], "1024 -> 1000")
    _check(gpu, qt, 1000, 1024, 1600, ROWS)


@pytest.mark.parametrize("n,k", [(1024, 4096), (96, 640), (200, 128), (130, 1184)],
                         ids=["four-rounds", "6chunks", "2chunks", "10chunks"])
def test_rounds_and_ragged_columns(gpu, n, k):
    say("few rows Q8_0", k, "->", n)
    _check(gpu, M.Q8_0, n, k, 1600 if n > 512 else 12100, [17, 64, 65, 750], act=1)


# the row counts on both sides of each line of the rule that chooses this form
# (256, 512, 640, 768, 1024, 1280, 1408 tiles of 32 x 32 by K and format)
EDGES = [(1024, 256, [256, 257]), (1024, 512, [512, 513, 768, 769]), (1024, 1024, [768, 769, 1024, 1025]),
         (640, 1280, [1024, 1025, 1632, 1633]), (1024, 2048, [1280, 1281, 1408, 1409])]


@pytest.mark.parametrize("qt", [M.F32, M.INT4, M.Q8_0, M.Q4_K, M.Q6_K], ids=lambda q: M.NAMES[q])
@pytest.mark.parametrize("n,k,rows", EDGES, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_rows_at_the_rules_edges(gpu, qt, n, k, rows):
    say("few rows, rule edges", M.NAMES[qt], k, "->", n)
    _check(gpu, qt, n, k, 2200, rows)


@pytest.mark.parametrize("qt", [M.Q4_0, M.Q8_0, M.Q2_K, M.Q5_K, M.Q6_K], ids=lambda q: M.NAMES[q])
def test_int8_activation_rows(gpu, qt):
    say("few rows, int8 activations", M.NAMES[qt])
    gpu.set_numerics(M.INT8ACT)
    try:
        _check(gpu, qt, 1000, 1024, 1600, ROWS)
    finally:
        gpu.set_numerics(M.EXACT)


@pytest.mark.parametrize("q1,q2", [(M.Q8_0, M.Q8_0), (M.F32, M.Q2_K), (M.Q6_K, M.Q4_K), (M.Q4_K, M.INT4)],
                         ids=lambda q: M.NAMES[q])
def test_ffn_hand_off(gpu, q1, q2):
    """The prepared hand-off against the larger FFN's (k_gemm's epilogue)."""
    import torch
    say("few rows FFN", M.NAMES[q1], M.NAMES[q2])
    d, f, big = 512, 1024, 2100   # (256 workgroups of the prepared output at 1024 rows)
    w1 = M.DeviceWeight(gpu, M.Weight.make(gpu, q1, gpu.randn(5, 0.05, (f, d))))
    w2 = M.DeviceWeight(gpu, M.Weight.make(gpu, q2, gpu.randn(6, 0.05, (d, f))))
    x = torch.from_numpy(gpu.randn(7, 1.0, (big, d))).cuda()
    torch.cuda.synchronize()

    def ffn(m):
        y = torch.full((m, d), float("nan"), device="cuda")
        torch.cuda.synchronize()
        M.ffn_dev(gpu, w1, w2, x.data_ptr(), y.data_ptr(), m)
        torch.cuda.synchronize()
        return y

    try:
        ref = _bits(ffn(big))
        assert np.isfinite(ref.view(np.float32)).all()
        for m in (17, 64, 65, 250, 512, 513, 1024, 1025):
            assert np.array_equal(_bits(ffn(m)), ref[:m]), f"M={m}"
    finally:
        w1.close()
        w2.close()


@pytest.mark.parametrize("qt", FMTS, ids=lambda q: M.NAMES[q])
def test_one_row_carries_the_larger_products_bits(gpu, qt):
    """One row is split by its whole wave: one and several chunks per wave, two
    column groups per workgroup, the split over workgroups, and the largest K."""
    import torch
    for n, k in [(1000, 1024), (8200, 512), (130, 1280), (1024, 4096), (2100, 4096), (96, 8192)]:
        say("one row", M.NAMES[qt], n, k)
        _check(gpu, qt, n, k, 40, [1])
    # rows off the 16-byte grid, whose elements are loaded one by one
    n, k = 200, 768
    dw = M.DeviceWeight(gpu, M.Weight.make(gpu, qt, gpu.randn(3, 0.02, (n, k))))
    x = torch.from_numpy(gpu.randn(4, 1.0, (1 + 40 * k,))).cuda()
    y = torch.empty((40, n), device="cuda")
    y1 = torch.empty((1, n), device="cuda")
    torch.cuda.synchronize()
    try:
        dw.gemm(x.data_ptr() + 4, y.data_ptr(), 40, 0)
        dw.gemm(x.data_ptr() + 4, y1.data_ptr(), 1, 0)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(y1), _bits(y)[:1])
    finally:
        dw.close()


@pytest.mark.parametrize("k", [1, 37, 129, 1027])
def test_one_row_of_odd_length(gpu, k):
    say("one row, K", k)
    _check(gpu, M.F32, 70, k, 40, [1])
