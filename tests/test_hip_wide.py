"""The many-row matmul tiles (33 rows and more), where their dispatch can go wrong: every tile size at
ragged rows, outputs and block counts, and weight scales that are not finite. Every output is one
in-order chain per (row, column), so the expected values are the same rows in calls of at most 16
rows (other kernels, held to the oracle by test_hip_kernels.py), and the oracle itself for the first
and the last row; all bit for bit."""
import ctypes as C

import numpy as np
import pytest

from tables import CTable, HipTable, QUANT_TYPES, random_floats, random_weights, same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def o():
    return CTable("oracle")


@pytest.fixture(scope="module")
def h():
    return HipTable()


def inputs(o, kind, m, n_out, n_in, seed=1):
    xq = np.concatenate([o.quantize_row_q8_0(random_floats(n_in, seed * 1000 + r, 3.0)) for r in range(m)])
    return random_weights(kind, n_out, n_in, seed), xq


def check(o, h, kind, w, xq, m, n_out, n_in):
    nb = n_in // 32
    y = h.matmul(kind + "_q8", w, xq, n_out, n_in, n_rows=m).reshape(m, n_out)
    for r0 in range(0, m, 16):
        rows = min(16, m - r0)
        want = h.matmul(kind + "_q8", w, xq[r0 * nb:(r0 + rows) * nb], n_out, n_in, n_rows=rows)
        assert same_bits(y[r0:r0 + rows].ravel(), want), f"rows from {r0}"
    for r in (0, m - 1):
        assert same_bits(y[r], o.matmul(kind + "_q8", w, xq[r * nb:(r + 1) * nb], n_out, n_in))


@pytest.mark.parametrize("kind", QUANT_TYPES)
@pytest.mark.parametrize("m,n_out,n_in", [
    (65, 33, 64),        # 32 x 32 tiles: one partial chunk of two blocks, ragged rows and columns
    (70, 100, 576),      # a whole chunk of 16 blocks and a partial one of 2
    (512, 1984, 320),    # 32 x 64 tiles, partial chunks only
    (130, 6700, 896),    # 64 x 64 tiles, ragged in all three
    (33, 8200, 320),     # 33 rows of a matrix wide enough to leave the few-rows kernel
    (257, 6500, 1600),   # 64 x 128 tiles: 50 blocks, a last chunk of 2
])
def test_many_rows_bit_exact(o, h, kind, m, n_out, n_in):
    w, xq = inputs(o, kind, m, n_out, n_in)
    check(o, h, kind, w, xq, m, n_out, n_in)


@pytest.mark.parametrize("kind", QUANT_TYPES)
@pytest.mark.parametrize("m,n_out", [(65, 96), (128, 5632)])
def test_scales_that_are_not_finite(o, h, kind, m, n_out):
    """Infinite and NaN weight scales (and an infinite activation scale) give what the products
    give: infinities of the right sign where a sum is not zero, NaN where it is, and every other
    output untouched."""
    n_in = 640
    w, xq = inputs(o, kind, m, n_out, n_in, seed=3)
    nb = n_in // 32
    for row, block, bits in ((5, 0, 0x7c00), (37, 19, 0xfc00), (n_out - 1, 7, 0x7e00)):
        w["d"][row * nb + block] = bits
    xq["d"][3 * nb + 2] = 0x7c00
    xq["qs"][40 * nb:41 * nb] = 0
    check(o, h, kind, w, xq, m, n_out, n_in)


@pytest.mark.parametrize("kind", QUANT_TYPES)
@pytest.mark.parametrize("m,n_out", [(65, 96), (128, 5632)])
def test_scales_at_the_ends_of_the_half_range(o, h, kind, m, n_out):
    """Subnormal and largest half scales on both sides, and zero weights under negative scales."""
    n_in = 320
    w, xq = inputs(o, kind, m, n_out, n_in, seed=4)
    nb = n_in // 32
    rng = np.random.default_rng(5)
    w["d"] = rng.choice(np.array([0x0001, 0x8001, 0x03ff, 0x0400, 0x7bff, 0xfbff, 0x8000, 0x2c00], np.uint16), len(w))
    xq["d"] = rng.choice(np.array([0x0001, 0x03ff, 0x7bff, 0x0000, 0x2c00], np.uint16), len(xq))
    w["qs"][7 * nb:8 * nb] = 0 if kind != "q4_0" else 0x88
    check(o, h, kind, w, xq, m, n_out, n_in)


@pytest.mark.parametrize("kind", QUANT_TYPES)
@pytest.mark.parametrize("m,n_in,n_ff", [(33, 320, 4096), (65, 576, 160), (130, 896, 4864), (257, 1600, 6560)])
def test_swiglu_tiles_bit_exact(o, h, kind, m, n_in, n_ff):
    """gate|up with the product and its blocks in the epilogue against the separate entries, at both
    tile sizes and at outputs that end inside a tile."""
    H = h.H
    wg, xq = inputs(o, kind, m, n_ff, n_in, seed=5)
    wu = random_weights(kind, n_ff, n_in, 6)
    t = {"q8_0": 8, "q4_0": 2, "q4_1": 3}[kind]
    g = h.matmul(kind + "_q8", wg, xq, n_ff, n_in, n_rows=m)
    u = h.matmul(kind + "_q8", wu, xq, n_ff, n_in, n_rows=m)
    want = h.silu_mul(g, u)
    dg, du, dx = (H.DeviceBuffer.of(a) for a in (wg, wu, xq))
    out, outq = H.DeviceBuffer(m * n_ff * 4), H.DeviceBuffer(m * n_ff // 32 * 34)
    H.call("matmul_q8_swiglu", C.c_int(t), dx, m, n_in, dg, du, n_ff, out, outq)
    assert same_bits(out.download(np.float32), want)
    assert outq.download(np.uint8).tobytes() == h.quantize_row_q8_0(want).tobytes()
