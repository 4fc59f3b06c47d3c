"""F32 / F16 / BF16 weights against float activations around the kernel's tiles (16 outputs x 16 or 32
rows, chunks of 256 elements, two loaded ahead): odd sizes, one to three chunks and more, strided
outputs, weights that pairs of elements are not aligned for, special values; bit for bit against the
oracle."""
import numpy as np
import pytest

from tables import CTable, HipTable, random_floats, same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def o():
    return CTable("oracle")


@pytest.fixture(scope="module")
def h():
    return HipTable()


def weights(kind, n, seed):
    w = random_floats(n, seed, 2.0)
    w[::97] = -0.0
    w[5::501] = 1e-7  # below the smallest normal half
    if kind == "f16":
        return w.astype(np.float16).view(np.uint16)
    return (w.view(np.uint32) >> 16).astype(np.uint16) if kind == "bf16" else w


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n_rows,n_out,n_in", [(1, 1, 1), (1, 17, 255), (3, 16, 256), (16, 33, 257), (17, 15, 513),
                                               (33, 50, 1031), (2, 300, 2048)])
def test_float_matmul_tiles(o, h, kind, n_rows, n_out, n_in):
    w, x = weights(kind, n_out * n_in, 1), random_floats(n_rows * n_in, 2, 3.0)
    stride = n_out + 2
    want = o.matmul(kind, w, x, n_out, n_in, n_rows=n_rows, y_stride=stride)
    got = h.matmul(kind, w, x, n_out, n_in, n_rows=n_rows, y_stride=stride)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    if n_rows == 1:
        assert np.array_equal(h.matmul(kind, w, x, n_out, n_in).view(np.uint32), want[:n_out].view(np.uint32))


# Either side of the lines between one lane per output and the tiles: 28 bytes a row of 16-bit weights, 36
# (but 32) of 32-bit ones, 416 bytes in all rows, and 100 or 128 bytes of one row against many outputs.
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n_rows,n_out,n_in", [(40, 300, 7), (40, 300, 8), (40, 300, 9), (40, 300, 10), (33, 270, 14), (33, 270, 15),
                                               (8, 257, 13), (8, 257, 26), (8, 257, 27), (1, 100, 40), (1, 100, 41), (1, 8192, 50),
                                               (1, 8191, 50), (1, 32000, 64), (1, 31999, 64), (1, 32001, 65)])
def test_float_matmul_short_rows(o, h, kind, n_rows, n_out, n_in):
    w, x = weights(kind, n_out * n_in, 9), random_floats(n_rows * n_in, 10, 3.0)
    want = o.matmul(kind, w, x, n_out, n_in, n_rows=n_rows, y_stride=n_out + 1)
    assert same_bits(h.matmul(kind, w, x, n_out, n_in, n_rows=n_rows, y_stride=n_out + 1), want)


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
def test_float_matmul_infinities_stay_in_their_row(o, h, kind):
    n_rows, n_out, n_in = 18, 20, 300
    w, x = weights(kind, n_out * n_in, 3), random_floats(n_rows * n_in, 4)
    x[7 * n_in + 299] = np.inf
    x[17 * n_in] = np.nan
    want = o.matmul(kind, w, x, n_out, n_in, n_rows=n_rows)
    assert same_bits(h.matmul(kind, w, x, n_out, n_in, n_rows=n_rows), want)


# Both row counts of a tile on whole and partial ones: 32 rows up to 16 rows of input, and from 256
# workgroups on; 16 rows between.
@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n_rows,n_out,n_in", [(16, 32, 512), (17, 32, 768), (31, 4100, 270), (33, 2049, 512), (65, 1366, 258)])
def test_float_matmul_tile_heights(o, h, kind, n_rows, n_out, n_in):
    w, x = weights(kind, n_out * n_in, 5), random_floats(n_rows * n_in, 6, 3.0)
    want = o.matmul(kind, w, x, n_out, n_in, n_rows=n_rows)
    got = h.matmul(kind, w, x, n_out, n_in, n_rows=n_rows)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("kind", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("n_rows", [3, 20])
def test_float_matmul_weights_off_pair_alignment(o, h, kind, n_rows):
    """Even rows from an address that is a whole element, not a whole pair; activations off 16 bytes."""
    n_out, n_in = 35, 514
    w, x = weights(kind, n_out * n_in + 1, 7), random_floats(n_rows * n_in + 1, 8, 3.0)
    dw, dx, y = h._dev(w), h._dev(x), h._dev(np.zeros(n_rows * n_out, np.float32))
    h.H.call(f"matmul_{kind}_rows", dw.at(w.itemsize), dx.at(4), y, n_rows, n_out, n_in, n_out)
    want = o.matmul(kind, w[1:].copy(), x[1:].copy(), n_out, n_in, n_rows=n_rows)
    assert np.array_equal(y.download(np.float32).view(np.uint32), want.view(np.uint32))
