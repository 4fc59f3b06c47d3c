"""Many-row attention with its products on the matrix cores (kv groups of 4 and 8 heads), where it
can go wrong: rows that end inside a block, positions around the 64- and 32-position stages, the
16-pair form of long contexts, spans that are not 16-byte aligned, blocks whose rows belong to
different sequences, and values that are not finite past a row's own positions. Workgroups take 16 (row, head)
pairs where there are 512 of them and two share a CU, else 32 where there are 256. Bit for bit against
the oracle, the Q8_0 blocks of the outputs too."""
import ctypes as C

import numpy as np
import pytest

from tables import CTable, HipTable

pytestmark = pytest.mark.gpu
HD = 64


@pytest.fixture(scope="module")
def o():
    return CTable("oracle")


@pytest.fixture(scope="module")
def h():
    return HipTable()


def run(h, q, pool, k_off, v_off, n_vis, n_head, n_kv, f16):
    H = h.H
    n = len(n_vis)
    bufs = [H.DeviceBuffer.of(a) for a in (q, pool, np.asarray(k_off, np.int64), np.asarray(v_off, np.int64),
                                           np.asarray(n_vis, np.int32))]
    out, outq = H.DeviceBuffer(n * n_head * HD * 4), H.DeviceBuffer(n * n_head * HD // 32 * 34)
    a = H.AttentionRowsArgs()
    a.q, a.kv, a.k_off, a.v_off, a.n_vis = (b.ptr for b in bufs)
    a.out, a.outq, a.q_stride, a.out_stride = out.ptr, outq.ptr, n_head * HD, n_head * HD
    a.n_head, a.n_kv, a.head_dim, a.scale, a.f16, a.max_vis = n_head, n_kv, HD, 0.125, int(f16), max(n_vis)
    scratch = H.DeviceBuffer(4 * max(1, H.lib().axon_hip_attention_scratch_floats(C.byref(a), C.c_size_t(n))))
    a.scratch = scratch.ptr
    H.call("attention_rows", C.c_void_p(C.addressof(a)), n)
    return out.download(np.float32).reshape(n, n_head, HD), outq.download(np.uint8)


def check(o, h, chunk, past, decode, n_head, n_kv, f16, shift=0, poison=False, seed=1, change=None):
    """A chunk of `chunk` rows behind `past` positions, then one row of each sequence in `decode`.
    `change` alters the queries and the chunk's keys and values in place."""
    rng = np.random.default_rng(seed)
    seqs = [past + chunk] + list(decode)
    n = chunk + len(decode)
    row = n_kv * HD
    q = rng.standard_normal((n, n_head, HD)).astype(np.float32)
    kv = [(rng.standard_normal((m, row)).astype(np.float32), rng.standard_normal((m, row)).astype(np.float32)) for m in seqs]
    if change is not None:
        change(rng, q, *kv[0])
    if f16:
        kv = [(k.astype(np.float16), v.astype(np.float16)) for k, v in kv]
    want = np.zeros((n, n_head, HD), np.float32)
    view = (lambda x: x.view(np.uint16)) if f16 else (lambda x: x)
    want[:chunk] = o.attention_kv_heads(q[:chunk], view(kv[0][0]), view(kv[0][1]), chunk, past, n_head, n_kv, HD, 0.125,
                                        0, n_head, f16=f16)
    for i, m in enumerate(decode):
        k, v = kv[1 + i]
        want[chunk + i] = o.attention_kv_heads(q[chunk + i:chunk + i + 1], view(k), view(v), 1, m - 1, n_head, n_kv, HD,
                                               0.125, 0, n_head, f16=f16)[0]
    if poison:
        # The last position is seen by the chunk's last row only: every other row's output must not
        # take anything from it.
        kv[0][0][-1] = np.nan
        kv[0][1][-1] = np.inf
    parts, k_off, v_off, at = [np.zeros(shift, kv[0][0].dtype)], [], [], shift
    for k, v in kv:
        k_off.append(at)
        v_off.append(at + k.size)
        parts += [k.ravel(), v.ravel()]
        at += 2 * k.size
    of = [0] * chunk + list(range(1, 1 + len(decode)))
    n_vis = [past + i + 1 for i in range(chunk)] + list(decode)
    got, blocks = run(h, q, np.concatenate(parts), [k_off[i] for i in of], [v_off[i] for i in of], n_vis, n_head, n_kv, f16)
    keep = [r for r in range(n) if not (poison and r == chunk - 1)]
    assert np.array_equal(got[keep].view(np.uint32), want[keep].view(np.uint32))
    per_row = n_head * HD // 32 * 34
    wq = h.quantize_row_q8_0(np.ascontiguousarray(want).ravel()).view(np.uint8).reshape(n, per_row)
    assert np.array_equal(blocks.reshape(n, per_row)[keep], wq[keep])


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("chunk,past,n_head,n_kv", [
    (250, 0, 32, 8),     # 32 pairs; a last block of two rows; contexts from one position up
    (385, 63, 32, 8),    # a last block of one row, contexts across the first K stage
    (257, 63, 32, 8),    # 16 pairs: a last block of one row
    (505, 31, 32, 4),    # groups of 8 heads: two or four rows per workgroup
    (128, 1100, 32, 8),  # 16 pairs' LDS, too few workgroups for them
    (128, 1030, 64, 8),  # the same with groups of 8
    (64, 1100, 128, 32),  # both again at the 512 workgroups that 16 pairs ask for
    (64, 1030, 128, 16),
    (256, 1500, 32, 4),  # rows too long for the blocked kernel's LDS: one per CU of 16 pairs, with a scratch
])
def test_chunk(o, h, chunk, past, n_head, n_kv, f16):
    check(o, h, chunk, past, [], n_head, n_kv, f16)


# Either side of the last position at which two workgroups of 16 pairs share a CU, and of the last
# that 32 pairs' scores fit.
@pytest.mark.parametrize("f16,total", [(False, 832), (False, 833), (False, 1024), (False, 1025), (True, 1024), (True, 1025),
                                       (True, 1152), (True, 1153)])
def test_positions_at_the_edges_of_lds(o, h, f16, total):
    check(o, h, 256, total - 256, [], 32, 8, f16)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("chunk", [250, 257])  # 32 pairs, 16 pairs
def test_unaligned_span(o, h, chunk, f16):
    check(o, h, chunk, 20, [], 32, 8, f16, shift=1)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("chunk,n_head,n_kv", [(243, 32, 8), (254, 32, 8), (243, 64, 8), (120, 64, 8)])
def test_rows_of_other_sequences(o, h, chunk, n_head, n_kv, f16):
    check(o, h, chunk, 9, [1, 64, 65, 300, 17, 128, 33], n_head, n_kv, f16)


def test_nothing_from_past_a_rows_positions(o, h):
    check(o, h, 248, 15, [], 32, 8, False, poison=True)  # 32 pairs
    check(o, h, 256, 15, [], 32, 8, False, poison=True)  # 16


def subnormal(rng, q, k, v):
    """Rows whose products with the keys lie below the smallest normal float, rows whose scores lie so
    far apart that most probabilities do, and values of every size."""
    q[::4] *= np.float32(1e-37)
    q[1::4] *= np.float32(1e-40)
    q[2::4] *= np.float32(40)
    k[:, ::2] *= np.float32(1e-3)
    v *= (np.float32(10) ** rng.integers(-40, 1, v.shape)).astype(np.float32)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("chunk", [248, 256])  # 32 pairs, 16 pairs
def test_subnormal_products(o, h, chunk, f16):
    check(o, h, chunk, 15, [], 32, 8, f16, change=subnormal)
