"""The oracle's forward pass splits columns and rows over threads: any number of them gives the same
bits, and a pass really uses them (on one thread the full-depth model tests take over ten minutes)."""
import ctypes as C
import os

import numpy as np
import pytest

from helpers import GOLDEN, OracleModel


def set_threads(n):
    C.CDLL("libgomp.so.1").omp_set_num_threads(n)


@pytest.fixture
def default_threads():
    n = C.CDLL("libgomp.so.1").omp_get_max_threads()
    yield
    set_threads(n)


def passes(path, f16):
    """A prompt, one row behind it, and a batch of three sequences of different lengths."""
    m = OracleModel(path)
    caches = [m.new_cache(64, f16=f16) for _ in range(3)]
    out = [m.forward(np.arange(1, 20 + i), c) for i, c in enumerate(caches)]
    out.append(m.forward([3], caches[0]))
    out.append(m.forward_batch([5, 6, 7], caches))
    if not f16:
        out.append(m.forward(np.arange(30)))
    return np.concatenate(out)


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("kind", ["", "-q4_0"])
def test_any_number_of_threads_gives_the_same_bits(default_threads, kind, f16):
    path = GOLDEN / "gguf" / f"synthetic-2l{kind}.gguf"
    set_threads(1)
    want = passes(path, f16).view(np.uint32)
    for n in (2, 5):
        set_threads(n)
        assert np.array_equal(passes(path, f16).view(np.uint32), want), n


def test_a_pass_uses_the_threads(default_threads):
    set_threads(23)  # more than anything else in this process has started
    before = len(os.listdir("/proc/self/task"))
    passes(GOLDEN / "gguf" / "synthetic-2l-q4_0.gguf", False)
    assert len(os.listdir("/proc/self/task")) > before
