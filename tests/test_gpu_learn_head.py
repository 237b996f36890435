"""The pruning network's head to the bit: each logit is the fmaf chain b[o], f = 0 .. 511 in ascending order, that a scalar
loop makes of the FP32 weights and BF16 features.  Item counts at and around the tiles of 16 items.  The chain is made in
NumPy: a float32 x BF16 product is exact in float64, and the sum is rounded to odd there (two-sum gives the part lost),
from which the rounding to float32 is that of the exact sum."""
import ctypes
import ctypes.util

import numpy as np
import pytest

from av1gpu_amd import learn as Ln


def fma32(a, b, c):
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)
    s = p + c
    t = s - p
    e = (p - (s - t)) + (c - t)
    even = (s.view(np.int64) & 1) == 0
    odd = np.nextafter(s, np.where(e > 0, np.inf, -np.inf))
    return np.where((e != 0) & even, odd, s).astype(np.float32)


def test_fma32_is_fmaf():
    f = ctypes.CDLL(ctypes.util.find_library("m")).fmaf
    f.argtypes, f.restype = [ctypes.c_float] * 3, ctypes.c_float
    rng = np.random.default_rng(3)
    a = (rng.standard_normal(20000) * 10.0 ** rng.integers(-6, 7, 20000)).astype(np.float32)
    b = (rng.standard_normal(20000) * 10.0 ** rng.integers(-2, 3, 20000)).astype(np.float32)
    b = (b.view(np.uint32) & 0xFFFF0000).view(np.float32)
    c = (rng.standard_normal(20000) * 10.0 ** rng.integers(-6, 7, 20000)).astype(np.float32)
    c[::4] = (-a[::4] * b[::4]).astype(np.float32)   # cancellation
    assert np.array_equal(fma32(a, b, c), np.array([f(*map(float, v)) for v in zip(a, b, c)], np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,shipped", [(1, True), (15, False), (16, True), (17, False), (300, True)])
def test_gpu_head_is_the_fmaf_chain(n, shipped):
    rng = np.random.default_rng(n)
    p = Ln.load_params() if shipped else Ln.init_params(21)
    L = Ln.Learner(p)
    logits = L.forward(rng.integers(0, 256, (n, 64, 64), dtype=np.uint8), rng.integers(1, 256, n).astype(np.uint8))
    x = L.activations(4, n).reshape(n, Ln.N_FEAT)
    L.close()
    _, w, b = Ln.unpack(p)
    z = np.broadcast_to(b.astype(np.float32), (n, Ln.N_OUT)).copy()
    for k in range(Ln.N_FEAT):
        z = fma32(np.broadcast_to(w[:, k], z.shape), np.broadcast_to(x[:, k:k + 1], z.shape), z)
    assert np.count_nonzero(x) > 0 and np.array_equal(logits, z)
