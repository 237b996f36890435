"""The matrix-core transforms of tx blocks with a side of 32 or 64 against the oracle, bit for bit, where their special cases
lie: residuals so large that a virtual lane's energy passes 2^24 (10-bit noise and hard steps: the order of the float sums
matters there), flat blocks (no coefficient), frame edges inside a 64x64 block, the quantizer's end points, 4:4:4 chroma."""
import numpy as np
import pytest

import av1gpu_amd as A
from test_gpu_parity import same_search

pytestmark = pytest.mark.gpu


def _planes(kind, W, H, bd, ss):
    rng = np.random.default_rng(W * 1000 + H)
    top = (1 << bd) - 1
    dt = np.uint16 if bd > 8 else np.uint8
    shapes = [(H, W)] + [((H + ss) >> ss, (W + ss) >> ss)] * 2
    if kind == "noise":     # full-range noise
        return [rng.integers(0, top + 1, s).astype(dt) for s in shapes]
    if kind == "steps":     # full-range columns of 8 samples
        return [np.tile(((np.arange(s[1]) // 8) % 2 * top).astype(dt), (s[0], 1)) for s in shapes]
    return [np.full(s, top // 2, dt) for s in shapes]


@pytest.mark.parametrize("kind,W,H,bd,q,ss", [("noise", 128, 64, 10, 120, 1), ("noise", 72, 136, 8, 20, 1), ("steps", 136, 72, 10, 255, 1),
                                              ("steps", 64, 128, 10, 200, 0), ("flat", 130, 70, 8, 1, 1), ("noise", 64, 64, 10, 255, 0)])
def test_gpu_wide_blocks_equal_oracle(oracle, kind, W, H, bd, q, ss):
    planes = _planes(kind, W, H, bd, ss)
    e = A.GpEncoder().init(A.GpConfig(qindex=q))
    e.set_search_export(True)
    f = A.DeviceFrame(planes, W, H, bd=bd, qindex=q, yuv444=not ss)
    g = e.encode([f])[0][0]
    ex = e.search_export(0)
    f.close()
    e.close()
    r = oracle.encode(planes, W, H, ssx=ss, bd=bd, qindex=q, threads=8, detail=True)
    same_search(ex, r)
    for k in ("blocks", "block_txb", "txb", "coeffs"):
        assert np.array_equal(getattr(g, k), r[k]), k
    for p in range(3):
        assert np.array_equal(g.recon[p].astype(np.uint16), r["recon"][p]), "recon plane %d" % p
