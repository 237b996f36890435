"""The persistent closed loop's item orders (luma and chroma of a superblock as separate items, progress published per
block or per superblock, from one workgroup to one per item) against one launch per wavefront step: the same records and
reconstruction at the edges of the rules (one superblock, one column, one row, ragged frame edges, frames without chroma,
4:4:4, several images whose chains differ in length)."""
import numpy as np
import pytest

import av1gpu_amd as A

pytestmark = pytest.mark.gpu


def _encode(frames, **kw):
    e = A.GpEncoder().init(A.GpConfig(qindex=100, **kw))
    try:
        out, t = e.encode(frames)
        return [(o.blocks.copy(), o.block_txb.copy(), o.txb.copy(), o.coeffs.copy(), [p.copy() for p in o.recon]) for o in out], t
    finally:
        e.close()


# (sizes, 4:4:4, bit depth, monochrome)
CASES = [([(40, 24)], False, 8, False), ([(72, 520)], False, 8, False), ([(520, 40)], False, 10, False), ([(201, 139)], False, 8, True),
         ([(201, 139)], True, 8, False), ([(64, 64), (264, 328), (130, 18)], False, 8, False)]


@pytest.mark.parametrize("sizes,yuv444,bd,mono", CASES)
def test_gpu_item_orders_agree(sizes, yuv444, bd, mono):
    frames = [A.DeviceFrame(A.synth_image(900 + k, W, H, ssx=0 if yuv444 else 1, bd=bd), W, H, bd=bd, yuv444=yuv444)
              for k, (W, H) in enumerate(sizes)]
    ins = [f.frame_in() for f in frames]
    for f in ins:
        f.mono = int(mono)
    ref, _ = _encode(ins, schedule=1)
    for qb, occ in ((0, 1), (0, 2), (1, 1), (2, 1), (5, 2)):
        print("queueBlocks", qb, "queueOcc", occ, flush=True)
        got, t = _encode(ins, queueBlocks=qb, queueOcc=occ)
        assert t.schedule == 0 and t.queueOcc == occ
        for g, r in zip(got, ref):
            for a, b in zip(g[:4], r[:4]):
                assert np.array_equal(a, b)
            for a, b in zip(g[4], r[4]):
                assert np.array_equal(a, b)
    for f in frames:
        f.close()
