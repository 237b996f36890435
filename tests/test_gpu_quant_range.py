"""Rounding offsets outside the usual range against the oracle, bit for bit: the quantizer truncates quotient + offset, so an
offset below -1 with a small dead zone gives levels of the other sign (-1, or -40 with every coefficient nonzero), whose
contexts and costs go by their magnitudes like any other's; an offset of 1 and more makes every level nonzero."""
import numpy as np
import pytest

import av1gpu_amd as A
from test_gpu_parity import _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rnd,zbin", [(-1.75, 0.5), (-40.0, 0.0), (1.5, 0.0), (20.0, 0.0)])
@pytest.mark.parametrize("W,H,bd,ss", [(72, 64, 8, 1), (64, 24, 10, 0)])
def test_gpu_quantizer_offsets_equal_oracle(oracle, rnd, zbin, W, H, bd, ss):
    print("case", rnd, zbin, W, H, bd, ss, flush=True)
    kw = dict(rnd=rnd, zbin=zbin, rndC=rnd, zbinC=zbin)
    planes = A.synth_image(1080, W, H, ssx=ss, bd=bd)
    e = A.GpEncoder().init(A.GpConfig(qindex=120, P=A.GpParams(**kw)))
    f = A.DeviceFrame(planes, W, H, bd=bd, yuv444=not ss)
    g = e.encode([f])[0][0]
    f.close()
    e.close()
    r = oracle.encode(planes, W, H, ssx=ss, bd=bd, qindex=120, params=oracle.params(**kw), threads=8)
    assert np.count_nonzero(r["coeffs"]) > 0
    _same(g, r)
