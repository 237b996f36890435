"""The device memory of an encode: it holds the list of its own closed-loop schedule only."""
import pytest

import av1gpu_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [0, 1])
def test_gpu_schedule_list(graph):
    """512 x 512: 64 superblocks.  The persistent schedule lists 128 items (512 bytes), one launch per step 64
    superblocks (256 bytes, the arena's granularity); everything else is the same."""
    W, H = 512, 512
    f = A.DeviceFrame(A.synth_image(1090, W, H), W, H)
    size, rec = {}, {}
    for sched in (0, 1):
        e = A.GpEncoder().init(A.GpConfig(qindex=200, schedule=sched, graph=graph))
        for _ in range(2 + graph):   # a captured plan replays with the list it was captured with
            (o,), t = e.encode([f])
            assert rec.setdefault("coeffs", o.coeffs.tobytes()) == o.coeffs.tobytes()
        size[sched] = t.deviceBytes
        e.close()
    f.close()
    assert size[0] - size[1] == 256
