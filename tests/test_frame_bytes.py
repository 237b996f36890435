"""av1mi_frame_bytes is an upper bound of a frame's device bytes: per superblock it covers every array that an encode's
arena holds for it.  Checked as the growth between two frames of whole superblocks, both above the pruning network's
chunk (65536 superblocks), where its activations no longer grow."""
import pytest

import av1gpu_amd as A

LEAVES, SHAPES = 256, [(4, 4), (4, 8), (8, 4), (8, 8), (8, 16), (16, 8), (16, 16), (16, 32), (32, 16), (32, 32), (32, 64), (64, 32),
                       (64, 64), (4, 16), (16, 4), (8, 32), (32, 8), (16, 64), (64, 16)]


@pytest.mark.parametrize("bd,yuv444", [(8, 0), (10, 1)])
def test_frame_bytes_cover_each_superblocks_arrays(bd, yuv444):
    f = A.lib().av1mi_frame_bytes
    n = 1024 * 128
    per_sb = (f(65536, 2 * 8192, bd, yuv444) - f(65536, 8192, bd, yuv444)) / n
    chroma = 2 * (64 * 64 if yuv444 else 32 * 32)
    planes = (64 * 64 + chroma) * (2 if bd == 10 else 1)
    txb, coef = (768, 12288) if yuv444 else (384, 6144)
    maps = 5 * 256 + 2 * (256 + 2 * (256 if yuv444 else 64))
    analysis = 12 * sum((64 // w) * (64 // h) for w, h in SHAPES)
    slots = LEAVES * (16 + 2) + txb * 16 + coef * 2            # block, its first tx block; tx blocks; coefficients
    search = LEAVES * 4 + 2 + 4 + 4 + 16 + 24                  # leaves and their count, image, cost, counts, pack offsets
    loop = 2 * 4 + 2 * 4                                       # closed loop: two progress words and two items
    records = LEAVES * (16 + 4) + txb * 16 + coef * 2
    network = 12 * 4                                           # masks
    assert per_sb >= 2 * planes + maps + analysis + slots + search + loop + records + network
