"""Performance cases of the intra RD core: the calls that a program using this package makes, from one thumbnail to
batches of camera images, exhaustive and with the learned pruning, 8-bit 4:2:0 and 10-bit 4:4:4, a whole request from
host planes to an AVIF file, and the pruning network's training gradient (forward and backward).

A case is a dict of plain values.  ``kind``:
  encode   one ``GpEncoder.encode`` call on ``n`` images resident in device memory.  The sizes are ``w`` x ``h``, or,
           with ``w`` 0, log-uniform over ``mp_lo`` .. ``mp_hi`` megapixels at an aspect ratio uniform over [0.5, 2]
           (drawn from ``spec``, sides rounded to ``step``).  ``qindex`` 0: drawn per image from 80, 120 and 160.
           ``conf`` > 0: the shipped pruning network at that confidence, else the exhaustive search.  ``graph``: the
           captured launch mode on four analysis streams.  ``post``: deblocking and CDEF.  ``recon``: the
           reconstruction is downloaded too.
  request  host planes of one image -> upload, encode with the pruning network, AVIF file (the serving loop's work for
           one request).
  train    loss and gradient of the pruning network over ``n`` superblocks.
"""
import math
import random
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import av1gpu_amd as A
from av1gpu_amd import learn

# Forward-transform FLOPs per luma sample of the searches, as the encoder's own work accounting counts them
# (av1mi_set_work_count) on 0.18-24 MP images at qindex 80/120/160: the exhaustive and the pruned analysis, the closed loop
FLOPS_EXHAUSTIVE, FLOPS_PRUNED, FLOPS_CLOSED = 9300.0, 2230.0, 1060.0


def _encode(name, n, w=0, h=0, mp_lo=0.0, mp_hi=0.0, spec=0, step=8, qindex=120, bd=8, yuv444=False, conf=0.0, graph=False,
            post=False, recon=True):
    c = {"kind": "encode", "n": n, "w": w, "h": h, "mp_lo": mp_lo, "mp_hi": mp_hi, "spec": spec, "step": step, "qindex": qindex,
         "bd": bd, "yuv444": yuv444, "conf": conf, "graph": graph, "post": post, "recon": recon}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one thumbnail of a few superblocks, exhaustive; launches, copies and one short chain
        _encode("thumb_96x64", 1, 96, 64),
        # one small web image, exhaustive: the configuration of the CPU baseline
        _encode("single_512", 1, 512, 512),
        # one ragged 10-bit 4:4:4 image through the post-filters: every sample type and filter the plain cases leave out
        _encode("odd_10b444_post", 1, 1021, 767, bd=10, yuv444=True, post=True),
        # one camera image, exhaustive: the plain path of the benchmark
        _encode("photo_12mp", 1, 4000, 3000),
        # one large image with the pruning network: the latency of the fast path
        _encode("photo_24mp_learned", 1, 6000, 4000, conf=0.8),
        # a fixed batch shape sent again and again: the captured launch mode (benchmark: launch modes)
        _encode("batch16_512_graph", 16, 512, 512, conf=0.8, graph=True, recon=False),
        # what a serving worker takes at once: a few images of very different sizes
        _encode("mixed9_learned", 9, mp_lo=0.18, mp_hi=24.0, spec=1000, qindex=0, conf=0.8),
        # a batch of small ragged images, exhaustive: the training data's and the quality baseline's path
        _encode("mixed16_exhaustive", 16, mp_lo=0.18, mp_hi=2.0, spec=1001, step=1, qindex=0, recon=False),
        # a folder of camera images: the throughput case, enough superblocks ready to fill the device
        _encode("photos16_12mp_learned", 16, 4000, 3000, qindex=0, spec=1002, conf=0.8, recon=False),
        # high-quality masters: the mixed batch at 10-bit 4:4:4
        _encode("mixed9_10b444", 9, mp_lo=0.18, mp_hi=6.0, spec=1003, qindex=0, bd=10, yuv444=True, conf=0.8),
        # one request of the serving loop, host planes to file
        {"name": "request_1mp", "kind": "request", "w": 1333, "h": 1001, "qindex": 120, "conf": 0.8},
        # one training step's gradient at the batch size of the training script
        {"name": "train_512", "kind": "train", "n": 512},
    ]


def draw(rng):
    def log(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def size(mp, step):
        a = rng.uniform(0.5, 2.0)
        return (max(8, int(round(math.sqrt(mp * 1e6 * a) / step)) * step), max(8, int(round(math.sqrt(mp * 1e6 / a) / step)) * step))

    kind = rng.choice(["single", "single", "single", "batch", "batch", "batch", "small", "request", "train"])
    q = rng.choice([60, 80, 100, 120, 140, 160, 180])
    step = rng.choice([1, 1, 8])
    if kind == "single":
        conf = rng.choice([0.0, 0.8, 0.8])
        deep = rng.random() < 0.25
        w, h = size(log(0.006, (3.0 if deep else 12.0) if conf == 0.0 else (6.0 if deep else 24.0)), step)
        return _encode(None, 1, w, h, step=step, qindex=q, bd=10 if deep else 8, yuv444=deep, conf=conf, post=rng.random() < 0.25)
    if kind == "batch":
        conf, deep, recon = rng.choice([0.0, 0.8, 0.8]), rng.random() < 0.25, rng.random() < 0.5
        hi = log(0.5, (2.0 if deep else 4.0) if conf == 0.0 else (4.0 if deep else 12.0))
        return _encode(None, rng.randint(2, 9 if recon else 16), mp_lo=0.18, mp_hi=hi, spec=rng.randrange(1 << 20), step=step, qindex=0,
                       bd=10 if deep else 8, yuv444=deep, conf=conf, post=rng.random() < 0.15, recon=recon)
    if kind == "small":
        w, h = size(log(0.01, 0.5), 8)
        return _encode(None, rng.randint(2, 16), w, h, qindex=q, conf=0.8, graph=rng.random() < 0.5, recon=False)
    if kind == "request":
        w, h = size(log(0.05, 4.0), 1)
        return {"kind": "request", "w": w, "h": h, "qindex": q, "conf": 0.8}
    return {"kind": "train", "n": rng.randint(32, 768)}


def _sizes(case):
    """[(W, H, qindex)] of the images of an encode case."""
    r, out = random.Random(case["spec"]), []
    for _ in range(case["n"]):
        w, h, s = case["w"], case["h"], case["step"]
        if not w:
            mp, a = math.exp(r.uniform(math.log(case["mp_lo"]), math.log(case["mp_hi"]))), r.uniform(0.5, 2.0)
            w = max(8, int(round(math.sqrt(mp * 1e6 * a) / s)) * s)
            h = max(8, int(round(math.sqrt(mp * 1e6 / a) / s)) * s)
        out.append((w, h, case["qindex"] or r.choice([80, 120, 160])))
    return out


def _images(sizes, seed, yuv444=False, bd=8):
    """Planes of the benchmark's synthetic images, one seed each."""
    with ThreadPoolExecutor(min(16, len(sizes))) as ex:
        return list(ex.map(lambda k: A.synth_image(seed * 4096 + k, sizes[k][0], sizes[k][1], ssx=0 if yuv444 else 1, bd=bd),
                           range(len(sizes))))


def _encoder(case):
    cfg = A.GpConfig(qindex=case["qindex"] or 120)
    if case.get("graph"):
        cfg.graph, cfg.anStreams = 1, 4
    if case.get("post"):
        cfg.lfMode, cfg.cdef, cfg.cdefYPri, cfg.cdefYSec, cfg.cdefUVPri, cfg.cdefUVSec = 1, 1, 2, 1, 1, 1
    enc = A.GpEncoder().init(cfg)
    if case["conf"]:
        learn.set_shortlist(enc, learn.load_params(), case["conf"])
    return enc


def _train_data(case, seed):
    """Tiles, qindex, labels and label masks of n superblocks: 512 x 512 images, node labels of a search's usual density."""
    n, tiles = case["n"], []
    for y in (p[0] for p in _images([(512, 512)] * (-(-n // 64)), seed)):
        tiles.append(learn.sb_tiles(y, 512, 512))
    rng = np.random.default_rng(seed)
    q = rng.choice(np.array([80, 120, 160], np.uint8), n)
    label = (rng.uniform(size=(n, learn.N_OUT)) < 0.4).astype(np.float32)
    mask = (rng.uniform(size=(n, learn.N_OUT)) < 0.95).astype(np.float32)
    return np.concatenate(tiles)[:n], q, label, mask


# A program keeps the records it gets: run() appends them to the program's own store, one array per record part with room
# for the most that the images can have, zero where nothing was written.  Large stores are filled by several threads.
_COPIERS = ThreadPoolExecutor(8)
_CHUNK = 4 << 20


def _store(images, yuv444):
    """The record store of images [(W, H)]: 256 blocks and 384 (4:4:4: 768) tx blocks per superblock, a level per sample."""
    sbs = sum(-(-w // 64) * -(-h // 64) for w, h in images)
    shapes = {"blocks": 16 * 256 * sbs, "block_txb": 256 * sbs + len(images), "txb": 16 * (768 if yuv444 else 384) * sbs,
              "coeffs": (12288 if yuv444 else 6144) * sbs, "counts": 3 * len(images)}
    kinds = {"blocks": np.uint8, "block_txb": np.uint32, "txb": np.uint8, "coeffs": np.int16, "counts": np.int64}
    return {k: np.full(n, 0, kinds[k]) for k, n in shapes.items()}


def _append(store, outs):
    """The records of outs back to back in the store."""
    at, jobs = {"blocks": 0, "block_txb": 0, "txb": 0, "coeffs": 0}, []
    for i, o in enumerate(outs):
        store["counts"][3 * i:3 * i + 3] = len(o.blocks), len(o.txb), len(o.coeffs)
        for k in at:
            a = getattr(o, k)
            a = a.view(np.uint8) if a.dtype.names else a
            for c in range(0, len(a), _CHUNK):
                part = a[c:c + _CHUNK]
                jobs.append((store[k][at[k] + c:at[k] + c + len(part)], part))
            at[k] += len(a)
    if len(jobs) > 64:
        list(_COPIERS.map(lambda j: np.copyto(*j), jobs))
    else:
        for j in jobs:
            np.copyto(*j)
    return store


def prepare(case, seed):
    if case["kind"] == "train":
        net = learn.Learner(learn.load_params())
        net.set_data(*_train_data(case, seed))
        return {"case": case, "net": net}
    enc = _encoder(case)
    if case["kind"] == "request":
        return {"case": case, "enc": enc, "planes": _images([(case["w"], case["h"])], seed)[0],
                "file": np.full(2 * case["w"] * case["h"] + 65536, 0, np.uint8)}
    sizes = _sizes(case)
    planes = _images(sizes, seed, case["yuv444"], case["bd"])
    frames = [A.DeviceFrame(p, w, h, bd=case["bd"], qindex=q, yuv444=case["yuv444"]) for p, (w, h, q) in zip(planes, sizes)]
    return {"case": case, "enc": enc, "frames": frames, "store": _store([s[:2] for s in sizes], case["yuv444"])}


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        loss, grads = state["net"].gradient(0, case["n"])
        return {"loss": loss, "grads": grads}
    if case["kind"] == "request":
        frame = A.DeviceFrame(state["planes"], case["w"], case["h"], qindex=case["qindex"])
        out = state["enc"].encode([frame], want_recon=False)[0][0]
        frame.close()
        data = np.frombuffer(A.write_bitstream(out), np.uint8)
        state["file"][:len(data)] = data
        return {"size": len(data), "file": state["file"]}
    out = state["enc"].encode(state["frames"], want_recon=case["recon"])[0]
    return {"records": _append(state["store"], out), "recon": [o.recon for o in out]}


def work(case):
    if case["kind"] == "train":
        # three contractions per layer (forward, weight gradient, input gradient; no input gradient for the first)
        macs = [32 * 32 * 32 * 18, 16 * 16 * 32 * 288, 8 * 8 * 32 * 288, 4 * 4 * 32 * 288, learn.N_OUT * learn.N_FEAT]
        flops = 2.0 * case["n"] * (2 * macs[0] + 3 * sum(macs[1:]))
        return {"bytes": case["n"] * (4096.0 + 1 + 8 * learn.N_OUT) + 8.0 * learn.param_count(), "flops": flops}
    if case["kind"] == "request":
        px, samples, bps, pruned = case["w"] * case["h"], 1.5 * case["w"] * case["h"], 1, True
    else:
        px = sum(w * h for w, h, _ in _sizes(case))
        samples, bps, pruned = (3.0 if case["yuv444"] else 1.5) * px, case["bd"] // 8 + (case["bd"] > 8), case["conf"] > 0
        if case["post"]:
            samples *= 2   # the filtered frame is written beside the unfiltered one, which predicts
    # the source read and the reconstruction written once, the levels of every tx block written once
    return {"bytes": samples * 2 * bps + samples * 2,
            "flops": px * ((FLOPS_PRUNED if pruned else FLOPS_EXHAUSTIVE) + FLOPS_CLOSED)}


def exact(case, seed):
    """The network's loss and gradient in float64 (no BF16 roundings); the encoder's outputs are whole numbers."""
    if case["kind"] != "train":
        return None
    tiles, q, label, mask = (torch.from_numpy(np.ascontiguousarray(a)) for a in _train_data(case, seed))
    n = case["n"]
    x = torch.empty(n, 2, 64, 64, dtype=torch.float64)
    x[:, 0] = tiles.reshape(n, 64, 64).double() / 255.0 - 0.5
    x[:, 1] = (q.double() / 255.0)[:, None, None]
    flat = torch.from_numpy(learn.load_params().astype(np.float64)).requires_grad_()
    off = 0
    for k, c in zip(learn.KP, learn.CIN):   # weights [32][taps x channels, padded], bias [32]
        w = flat[off:off + 32 * k].reshape(32, k)[:, :9 * c].reshape(32, 3, 3, c).permute(0, 3, 1, 2)
        x = torch.relu(torch.nn.functional.conv2d(x, w, flat[off + 32 * k:off + 32 * k + 32], stride=2, padding=1))
        off += 32 * k + 32
    w5 = flat[off:off + learn.N_OUT * learn.N_FEAT].reshape(learn.N_OUT, learn.N_FEAT)
    z = x.permute(0, 2, 3, 1).reshape(n, -1) @ w5.T + flat[off + learn.N_OUT * learn.N_FEAT:]
    loss = (mask.double() * torch.nn.functional.binary_cross_entropy_with_logits(z, label.double(), reduction="none")).sum() / n
    loss.backward()
    return {"loss": float(loss), "grads": flat.grad.numpy()}
