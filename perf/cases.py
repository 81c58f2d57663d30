"""What the encoder backend's speed is measured on: the calls a program makes
through the Python binding (mav1-encoder_amd/mav1hip.py), over the sizes,
presets and options the tests and the benchmark use.

  stream    one video through the sequence driver, frames from host or device
            memory: the first `frames` frames of a group that starts with a
            key frame (keyint = frames, so a pass codes one whole group and
            the driver goes on with the next, as a running encoder does)
  batch     several videos fed in step through the batched driver
  stages    one frame through the host-buffer stage calls, as a mav1 build
            that binds them as its backend codes a frame
  motion    motion search alone through its host-buffer call
  restore   the loop-restoration search on device buffers, without allocation
  infer     the pruner network's logits of a loaded set of superblocks
  train     one training step of the network: a batch loaded, forward,
            backward, Adam

Contents are synthetic, made on the GPU: a panned sum of sinusoids, opaque
rectangles moving at multiples of 1/8 px and Gaussian noise, in the manner of
synth.py (which makes the same kind of content on the host, slowly). Coded
frames are whole numbers and have to be the same; the network's outputs are
floating point.
"""
import ctypes as C
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mav1-encoder_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import autotune  # noqa: E402
import mav1hip  # noqa: E402
import synth  # noqa: E402

DEV = "cuda:0"

# Presets: keyword arguments of mav1hip.default_config. "turbo" is the
# real-time preset with loop restoration as the 1080p benchmark sets it,
# "plain" the same without restoration (the batched workload), "rd" the full
# rate-distortion search with a pyramid mini-GOP.
PRESETS = {
    "turbo": dict(turbo=1, restoration=1),
    "plain": dict(turbo=1),
    "rd": dict(turbo=0, leaf=1, tile_cols_log2=1),
}

# The batched workload's sizes (synth.BATCH_STREAMS), and smaller sets.
BATCH_SETS = {
    "sixteen": [(1920, 1080)] * 4 + [(1280, 720)] * 4 + [(854, 480)] * 8,
    "four": [(1280, 720), (854, 480), (640, 360), (352, 288)],
}


def listed():
    return [
        # motion search of one small frame with two references: the smallest call, bound by launches and copies
        dict(name="motion 352x288", kind="motion", w=352, h=288, q=125, turbo=True),
        # a thumbnail-sized real-time stream from host memory: launches and latency of every stage
        dict(name="stream 204x116 turbo", kind="stream", w=204, h=116, preset="turbo", q=90, altref=2, frames=8,
             host=True),
        # a 360p real-time stream from device memory
        dict(name="stream 640x360 turbo", kind="stream", w=640, h=360, preset="turbo", q=170, altref=2, frames=16,
             host=False),
        # the benchmark's stream: 1080p real-time, sources resident in HBM
        dict(name="stream 1920x1080 turbo", kind="stream", w=1920, h=1080, preset="turbo", q=125, altref=2, frames=25,
             host=False),
        # an all-intra 1080p stream (every frame a key frame) from host memory: the intra path alone
        dict(name="stream 1920x1080 intra", kind="stream", w=1920, h=1080, preset="turbo", q=125, altref=2, frames=1,
             host=True),
        # full rate-distortion search, pyramid of 8, CIF
        dict(name="stream 352x288 rd", kind="stream", w=352, h=288, preset="rd", q=125, altref=8, frames=9, host=True),
        # full rate-distortion search, pyramid of 4, 720p
        dict(name="stream 1280x720 rd", kind="stream", w=1280, h=720, preset="rd", q=125, altref=4, frames=5,
             host=False),
        # a frame through the host-buffer stage calls (the drop-in backend)
        dict(name="stages 854x480", kind="stages", w=854, h=480, q=125, inter=True),
        # the 16 uneven streams of the batched workload, a group of 5 frames each
        dict(name="batch of 16", kind="batch", set="sixteen", q=125, frames=5),
        # the restoration search of one 1080p frame on device buffers
        dict(name="restore 1920x1080", kind="restore", w=1920, h=1080, q=125),
        # the network's logits for four 1080p frames' superblocks
        dict(name="infer 2040", kind="infer", batch=2040),
        # a training step at the training program's batch size
        dict(name="train 256", kind="train", batch=256),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, wmax):
    """A frame size: widths of 160 .. wmax, odd ones among them, the usual shapes."""
    w = _log(rng, 160, wmax)
    h = int(w * rng.choice((9 / 16, 2 / 3, 3 / 4)))
    if w * h > 1920 * 1080:
        h = 1920 * 1080 // w
    return w, max(h, 96)


def draw(rng):
    kind = rng.choice(("stream", "stream", "stream", "rd", "batch", "stages", "motion", "restore", "infer", "train"))
    q = rng.randint(60, 215)
    if kind == "stream":
        w, h = _size(rng, 1920)
        frames = rng.choice((1, 6, 9, 16)) if w <= 1280 else rng.choice((1, 5, 8))
        return dict(kind="stream", w=w, h=h, preset=rng.choice(("turbo", "turbo", "plain")), q=q, altref=2,
                    frames=frames, host=rng.random() < 0.5)
    if kind == "rd":
        w, h = _size(rng, 854)
        altref = rng.choice((2, 4, 8))
        return dict(kind="stream", w=w, h=h, preset="rd", q=q, altref=altref, frames=altref + 1,
                    host=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind="batch", set=rng.choice(("sixteen", "four")), q=q, frames=rng.choice((3, 5)))
    if kind == "stages":
        w, h = _size(rng, 1280)
        return dict(kind="stages", w=w, h=h, q=q, inter=rng.random() < 0.7)
    if kind == "motion":
        w, h = _size(rng, 1920)
        return dict(kind="motion", w=w, h=h, q=q, turbo=rng.random() < 0.7)
    if kind == "restore":
        w, h = _size(rng, 1920)
        return dict(kind="restore", w=w, h=h, q=q)
    return dict(kind=kind, batch=_log(rng, 32, 2040 if kind == "infer" else 512))


# ---------------------------------------------------------------- contents


class Content:
    """Frames of one synthetic video on the GPU: frame(t) is (Y, U, V)."""

    def __init__(self, w, h, seed, objects, max_vel, sigma):
        self.w, self.h, self.cw, self.ch = w, h, (w + 1) >> 1, (h + 1) >> 1
        self.sigma = sigma
        rng = np.random.default_rng(seed)
        waves = lambda n, lo, hi: [(rng.uniform(8, 64), rng.uniform(0, math.pi), rng.uniform(0, 2 * math.pi),
                                    rng.uniform(lo, hi)) for _ in range(n)]
        self.bg = [waves(6, 8, 22), waves(3, 6, 12), waves(3, 6, 12)]
        self.objs = [(int(rng.integers(16, 97)), int(rng.integers(16, 97)), int(rng.integers(0, w)),
                      int(rng.integers(0, h)), int(rng.integers(-8 * max_vel, 8 * max_vel + 1)),
                      int(rng.integers(-8 * max_vel, 8 * max_vel + 1)),
                      (int(rng.integers(20, 236)), int(rng.integers(40, 217)), int(rng.integers(40, 217))))
                     for _ in range(objects)]
        self.gen = torch.Generator(DEV)
        self.gen.manual_seed(seed * 7919 + 17)

    def plane(self, p, t):
        w, h, s = (self.w, self.h, 1) if p == 0 else (self.cw, self.ch, 2)
        xx = torch.arange(w, device=DEV, dtype=torch.float32)
        yy = torch.arange(h, device=DEV, dtype=torch.float32)
        v = torch.full((h, w), 128.0, device=DEV)
        for period, angle, phase, amp in self.bg[p]:
            f = 2 * math.pi / period
            px, py = f * math.cos(angle), f * math.sin(angle)
            v += amp * torch.sin((yy[:, None] + 0.5 * t / s) * py + (xx[None, :] - 1.25 * t / s) * px + phase)
        for ow, oh, x0, y0, vx8, vy8, col in self.objs:
            x = ((8 * x0 + vx8 * t) % (8 * (self.w + ow)) - 8 * ow) / 8 / s
            y = ((8 * y0 + vy8 * t) % (8 * (self.h + oh)) - 8 * oh) / 8 / s
            cx = (torch.clamp(torch.minimum(xx + 1, torch.full_like(xx, x + ow / s)) - torch.clamp(xx, min=x), 0, 1))
            cy = (torch.clamp(torch.minimum(yy + 1, torch.full_like(yy, y + oh / s)) - torch.clamp(yy, min=y), 0, 1))
            cov = cy[:, None] * cx[None, :]
            v = v * (1 - cov) + col[p] * cov
        v += torch.randn((h, w), device=DEV, generator=self.gen) * (self.sigma / s)
        return torch.clamp(torch.round(v), 0, 255).to(torch.uint8)

    def frame(self, t):
        return [self.plane(p, t) for p in range(3)]


def _pad(geo, planes):
    """The encoder's padded frame (synth.pad_frame) on the GPU."""
    out = []
    for p in range(3):
        v = planes[p]
        rows = torch.clamp(torch.arange(geo.plane_h[p], device=DEV), max=v.shape[0] - 1)
        cols = torch.clamp(torch.arange(geo.stride[p], device=DEV), max=v.shape[1] - 1)
        out.append(v[rows][:, cols].reshape(-1))
    return torch.cat(out)


def _video(w, h, seed, n):
    """Objects and speeds grow with the frame, as in the repository's configurations."""
    big = w * h >= 1280 * 720
    c = Content(w, h, seed, 12 if big else 6, 48 if big else 10, 3.0 if big else 2.0)
    return [c.frame(t) for t in range(n)]


def _degraded(padded, seed, sigma):
    """A coded-looking copy of a frame: low-passed with a little noise."""
    g = torch.Generator(DEV)
    g.manual_seed(seed)
    f = padded.to(torch.float32)
    f = 0.25 * torch.roll(f, 1) + 0.5 * f + 0.25 * torch.roll(f, -1)
    f += torch.randn(f.shape, device=DEV, generator=g) * sigma
    return torch.clamp(torch.round(f), 0, 255).to(torch.uint8)


# ---------------------------------------------------------------- states


def _config(w, h, preset, q, altref, frames):
    kw = dict(PRESETS[preset])
    return mav1hip.default_config(w, h, qindex=q, altref=altref, keyint=frames, **kw)


class Outputs:
    """Host buffers that take the outputs of `frames` coded frames of every
    video, as the entropy coder behind the driver reads them: one buffer per
    kind of output, a video's frames one after another."""

    def __init__(self, geos, frames):
        self.flat, self.views, self.k = [], [[] for _ in geos], [0] * len(geos)
        units = []
        for g in geos:
            fp, _ = mav1hip.setup_params(mav1hip.default_config(g.w, g.h), mav1hip.turbo_frame("key", 0))
            units.append(sum(fp.lr_unit_rows[p] * fp.lr_unit_cols[p] for p in range(3)))
        # blocks, superblock records, levels, picture, CDEF choices, restoration units, frame kind and types
        for dtype, sizes in ((torch.int32, [g.num_sbs * 64 * 27 for g in geos]),
                             (torch.int32, [g.num_sbs * 89 for g in geos]),
                             (torch.int32, [g.num_sbs * 6144 for g in geos]),
                             (torch.uint8, [g.frame_bytes for g in geos]),
                             (torch.int8, [g.num_sbs for g in geos]),
                             (torch.int32, [12 * n for n in units]),
                             (torch.int32, [4] * len(geos))):
            flat = torch.zeros(frames * sum(sizes), dtype=dtype)
            self.flat.append(flat)
            at = 0
            for i, n in enumerate(sizes):
                self.views[i].append(flat[at:at + frames * n].reshape(frames, n))
                at += frames * n

    @staticmethod
    def _copy(dst, ptr):
        n = dst.numel() * dst.element_size()
        dst.view(torch.uint8).copy_(torch.frombuffer((C.c_uint8 * n).from_address(ptr), dtype=torch.uint8))

    def start(self):
        self.k = [0] * len(self.k)

    def take(self, i, r):
        k, v = self.k[i], self.views[i]
        self.k[i] += 1
        for dst, ptr in zip(v, (r.blocks, r.sbs, r.coefs, r.recon, r.cdef_choice, r.lr_units)):
            if ptr:
                self._copy(dst[k], ptr)
        v[6][k] = torch.tensor([r.frame_kind, r.fp.lr_type[0], r.fp.lr_type[1], r.fp.lr_type[2]], dtype=torch.int32)


def _parameters(seed):
    """Network parameters as the training program starts from (He-normal convolutions and heads)."""
    rng = np.random.default_rng(seed)
    parts = []
    for shape, fan in (((32, 9, 2), 18), ((32,), 0), ((64, 9, 32), 288), ((64,), 0), ((64, 9, 64), 576), ((64,), 0)):
        parts.append(rng.standard_normal(shape).ravel() * math.sqrt(2.0 / fan) if fan
                     else 0.02 * rng.standard_normal(shape))
    parts += [rng.standard_normal(64) * 0.1, np.zeros(64), rng.standard_normal(256) / 8, np.zeros(4),
              rng.standard_normal(512) / 8, np.zeros(8)]
    return np.concatenate(parts).astype(np.float32)


def _samples(batch, seed):
    """Superblock samples (luma and its residual against the frame before, over 255), quantisers, labels."""
    per = 510  # the superblocks of a 1920 x 1088 area
    xs = []
    for k in range((batch + per - 1) // per):
        y0, y1 = (f[0][:1088, :1920].to(torch.float32) for f in _video(1920, 1088, seed + 1000 * k, 2))
        x = torch.stack([y1, y1 - y0], -1) / 255.0
        xs.append(x.reshape(17, 64, 30, 64, 2).permute(0, 2, 1, 3, 4).reshape(per, 64, 64, 2))
    x = torch.cat(xs)[:batch].contiguous().cpu().numpy()
    rng = np.random.default_rng(seed)
    qs = (rng.choice((80, 125, 170, 215), batch) / 255.0).astype(np.float32)
    labels = np.stack([rng.integers(0, 4, batch), rng.integers(0, 8, batch)], 1).astype(np.int32)
    return x, qs, labels


def prepare(case, seed):
    kind = case["kind"]
    if kind == "stream":
        cfg = _config(case["w"], case["h"], case["preset"], case["q"], case["altref"], case["frames"])
        geo = synth.Geometry(cfg.width, cfg.height, cfg.tile_cols_log2)
        video = _video(cfg.width, cfg.height, seed, case["frames"])
        if case["host"]:
            frames = [[p.cpu().numpy() for p in f] for f in video]
        else:
            frames = [_pad(geo, f) for f in video]
        return dict(kind=kind, host=case["host"], seq=mav1hip.Sequence(cfg), frames=frames,
                    out=Outputs([geo], case["frames"]))
    if kind == "batch":
        sizes = BATCH_SETS[case["set"]]
        cfgs = [_config(w, h, "plain", case["q"], 2, case["frames"]) for w, h in sizes]
        geos = [synth.Geometry(c.width, c.height, c.tile_cols_log2) for c in cfgs]
        frames = [[_pad(g, f) for f in _video(c.width, c.height, seed * 31 + i, case["frames"])]
                  for i, (c, g) in enumerate(zip(cfgs, geos))]
        b = mav1hip.Batch(cfgs)
        b.set_knobs(autotune.load_tuned())
        return dict(kind=kind, batch=b, frames=frames, n=case["frames"], out=Outputs(geos, case["frames"]))
    if kind in ("stages", "motion"):
        turbo = case.get("turbo", True)
        cfg = mav1hip.default_config(case["w"], case["h"], qindex=case["q"], altref=2, leaf=1,
                                     **(PRESETS["turbo"] if turbo else dict(turbo=0)))
        geo = synth.Geometry(cfg.width, cfg.height, cfg.tile_cols_log2)
        video = [_pad(geo, f) for f in _video(cfg.width, cfg.height, seed, 3)]
        # the frames before and after it, coded
        ref, gold = (_degraded(video[t], seed + t, 1.0).cpu().numpy() for t in (0, 2))
        what = "leaf" if kind == "motion" else "arf" if case["inter"] else "key"
        fr = mav1hip.turbo_frame(what, 0 if what == "key" else 1)
        fp, presets = mav1hip.setup_params(cfg, fr)
        return dict(kind=kind, ctx=mav1hip.Context(cfg), fp=fp, sets=presets, src=video[1].cpu().numpy(), ref=ref,
                    gold=gold)
    if kind == "restore":
        cfg = mav1hip.default_config(case["w"], case["h"], qindex=case["q"], **PRESETS["turbo"])
        geo = synth.Geometry(cfg.width, cfg.height, cfg.tile_cols_log2)
        src = _pad(geo, _video(cfg.width, cfg.height, seed, 1)[0])
        fp, _ = mav1hip.setup_params(cfg, mav1hip.turbo_frame("arf", 1))
        n = sum(fp.lr_unit_rows[p] * fp.lr_unit_cols[p] for p in range(3))
        return dict(kind=kind, fp=fp, src=src, cdef=_degraded(src, seed + 1, 1.5), dbk=_degraded(src, seed + 1, 2.0),
                    units=torch.zeros((n, 12), dtype=torch.int32, device=DEV),
                    types=torch.zeros(3, dtype=torch.int32, device=DEV))
    x, q, labels = _samples(case["batch"], seed)
    net = mav1hip.Pruner(max_batch=case["batch"])
    net.set_params(_parameters(seed))
    state = dict(kind=kind, net=net, x=x, q=q, labels=labels, step=0)
    if kind == "infer":
        net.load(x, q)
    return state


# ---------------------------------------------------------------- passes


def _run_stream(s):
    seq, out, n = s["seq"], s["out"], len(s["frames"])
    out.start()
    for f in s["frames"]:
        while not (seq.send(f) if s["host"] else seq.send_device(f.data_ptr())):
            out.take(0, seq.receive_raw(True))
        while True:
            r = seq.receive_raw(False)
            if r is None:
                break
            out.take(0, r)
    while out.k[0] < n:
        out.take(0, seq.receive_raw(True))
    return out.flat


def _run_batch(s):
    b, out, n = s["batch"], s["out"], s["n"]
    out.start()
    for t in range(n):
        for i, frames in enumerate(s["frames"]):
            while not b.send_device(i, frames[t].data_ptr()):
                out.take(i, b.receive_raw(i, True))
        for i in range(len(s["frames"])):
            while True:
                r = b.receive_raw(i, False)
                if r is None:
                    break
                out.take(i, r)
    for i in range(len(s["frames"])):
        while out.k[i] < n:
            out.take(i, b.receive_raw(i, True))
    return out.flat


def _run_stages(s):
    ctx, fp, src = s["ctx"], s["fp"], s["src"]
    ref = gold = mv = mvg = None
    if not fp.frame_is_intra:
        ref = s["ref"]
        mv, mvg = ctx.motion_search(fp, src, ref)
    _, _, blocks, sbs = ctx.analyze(fp, src, ref, gold, mv, mvg, tables=False)
    blocks = ctx.edge_types(fp, blocks, sbs)
    rec, coefs, blocks = ctx.recon(fp, blocks, sbs, src, ref, gold)
    info = ctx.filter_info(fp, blocks, sbs)
    dbk, sets = ctx.filter(fp, info, rec, s["sets"])
    cdef, choice = ctx.cdef_select(fp, src, sets, dbk)
    units, types, _ = ctx.lr_select(fp, src, cdef, dbk)
    for p in range(3):
        fp.lr_type[p] = types[p]
    final = ctx.restore(fp, cdef, dbk, units)
    return [a for a in (mv, blocks, sbs, rec, coefs, info, dbk, sets, cdef, choice, units, np.array(types), final)
            if a is not None]


def run(s):
    kind = s["kind"]
    if kind == "stream":
        return _run_stream(s)
    if kind == "batch":
        return _run_batch(s)
    if kind == "stages":
        return _run_stages(s)
    if kind == "motion":
        return list(s["ctx"].motion_search(s["fp"], s["src"], s["ref"], s["gold"]))
    if kind == "restore":
        mav1hip.lr_select_static(s["fp"], s["src"].data_ptr(), s["cdef"].data_ptr(), s["dbk"].data_ptr(), 0,
                                 s["units"].data_ptr(), s["types"].data_ptr(),
                                 torch.cuda.current_stream().cuda_stream)
        return [s["units"], s["types"]]
    net = s["net"]
    if kind == "infer":
        return {"logits": net.forward()[0]}
    net.load(s["x"], s["q"], s["labels"])
    logits, loss = net.forward()
    grads = net.backward()
    s["step"] += 1
    net._chk("adam", mav1hip.lib().mav1hip_pruner_adam(net.h, 1e-4, 0.9, 0.999, 1e-8, s["step"]))
    return {"logits": logits, "loss": loss, "grads": grads}


# ---------------------------------------------------------------- work and tolerance


def _frame_work(w, h, refs, rd):
    """Bytes of one coded frame that any implementation moves (source and
    references read, picture, levels and records written) and a floor of its
    arithmetic: full-pel and sub-pel candidates, predictions and transforms
    of every sample at one operation each."""
    geo = synth.Geometry(w, h)
    n, f = geo.num_sbs, geo.frame_bytes
    b = f * (2 + refs) + n * (6144 * 4 + 64 * 108 + 356)
    return b, f * (60 + 400 * refs + (600 if rd else 0))


def work(case):
    kind = case["kind"]
    b = o = 0
    if kind == "stream":
        for k in range(case["frames"]):
            x, y = _frame_work(case["w"], case["h"], 0 if k == 0 else 1.5, case["preset"] == "rd")
            b, o = b + x, o + y
    elif kind == "batch":
        for w, h in BATCH_SETS[case["set"]]:
            for k in range(case["frames"]):
                x, y = _frame_work(w, h, 0 if k == 0 else 1.5, False)
                b, o = b + x, o + y
    elif kind == "stages":
        b, o = _frame_work(case["w"], case["h"], 1 if case["inter"] else 0, False)
    elif kind == "motion":
        geo = synth.Geometry(case["w"], case["h"])
        b, o = 3 * geo.frame_bytes + 2 * geo.num_sbs * 85 * 8, 600 * geo.frame_bytes
    elif kind == "restore":
        geo = synth.Geometry(case["w"], case["h"])
        # per sample: the Wiener fit's normal equations, 16 self-guided sets of two passes, the refinement
        b, o = 3 * geo.frame_bytes, (4 * 2 * 12 + 16 * 60 + 12 * 28) * geo.frame_bytes
    else:
        # the three convolutions' multiply-adds; a training step has two more products of each
        n = case["batch"]
        conv = 2.0 * n * (32 * 32 * 32 * 18 + 16 * 16 * 64 * 288 + 8 * 8 * 64 * 576)
        b = n * (64 * 64 * 2 * (4 if kind == "train" else 2) + 48) + 4 * 56940 * (4 if kind == "train" else 1)
        o = conv * (3 if kind == "train" else 1)
    return {"bytes": float(b), "flops": float(o)}


def tolerance(case):
    if case["kind"] in ("infer", "train"):
        # the sums are 32-bit, but what they round to 16 bits between the layers changes with their order:
        # logits and gradients of a path with its sums in another order are up to 5e-5 apart
        return {"rel": 3e-4, "max": 0.02}
    return "exact"


def exact(case, seed):
    """The network's outputs in 64 bits, without the 16-bit roundings."""
    if case["kind"] not in ("infer", "train"):
        return None
    x, q, labels = _samples(case["batch"], seed)
    p = torch.from_numpy(_parameters(seed)).to(DEV, torch.float64)
    train = case["kind"] == "train"
    p.requires_grad_(train)
    at, parts = 0, []
    for shape in ((32, 9, 2), (32,), (64, 9, 32), (64,), (64, 9, 64), (64,), (64,), (64,), (64, 4), (4,), (64, 8), (8,)):
        n = int(np.prod(shape))
        parts.append(p[at:at + n].reshape(shape))
        at += n
    w1, b1, w2, b2, w3, b3, wq, bq, wp, bp, wm, bm = parts

    def conv(v, w, b):
        # 3x3, stride 2, one sample of padding, as a product over the gathered taps
        n, c, h, ww = v.shape
        cols = torch.nn.functional.unfold(v, 3, padding=1, stride=2).reshape(n, c, 9, -1)
        cols = cols.permute(0, 3, 2, 1).reshape(-1, 9 * c)
        r = cols @ w.reshape(w.shape[0], -1).t() + b
        return torch.relu(r).reshape(n, h // 2, ww // 2, -1).permute(0, 3, 1, 2)

    logits, losses = [], []
    for i in range(0, case["batch"], 64):
        v = torch.from_numpy(x[i:i + 64]).to(DEV, torch.float64).permute(0, 3, 1, 2)
        v = conv(conv(conv(v, w1, b1), w2, b2), w3, b3)
        hid = v.mean((2, 3)) + torch.from_numpy(q[i:i + 64]).to(DEV, torch.float64)[:, None] * wq + bq
        lg = torch.cat([hid @ wp + bp, hid @ wm + bm], 1)
        logits.append(lg.detach())
        if train:
            y = torch.from_numpy(labels[i:i + 64]).to(DEV).long()
            part = (torch.nn.functional.cross_entropy(lg[:, :4], y[:, 0], reduction="sum")
                    + torch.nn.functional.cross_entropy(lg[:, 4:], y[:, 1], reduction="sum")) / case["batch"]
            part.backward()
            losses.append(float(part.detach()))
    out = {"logits": torch.cat(logits)}
    if train:
        out["loss"] = sum(losses)
        out["grads"] = p.grad
    return out
