"""Timing cases of the framework: what a program does with it, one kind of work per case.

Eleven kinds cover an evaluation from the detector's raw frames to the normalised
correlation, and the simulator that makes such frames:

  eval      a whole small evaluation: frames to hit lists, AC_uw, flat-field C(q)
  events    the per-event call, one hit list after the other into one mesh
  batch     a prepared batch of sparse frames, launched again and again
  orient    a one-call batch whose frames carry a crystal orientation each
  uneven    a one-call batch of very uneven frames, any interpolation of the two maps
  cq        the pixel-pair normalisation C(q) of dense images
  merge     the rotation merge of C(q), to double, and the final division
  radial    the angular averaged evaluation: C(q), AC_uw and their quotient in 1D
  photons   detector frames to photons: mask, offset, gain, photon finder, counts
  ingest    averaged intensity of a frame stack and its sparse hit lists
  simulate  the emitter speckle field of a detector, then photon sampling

Sizes are those of the repository's configurations and benchmark, scaled to a pass of
at most some tens of milliseconds, and odd ones around them.  Inputs are made on the GPU
from the seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import incohautocorrelate_amd as iac
from incohautocorrelate_amd import workloads as W

MODES = {"bf16x3": iac.SIM_BF16X3, "fp16x3": iac.SIM_FP16X3, "fp16": iac.SIM_FP16}


def listed() -> list[dict]:
    return [
        # a small detector from frames to meshes: every launch and read-back counts
        dict(name="eval_128", kind="eval", rows=128, cols=128, frames=100, mean=0.01, edge=63),
        # the per-event call of the reference's frame loop on a full detector, oriented hits
        dict(name="events_1024", kind="events", rows=1024, cols=1024, events=16, mean=0.002, edge=255, rotated=True),
        # the sparse photon-list workload (the benchmark's headline), fewer frames
        dict(name="batch_1024", kind="batch", rows=1024, cols=1024, frames=3000, mean=0.002, edge=255),
        # the same frames with an orientation each, as a crystal's hits have
        dict(name="orient_1024", kind="orient", rows=1024, cols=1024, frames=800, mean=0.002, edge=255),
        # lognormal photon numbers (10..20,000 per frame), linear in both maps
        dict(name="uneven_linear", kind="uneven", rows=1024, cols=1024, frames=300, median=1500, edge=255, interp1=1,
             interp2=1, double_map=True),
        # C(q) of the averaged intensity of a medium detector, nearest neighbour
        dict(name="cq_384x360", kind="cq", rows=384, cols=360, images=1, groups=1, edge=127, interp=0),
        # the same, linear, on a small odd detector
        dict(name="cq_linear_191x173", kind="cq", rows=191, cols=173, images=1, groups=1, edge=95, interp=1),
        # one averaged C(q) merged over the orientations of a run, then the final division
        dict(name="merge_1000", kind="merge", events=1000, edge=127, interp=0, multi=False),
        # the angular averaged evaluation, linear bins as RunIAC takes them
        dict(name="radial_256", kind="radial", rows=256, cols=256, frames=500, mean=0.02, bins=4096, interp=1),
        # raw frames of a panelled detector through the photon finder with its maps
        dict(name="photons_1024", kind="photons", rows=1024, cols=1024, frames=100, panels=8, maps=True, gain_only=False),
        # a stack of calibrated frames averaged and made sparse, odd rows
        dict(name="ingest_517x512", kind="ingest", rows=517, cols=512, frames=200, mean=0.01, step=0.0, masked=True),
        # speckle frames of a 256^2 detector from 4,000 emitters, then Poisson photons
        dict(name="simulate_256", kind="simulate", rows=256, cols=256, emitters=4000, frames=250, mode="bf16x3",
             subsampling=0, modes=1, photons=0.05),
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(sorted(KINDS))
    rows = _log(rng, 96, 1024)
    cols = max(64, min(1024, int(rows * rng.uniform(0.7, 1.3))))
    sparse = dict(rows=rows, cols=cols, mean=round(min(0.05, _log(rng, 100, 2200) / (rows * cols)), 7),
                  edge=2 * rng.randint(24, 127) + 1)
    if kind == "eval":
        rows, cols = rng.randint(48, 128), rng.randint(48, 128)
        return dict(kind=kind, rows=rows, cols=cols, frames=_log(rng, 8, 100), mean=round(rng.uniform(0.003, 0.01), 4),
                    edge=2 * rng.randint(12, 31) + 1)
    if kind == "events":
        return dict(kind=kind, **sparse, events=_log(rng, 1, 16), rotated=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind=kind, **sparse, frames=_log(rng, 30, 2500))
    if kind == "orient":
        return dict(kind=kind, **sparse, frames=_log(rng, 10, 600))
    if kind == "uneven":
        i1, i2 = rng.choice([(0, 0), (0, 1), (1, 0), (1, 1)])
        return dict(kind=kind, rows=rows, cols=cols, frames=_log(rng, 20, 250), median=_log(rng, 200, 1500),
                    edge=sparse["edge"], interp1=i1, interp2=i2, double_map=rng.random() < 0.7)
    if kind == "cq":
        lin = rng.random() < 0.3
        rows, cols = (_log(rng, 48, 170), _log(rng, 48, 170)) if lin else (_log(rng, 64, 350), _log(rng, 64, 350))
        images = 1 if rng.random() < 0.5 or rows * cols > 20000 else rng.randint(2, 7)
        return dict(kind=kind, rows=rows, cols=cols, images=images, groups=rng.randint(1, images),
                    edge=2 * rng.randint(16, 63) + 1, interp=int(lin))
    if kind == "merge":
        lin = rng.random() < 0.4
        return dict(kind=kind, events=_log(rng, 10, 250 if lin else 900), edge=2 * rng.randint(24, 63) + 1, interp=int(lin),
                    multi=rng.random() < 0.3)
    if kind == "radial":
        rows, cols = _log(rng, 64, 250), _log(rng, 64, 250)
        return dict(kind=kind, rows=rows, cols=cols, frames=_log(rng, 20, 450), mean=round(rng.uniform(0.005, 0.02), 4),
                    bins=_log(rng, 200, 4096), interp=int(rng.random() < 0.7))
    if kind == "photons":
        return dict(kind=kind, rows=8 * _log(rng, 10, 100), cols=_log(rng, 100, 1000), frames=_log(rng, 4, 100),
                    panels=rng.choice([1, 2, 4, 8]), maps=rng.random() < 0.7, gain_only=rng.random() < 0.25)
    if kind == "ingest":
        return dict(kind=kind, rows=_log(rng, 64, 510), cols=_log(rng, 64, 510), frames=_log(rng, 10, 200),
                    mean=round(rng.uniform(0.002, 0.03), 4), step=rng.choice([0.0, 1.0]), masked=rng.random() < 0.6)
    sub, modes = rng.choice([(0, 1), (0, 1), (0, 2), (1, 1)])
    shrink = modes * (2 * sub + 1)
    return dict(kind=kind, rows=_log(rng, 32, 256 // (2 * sub + 1)), cols=_log(rng, 32, 256 // (2 * sub + 1)),
                emitters=_log(rng, 200, 4000), frames=_log(rng, 8, 250 // shrink), mode=rng.choice(sorted(MODES)),
                subsampling=sub, modes=modes, photons=round(rng.uniform(0.01, 0.2), 3))


# ---- inputs ------------------------------------------------------------------------------


def _rng(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + 17)
    return g


def _rand(g, *shape) -> torch.Tensor:
    return torch.rand(shape, device="cuda", generator=g)


def _pixmap(case) -> np.ndarray:
    """A flat detector of 75 um pixels, half a metre behind the sample."""
    r, c = case["rows"], case["cols"]
    pm = np.empty((r, c, 3), np.float32)
    pm[..., 0] = ((np.arange(r) - (r - 1) / 2.0) * W.PIXEL_UM)[:, None]
    pm[..., 1] = ((np.arange(c) - (c - 1) / 2.0) * W.PIXEL_UM)[None, :]
    pm[..., 2] = W.DIST_UM
    return pm.reshape(-1, 3)


def _photon_lists(npix: int, per_frame: torch.Tensor, mean: float, g):
    """Per frame, sorted distinct pixels with their counts, and the frames' offsets."""
    nf = per_frame.numel()
    frame = torch.repeat_interleave(torch.arange(nf, device="cuda"), per_frame)
    key = torch.unique(frame * npix + torch.randint(0, npix, (frame.numel(),), device="cuda", generator=g))
    cnt = (1 + (_rand(g, key.numel()) < mean / 2)).to(torch.int16)
    off = torch.zeros(nf + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(key // npix, minlength=nf), 0)
    return (key % npix).to(torch.int32), cnt, off


def _poisson_lists(case, frames: int, g):
    npix = case["rows"] * case["cols"]
    lam = torch.full((frames,), npix * -math.expm1(-case["mean"]), device="cuda")
    per = torch.poisson(lam, generator=g).clamp_(1, npix // 2).long()
    return _photon_lists(npix, per, case["mean"], g)


def _rotations(n: int, seed: int) -> np.ndarray:
    return W.random_rotations(n, seed + 5)


def _records(kmap, pix, cnt) -> torch.Tensor:
    return torch.cat([kmap[pix.long()], cnt.float()[:, None]], 1).contiguous()


def _mask(npix: int, g) -> torch.Tensor:
    return (_rand(g, npix) > 0.03).to(torch.int32)


def _u64(n: int) -> torch.Tensor:
    return torch.zeros(n, dtype=torch.int64, device="cuda")


def _geometry(case):
    """The k-map on the GPU and the detector's largest q, as Detector::Calc_kMap gives them."""
    kmap, _, _, max_q = iac.calc_kmap(_pixmap(case))
    return torch.from_numpy(kmap).cuda(), max_q


def _big(s: dict, max_q, edge: int) -> None:
    s["shape"] = iac.mesh_shape_big(max_q, edge)
    s["mesh"] = _u64(s["shape"].size_ab ** 3)


# ---- eval: a whole small evaluation ----------------------------------------------------------


def _eval_prepare(case, seed):
    g = _rng(seed)
    npix, nf = case["rows"] * case["cols"], case["frames"]
    kmap, max_q = _geometry(case)
    s = dict(ctx=iac.Context(0), kmap=kmap, mask=_mask(npix, g))
    s["frames"] = torch.poisson(torch.full((nf, npix), case["mean"], device="cuda"), generator=g)
    s["flat"] = s["mask"].float()
    s["mult"] = iac.cq_small_multiplicator(s["flat"].cpu().numpy())
    s["rec"] = torch.zeros((nf * npix, 4), device="cuda")
    s["off"] = _u64(nf + 1)
    _big(s, max_q, case["edge"])
    s["small"] = iac.mesh_shape_small_cofq(max_q, case["edge"])
    s["cq"] = _u64(s["small"].size_ab ** 2 * s["small"].size_c)
    return s


def _eval_run(s):
    ctx = s["ctx"]
    s["mesh"].zero_()
    s["cq"].zero_()
    n = ctx.sparse_hit_list(s["kmap"], s["frames"], s["mask"], 0.0, 1.0, s["rec"], s["off"])
    ctx.ac3d_records_batch(s["kmap"], s["rec"], s["off"], n, s["shape"], s["mesh"])
    ctx.cq_small(s["kmap"], s["flat"], s["small"], s["cq"], iac.NEAREST, s["mult"])
    return {"mesh": s["mesh"], "cq": s["cq"], "n": n}


def _eval_work(c):
    npix = c["rows"] * c["cols"]
    hits = npix * c["mean"]
    return dict(bytes=4.0 * npix * c["frames"] + 8.0 * (c["edge"] + 2) ** 3,
                flops=20.0 * (npix ** 2 / 2 + c["frames"] * hits ** 2 / 2))


# ---- events: one call per event ----------------------------------------------------------------


def _events_prepare(case, seed):
    g = _rng(seed)
    kmap, max_q = _geometry(case)
    pix, cnt, off = _poisson_lists(case, case["events"], g)
    rec, o = _records(kmap, pix, cnt), off.tolist()
    rots = _rotations(case["events"], seed) if case["rotated"] else np.tile(np.eye(3, dtype=np.float32).ravel(),
                                                                            (case["events"], 1))
    s = dict(ctx=iac.Context(0), hits=[rec[a:b].contiguous() for a, b in zip(o, o[1:])], rots=list(rots))
    _big(s, max_q, case["edge"])
    return s


def _events_run(s):
    s["mesh"].zero_()
    for hits, rot in zip(s["hits"], s["rots"]):
        s["ctx"].ac3d_sparse(hits, rot, s["shape"], s["mesh"])
    return s["mesh"]


def _sparse_work(c, frames):
    hits = c["rows"] * c["cols"] * c["mean"]
    return dict(bytes=frames * hits * 16.0 + 8.0 * (c["edge"] + 2) ** 3, flops=20.0 * frames * hits ** 2 / 2)


# ---- batch, orient, uneven: many frames in one call -----------------------------------------------


def _batch_prepare(case, seed):
    kmap, max_q = _geometry(case)
    pix, cnt, off = _poisson_lists(case, case["frames"], _rng(seed))
    s = dict(ctx=iac.Context(0))
    _big(s, max_q, case["edge"])
    s["batch"] = s["ctx"].ac3d_batch(kmap, pix, cnt, off, pix.numel(), s["shape"])
    return s


def _batch_run(s):
    s["batch"].launch(s["mesh"], zero_mesh=True)
    return s["mesh"]


def _orient_prepare(case, seed):
    kmap, max_q = _geometry(case)
    pix, cnt, off = _poisson_lists(case, case["frames"], _rng(seed))
    s = dict(ctx=iac.Context(0), lists=(kmap, pix, cnt, off, pix.numel()),
             opt=dict(rots=torch.from_numpy(_rotations(case["frames"], seed)).cuda()))
    _big(s, max_q, case["edge"])
    return s


def _uneven_prepare(case, seed):
    g = _rng(seed)
    npix = case["rows"] * case["cols"]
    kmap, max_q = _geometry(case)
    per = torch.exp(torch.randn(case["frames"], device="cuda", generator=g)) * case["median"]
    pix, cnt, off = _photon_lists(npix, per.clamp_(10, min(20000, npix // 4)).long(), 0.01, g)
    s = dict(ctx=iac.Context(0), lists=(kmap, pix, cnt, off, pix.numel()),
             opt=dict(interp1=case["interp1"], interp2=case["interp2"], double_map=case["double_map"]))
    _big(s, max_q, case["edge"])
    return s


def _lists_run(s):
    s["mesh"].zero_()
    s["ctx"].ac3d_sparse_batch(*s["lists"], s["shape"], s["mesh"], **s["opt"])
    return s["mesh"]


def _uneven_work(c):
    pairs = c["frames"] * c["median"] ** 2 * math.e ** 2 / 2  # the lognormal's second moment, sigma 1
    corners = 8 if c["interp1"] or c["interp2"] else 1
    return dict(bytes=c["frames"] * c["median"] * 1.65 * 10.0 + 8.0 * (c["edge"] + 2) ** 3,
                flops=(14.0 + 6.0 * corners) * pairs)


# ---- cq: the pixel-pair normalisation -----------------------------------------------------------------


def _cq_prepare(case, seed):
    g = _rng(seed)
    npix, ni, ng = case["rows"] * case["cols"], case["images"], case["groups"]
    kmap, max_q = _geometry(case)
    frames = _rand(g, ni, npix).clamp_(min=1e-7).log_().mul_(-0.5)  # Gamma(1, 0.5)
    shape = iac.mesh_shape_small_cofq(max_q, case["edge"])
    return dict(ctx=iac.Context(0), kmap=kmap, frames=frames, shape=shape, interp=case["interp"],
                groups=[ni * i // ng for i in range(ng + 1)], cq=_u64(ng * shape.size_ab ** 2 * shape.size_c),
                mult=iac.cq_small_multiplicator(frames[0].cpu().numpy()))


def _cq_run(s):
    s["cq"].zero_()
    if s["frames"].shape[0] == 1:
        s["ctx"].cq_small(s["kmap"], s["frames"][0], s["shape"], s["cq"], s["interp"], s["mult"])
    else:
        s["ctx"].cq_dense_frames(s["kmap"], s["frames"], s["groups"], s["shape"], s["cq"], s["interp"], s["mult"])
    return s["cq"]


def _cq_work(c):
    npix = c["rows"] * c["cols"]
    pairs = c["images"] * npix ** 2 / (1 if c["interp"] else 2)
    return dict(bytes=4.0 * npix * (3 + c["images"]) + 8.0 * c["groups"] * (c["edge"] + 2) ** 2 * 3,
                flops=pairs * (40.0 if c["interp"] else 20.0))


# ---- merge: rotate C(q) into the lab frame, divide --------------------------------------------------------


def _merge_inputs(case, seed):
    """A triangle-like C(q) of a flat square detector (thin along the beam), zero past Max_Q."""
    g = _rng(seed)
    sab, nev = case["edge"] + 2, case["events"]
    r = (sab - 1) // 2
    x = (torch.arange(sab, device="cuda") - r).double()
    tri = (1 - x.abs() / r).clamp_(min=0)
    plane = tri[:, None] * tri[None, :] * (x[:, None] ** 2 + x[None, :] ** 2 < (r - 1) ** 2)
    depth = torch.tensor([0.1, 1.0, 0.1], device="cuda", dtype=torch.float64)
    nm = nev if case["multi"] else 1
    small = depth[None, :, None, None] * plane[None, None] * (0.8 + 0.4 * _rand(g, nm, 3, sab, sab).double())
    rot = _rotations(nev, seed)
    mean_i = (0.02 + 0.01 * _rand(g, nev)).cpu().numpy()
    ac = (_rand(g, sab ** 3) < 0.7).long() * torch.randint(1, 4000, (sab ** 3,), device="cuda", generator=g) * 1000
    return small.reshape(nm, -1).contiguous(), rot, mean_i, ac


def _merge_prepare(case, seed):
    small, rot, mean_i, ac = _merge_inputs(case, seed)
    sab = case["edge"] + 2
    shape = iac.MeshShape(k_a=0, k_b=1, k_c=2, size_ab=sab, size_c=3)
    rw, mult = iac.merge_prepare(rot, mean_i, small.mean(0).cpu().numpy())
    n = sab ** 3
    f64 = dict(dtype=torch.float64, device="cuda")
    return dict(ctx=iac.Context(0), small=small, shape=shape, rw=torch.from_numpy(rw).cuda(), mult=mult, ac=ac,
                interp=case["interp"], multi=case["multi"], big=_u64(n), cq=torch.zeros(n, **f64),
                out=torch.zeros(n, **f64))


def _merge_run(s):
    ctx = s["ctx"]
    s["big"].zero_()
    call = ctx.merge_cq_multi if s["multi"] else ctx.merge_cq
    call(s["small"], s["shape"], s["rw"], s["interp"], s["mult"], s["big"])
    ctx.u64_to_f64(s["big"], s["mult"], s["cq"])
    ctx.merge_ac_cq(s["ac"], s["cq"], s["out"])
    return {"big": s["big"], "cq": s["cq"], "out": s["out"]}


def _merge_work(c):
    sab = c["edge"] + 2
    voxels = 3.0 * sab ** 2 * 0.75 * c["events"]
    return dict(bytes=8.0 * 3 * sab ** 2 * (c["events"] if c["multi"] else 1) + 8.0 * 4 * sab ** 3,
                flops=voxels * (80.0 if c["interp"] else 25.0))


def _merge_exact(case, seed):
    small, rot, mean_i, ac = _merge_inputs(case, seed)
    sab = case["edge"] + 2
    r = (sab - 1) // 2
    x = (torch.arange(sab, device="cuda") - r).double()
    z = (torch.arange(3, device="cuda") - 1).double()
    q = torch.stack([x[None, None, :].expand(3, sab, sab), x[None, :, None].expand(3, sab, sab),
                     z[:, None, None].expand(3, sab, sab)], -1).reshape(-1, 3)
    big = torch.zeros(sab ** 3, dtype=torch.float64, device="cuda")

    def add(at, v):
        ok = ((at >= 0) & (at < sab)).all(1)
        at = at[ok].long()
        big.index_add_(0, (at[:, 2] * sab + at[:, 1]) * sab + at[:, 0], v[ok])

    for i in range(case["events"]):
        v = small[i if case["multi"] else 0] * float(mean_i[i]) ** 2
        R = torch.from_numpy(rot[i].astype(np.float64).reshape(3, 3)).cuda()
        p = q @ R.T
        if not case["interp"]:
            add(torch.sign(p) * torch.floor(p.abs() + 0.5) + r, v)
            continue
        f = torch.floor(p)
        t = p - f
        for c in range(8):
            e = torch.tensor([c & 1, c >> 1 & 1, c >> 2 & 1], device="cuda", dtype=torch.float64)
            add(f + e + r, v * (e * t + (1 - e) * (1 - t)).prod(1))
    out = torch.where(big > 0, ac.double() * 0.001 / big, torch.zeros_like(big))
    # a linear merge leaves voxels of next to no weight, whose quotient is the fixed point's rounding
    return {"big": None, "cq": big, "out": None if case["interp"] else out}


# ---- radial: the angular averaged evaluation ---------------------------------------------------------------


def _radial_inputs(case, seed):
    g = _rng(seed)
    npix = case["rows"] * case["cols"]
    image = _rand(g, npix).mul_(0.4).add_(0.8).mul_(case["mean"])  # an averaged intensity
    return (image, *_poisson_lists(case, case["frames"], g))


def _radial_prepare(case, seed):
    image, pix, cnt, off = _radial_inputs(case, seed)
    kmap, max_q = _geometry(case)
    n = case["bins"]
    f64 = dict(dtype=torch.float64, device="cuda")
    return dict(ctx=iac.Context(0), kmap=kmap, image=image, rec=_records(kmap, pix, cnt), off=off, bins=n,
                interp=case["interp"], shape=iac.ac1d_shape(max_q, n),
                mult=iac.ac1d_cq_multiplicator(image.cpu().numpy()), hist=_u64(n), cq=torch.zeros(n, **f64),
                acuw=torch.zeros(n, **f64), ac=torch.zeros(n, **f64))


def _radial_run(s):
    ctx, (max_q, dq) = s["ctx"], s["shape"]
    s["hist"].zero_()
    s["acuw"].zero_()
    ctx.ac1d_cq(s["kmap"], s["image"], s["bins"], max_q, dq, s["interp"], s["mult"], s["hist"])
    ctx.u64_to_f64(s["hist"], s["mult"], s["cq"])
    ctx.ac1d_acuw_records(s["rec"], s["off"], s["rec"].shape[0], s["bins"], max_q, dq, s["interp"], s["acuw"])
    ctx.ac1d_calc_ac(s["acuw"], s["cq"], s["ac"])
    return {"hist": s["hist"], "cq": s["cq"], "acuw": s["acuw"], "ac": s["ac"]}


def _radial_work(c):
    npix = c["rows"] * c["cols"]
    hits = npix * c["mean"]
    return dict(bytes=16.0 * npix + c["frames"] * hits * 16.0 + 32.0 * c["bins"],
                flops=(20.0 + 6.0 * c["interp"]) * (npix ** 2 / 2 + c["frames"] * hits ** 2 / 2))


def _radial_exact(case, seed):
    image, pix, cnt, off = _radial_inputs(case, seed)
    npix = image.numel()
    if npix ** 2 > 4.4e9:  # over about 20 s
        return None
    kmap = torch.from_numpy(_pixmap(case).astype(np.float32))
    norm = (kmap[:, 0] * kmap[:, 0] + kmap[:, 1] * kmap[:, 1] + kmap[:, 2] * kmap[:, 2]).sqrt()
    kmap = (kmap / norm[:, None]).cuda()
    span = (kmap.max(0).values - kmap.min(0).values).cpu().numpy()
    max_q = np.float32(np.sqrt(np.float32(span[0] ** 2) + np.float32(span[1] ** 2) + np.float32(span[2] ** 2)))
    dq = float(max_q / np.float32(case["bins"] - 2))
    hist = [torch.zeros(case["bins"], dtype=torch.float64, device="cuda") for _ in range(2)]

    def add(h, ka, va, kb, vb, twice_self):
        d = ka[:, None, :] - kb[None, :, :]
        b = d.square().sum(-1).sqrt() / dq
        w = va[:, None] * vb[None, :]
        if twice_self is not None:
            w = w + torch.diag_embed(torch.diagonal(w, twice_self), twice_self)[: w.shape[0], : w.shape[1]]
        low = torch.floor(b) if case["interp"] else torch.floor(b + 0.5)
        f = (b - low) if case["interp"] else torch.zeros_like(b)
        low = low.long().flatten()
        h += torch.bincount(low, ((1 - f) * w).flatten(), minlength=h.numel())[: h.numel()]
        if case["interp"]:
            h += torch.bincount(low + 1, (f * w).flatten(), minlength=h.numel())[: h.numel()]

    k = kmap.double()
    img = image.double()
    for a in range(0, npix, 1024):
        add(hist[0], k[a:a + 1024], img[a:a + 1024], k, img, None)
    o = off.tolist()
    for a, b in zip(o, o[1:]):
        kf, c = k[pix[a:b].long()], cnt[a:b].double()
        add(hist[1], kf, c, kf, c, 0)  # photon pairs weigh 2, a photon with itself too
    ac = hist[1] / hist[0]
    return {"hist": None, "cq": hist[0], "acuw": hist[1], "ac": torch.where(ac.isnan(), torch.zeros_like(ac), ac)}


# ---- photons: raw frames through the photon finder -----------------------------------------------------------


def _photons_inputs(case, seed):
    g = _rng(seed)
    npix, nf = case["rows"] * case["cols"], case["frames"]
    frames = torch.poisson(torch.full((nf, npix), 0.4, device="cuda"), generator=g)
    frames.add_(_rand(g, nf, npix).mul_(1.3).sub_(0.3)).mul_(37.0)
    maps = {}
    if case["maps"]:
        maps = dict(mask=_mask(npix, g), offset=_rand(g, npix) * 3.0, gain=0.8 + 0.4 * _rand(g, npix))
    return frames, maps


def _photons_prepare(case, seed):
    frames, maps = _photons_inputs(case, seed)
    nf, rows, cols, np_ = case["frames"], case["rows"], case["cols"], case["panels"]
    h = rows // np_
    return dict(ctx=iac.Context(0), frames=frames, maps=maps, gain_only=case["gain_only"],
                panels=[(i * h * cols, cols, h) for i in range(np_)], out=torch.zeros_like(frames),
                count=torch.zeros(nf, dtype=torch.int32, device="cuda"), mean=torch.zeros(nf, device="cuda"))


def _photons_run(s):
    s["ctx"].ppp_lap(s["frames"], s["out"], s["panels"], 37.0, gain_only=s["gain_only"], photon_count=s["count"],
                     mean_intensity=s["mean"], **s["maps"])
    return {"out": s["out"], "count": s["count"], "mean": s["mean"]}


def _photons_work(c):
    n = float(c["rows"] * c["cols"]) * c["frames"]
    return dict(bytes=8.0 * n, flops=20.0 * n)


def _photons_exact(case, seed):
    """Gain-corrected frames have a value in 64 bits; found photons are whole numbers."""
    if not case["gain_only"]:
        return None
    frames, maps = _photons_inputs(case, seed)
    v = frames.double()
    if maps:
        m = maps["mask"].double()
        v = (v * m - maps["offset"].double()) / maps["gain"].double() * (m == 1)
    return {"out": v, "count": None, "mean": v.mean(1)}


# ---- ingest: averaged intensity and hit lists -------------------------------------------------------------------


def _ingest_inputs(case, seed):
    """Frames of analogue values around 1 or 2 photons; masked pixels are hot in every frame."""
    g = _rng(seed)
    npix, nf = case["rows"] * case["cols"], case["frames"]
    order = torch.randperm(npix, device="cuda", generator=g)
    hot = order[: npix // 40] if case["masked"] else order[:0]
    good = order[hot.numel():]
    mask = torch.ones(npix, dtype=torch.int32, device="cuda")
    mask[hot] = 0
    frames = torch.zeros((nf, npix), device="cuda")
    frames[:, hot] = 5.0
    at = torch.randperm(nf * good.numel(), device="cuda", generator=g)[: int(nf * good.numel() * case["mean"])]
    value = (1.0 + (_rand(g, at.numel()) < 0.02)) * (0.8 + 0.4 * _rand(g, at.numel()))
    frames[at // good.numel(), good[at % good.numel()]] = value
    return frames, mask if case["masked"] else None


def _ingest_prepare(case, seed):
    frames, mask = _ingest_inputs(case, seed)
    nf, npix = frames.shape
    kmap, _ = _geometry(case)
    return dict(ctx=iac.Context(0), kmap=kmap, frames=frames, mask=mask, step=case["step"],
                avg=torch.zeros(npix, device="cuda"), mean=torch.zeros(nf, device="cuda"),
                count=torch.zeros(nf, dtype=torch.int32, device="cuda") if case["step"] > 0 else None,
                rec=torch.zeros((nf * npix, 4), device="cuda"), off=_u64(nf + 1))


def _ingest_run(s):
    s["ctx"].average_intensity(s["frames"], s["mask"], 0.1, s["step"], s["avg"], s["mean"], s["count"])
    n = s["ctx"].sparse_hit_list(s["kmap"], s["frames"], s["mask"], 0.1, s["step"], s["rec"], s["off"])
    out = {"avg": s["avg"], "mean": s["mean"], "off": s["off"], "hits": s["rec"][:n]}
    return out if s["count"] is None else {**out, "count": s["count"]}


def _ingest_work(c):
    n = float(c["rows"] * c["cols"]) * c["frames"]
    return dict(bytes=4.0 * n + 16.0 * n * c["mean"], flops=4.0 * n)


def _ingest_exact(case, seed):
    frames, mask = _ingest_inputs(case, seed)
    v = frames.double() if mask is None else frames.double() * mask.double()
    t, step = float(np.float32(0.1)), case["step"]
    if step > 0:
        v = torch.where(v >= t, torch.ceil((v - t) / step), torch.zeros_like(v))
    else:
        v = torch.where(v >= t, v, torch.zeros_like(v))
    out = {"avg": v.mean(0), "mean": v.mean(1), "off": None, "hits": None}
    return {**out, "count": None} if step > 0 else out


# ---- simulate: speckle frames, then photons -----------------------------------------------------------------------


def _simulate_inputs(case, seed):
    g = _rng(seed)
    f64 = dict(dtype=torch.float64, device="cuda", generator=g)
    em = (torch.rand((case["emitters"], 3), **f64) - 0.5) * 500.0  # a 50 nm cube, in Angstrom
    ph = torch.rand((case["frames"] * case["modes"], case["emitters"]), **f64) * (2 * math.pi)
    step = W.PIXEL_UM / (2 * case["subsampling"] + 1)
    return torch.from_numpy(_pixmap(case)).cuda(), em, ph, (step, 0.0, 0.0), (0.0, step, 0.0)


def _simulate_prepare(case, seed):
    pm, em, ph, u, v = _simulate_inputs(case, seed)
    ctx = iac.Context(0)
    plan = ctx.sim_plan(pm, em, W.WAVELENGTH_A, MODES[case["mode"]], case["subsampling"], u, v)
    n = case["rows"] * case["cols"]
    return dict(ctx=ctx, plan=plan, phases=ph, modes=case["modes"], expected=n * case["photons"], seed=seed,
                field=torch.zeros((case["frames"], n), device="cuda"),
                shot=torch.zeros((case["frames"], n), device="cuda"))


def _simulate_run(s):
    ctx = s["ctx"]
    ctx.sim_run(s["plan"], s["phases"], s["field"], modes=s["modes"])
    s["shot"].copy_(s["field"])  # the program keeps the noiseless field beside the photons
    ctx.sim_postprocess(s["shot"], s["expected"], seed=s["seed"])
    return {"field": s["field"], "shot": s["shot"]}


def _simulate_work(c):
    rows = float(c["rows"] * c["cols"]) * (2 * c["subsampling"] + 1) ** 2
    cols = float(c["frames"] * c["modes"])
    split = 1 if c["mode"] == "fp16" else 2
    return dict(bytes=rows * c["emitters"] * 4.0 * split + cols * c["emitters"] * 8.0 + 16.0 * c["rows"] * c["cols"] * c["frames"],
                flops=8.0 * rows * cols * c["emitters"] * (1 if split == 1 else 3))


def _simulate_exact(case, seed):
    pm, em, ph, u, v = _simulate_inputs(case, seed)
    s, m, nf = case["subsampling"], case["modes"], case["frames"]
    phase = torch.polar(torch.ones_like(ph), ph).T.contiguous()
    field = torch.zeros((nf, pm.shape[0]), dtype=torch.float64, device="cuda")
    U, V = torch.tensor(u, dtype=torch.float64, device="cuda"), torch.tensor(v, dtype=torch.float64, device="cuda")
    for p0 in range(0, pm.shape[0], 8192):
        p = pm[p0:p0 + 8192].double()
        for a in range(-s, s + 1):
            for b in range(-s, s + 1):
                x = p + a * V + b * U
                k = x * (2 * math.pi / W.WAVELENGTH_A) / x.square().sum(1).sqrt()[:, None]
                arg = k @ em.T
                amp = (torch.polar(torch.ones_like(arg), arg) @ phase).abs()
                field[:, p0:p0 + 8192] += amp.reshape(p.shape[0], nf, m).sum(2).T / (2 * s + 1) ** 2
    return {"field": field, "shot": None}


KINDS = {
    "eval": (_eval_prepare, _eval_run, _eval_work, None),
    "events": (_events_prepare, _events_run, lambda c: _sparse_work(c, c["events"]), None),
    "batch": (_batch_prepare, _batch_run, lambda c: _sparse_work(c, c["frames"]), None),
    "orient": (_orient_prepare, _lists_run, lambda c: _sparse_work(c, c["frames"]), None),
    "uneven": (_uneven_prepare, _lists_run, _uneven_work, None),
    "cq": (_cq_prepare, _cq_run, _cq_work, None),
    "merge": (_merge_prepare, _merge_run, _merge_work, _merge_exact),
    "radial": (_radial_prepare, _radial_run, _radial_work, _radial_exact),
    "photons": (_photons_prepare, _photons_run, _photons_work, _photons_exact),
    "ingest": (_ingest_prepare, _ingest_run, _ingest_work, _ingest_exact),
    "simulate": (_simulate_prepare, _simulate_run, _simulate_work, _simulate_exact),
}


def prepare(case: dict, seed: int) -> dict:
    return {"run": KINDS[case["kind"]][1], **KINDS[case["kind"]][0](case, seed)}


def run(state: dict):
    return state["run"](state)


def work(case: dict) -> dict:
    return KINDS[case["kind"]][2](case)


def exact(case: dict, seed: int):
    f = KINDS[case["kind"]][3]
    return f(case, seed) if f else None
