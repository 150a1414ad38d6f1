#!/usr/bin/env python3
"""Benchmark of the sparse 3D pixel-pair accumulation and of the speckle
simulator on one MI355X.

Workload (the sparse photon-list configuration): flat 1024x1024 detector,
75 um pixels at 0.5 m; 10,000 frames of Poisson(0.002) photons per pixel
(~2,100 photons/frame) stored as (uint32 pixel, uint16 count) lists; every
ordered photon pair of a frame is binned (nearest neighbour, double mapping,
identity rotation) into a 257^3 uint64 q-difference mesh with the reference
CPU path's fixed point.  One step = zero the mesh + one pass over all frames
(mesh clear + gather + cell sort + pair pass + mirror of a prepared frame batch,
iac_ac3d_batch_launch: no host synchronisation or planning inside the step).  Inputs are resident in HBM before
timing starts.  Every run checks the first 20 frames bit for bit against the
oracle and the full timed mesh for point symmetry.

metric: ordered pair-updates (pairs within Max_Q, self pairs once) per second.

Simulator leg (the "simulator" object of the JSON line): 512x512 detector with
the same geometry, 10,000 emitters uniform in a 500 A cube, lambda 1.5 A, 1,000
frames of uniform random phases; one step = the complex GEMM field (split bf16
or fp16) -> subpixel |psi| -> rescale to 0.01 photons/pixel -> Poisson, for all
frames; frames/s next to the FP32 direct sum, errors against the FP64 oracle on
a pixel/frame subset.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0  # MI355X HBM3E, public spec
# LDS bandwidth: 128 bytes per clock per CU, 256 CUs at 2.4 GHz (MI355X public figures)
LDS_PEAK_GBS = 128 * 256 * 2.4
BYTES_PER_UPDATE = 16  # one 8 B bin read + one 8 B bin write per pair-update
# Measured HBM bytes per pair-kernel launch on this workload, keyed by the engine settings
# (pair mode, box, cell_vox, frame_chunk): FETCH_SIZE x2.0 + WRITE_SIZE x1.0 KiB from two
# rocprofv3 --pmc passes, scaled by a 2 GiB copy kernel (profiles/pairs_lds_sparse1024_10k.md).
MEASURED_TRAFFIC = {(1, 1920, 6, 32): (2 * 1511764 + 3118483) * 1024}
# strip_kernel's, of the 10,000 frames (profiles/strips_sparse1024_10k.md)
STRIP_TRAFFIC = (2 * 7521047 + 794909) * 1024
# The same for sim_gemm_kernel per launch of 1,000 frames (profiles/sim_gemm_mfma_512_10k_1000.md)
SIM_TRAFFIC = {"bf16x3": (2 * 70271911 + 1025181) * 1024}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--frames", type=int, default=10000)
    ap.add_argument("--seed", type=int, default=2)
    ap.add_argument("--cpu-seconds", type=float, default=15.0,
                    help="target CPU work of the bounded CPU-baseline sample")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-queue", action="store_true", help="skip the per-frame queue leg")
    ap.add_argument("--kernel", type=int, default=0, help="0 auto, 1 global-atomic tiles, 2 LDS boxes")
    ap.add_argument("--no-tune", action="store_true", help="skip the cell-size / frame-chunk sweep")
    ap.add_argument("--cell-vox", type=int, default=0, help="fix the LDS cell side (skips the sweep)")
    ap.add_argument("--frame-chunk", type=int, default=0, help="fix the LDS frames per block (skips the sweep)")
    ap.add_argument("--box", type=int, default=0, help="fix the LDS box capacity 1024/1920/4096 (with the above)")
    ap.add_argument("--cell-vox-v", type=int, default=0, help="fix the cell side along the second k axis")
    ap.add_argument("--region", type=int, default=0, help="fix the task region side in cells (0: whole grid)")
    ap.add_argument("--mode", type=int, default=0, help="fix the LDS pair mode (1 lanes on consecutive pairs, "
                    "2 range per thread)")
    ap.add_argument("--no-sim", action="store_true", help="skip the simulator leg")
    ap.add_argument("--no-uneven", action="store_true", help="skip the uneven-batch leg")
    ap.add_argument("--no-rotated", action="store_true", help="skip the per-frame rotation leg")
    ap.add_argument("--no-cfg1", action="store_true", help="skip the small dense-frame pipeline leg")
    ap.add_argument("--no-cfg3", action="store_true", help="skip the dense float + rotation merge leg")
    ap.add_argument("--no-ac1d", action="store_true", help="skip the AC1D leg")
    ap.add_argument("--no-cq", action="store_true", help="skip the dense C(q) leg")
    ap.add_argument("--no-ppp", action="store_true", help="skip the LAP photon finder leg")
    ap.add_argument("--no-eval", action="store_true", help="skip the end-to-end iac_eval leg")
    ap.add_argument("--no-probes", action="store_true", help="skip the copy / atomic ceiling probes")
    ap.add_argument("--uneven-only", action="store_true", help="run only the uneven-batch leg")
    ap.add_argument("--eval-only", action="store_true", help="run only the end-to-end iac_eval leg")
    ap.add_argument("--sim-only", action="store_true", help="run only the simulator leg (prints its JSON object)")
    ap.add_argument("--sim-frames", type=int, default=1000)
    ap.add_argument("--sim-steps", type=int, default=3)
    ap.add_argument("--sim-direct-frames", type=int, default=8)
    ap.add_argument("--sim-modes", default="bf16x3,fp16x3,fp16", help="GEMM modes of the simulator leg")
    return ap.parse_args()


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported "
              "(frames would shard across GPUs, each accumulating a partial uint64 mesh, then one sum "
              "reduction)", file=sys.stderr)
        sys.exit(2)

    import torch

    import incohautocorrelate_amd as iac
    from incohautocorrelate_amd import workloads as W

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.sim_only:
        print(json.dumps(sim_leg(args, iac, W, dev)), flush=True)
        return
    if args.uneven_only:
        print(json.dumps(uneven_leg(args, iac, W, dev)), flush=True)
        return
    if args.eval_only:
        print(json.dumps(eval_leg(args, W)), flush=True)
        return
    t0 = time.time()
    _, kmap, max_q = W.detector(1024)
    shape = iac.mesh_shape_big(max_q, 255)
    data = W.poisson_photon_frames(1024 * 1024, args.frames, 0.002, args.seed)
    n_total = int(data["frame_off"][-1])
    log(f"[bench] workload generated in {time.time() - t0:.1f}s: {args.frames} frames, "
        f"{n_total} photons ({n_total / args.frames:.1f}/frame), mesh {shape.size_ab}^3")

    d_kmap = torch.from_numpy(kmap).to(dev)
    d_pix = torch.from_numpy(data["pix"].view(np.int32)).to(dev)
    d_cnt = torch.from_numpy(data["cnt"].view(np.int16)).to(dev)
    d_off = torch.from_numpy(data["frame_off"].view(np.int64)).to(dev)
    nvox = shape.size_ab * shape.size_ab * shape.size_c
    d_mesh = torch.zeros(nvox, dtype=torch.int64, device=dev)
    ctx = iac.Context(0)

    # pair-updates of the workload: the same pass with unit counts (val(1) = 1000)
    d_one = torch.ones_like(d_cnt)
    ctx.ac3d_sparse_batch(d_kmap, d_pix, d_one, d_off, n_total, shape, d_mesh)
    torch.cuda.synchronize()
    updates = int(d_mesh.sum().item()) // 1000
    del d_one
    log(f"[bench] ordered pair-updates per step: {updates:.4e} ({updates / args.frames:.4e}/frame)")

    ctx.set_option(iac.OPT_AC3D_KERNEL, args.kernel)
    tuned = None
    if args.cell_vox or args.frame_chunk or args.box or args.cell_vox_v or args.region or args.mode:
        tuned = {"cell_vox": args.cell_vox, "cell_vox_v": args.cell_vox_v, "frame_chunk": args.frame_chunk,
                 "box": args.box, "region": args.region, "mode": args.mode}
        apply_lds_config(ctx, iac, tuned)
        tuned["fixed"] = True
    elif args.kernel != 1 and not args.no_tune:
        tuned = autotune(ctx, iac, d_kmap, d_pix, d_cnt, d_off, shape)

    # the prepared batch with the tuned settings: plan, chunk table and buffers made once;
    # each step enqueues mesh clear + gather + cell sort + pair pass + mirror with no host
    # synchronisation (the pair kernel bracketed by HIP events)
    batch = ctx.ac3d_batch(d_kmap, d_pix, d_cnt, d_off, n_total, shape)

    def step():
        batch.launch(d_mesh, zero_mesh=True)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    log("[bench] warmup done")

    ctx.enable_timing(True)
    ctx.kernel_time(reset=True)
    before = ctx.pair_paths()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    kms, klaunch = ctx.kernel_time(reset=True)
    ctx.enable_timing(False)
    path = path_since(ctx, before)  # what took the timed steps' pairs
    ms_per_step = (t2 - t1) * 1e3 / args.steps
    value = updates / ((t2 - t1) / args.steps)
    k_avg_ms = kms / max(klaunch, 1)
    achieved = updates * BYTES_PER_UPDATE / (k_avg_ms * 1e-3) / 1e9
    log(f"[bench] {ms_per_step:.3f} ms/step, kernel {k_avg_ms:.3f} ms avg over {klaunch} launches, "
        f"{value:.4e} pair-updates/s")

    if ctx.dropped():
        log(f"[bench] WARNING: {ctx.dropped()} updates fell outside the mesh")

    parity = check_headline(ctx, iac, kmap, data, shape, dev, d_mesh, path, (d_kmap, d_pix, d_cnt, d_off))
    batch.destroy()
    # the one-call entry point (plans the chunks on every call) for comparison
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(2):
        d_mesh.zero_()
        ctx.ac3d_sparse_batch(d_kmap, d_pix, d_cnt, d_off, n_total, shape, d_mesh)
    torch.cuda.synchronize()
    oneshot_ms = (time.perf_counter() - t) * 1e3 / 2

    queue = None if args.no_queue else queue_leg(args, iac, dev, kmap, d_kmap, data, shape, d_mesh, updates,
                                                    ms_per_step)
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(kmap, data, shape, ctx, iac, d_kmap, dev, args)

    ac1d = None if args.no_ac1d else ac1d_leg(args, iac, W, dev, kmap, d_kmap, d_pix, d_cnt, d_off, data, max_q)
    rotated = None if args.no_rotated else rotated_leg(args, iac, W, dev, d_kmap, d_pix, d_cnt, d_off, data, shape,
                                                       updates)
    del d_pix, d_cnt, d_off, d_mesh
    torch.cuda.empty_cache()
    cq = None if args.no_cq else cq_dense_leg(args, iac, W, dev)
    cfg1 = None if args.no_cfg1 else cfg1_leg(args, iac, W, dev)
    cfg3 = None if args.no_cfg3 else cfg3_leg(args, iac, W, dev)
    ev = None if args.no_eval else eval_leg(args, W)
    probes = None if args.no_probes else probe_leg(iac, dev, nvox)
    if probes and ac1d:
        # AC1D bins in LDS: each unordered pair (twice-weighted) is two linear-split LDS adds, doubles
        # for AC_uw (float values), uint64 for C(q) (its fixed point)
        for leg, kind in ((ac1d, "lds_box_f64"), (ac1d["cq"], "lds_box")):
            upairs = leg["value"] / 2 if leg is ac1d else leg["value"]
            leg["lds_adds_per_s"] = 2 * upairs
            leg["lds_probe"] = kind
            leg["frac_of_lds_atomic_probe"] = 2 * upairs / probes["atomic_u64_per_s"][kind]
    ppp = None if args.no_ppp else ppp_leg(args, iac, dev, probes)
    uneven = None if args.no_uneven else uneven_leg(args, iac, W, dev)
    sim = None if args.no_sim else sim_leg(args, iac, W, dev)

    traffic = None
    strips = path == "strips"
    if strips:
        traffic = STRIP_TRAFFIC if args.frames == 10000 and args.seed == 2 else None
    elif tuned and args.kernel != 1:
        key = (tuned.get("mode") or 1, tuned.get("box") or 1920, tuned.get("cell_vox") or 6,
               tuned.get("frame_chunk") or 32)
        if (tuned.get("cell_vox_v") or key[2]) != key[2] or tuned.get("region"):
            key = None
        traffic = MEASURED_TRAFFIC.get(key) if key else None
    out = {
        "metric": "pixel-pair updates/sec into q-mesh (sparse 1024^2, 257^3 uint64, bit-exact)",
        "value": value,
        "unit": "pair-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u64",
        "data": "synthetic",
        "config": {
            "workload": "sparse photon-list AC_uw: 1024x1024 detector, 10,000 frames Poisson(0.002) "
                        "as (uint32 pixel, uint16 count), 257^3 uint64 mesh, NN/NN double-map, identity R",
            "frames": args.frames,
            "photons": n_total,
            "pair_updates_per_step": updates,
            "seed": args.seed,
            "kernel": "tile (global atomics)" if args.kernel == 1 else "LDS strips" if strips else "LDS cell boxes",
            "step": "prepared frame batch (iac_ac3d_batch_launch): clear + gather + sort + pairs + mirror",
            "tuned": tuned,
            "path": path,
        },
        # The 16 B read-modify-write of each pair-update lands in an LDS box, not in HBM
        # (measured HBM traffic is under 1 % of it): the bound is the LDS, against its
        # published bandwidth; the HBM view and the measured LDS-atomic ceiling beside it.
        "roofline": {
            "bound": "lds" if args.kernel != 1 else "hbm",
            "achieved": achieved,
            "peak": LDS_PEAK_GBS if args.kernel != 1 else HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / (LDS_PEAK_GBS if args.kernel != 1 else HBM_PEAK_GBS),
            "traffic": traffic,
            "traffic_unit": "HBM bytes per launch (rocprofv3 FETCH_SIZE + WRITE_SIZE, copy-scaled)",
            "traffic_over_algorithmic": (traffic / (updates * BYTES_PER_UPDATE)) if traffic else None,
            "kernel": ("ac3d_tiles_kernel<true>" if args.kernel == 1 else
                       "strip_kernel (32-bit LDS boxes of strips)" if strips else "pairs_kernel (LDS cell boxes)"),
            "kernel_avg_ms": k_avg_ms,
            "bytes_per_update": BYTES_PER_UPDATE,
            "peak_basis": "LDS 128 B/clk/CU x 256 CUs x 2.4 GHz" if args.kernel != 1 else "HBM3E 8 TB/s",
            "hbm_view": {"achieved_algorithmic_GBps": achieved, "peak": HBM_PEAK_GBS,
                         "note": "algorithmic bytes over HBM peak; above 1 because the boxes absorb the "
                                 "read-modify-write (see traffic)"},
            "frac_of_measured_copy": achieved / probes["hbm_copy_GBps"] if probes else None,
            "updates_vs_uniform_u64_atomics": value / probes["atomic_u64_per_s"]["uniform"] if probes else None,
            # the kernel's LDS adds (one per distinct unordered pair: (updates - photons) / 2, the self
            # pairs go to the centre separately) against random uint64 adds into a 4096-voxel LDS box
            # (the strips' adds are 32 bits wide)
            "lds_adds_per_s": (updates - n_total) / 2 / (k_avg_ms * 1e-3) if k_avg_ms > 0 else None,
            "frac_of_lds_atomic_probe": ((updates - n_total) / 2 / (k_avg_ms * 1e-3)
                                         / probes["atomic_u64_per_s"]["lds_box"]
                                         if probes and k_avg_ms > 0 else None),
        },
        "parity": parity,
        "oneshot_call_ms": oneshot_ms,
        "cpu_baseline": cpu,
        "probes": probes,
        "per_frame_queue": queue,
        "uneven_batch": uneven,
        "rotated": rotated,
        "cfg1": cfg1,
        "cfg3": cfg3,
        "ac1d": ac1d,
        "cq_dense": cq,
        "ppp_lap": ppp,
        "eval_e2e": ev,
        "simulator": sim,
    }
    print(json.dumps(out), flush=True)
    ctx.close()


TUNE_KEYS = ("box", "cell_vox", "cell_vox_v", "region", "frame_chunk", "mode")


def path_since(ctx, before):
    """What took the pairs of the engine's passes since `before` (pair_paths): one name, or both."""
    names = [n for n, a, b in zip(("walk", "strips", "region tiles"), before, ctx.pair_paths()) if b > a]
    return " and ".join(names) if names else "tile kernel"


def apply_lds_config(ctx, iac, cfg):
    """Set the LDS kernel options of one tuning point (0 = library default; all 0 leaves the engine its
    strips and region tiles)."""
    ctx.set_option(iac.OPT_BOX_CAP, cfg.get("box", 0))
    ctx.set_option(iac.OPT_PAIR_PREFETCH, 0)
    ctx.set_option(iac.OPT_CELL_VOX, cfg.get("cell_vox", 0))
    ctx.set_option(iac.OPT_CELL_VOX_V, cfg.get("cell_vox_v", 0))
    ctx.set_option(iac.OPT_TASK_REGION, cfg.get("region", 0))
    ctx.set_option(iac.OPT_FRAME_CHUNK, cfg.get("frame_chunk", 0))
    ctx.set_option(iac.OPT_PAIR_MODE, cfg.get("mode", 0))


def cfg_str(cfg):
    return " ".join(f"{k}={cfg.get(k, 0)}" for k in TUNE_KEYS)


# the engine's own choice, then the walk around its defaults (mode 2, 3-voxel cells, 1920-voxel boxes,
# 2x2-cell regions); frames per block do not matter here (a dense frame is one chunk)
CQ_GRID = [{}] + [dict(mode=m, box=b, cell_vox=c, cell_vox_v=c, frame_chunk=32, region=r)
           for m in (1, 2) for b, c in ((1920, 3), (1024, 3), (1920, 4), (4096, 4), (1920, 5)) for r in (2, 4)]


def autotune(ctx, iac, d_kmap, d_pix, d_cnt, d_off, shape, label="tune"):
    """The library's autotuner (iac_ac3d_tune) on a 1,000-frame prefix: it times the pair
    kernel of each candidate setting and leaves the fastest applied to the context."""
    best, cands = ctx.ac3d_tune(d_kmap, d_pix, d_cnt, d_off, shape, prefix_frames=1000, force=True)
    for c in cands:
        log(f"[{label}] mode={c['pair_mode']} box={c['box_cap']} cell_vox={c['cell_vox']} "
            f"frame_chunk={c['frame_chunk']}: {c['ms']:.3f} ms / 1000 frames")
    log(f"[{label}] library tuner chose mode={best['pair_mode']} box={best['box_cap']} cell_vox={best['cell_vox']} "
        f"frame_chunk={best['frame_chunk']}")
    return {"mode": best["pair_mode"], "box": best["box_cap"], "cell_vox": best["cell_vox"],
            "cell_vox_v": best["cell_vox_v"], "region": best["task_region"], "frame_chunk": best["frame_chunk"],
            "by": "iac_ac3d_tune (library)", "candidates": cands}


def check_headline(ctx, iac, kmap, data, shape, dev, d_mesh, path, d_in):
    """Parity of the headline pass: the first 20 frames through the same prepared-batch
    code path and tuned settings (so few frames go by the walk), bit for bit against the
    oracle; the full timed mesh (all frames, identity rotation, nearest-neighbour levels) bit for
    bit against the walk's where another path took the timed steps, for point symmetry,
    mesh[C + d] == mesh[C - d], and a centre voxel of at least 1000 sum c^2 (every self
    pair lands there; so do neighbours closer than half a voxel)."""
    import torch

    O = _oracle()
    nf = 20
    off = data["frame_off"][: nf + 1]
    n = int(off[-1])
    t = time.perf_counter()
    ref, _ = O.ac3d_frames(kmap, data["pix"][:n], data["cnt"][:n], off, shape)
    dt = time.perf_counter() - t
    m = torch.zeros(ref.size, dtype=torch.int64, device=dev)
    sub = ctx.ac3d_batch(torch.from_numpy(kmap).to(dev), torch.from_numpy(data["pix"][:n].view(np.int32)).to(dev),
                         torch.from_numpy(data["cnt"][:n].view(np.int16)).to(dev),
                         torch.from_numpy(off.view(np.int64)).to(dev), n, shape)
    sub.launch(m, zero_mesh=True)
    torch.cuda.synchronize()
    sub.destroy()
    ok = bool((m.cpu().numpy().view(np.uint64) == ref).all())
    same = None
    if path != "walk":
        with iac.Context(0) as walk:
            walk.set_option(iac.OPT_AC3D_KERNEL, 2)
            walk.set_option(iac.OPT_PAIR_MODE, 1)
            mw = torch.zeros_like(d_mesh)
            walk.ac3d_sparse_batch(*d_in, int(data["frame_off"][-1]), shape, mw)
            walk.sync()
            if walk.pair_paths() != (1, 0, 0):
                raise SystemExit("headline check: the reference pass was not the walk's")
            same = bool(torch.equal(mw, d_mesh))
            del mw
    # the full timed mesh (the last replay)
    full = d_mesh.cpu().numpy().view(np.uint64).reshape(shape.size_c, shape.size_ab, shape.size_ab)
    sym = bool(np.array_equal(full, full[::-1, ::-1, ::-1]))
    cnt = data["cnt"].astype(np.uint64)
    centre = int(full[shape.center[2], shape.center[1], shape.center[0]])
    centre_ok = centre >= 1000 * int((cnt * cnt).sum())
    log(f"[bench] bit-exact check on {nf} frames: {'OK' if ok else 'MISMATCH'} (oracle {dt:.1f}s); full mesh by {path} "
        f"equals the walk's: {same}; point symmetric: {sym}; centre voxel >= 1000 sum c^2: {centre_ok}")
    if not (ok and sym and centre_ok and same is not False):
        raise SystemExit("headline parity check failed")
    return {"oracle_frames": nf, "bit_exact_vs_oracle": ok, "timed_path": path, "full_mesh_equals_walk": same,
            "full_mesh_point_symmetric": sym,
            "full_mesh_centre_at_least_1000_sum_c2": centre_ok,
            "path": "oracle: the prepared-batch path with the tuned settings; the walk: the timed full mesh"}


def queue_leg(args, iac, dev, kmap, d_kmap, data, shape, d_ref, updates, batch_ms):
    """Detector::AutoCorrelateSparseList once per event (the reference's frame loop,
    RunIAC.cpp:524-550): every headline frame pushed on its own from a host hit list
    {k, count} into a frame queue (iac_ac3d_queue_push: a copy into pinned staging, no
    device call), binned by the LDS engine each time 2^22 records have queued; one pass =
    all pushes + the last flush + a synchronisation.  The mesh must equal the batched
    pass's (d_ref) bit for bit."""
    import ctypes as C

    import torch

    off = data["frame_off"]
    nf = len(off) - 1
    hl = np.empty((int(off[-1]), 4), np.float32)
    hl[:, :3] = kmap[data["pix"]]
    hl[:, 3] = data["cnt"]
    base = hl.ctypes.data
    starts = [int(x) for x in off]
    rot = (C.c_float * 9)(1, 0, 0, 0, 1, 0, 0, 0, 1)
    push = iac.lib().iac_ac3d_queue_push
    ctx = iac.Context(0)
    mesh = torch.zeros_like(d_ref)
    q = ctx.ac3d_queue(d_kmap, shape, mesh, max_records=1 << 22, max_frames=4096)
    h = q.handle

    def one_pass():
        mesh.zero_()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for f in range(nf):
            a = starts[f]
            rc = push(h, base + 16 * a, starts[f + 1] - a, rot)
            if rc:
                raise RuntimeError(f"iac_ac3d_queue_push failed: {rc}")
        q.flush()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) * 1e3

    one_pass()
    ms = min(one_pass() for _ in range(2))
    equal = bool(torch.equal(mesh, d_ref))
    q.destroy()
    ctx.close()
    rate = updates / (ms * 1e-3)
    log(f"[queue] {nf} per-frame pushes + flush: {ms:.2f} ms ({rate:.4e} pair-updates/s, "
        f"{batch_ms / ms:.2f}x the batched pass), mesh equals the batched pass: {equal}")
    if not equal:
        raise SystemExit("per-frame queue mesh differs from the batched pass")
    mirror = queue_mirror(data, d_ref, updates, batch_ms)
    return {"workload": f"the headline {nf} frames, one iac_ac3d_queue_push per frame from host hit lists "
                        "(Detector::AutoCorrelateSparseList per event), flush every 2^22 records",
            "value": rate, "unit": "pair-updates/s", "ms_per_pass": ms, "frac_of_batched_rate": batch_ms / ms,
            "mesh_equals_batched_pass": equal, "cpp_mirror": mirror}


def queue_mirror(data, d_ref, updates, batch_ms):
    """The same per-event loop through the C++ host mirror: `iac_eval --queue` calls
    Detector::AutoCorrelateSparseList once per frame (a device reservation, the mesh's queue,
    a push into pinned staging) on hit lists it builds from the photon lists, then flushes;
    its mesh must equal the batched pass's."""
    import subprocess
    import tempfile

    from incohautocorrelate_amd import workloads as W

    exe = ROOT / "incohautocorrelate_amd" / "iac_eval"
    tmp = Path(tempfile.mkdtemp(prefix="iac_queue_bench_"))
    try:
        pm, _, _ = W.detector(1024)
        pm.astype(np.float32).tofile(tmp / "pm.bin")
        data["pix"].astype(np.uint32).tofile(tmp / "pix.bin")
        data["cnt"].astype(np.uint16).tofile(tmp / "cnt.bin")
        data["frame_off"].astype(np.uint64).tofile(tmp / "off.bin")
        nf = len(data["frame_off"]) - 1
        cmd = [str(exe), "--queue", str(tmp / "pm.bin"), "1024", "1024", str(tmp / "pix.bin"), str(tmp / "cnt.bin"),
               str(tmp / "off.bin"), str(nf), "255", str(tmp / "mesh.bin")]
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
        if r.returncode != 0:
            raise RuntimeError("iac_eval --queue failed: " + r.stderr[-2000:])
        ms = float(r.stdout.split("queue ms ")[1].split()[0])
        got = np.fromfile(tmp / "mesh.bin", dtype=np.uint64)
        equal = bool(np.array_equal(got, d_ref.cpu().numpy().view(np.uint64)))
    finally:
        for f in tmp.iterdir():
            f.unlink()
        tmp.rmdir()
    rate = updates / (ms * 1e-3)
    log(f"[queue] C++ mirror, Detector::AutoCorrelateSparseList per frame: {ms:.2f} ms ({rate:.4e} pair-updates/s, "
        f"{batch_ms / ms:.2f}x the batched pass), mesh equals the batched pass: {equal}")
    if not equal:
        raise SystemExit("C++ mirror per-event mesh differs from the batched pass")
    return {"value": rate, "unit": "pair-updates/s", "ms_per_pass": ms, "frac_of_batched_rate": batch_ms / ms,
            "mesh_equals_batched_pass": equal,
            "timed": "the calls and the last flush to the device's completion (the second pass of the process)"}


def cpu_baseline(kmap, data, shape, ctx, iac, d_kmap, dev, args):
    """The oracle's restatement of the reference CPU path (OpenMP over the outer
    photon, omp atomic uint64 adds) on a bounded prefix of the same frames."""
    import torch

    sys.path.insert(0, str(ROOT / "oracle"))
    import oracle as O

    cores = len(os.sched_getaffinity(0))
    host = _host_cpu()
    off = data["frame_off"]
    # calibrate on a few frames, then size the sample to ~cpu_seconds
    nf = 4
    t = time.perf_counter()
    O.ac3d_frames(kmap, data["pix"][: off[nf]], data["cnt"][: off[nf]], off[: nf + 1], shape,
                  nthreads=cores)
    per = (time.perf_counter() - t) / nf
    nf = int(max(8, min(len(off) - 1, args.cpu_seconds / max(per, 1e-6))))
    n = int(off[nf])
    t = time.perf_counter()
    O.ac3d_frames(kmap, data["pix"][:n], data["cnt"][:n], off[: nf + 1], shape, nthreads=cores)
    dt = time.perf_counter() - t
    # pair-updates of the sample (unit counts on the GPU, val(1) = 1000)
    m = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)
    ctx.ac3d_sparse_batch(d_kmap, torch.from_numpy(data["pix"][:n].view(np.int32)).to(dev),
                          torch.ones(n, dtype=torch.int16, device=dev),
                          torch.from_numpy(off[: nf + 1].view(np.int64)).to(dev), n, shape, m)
    upd = int(m.sum().item()) // 1000
    log(f"[bench] CPU oracle: {nf} frames, {upd:.3e} updates in {dt:.2f}s on {cores} threads")
    # the same restatement on one thread, calibrated on 2 frames, over a prefix of about a
    # third of that time
    t = time.perf_counter()
    O.ac3d_frames(kmap, data["pix"][: off[2]], data["cnt"][: off[2]], off[:3], shape, nthreads=1)
    per1 = (time.perf_counter() - t) / 2
    nf1 = int(max(2, min(nf, (args.cpu_seconds / 3) / max(per1, 1e-6))))
    n1 = int(off[nf1])
    t = time.perf_counter()
    O.ac3d_frames(kmap, data["pix"][:n1], data["cnt"][:n1], off[: nf1 + 1], shape, nthreads=1)
    dt1 = time.perf_counter() - t
    m.zero_()
    ctx.ac3d_sparse_batch(d_kmap, torch.from_numpy(data["pix"][:n1].view(np.int32)).to(dev),
                          torch.ones(n1, dtype=torch.int16, device=dev),
                          torch.from_numpy(off[: nf1 + 1].view(np.int64)).to(dev), n1, shape, m)
    upd1 = int(m.sum().item()) // 1000
    log(f"[bench] CPU oracle, 1 thread: {nf1} frames, {upd1:.3e} updates in {dt1:.2f}s")
    # thread scaling on a fixed 12-frame sample (omp atomics on a shared mesh)
    scaling = {}
    n12 = int(off[12])
    for th in sorted({1, 2, 4, 8, 16, cores}):
        if th > cores:
            continue
        t = time.perf_counter()
        O.ac3d_frames(kmap, data["pix"][:n12], data["cnt"][:n12], off[:13], shape, nthreads=th)
        scaling[str(th)] = (time.perf_counter() - t)
    t1s = scaling["1"]
    log("[bench] CPU thread scaling (speedup over 1 thread, 12 frames): " +
        ", ".join(f"{k}: {t1s / v:.2f}x" for k, v in scaling.items()))
    return {
        "value": upd / dt,
        "unit": "pair-updates/s",
        "cores": cores,
        "kind": "port",
        "sample": f"first {nf} of the {len(off) - 1} frames ({upd} pair-updates), "
                  f"OpenMP {cores} threads, -O3 -fopenmp -ffp-contract=off",
        "single_thread": {"value": upd1 / dt1, "cores": 1,
                          "sample": f"first {nf1} frames ({upd1} pair-updates), 1 thread"},
        "host": host,
        "thread_scaling_speedup": {k: t1s / v for k, v in scaling.items()},
    }


def _host_cpu():
    """The host CPU as the bench process sees it: model, logical CPUs, affinity, cgroup quota."""
    info = {"logical_cpus": os.cpu_count(), "affinity_cpus": len(os.sched_getaffinity(0))}
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                info["model"] = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    try:
        q = open("/sys/fs/cgroup/cpu.max").read().split()
        if q[0] != "max":
            info["cgroup_cpu_quota"] = int(q[0]) / int(q[1])
    except (OSError, ValueError, IndexError):
        pass
    return info


def cfg1_leg(args, iac, W, dev):
    """The small dense-frame pipeline (cfg1 shape): 100 dense 128^2 uint32 Poisson(0.01)
    frames as float32 on the device, sparsified there (CreateSparseHitList, threshold 0,
    step 1), AC_uw of the hit lists into the 65^3 mesh (NN/NN double map), and C(q) small
    of the flat-field mask into 65x65x3.  Reported per step as the reference plain
    method's dense pixel-pair visits per second (16,384^2 per frame): the job the
    pipeline does, not the pairs it touches.  The mesh is checked against the oracle."""
    import torch

    n, nf = 128, 100
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 63)
    s = iac.mesh_shape_small_cofq(mq, 63)
    d = W.dense_poisson_frames(n * n, nf, 0.01, seed=args.seed + 31)
    flat = np.ones(n * n, np.float32)
    mult = iac.cq_small_multiplicator(flat)
    ctx = iac.Context(0)
    d_km = torch.from_numpy(km).to(dev)
    frames = torch.from_numpy(d["frames"].astype(np.float32)).to(dev)
    d_flat = torch.from_numpy(flat).to(dev)
    rec = torch.zeros((nf * n * n, 4), dtype=torch.float32, device=dev)
    off = torch.zeros(nf + 1, dtype=torch.int64, device=dev)
    mesh = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)
    cqm = torch.zeros(s.size_ab ** 2 * s.size_c, dtype=torch.int64, device=dev)

    def run():
        mesh.zero_()
        cqm.zero_()
        nt = ctx.sparse_hit_list(d_km, frames, None, 0.0, 1.0, rec, off)
        ctx.ac3d_records_batch(d_km, rec, off, nt, shape, mesh)
        ctx.cq_small(d_km, d_flat, s, cqm, 0, mult)

    run()
    torch.cuda.synchronize()
    steps = max(1, args.steps)
    t = time.perf_counter()
    for _ in range(steps):
        run()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) * 1e3 / steps
    ctx.close()
    visits = float(n * n) ** 2 * nf
    O = _oracle()
    t = time.perf_counter()
    ref, _ = O.ac3d_frames(km, d["pix"], d["cnt"], d["frame_off"], shape, nthreads=_cpu_cores())
    ref_cq, _ = O.cq_small(flat, km, s, 0, mult, nthreads=_cpu_cores())
    cpu_s = time.perf_counter() - t
    parity = bool(np.array_equal(mesh.cpu().numpy().view(np.uint64), ref) and
                  np.array_equal(cqm.cpu().numpy().view(np.uint64), ref_cq))
    log(f"[cfg1] {ms:.2f} ms/step ({visits / (ms * 1e-3):.4e} dense pixel-pair visits/s), oracle {cpu_s * 1e3:.1f} ms "
        f"on {_cpu_cores()} threads, bit exact: {parity}")
    return {"workload": f"{nf} dense {n}x{n} uint32 Poisson(0.01) frames: device sparsify, AC_uw into "
                        f"{shape.size_ab}^3 (NN/NN double map), C(q) small of the flat field into "
                        f"{s.size_ab}x{s.size_ab}x{s.size_c}",
            "value": visits / (ms * 1e-3), "unit": "dense pixel-pair visits/s (job equivalent)", "ms_per_step": ms,
            "steps": steps, "bit_exact_vs_oracle": parity,
            "cpu_baseline": {"value": visits / cpu_s, "unit": "dense pixel-pair visits/s (job equivalent)",
                             "cores": _cpu_cores(), "kind": "port",
                             "sample": f"the whole workload (AC_uw of the {nf} hit lists and the flat-field "
                                       f"C(q)) in {cpu_s:.3f} s; hit lists built outside the clock"}}


def cfg3_leg(args, iac, W, dev):
    """Dense float frames with the rotation merge (cfg3): 2,000 256^2 FP32 Gamma(1, 0.5)
    frames over 360 uniform random rotations, frame f in orientation f mod 360 (uploaded
    orientation by orientation, so each orientation's 5 or 6 frames are one group), each
    orientation's C(q) small summed into its own 129x129x3 uint64 mesh (M = 1e10), to
    double, then Merge_CQ of mesh o with orientation o (weight 1) into the 129^3 lab
    mesh, to double.  M = 1e10 for the small
    meshes instead of the reference's 1e6 (Detector.cpp:1215-1227): at 1e6 the truncation
    of each pair value alone moves a voxel by about 2e-6, above the 1e-6 bar.  Parity: the
    first orientation's frame through the same chain against the FP64 oracle, every
    populated lab voxel within 1e-6 relative."""
    import torch

    n, norient, nframes = 256, 360, 2000
    _, km, mq = W.detector(n)
    s = iac.mesh_shape_small_cofq(mq, 127)
    orient = np.arange(nframes) % norient
    order = np.argsort(orient, kind="stable")  # frames of orientation 0, then 1, ...
    frames = torch.from_numpy(W.gamma_frames(n * n, nframes, 1.0, 0.5, seed=args.seed + 41)[order]).to(dev)
    rw = np.zeros((norient, 10), np.float32)
    rw[:, :9] = W.random_rotations(norient, args.seed + 43)
    rw[:, 9] = 1.0
    goff = np.concatenate([[0], np.cumsum(np.bincount(orient, minlength=norient))]).astype(np.uint32)
    nsmall = s.size_ab ** 2 * s.size_c
    ctx = iac.Context(0)
    d_km = torch.from_numpy(km).to(dev)
    d_rw = torch.from_numpy(rw).to(dev)
    small_u = torch.zeros(norient * nsmall, dtype=torch.int64, device=dev)
    small = torch.zeros(norient * nsmall, dtype=torch.float64, device=dev)
    big_u = torch.zeros(s.size_ab ** 3, dtype=torch.int64, device=dev)
    big = torch.zeros(s.size_ab ** 3, dtype=torch.float64, device=dev)
    m1, m2 = 1e10, 1e6

    def run():
        small_u.zero_()
        big_u.zero_()
        ctx.cq_dense_frames(d_km, frames, goff, s, small_u, iac.NEAREST, m1)
        ctx.u64_to_f64(small_u, m1, small)
        ctx.merge_cq_multi(small, s, d_rw, iac.NEAREST, m2, big_u)
        ctx.u64_to_f64(big_u, m2, big)

    run()
    torch.cuda.synchronize()
    t = time.perf_counter()
    run()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) * 1e3
    # parity: the first frame of orientation 0 alone against the FP64 oracle
    O = _oracle()
    g1 = np.array([0, 1], np.uint32)
    small_u.zero_()
    big_u.zero_()
    ctx.cq_dense_frames(d_km, frames[:1].contiguous(), g1, s, small_u[:nsmall], iac.NEAREST, m1)
    ctx.u64_to_f64(small_u[:nsmall], m1, small[:nsmall])
    ctx.merge_cq_multi(small[:nsmall], s, d_rw[:1].contiguous(), iac.NEAREST, m2, big_u)
    ctx.u64_to_f64(big_u, m2, big)
    got = big.cpu().numpy()
    t = time.perf_counter()
    ref = O.merge_f64(O.cq_small_f64(frames[0].cpu().numpy(), km, s), s, rw[0])
    odt = time.perf_counter() - t
    pop = ref > 1e-3 * ref.max()
    rel = float((np.abs(got[pop] - ref[pop]) / ref[pop]).max())
    ctx.close()
    log(f"[cfg3] parity: orientation 0 vs the FP64 oracle, max relative error {rel:.3e} over {int(pop.sum())} "
        f"populated voxels (oracle {odt:.1f}s)")
    if not rel <= 1e-6:
        raise SystemExit("cfg3 parity above 1e-6")
    pairs = float(n * n) ** 2 * nframes
    log(f"[cfg3] {nframes} dense {n}^2 frames in {norient} orientations + merge: {ms:.1f} ms "
        f"({pairs / (ms * 1e-3):.4e} pixel pairs/s, {nframes / (ms * 1e-3):.1f} frames/s)")
    return {"workload": f"{nframes} dense {n}x{n} FP32 Gamma(1, 0.5) frames, frame f in orientation f mod {norient}: "
                        f"C(q) small into {s.size_ab}x{s.size_ab}x{s.size_c} per orientation, Merge_CQ of the "
                        f"{norient} meshes into {s.size_ab}^3",
            "value": pairs / (ms * 1e-3), "unit": "ordered pixel pairs/s (merge included)", "ms_per_step": ms,
            "frames_per_s": nframes / (ms * 1e-3), "steps": 1,
            "multiplicators": {"small_cq": m1, "merge": m2,
                               "note": "small C(q) M = 1e10 (reference rule gives 1e6, whose per-pair "
                                       "truncation alone is ~2e-6 relative); tests pin the reference M bit for "
                                       "bit at this shape"},
            "parity": {"subset": "orientation 0 (one 256^2 frame) through the timed chain",
                       "max_rel_err_vs_fp64": rel, "populated_voxels": int(pop.sum()), "bar": 1e-6}}


def rotated_leg(args, iac, W, dev, d_kmap, d_pix, d_cnt, d_off, data, shape, updates):
    """The headline frames with a distinct uniform random rotation each (the event
    orientations of RunIAC's frame loop): the LDS engine rotates first-level voxels at
    the box flush; the global-atomic tile kernel is timed once beside it."""
    import torch

    nf = len(data["frame_off"]) - 1
    rots = torch.from_numpy(W.random_rotations(nf, args.seed + 21).astype(np.float32)).to(dev)
    n_total = int(data["frame_off"][-1])
    ctx = iac.Context(0)
    mesh = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)

    def run():
        mesh.zero_()
        ctx.ac3d_sparse_batch(d_kmap, d_pix, d_cnt, d_off, n_total, shape, mesh, rots=rots)

    def timed(k):
        run()
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(k):
            run()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) * 1e3 / k

    ms = timed(max(1, min(args.steps, 3)))
    engine_mesh = mesh.clone()
    ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
    ms_tiles = timed(1)
    same = bool(torch.equal(mesh, engine_mesh))
    ctx.close()
    log(f"[rotated] {ms:.2f} ms/step on the engine ({updates / (ms * 1e-3):.4e} pair-updates/s), tile kernel "
        f"{ms_tiles:.2f} ms, meshes equal: {same}")
    if not same:
        raise SystemExit("rotated leg: the engine and the tile kernel differ")
    return {"workload": f"the headline frames ({nf}) with a distinct uniform random rotation each",
            "value": updates / (ms * 1e-3), "unit": "pair-updates/s", "ms_per_step": ms,
            "tile_kernel_ms": ms_tiles, "full_meshes_equal_engine_vs_tile_kernel": same}


def _oracle():
    sys.path.insert(0, str(ROOT / "oracle"))
    import oracle as O

    return O


def _cpu_cores():
    return min(len(os.sched_getaffinity(0)), 16)


def ac1d_acuw_cpu(args, kmap, data, size, max_q, dq):
    """The oracle's AC1D AC_uw restatement (the reference CPU branch, one thread, linear
    split, self pairs weighted 2) on a prefix of the same frames, about a fifth of
    --cpu-seconds; hit lists built before the clock starts."""
    O = _oracle()
    off = data["frame_off"]
    hls = []

    def run(nf):
        while len(hls) < nf:
            f = len(hls)
            hls.append(O.hit_list_from_photons(kmap, data["pix"][off[f]:off[f + 1]], data["cnt"][off[f]:off[f + 1]]))
        ac = np.zeros(size)
        t = time.perf_counter()
        for f in range(nf):
            O.ac1d_acuw(hls[f], size, max_q, dq, 1, 2, ac=ac)
        return time.perf_counter() - t

    per = run(2) / 2
    nf = int(max(2, min(len(off) - 1, args.cpu_seconds / 5 / max(per, 1e-6))))
    dt = run(nf)
    pairs = float((np.diff(off[: nf + 1].astype(np.int64)).astype(np.float64) ** 2).sum())
    log(f"[ac1d] CPU oracle: {nf} frames, {pairs:.3e} ordered pairs in {dt:.2f}s on 1 thread")
    return {"value": pairs / dt, "unit": "ordered photon pairs/s", "cores": 1, "kind": "port",
            "sample": f"first {nf} frames ({pairs:.4e} ordered pairs) in {dt:.2f} s"}


def dense_cpu(args, label, run_k, npix, unordered):
    """Time an oracle pass over the first K pixels of an image (K^2 ordered pixel
    pairs, OpenMP over the outer pixel), K sized to about a fifth of --cpu-seconds.
    `unordered`: report the job-equivalent K(K+1)/2 unordered pairs per second (the
    unit of the GPU leg, whose symmetric kernel visits each unordered pair once)."""
    cores = _cpu_cores()
    k = min(npix, 4096)
    t = time.perf_counter()
    run_k(k, cores)
    dt = time.perf_counter() - t
    k = int(min(npix, max(k, k * (args.cpu_seconds / 5 / max(dt, 1e-6)) ** 0.5)))
    t = time.perf_counter()
    run_k(k, cores)
    dt = time.perf_counter() - t
    pairs = k * (k + 1) / 2 if unordered else float(k) * k
    log(f"[{label}] CPU oracle: {k} pixels, {pairs:.3e} pairs in {dt:.2f}s on {cores} threads")
    return {"value": pairs / dt, "unit": ("unordered" if unordered else "ordered") + " pixel pairs/s",
            "cores": cores, "kind": "port",
            "sample": f"the first {k} pixels of the image ({k}^2 ordered pairs visited) in {dt:.2f} s"}


def ac1d_leg(args, iac, W, dev, kmap, d_kmap, d_pix, d_cnt, d_off, data, max_q_vec):
    """AC1D AC_uw on the headline workload: the radial |q| histogram of every frame's
    ordered photon pairs (4096 bins, linear split as the evaluation forces), timed
    against the measured LDS-atomic ceiling."""
    import torch

    size = 4096
    max_q, dq = iac.ac1d_shape(max_q_vec, size)
    ctx = iac.Context(0)
    n_total = int(data["frame_off"][-1])
    sizes = np.diff(data["frame_off"].astype(np.int64))
    pairs = int((sizes.astype(np.float64) ** 2).sum())  # ordered pairs, a = b included
    h = torch.zeros(size, dtype=torch.float64, device=dev)

    def run():
        h.zero_()
        ctx.ac1d_acuw(d_kmap, d_pix, d_cnt, d_off, n_total, size, max_q, dq, 1, h)

    run()
    torch.cuda.synchronize()
    steps = max(1, args.steps)
    t = time.perf_counter()
    for _ in range(steps):
        run()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) * 1e3 / steps
    log(f"[ac1d] {ms:.2f} ms/step, {pairs:.4e} ordered pairs, {pairs / (ms * 1e-3):.4e} pairs/s")
    out = {"workload": f"AC1D AC_uw of the headline frames: {len(sizes)} frames, {size} bins, linear split, "
                       f"self pairs weighted 2",
           "value": pairs / (ms * 1e-3), "unit": "ordered photon pairs/s", "ms_per_step": ms, "steps": steps,
           "pairs_per_step": pairs,
           "cpu_baseline": None if args.no_cpu else ac1d_acuw_cpu(args, kmap, data, size, max_q, dq)}

    # AC1D C(q): every unordered pixel pair of one averaged-intensity image of the same detector
    npix = int(d_kmap.shape[0])
    img = W.gamma_frames(npix, 1, 1.0, 0.5, seed=args.seed + 11)[0]
    mult = iac.ac1d_cq_multiplicator(img)
    d_img = torch.from_numpy(img).to(dev)
    hq = torch.zeros(size, dtype=torch.int64, device=dev)

    def run_cq():
        hq.zero_()
        ctx.ac1d_cq(d_kmap, d_img, size, max_q, dq, 1, mult, hq)

    run_cq()
    torch.cuda.synchronize()
    cq_steps = max(1, min(args.steps, 3))
    t = time.perf_counter()
    for _ in range(cq_steps):
        run_cq()
    torch.cuda.synchronize()
    cq_ms = (time.perf_counter() - t) * 1e3 / cq_steps
    ctx.close()
    cq_pairs = npix * (npix + 1) // 2
    log(f"[ac1d-cq] {cq_ms:.2f} ms/step, {cq_pairs:.4e} pixel pairs, {cq_pairs / (cq_ms * 1e-3):.4e} pairs/s")
    cq_cpu = None
    if not args.no_cpu:
        O = _oracle()
        km = kmap.reshape(-1, 3)
        cq_cpu = dense_cpu(args, "ac1d-cq", lambda k, c: O.ac1d_cq(img[:k], km[:k], size, max_q, dq, 1, mult,
                                                                    nthreads=c), npix, True)
    out["cq"] = {"workload": f"AC1D C(q) of one {npix}-pixel Gamma(1, 0.5) image: {size} bins, linear split",
                 "value": cq_pairs / (cq_ms * 1e-3), "unit": "unordered pixel pairs/s", "ms_per_step": cq_ms,
                 "steps": cq_steps, "pairs_per_step": cq_pairs, "cpu_baseline": cq_cpu}
    return out


def cq_dense_leg(args, iac, W, dev):
    """Dense pixel-pair C(q) (cfg3 shape): 256^2 FP32 Gamma(1, 0.5) frames into the
    129^3 small C(q) mesh, every ordered pixel pair of each frame."""
    import torch

    n, nf = 256, 8
    _, kmap, mq = W.detector(n)
    s = iac.mesh_shape_small_cofq(mq, 127)
    frames = W.gamma_frames(n * n, nf, 1.0, 0.5, seed=args.seed + 7)
    ctx = iac.Context(0)
    d_kmap = torch.from_numpy(kmap).to(dev)
    d_frames = torch.from_numpy(frames).to(dev)
    mesh = torch.zeros(s.size_ab ** 2 * s.size_c, dtype=torch.int64, device=dev)
    goff = np.array([0, nf], np.uint32)
    mult = iac.cq_small_multiplicator(frames[0])

    def run():
        mesh.zero_()
        ctx.cq_dense_frames(d_kmap, d_frames, goff, s, mesh, iac.NEAREST, mult)

    tuned = None
    if not args.no_tune:
        best = None
        ctx.enable_timing(True)
        for cfg in CQ_GRID:
            apply_lds_config(ctx, iac, cfg)
            run()
            ctx.kernel_time(reset=True)
            run()
            ms, _ = ctx.kernel_time(reset=True)
            log(f"[cq tune] {cfg_str(cfg)}: {ms:.2f} ms")
            if best is None or ms < best[0]:
                best = (ms, cfg)
        ctx.enable_timing(False)
        apply_lds_config(ctx, iac, best[1])
        tuned = dict(best[1])
    before = ctx.pair_paths()
    run()
    torch.cuda.synchronize()
    path = path_since(ctx, before)
    steps = max(1, min(args.steps, 3))
    t = time.perf_counter()
    for _ in range(steps):
        run()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) * 1e3 / steps
    ctx.close()
    pairs = float(n * n) ** 2 * nf
    log(f"[cq] dense {n}^2 x {nf} frames: {ms:.2f} ms/step, {pairs / (ms * 1e-3):.4e} pixel pairs/s")
    cpu = None
    if not args.no_cpu:
        O = _oracle()
        km = kmap.reshape(-1, 3)
        cpu = dense_cpu(args, "cq", lambda k, c: O.cq_small(frames[0][:k], km[:k], s, 0, mult, nthreads=c),
                        n * n, False)
    return {"workload": f"dense C(q) small (AutoCorr_CQ_small): {n}x{n} detector, {nf} FP32 Gamma(1, 0.5) frames, "
                        f"{s.size_ab}x{s.size_ab}x{s.size_c} uint64 mesh, nearest neighbour",
            "value": pairs / (ms * 1e-3), "unit": "ordered pixel pairs/s", "ms_per_step": ms, "steps": steps,
            "pairs_per_step": pairs, "path": path, "tuned": tuned, "cpu_baseline": cpu}


def ppp_leg(args, iac, dev, probes):
    """LAP photon finder chain (PPP::ProcessData_PF_LAP per frame: pixel mask, offset and
    gain correction, largest-adjacent-pixel photon finder, photon counts) over 500 frames
    of a 1024x1024 detector laid out as eight 1024x128 modules; 37 ADU per photon."""
    import torch

    side, nf, adu = 1024, 500, 37.0
    npix = side * side
    panels = [(k * side * 128, side, 128) for k in range(8)]
    g = torch.Generator(device=dev)
    g.manual_seed(args.seed + 13)
    frames = torch.poisson(torch.full((nf, npix), 0.4, device=dev), generator=g)
    frames.add_(torch.rand((nf, npix), device=dev, generator=g) * 1.3 - 0.3).mul_(adu)
    mask = (torch.rand(npix, device=dev, generator=g) > 0.05).to(torch.int32)
    offset = torch.rand(npix, device=dev, generator=g) * 3.0
    gain = 0.8 + 0.4 * torch.rand(npix, device=dev, generator=g)
    out = torch.empty_like(frames)
    pc = torch.empty(nf, dtype=torch.int32, device=dev)
    mi = torch.empty(nf, dtype=torch.float32, device=dev)
    ctx = iac.Context(0)

    def run():
        ctx.ppp_lap(frames, out, panels, adu, mask=mask, offset=offset, gain=gain, photon_count=pc,
                    mean_intensity=mi)

    run()
    torch.cuda.synchronize()
    steps = max(1, min(args.steps, 5))
    ctx.enable_timing(True)
    ctx.kernel_time(reset=True)
    t = time.perf_counter()
    for _ in range(steps):
        run()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) * 1e3 / steps
    kms, kn = ctx.kernel_time(reset=True)
    ctx.enable_timing(False)
    k_ms = kms / max(kn, 1)
    # bit-exact check of the first two frames against the oracle
    O = _oracle()
    h_in = frames[:2].cpu().numpy()
    ref, rpc, _ = O.ppp_lap(h_in, panels, adu=adu, mask=mask.cpu().numpy(), offset=offset.cpu().numpy(),
                            gain=gain.cpu().numpy())
    exact = bool(np.array_equal(out[:2].cpu().numpy().view(np.int32), ref.view(np.int32))
                 and np.array_equal(pc[:2].cpu().numpy(), rpc))
    ctx.close()
    nbytes = nf * npix * 8  # each frame pixel read once and written once
    gbs = nbytes / (k_ms * 1e-3) / 1e9
    log(f"[ppp] LAP {side}^2 x {nf} frames: {ms:.3f} ms/step (finder kernel {k_ms:.3f} ms, {gbs:.0f} GB/s), "
        f"oracle match {exact}")
    cpu = None
    if not args.no_cpu:
        h = frames[:1].cpu().numpy()
        hm, ho, hg = mask.cpu().numpy(), offset.cpu().numpy(), gain.cpu().numpy()
        n, t0 = 0, time.perf_counter()
        while n == 0 or (time.perf_counter() - t0 < min(5.0, args.cpu_seconds / 5) and n < 200):
            O.ppp_lap(h, panels, adu=adu, mask=hm, offset=ho, gain=hg)
            n += 1
        cpu = {"value": n / (time.perf_counter() - t0), "unit": "frames/s", "cores": 1, "kind": "port",
               "sample": f"{n} frames of {side}x{side}, one thread (the reference loops frames serially)"}
    del frames, out
    torch.cuda.empty_cache()
    return {"workload": f"LAP photon finder chain: {side}x{side} detector as eight {side}x128 modules, {nf} FP32 "
                        f"frames, pixel mask, offset and gain maps, {adu} ADU per photon, per-event photon counts",
            "value": nf / (ms * 1e-3), "unit": "frames/s", "ms_per_step": ms, "steps": steps,
            "bit_exact_first_frames": exact,
            "roofline": {"bound": "hbm", "kernel": "lap_rows_kernel", "kernel_avg_ms": k_ms, "achieved": gbs,
                         "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": gbs / HBM_PEAK_GBS,
                         "bytes_per_pixel": 8,
                         "frac_of_measured_copy": gbs / probes["hbm_copy_GBps"] if probes else None},
            "cpu_baseline": cpu}


def eval_leg(args, W):
    """RunIAC::Run_AutoCorr_DataEval end to end through the C++ host mirror (the
    iac_eval driver): a raw float32 stack of photon frames is read event by event,
    averaged, sparsified, C(q) small and its merge computed, the frames binned by
    batched AC_uw, the final mesh normalised and written."""
    import shutil
    import subprocess
    import tempfile

    exe = ROOT / "incohautocorrelate_amd" / "iac_eval"
    n, nf, edge = 512, 1000, 255
    pm, _, _ = W.detector(n)
    tmp = Path(tempfile.mkdtemp(prefix="iac_eval_bench_"))
    try:
        pm.astype(np.float32).tofile(tmp / "pm.bin")
        rng = np.random.default_rng(args.seed + 11)
        with open(tmp / "frames.bin", "wb") as fh:  # photons of 6.4 ADU with 0.8 ADU noise, Poisson(0.01)
            for f0 in range(0, nf, 100):
                ph = rng.poisson(0.01, (min(100, nf - f0), n * n))
                fr = ph * 6.4 + rng.normal(0.0, 0.8, ph.shape) * (ph > 0)
                fh.write(fr.astype(np.float32).tobytes())
        cmd = [str(exe), "--pixelmap", str(tmp / "pm.bin"), "--size", str(n), str(n), "--frames",
               str(tmp / "frames.bin"), "--nframes", str(nf), "--mesh-size", str(edge), "--photon-offset", "3.2",
               "--photon-step", "6.4", "--out-final", str(tmp / "final.bin"), "--out-acuw", str(tmp / "acuw.bin"),
               "--out-cq", str(tmp / "cq.bin")]
        t = time.perf_counter()
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
        dt = time.perf_counter() - t
        if r.returncode != 0:
            raise RuntimeError("iac_eval failed: " + r.stderr[-2000:])
        report = json.loads(r.stdout.strip().splitlines()[-1])
        # the file-read bound: one plain sequential pass over the stack (page cache as warm as for the run)
        buf = bytearray(64 << 20)
        t = time.perf_counter()
        with open(tmp / "frames.bin", "rb", buffering=0) as fh:
            while fh.readinto(buf):
                pass
        read_pass = time.perf_counter() - t
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    ing = report.get("ingest", {})
    passes = ing.get("frames", 0) / nf if nf else 0
    bound = nf / (passes * read_pass) if passes else None
    overlap = 1.0 - ing["wait_s"] / ing["read_s"] if ing.get("read_s") else None
    log(f"[eval] {nf} frames of {n}^2 end to end in {dt:.2f} s ({nf / dt:.1f} frames/s), report {report}")
    log(f"[eval] {passes:.0f} streamed passes: reads {ing.get('read_s', 0):.3f} s on the reader thread, device loop "
        f"waited {ing.get('wait_s', 0):.3f} s (overlap {overlap}), uploads {ing.get('upload_s', 0):.3f} s; one plain "
        f"read pass {read_pass:.3f} s -> file-read bound {bound} frames/s")
    return {"workload": f"Run_AutoCorr_DataEval (3D) through iac_eval: {nf} float32 frames of {n}x{n} "
                        f"(Poisson(0.01) photons of 6.4 ADU + 0.8 ADU noise) from a raw stack, identity "
                        f"orientations, {edge + 2}^3 mesh, averaged intensity, C(q) small + merge, AC_uw, "
                        f"normalisation, three raw float64 outputs",
            "value": nf / dt, "unit": "frames/s (process wall time, file reads and writes included)",
            "seconds": dt, "report": report,
            "ingest": {"streamed_passes": passes, "reader_busy_s": ing.get("read_s"),
                       "device_loop_waited_s": ing.get("wait_s"), "upload_s": ing.get("upload_s"),
                       "streamed_loop_s": ing.get("loop_s"), "read_overlap_frac": overlap,
                       "plain_read_pass_s": read_pass, "file_read_bound_frames_per_s": bound,
                       "streamed_frames_per_s": ing["frames"] / ing["loop_s"] if ing.get("loop_s") else None,
                       "streamed_frac_of_file_read_bound": (ing["frames"] / ing["loop_s"]) / (nf / read_pass)
                       if ing.get("loop_s") else None,
                       "note": "frames are read one stack ahead on a reader thread into page-locked stacks; "
                               "read_overlap_frac = 1 - waited / reader busy"}}


def probe_leg(iac, dev, nvox):
    """Measured ceilings: a 2 GiB device copy (HBM), uint64 atomic adds uniform over
    the 257^3 mesh, over a hot window of the occupied slab's size (7.3e5 voxels), in runs
    of 8 consecutive voxels (one 64-byte segment per 8 lanes), and into LDS boxes."""
    import torch

    ctx = iac.Context(0)
    src = torch.empty(2 << 30, dtype=torch.uint8, device=dev)
    dst = torch.empty_like(src)
    ctx.probe_copy(src, dst)
    ms = min(ctx.probe_copy(src, dst) for _ in range(5))
    copy_gbs = 2 * src.numel() / (ms * 1e-3) / 1e9
    del src, dst
    mesh = torch.zeros(nvox, dtype=torch.int64, device=dev)
    n = 1 << 30
    rates = {}
    for mode, name, hot in ((0, "uniform", 0), (1, "hot_slab", 730000), (3, "runs_of_8", 0), (2, "lds_box", 0),
                            (4, "lds_box_f64", 0)):
        adds = n << 2 if name.startswith("lds") else n  # the boxes' clear and flush below 2 %
        ctx.probe_atomics(mesh, n >> 4, mode, hot)
        t = min(ctx.probe_atomics(mesh, adds, mode, hot) for _ in range(3))
        rates[name] = adds / (t * 1e-3)
    log(f"[probe] copy {copy_gbs:.0f} GB/s; u64 atomics/s uniform {rates['uniform']:.3e}, "
        f"hot slab {rates['hot_slab']:.3e}, runs of 8 {rates['runs_of_8']:.3e}, LDS {rates['lds_box']:.3e}, "
        f"LDS double {rates['lds_box_f64']:.3e}")
    ctx.close()
    return {"hbm_copy_GBps": copy_gbs, "atomic_u64_per_s": rates,
            "copy": "2 GiB device-to-device, 16-byte vector loads/stores, best of 5",
            "atomics": "2^30 adds of 1 (LDS boxes: 2^32), best of 3"}


def uneven_leg(args, iac, W, dev):
    """4,096 frames on the 1024^2 detector, photons/frame lognormal (median 1,500,
    sigma 1, clipped to 10..20,000, count 1 at distinct pixels) into the 257^3
    uint64 mesh: one prepared batch, its graph replayed per step (mesh cleared
    inside the graph)."""
    import torch

    _, kmap, max_q = W.detector(1024)
    shape = iac.mesh_shape_big(max_q, 255)
    t0 = time.time()
    data = W.lognormal_photon_frames(1024 * 1024, 4096, 1500, 1.0, 10, 20000, seed=0)
    n_total = int(data["frame_off"][-1])
    sizes = np.diff(data["frame_off"].astype(np.int64))
    log(f"[uneven] {n_total} photons in {len(sizes)} frames (mean {sizes.mean():.0f}, max {sizes.max()}), "
        f"generated in {time.time() - t0:.1f}s")
    d_kmap = torch.from_numpy(kmap).to(dev)
    d_pix = torch.from_numpy(data["pix"].view(np.int32)).to(dev)
    d_cnt = torch.from_numpy(data["cnt"].view(np.int16)).to(dev)
    d_off = torch.from_numpy(data["frame_off"].view(np.int64)).to(dev)
    nvox = shape.size_ab ** 2 * shape.size_c
    d_mesh = torch.zeros(nvox, dtype=torch.int64, device=dev)
    ctx = iac.Context(0)
    tuned = None
    if not args.no_tune:
        tuned = autotune(ctx, iac, d_kmap, d_pix, d_cnt, d_off, shape, label="uneven tune")
    b = ctx.ac3d_batch(d_kmap, d_pix, d_cnt, d_off, n_total, shape)
    b.capture(d_mesh, True)
    b.launch(d_mesh, True)
    torch.cuda.synchronize()
    updates = int(d_mesh.sum().item()) // 1000  # counts are 1: val(1) = 1000 per update
    steps = max(1, args.steps)
    ctx.enable_timing(True)
    ctx.kernel_time(reset=True)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    for _ in range(steps):
        b.launch(d_mesh, True)
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    gms, gl = ctx.kernel_time(reset=True)
    ctx.enable_timing(False)
    ms = (t2 - t1) * 1e3 / steps
    rate = updates / (ms * 1e-3)
    log(f"[uneven] {ms:.2f} ms/step (graph {gms / max(gl, 1):.2f} ms), {updates:.4e} updates, {rate:.4e} updates/s")
    b.destroy()
    ctx.close()
    return {
        "workload": "4,096 frames, 1024x1024 detector, photons/frame lognormal(median 1500, sigma 1) clipped "
                    "10..20,000, count 1 at distinct pixels, 257^3 uint64 mesh, NN/NN double-map, identity R",
        "value": rate, "unit": "pair-updates/s", "ms_per_step": ms, "graph_ms": gms / max(gl, 1),
        "steps": steps, "photons": n_total, "pair_updates_per_step": updates, "tuned": tuned,
        "launch": "hipGraph replay of one prepared batch (zero + gather + cell sort + pairs + mirror)",
    }


MFMA_PEAK_TFLOPS = {"bf16": 2500.0, "fp16": 2500.0}  # MI355X dense, public spec


def sim_leg(args, iac, W, dev):
    """Speckle simulator: 512^2 pixels x 10,000 emitters x sim_frames frames."""
    import torch

    sys.path.insert(0, str(ROOT / "oracle"))
    import oracle as O

    n, nem, nf, wl = 512, 10000, args.sim_frames, 1.5
    npix = n * n
    pm, _, _ = W.detector(n)
    em = W.emitters_cube(nem, 500.0, args.seed)
    ph = W.emitter_phases(nf, nem, args.seed + 1)
    d_pm = torch.from_numpy(pm).to(dev)
    d_em = torch.from_numpy(em).to(dev)
    d_ph = torch.from_numpy(ph).to(dev)
    out = torch.empty((nf, npix), dtype=torch.float32, device=dev)
    ctx = iac.Context(0)
    # FP64 oracle on 8 central detector rows x 4 frames
    p0, npx, nfe = (n // 2 - 4) * n, 8 * n, min(4, nf)
    t = time.perf_counter()
    ref = {k: O.simulate_fp64(pm, em, ph, wl, out_kind=k, pixels=(p0, npx), frames=(0, nfe)) for k in (0, 1)}
    log(f"[sim] FP64 oracle subset ({npx} px x {nfe} frames x {nem} emitters, both kinds) "
        f"in {time.perf_counter() - t:.1f}s")

    def rel(a, b):
        return float(np.linalg.norm(a - b) / np.linalg.norm(b))

    res = {}
    want = set(args.sim_modes.split(","))
    for mode, name, dt, nterms in ((iac.SIM_BF16X3, "bf16x3", "bf16", 3), (iac.SIM_FP16X3, "fp16x3", "fp16", 3),
                                   (iac.SIM_FP16, "fp16", "fp16", 1)):
        if name not in want:
            continue
        flops = 8.0 * npix * nem * nf  # algorithmic: one complex multiply-add per (pixel, emitter, frame)
        issued = nterms * flops  # the split products the MFMAs execute
        torch.cuda.synchronize()
        t = time.perf_counter()
        plan = ctx.sim_plan(d_pm, d_em, wl, mode)
        torch.cuda.synchronize()
        plan_s = time.perf_counter() - t
        errs = {}
        for k, kname in ((0, "amplitude"), (1, "intensity")):
            ctx.sim_run(plan, d_ph, out, 1, k)
            got = out[:nfe, p0:p0 + npx].cpu().numpy().astype(np.float64)
            errs[kname] = rel(got, ref[k])

        def step():
            ctx.sim_run(plan, d_ph, out, 1, iac.SIM_AMPLITUDE)
            ctx.sim_postprocess(out, 0.01 * npix, True, seed=args.seed)

        step()
        torch.cuda.synchronize()
        ctx.enable_timing(True)
        ctx.kernel_time(reset=True)
        t1 = time.perf_counter()
        for _ in range(args.sim_steps):
            step()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        gms, gl = ctx.kernel_time(reset=True)
        ctx.enable_timing(False)
        gemm_ms = gms / max(gl, 1)
        ms = (t2 - t1) * 1e3 / args.sim_steps
        ach = flops / (gemm_ms * 1e-3) / 1e12
        ach_issued = issued / (gemm_ms * 1e-3) / 1e12
        photons = float(out.sum().item()) / nf
        res[name] = {
            "frames_per_s": nf / (ms * 1e-3), "ms_per_step": ms, "gemm_ms": gemm_ms, "plan_s": plan_s,
            "err_vs_fp64": errs, "photons_per_frame": photons,
            "roofline": {"bound": "mfma", "achieved": ach, "peak": MFMA_PEAK_TFLOPS[dt], "unit": "TFLOP/s",
                         "frac": ach / MFMA_PEAK_TFLOPS[dt], "traffic": SIM_TRAFFIC.get(name),
                         "traffic_unit": "HBM bytes per launch (rocprofv3 FETCH_SIZE x2 + WRITE_SIZE, copy-scaled)",
                         "kernel": f"sim_gemm_kernel ({dt} v_mfma_f32_32x32x16, {nterms} product(s) per term, "
                                   "fused |psi| epilogue)",
                         "flops_per_step": flops, "flops_basis": "algorithmic 8 P E per frame",
                         "issued_flops_per_step": issued, "issued_tflops": ach_issued,
                         "issued_frac": ach_issued / MFMA_PEAK_TFLOPS[dt]},
        }
        log(f"[sim] {name}: {ms:.2f} ms/step ({nf / (ms * 1e-3):.1f} frames/s), GEMM region {gemm_ms:.2f} ms "
            f"= {ach:.0f} TFLOP/s algorithmic ({ach_issued:.0f} issued), plan {plan_s:.2f}s, "
            f"err amp {errs['amplitude']:.2e} "
            f"int {errs['intensity']:.2e}, {photons:.1f} photons/frame")
        plan.destroy()
        del plan
        torch.cuda.empty_cache()

    # the plain FP32 direct sum (reference arithmetic, float positions and phases)
    nd = min(args.sim_direct_frames, nf)
    em32 = em.astype(np.float32)
    ph32 = np.ascontiguousarray(ph[:nd]).astype(np.float32)
    d_em32 = torch.from_numpy(em32).to(dev)
    d_ph32 = torch.from_numpy(ph32).to(dev)
    od = torch.empty((nd, npix), dtype=torch.float32, device=dev)
    ctx.sim_direct_fp32(d_pm, d_em32, d_ph32[:1], wl, od[:1])
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    ctx.sim_direct_fp32(d_pm, d_em32, d_ph32, wl, od)
    torch.cuda.synchronize()
    dms = (time.perf_counter() - t1) * 1e3
    nfe32 = min(nfe, nd)
    ref32 = O.simulate_fp64(pm, em32.astype(np.float64), ph32.astype(np.float64), wl, out_kind=0,
                            pixels=(p0, npx), frames=(0, nfe32))
    e32 = rel(od[:nfe32, p0:p0 + npx].cpu().numpy().astype(np.float64), ref32)
    direct_fps = nd / (dms * 1e-3)
    log(f"[sim] fp32 direct: {dms / nd:.2f} ms/frame ({direct_fps:.1f} frames/s), err amp {e32:.2e}")
    ctx.close()
    # the headline mode: the fastest whose intensity error against FP64 is within 1e-3
    ok = [k for k, v in res.items() if v["err_vs_fp64"]["intensity"] <= 1e-3]
    best_mode = max(ok, key=lambda k: res[k]["frames_per_s"])
    best = res[best_mode]["frames_per_s"]
    return {
        "workload": f"{n}x{n} detector (75 um, 0.5 m), {nem} emitters uniform in a 500 A cube, lambda {wl} A, "
                    f"{nf} frames of uniform phases, |psi| output, rescale to 0.01 photons/pixel + Poisson",
        "unit": "frames/s",
        "value": best,
        "mode": best_mode,
        "error_bar": "normwise relative |psi|^2 error vs FP64 <= 1e-3",
        "algorithmic_flop_per_frame": 8.0 * npix * nem,
        "modes": res,
        "fp32_direct": {"frames_per_s": direct_fps, "ms_per_frame": dms / nd, "frames_timed": nd,
                        "err_vs_fp64": {"amplitude": e32}},
        "speedup_vs_fp32_direct": {k: v["frames_per_s"] / direct_fps for k, v in res.items()},
        "speedup_best_vs_fp32_direct": best / direct_fps,
        "err_subset": f"pixels [{p0}, {p0 + npx}) (8 central rows) x frames [0, {nfe}), normwise relative",
    }


if __name__ == "__main__":
    main()
