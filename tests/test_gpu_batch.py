"""Prepared frame batches (iac_ac3d_batch_*): one launch or a replayed graph equals
the unbatched per-frame GPU kernel, the one-call batch and the CPU oracle,
bit for bit -- including the uneven lognormal workload at full size."""
import numpy as np
import pytest

import oracle as O
from gpu_helpers import mesh_np, to_dev
from incohautocorrelate_amd import workloads as W

pytestmark = pytest.mark.gpu


def _dev_frames(data, dev):
    return (to_dev(data["pix"], dev), to_dev(data["cnt"], dev), to_dev(data["frame_off"], dev))


def _per_frame(ctx, dev, km, data, shape, frames):
    """The unbatched GPU path: iac_ac3d_sparse once per frame (tile kernel)."""
    import torch

    m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
    off = data["frame_off"]
    eye = np.eye(3, dtype=np.float32).reshape(9)
    for f in frames:
        a, b = int(off[f]), int(off[f + 1])
        if a == b:
            continue
        hl = O.hit_list_from_photons(km, data["pix"][a:b], data["cnt"][a:b])
        ctx.ac3d_sparse(to_dev(hl, dev), eye, shape, m)
    return mesh_np(m)


@pytest.mark.parametrize("interp1,interp2,dm", [(0, 0, True), (1, 1, True), (0, 1, False)])
def test_batch_equals_per_frame_and_oracle(ctx, dev, interp1, interp2, dm):
    import torch

    import incohautocorrelate_amd as iac

    n = 128
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 63)
    data = W.lognormal_photon_frames(n * n, 40, 60, 1.0, 2, 600, seed=5 + interp1)
    n_total = int(data["frame_off"][-1])
    d_km = to_dev(km, dev)
    pix, cnt, off = _dev_frames(data, dev)
    b = ctx.ac3d_batch(d_km, pix, cnt, off, n_total, shape, interp1, interp2, dm)
    m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
    b.launch(m, zero_mesh=True)
    got = mesh_np(m)
    ref, _ = O.ac3d_frames(km, data["pix"], data["cnt"], data["frame_off"], shape, None, interp1, interp2, dm)
    assert np.array_equal(got, ref)
    if (interp1, interp2, dm) == (0, 0, True):
        assert np.array_equal(got, _per_frame(ctx, dev, km, data, shape, range(40)))
    b.destroy()


def test_graph_replays_match_eager(ctx, dev):
    """Replays of the captured graph, with eager work and syncs in between, each
    equal the eager launch (the mesh is cleared inside the graph by a kernel)."""
    import torch

    import incohautocorrelate_amd as iac

    n = 192
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 95)
    data = W.lognormal_photon_frames(n * n, 64, 150, 1.0, 5, 1500, seed=8)
    n_total = int(data["frame_off"][-1])
    d_km = to_dev(km, dev)
    pix, cnt, off = _dev_frames(data, dev)
    b = ctx.ac3d_batch(d_km, pix, cnt, off, n_total, shape)
    eager = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)
    b.launch(eager, zero_mesh=True)
    want = mesh_np(eager)
    m = torch.zeros_like(eager)
    b.capture(m, zero_mesh=True)
    for r in range(4):
        m.fill_(12345)  # stale content the graph must clear
        b.launch(m, zero_mesh=True)
        torch.cuda.synchronize()
        assert np.array_equal(mesh_np(m), want), f"replay {r}"
        # eager work between replays
        other = torch.zeros_like(eager)
        ctx.ac3d_sparse_batch(d_km, pix, cnt, off, n_total, shape, other)
        torch.cuda.synchronize()
        assert np.array_equal(mesh_np(other), want)
    # new photon counts in the same buffers: the graph reads the current contents
    cnt2 = np.minimum(data["cnt"].astype(np.int64) * 3, 65535).astype(np.uint16)
    cnt.copy_(to_dev(cnt2, dev))
    b.launch(m, zero_mesh=True)
    ref, _ = O.ac3d_frames(km, data["pix"], cnt2, data["frame_off"], shape)
    assert np.array_equal(mesh_np(m), ref)
    b.destroy()


def test_accumulating_launches(ctx, dev):
    import torch

    import incohautocorrelate_amd as iac

    n = 96
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 47)
    data = W.poisson_photon_frames(n * n, 30, 0.01, 3)
    n_total = int(data["frame_off"][-1])
    pix, cnt, off = _dev_frames(data, dev)
    b = ctx.ac3d_batch(to_dev(km, dev), pix, cnt, off, n_total, shape)
    m = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)
    for _ in range(3):
        b.launch(m, zero_mesh=False)
    ref, _ = O.ac3d_frames(km, data["pix"], data["cnt"], data["frame_off"], shape)
    assert np.array_equal(mesh_np(m), ref * np.uint64(3))
    b.destroy()


def test_uneven_lognormal_full_size(ctx, dev):
    """4,096 frames on a 1024^2 detector, photons/frame lognormal (median 1,500,
    sigma 1, clipped to 10..20,000): the graph-replayed batch equals the
    global-atomic tile kernel over all frames, the per-frame kernel on a frame
    subset and the CPU oracle on a smaller subset."""
    import torch

    import incohautocorrelate_amd as iac

    n = 1024
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 255)
    data = W.lognormal_photon_frames(n * n, 4096, 1500, 1.0, 10, 20000, seed=0)
    n_total = int(data["frame_off"][-1])
    print(f"uneven workload: {n_total} photons, max frame {np.diff(data['frame_off'].astype(np.int64)).max()}")
    d_km = to_dev(km, dev)
    pix, cnt, off = _dev_frames(data, dev)
    nvox = shape.size_ab ** 2 * shape.size_c
    dropped0 = ctx.dropped()  # the context's counter is cumulative over the session
    b = ctx.ac3d_batch(d_km, pix, cnt, off, n_total, shape)
    m = torch.zeros(nvox, dtype=torch.int64, device=dev)
    b.capture(m, zero_mesh=True)
    b.launch(m, zero_mesh=True)
    got = mesh_np(m)
    tiles = torch.zeros(nvox, dtype=torch.int64, device=dev)
    ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
    try:
        ctx.ac3d_sparse_batch(d_km, pix, cnt, off, n_total, shape, tiles)
    finally:
        ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
    assert np.array_equal(got, mesh_np(tiles))
    assert got.sum() > 0 and ctx.dropped() == dropped0
    b.destroy()
    # subsets: per-frame GPU kernel (24 frames incl. the largest) and the CPU oracle (6 frames)
    sizes = np.diff(data["frame_off"].astype(np.int64))
    sub = sorted(set(range(16)) | set(np.argsort(sizes)[-8:].tolist()))
    sub_off = np.zeros(len(sub) + 1, np.uint64)
    sub_pix, sub_cnt = [], []
    for i, f in enumerate(sub):
        a, c = int(data["frame_off"][f]), int(data["frame_off"][f + 1])
        sub_pix.append(data["pix"][a:c])
        sub_cnt.append(data["cnt"][a:c])
        sub_off[i + 1] = sub_off[i] + (c - a)
    sd = {"pix": np.concatenate(sub_pix), "cnt": np.concatenate(sub_cnt), "frame_off": sub_off}
    spix, scnt, soff = _dev_frames(sd, dev)
    bs = ctx.ac3d_batch(d_km, spix, scnt, soff, int(sub_off[-1]), shape)
    ms = torch.zeros(nvox, dtype=torch.int64, device=dev)
    bs.launch(ms, zero_mesh=True)
    assert np.array_equal(mesh_np(ms), _per_frame(ctx, dev, km, data, shape, sub))
    bs.destroy()
    six = {"pix": sd["pix"][: int(sub_off[6])], "cnt": sd["cnt"][: int(sub_off[6])], "frame_off": sub_off[:7]}
    ref, _ = O.ac3d_frames(km, six["pix"], six["cnt"], six["frame_off"], shape)
    p6, c6, o6 = _dev_frames(six, dev)
    b6 = ctx.ac3d_batch(d_km, p6, c6, o6, int(sub_off[6]), shape)
    m6 = torch.zeros(nvox, dtype=torch.int64, device=dev)
    b6.launch(m6, zero_mesh=True)
    assert np.array_equal(mesh_np(m6), ref)
    b6.destroy()


@pytest.mark.parametrize("mode,cell,box", [(1, 5, 4096), (1, 4, 1920), (2, 4, 4096), (1, 3, 1024)])
def test_linear_modes_pair_walks(ctx, dev, mode, cell, box):
    """Linear AC_uw (ordered pairs, 8 or 64 corner adds each; a linear first level with a
    nearest second level bins in-box tasks inline) through the engine with lanes on
    consecutive pairs and with a pair range per thread: the oracle's bits."""
    import torch

    import incohautocorrelate_amd as iac

    n = 96
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 47)
    data = W.lognormal_photon_frames(n * n, 12, 50, 1.0, 1, 400, seed=31)
    n_total = int(data["frame_off"][-1])
    ref = {}
    for i1, i2 in ((1, 1), (0, 1), (1, 0)):
        ref[i1, i2], _ = O.ac3d_frames(km, data["pix"], data["cnt"], data["frame_off"], shape, None, i1, i2, True)
    ctx.set_option(iac.OPT_AC3D_KERNEL, 2)
    ctx.set_option(iac.OPT_PAIR_MODE, mode)
    ctx.set_option(iac.OPT_CELL_VOX, cell)
    ctx.set_option(iac.OPT_BOX_CAP, box)
    try:
        pix, cnt, off = _dev_frames(data, dev)
        for (i1, i2), r in ref.items():
            m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
            ctx.ac3d_sparse_batch(to_dev(km, dev), pix, cnt, off, n_total, shape, m, interp1=i1, interp2=i2)
            assert np.array_equal(mesh_np(m), r), (i1, i2)
    finally:
        for o in (iac.OPT_AC3D_KERNEL, iac.OPT_PAIR_MODE, iac.OPT_CELL_VOX, iac.OPT_BOX_CAP):
            ctx.set_option(o, 0)


@pytest.mark.parametrize("mode", [1, 2])
def test_nn_linear_double_map_symmetric(ctx, dev, mode):
    """Double map, nearest first level, linear second level, identity rotation: the
    engine bins it point-symmetrically on the voxel itself, valued FloatToInt(double).
    Float weights and integer counts whose products pass 10,527 (where the double and
    float fixed points part) pin that value against the oracle's ordered 8-corner loop."""
    import torch

    import incohautocorrelate_amd as iac

    n = 96
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 47)
    rng = np.random.default_rng(77)
    hls = []
    for f in range(6):
        npho = int(rng.integers(20, 120))
        pix = rng.choice(n * n, npho, replace=False)
        w = (rng.gamma(1.0, 3.0, npho) if f % 2 == 0 else rng.integers(1, 300, npho)).astype(np.float32)
        hl = np.empty((npho, 4), np.float32)
        hl[:, :3] = km[pix]
        hl[:, 3] = w
        hls.append(hl)
    ref = np.zeros(shape.size_ab ** 3, np.uint64)
    ref_nn = np.zeros(shape.size_ab ** 3, np.uint64)
    for hl in hls:
        ref, _ = O.ac3d_sparse(hl, shape, None, 0, 1, True, mesh=ref)
        ref_nn, _ = O.ac3d_sparse(hl, shape, None, 0, 0, True, mesh=ref_nn)
    assert not np.array_equal(ref, ref_nn)  # the value function matters for these weights
    rec = np.concatenate(hls)
    off = np.concatenate([[0], np.cumsum([len(h) for h in hls])]).astype(np.uint64)
    ctx.set_option(iac.OPT_AC3D_KERNEL, 2)
    ctx.set_option(iac.OPT_PAIR_MODE, mode)
    try:
        m = torch.zeros(shape.size_ab ** 3, dtype=torch.int64, device=dev)
        ctx.ac3d_records_batch(to_dev(km, dev), to_dev(rec, dev), to_dev(off, dev), len(rec), shape, m,
                               interp1=0, interp2=1)
        assert np.array_equal(mesh_np(m), ref)
    finally:
        ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
        ctx.set_option(iac.OPT_PAIR_MODE, 0)


@pytest.mark.parametrize("interp1,interp2", [(0, 0), (1, 1)])
def test_library_tuner(ctx, dev, interp1, interp2):
    """iac_ac3d_tune times every candidate on a frame prefix, applies the fastest, caches it
    per (k-map, mesh, modes); every setting it tries gives the oracle's mesh (the tuner is
    also how the benchmark picks its settings)."""
    import torch

    import incohautocorrelate_amd as iac

    n = 128
    _, km, mq = W.detector(n)
    shape = iac.mesh_shape_big(mq, 63)
    data = W.lognormal_photon_frames(n * n, 60, 80, 1.0, 2, 800, seed=23)
    d_km = to_dev(km, dev)
    pix, cnt, off = _dev_frames(data, dev)
    c = iac.Context(0)
    try:
        best, cands = c.ac3d_tune(d_km, pix, cnt, off, shape, interp1, interp2, True, prefix_frames=40)
        assert len(cands) >= 5 and all(x["ms"] > 0 for x in cands)
        assert best["ms"] == min(x["ms"] for x in cands)
        if interp1 == 1:  # linear binning: the 4096-voxel boxes lead the candidates
            assert cands[0]["box_cap"] == 4096
        again, none = c.ac3d_tune(d_km, pix, cnt, off, shape, interp1, interp2, True, prefix_frames=40)
        assert none == [] and again["ms"] == -1.0
        assert {k: v for k, v in again.items() if k != "ms"} == {k: v for k, v in best.items() if k != "ms"}
        ref, _ = O.ac3d_frames(km, data["pix"], data["cnt"], data["frame_off"], shape, None, interp1, interp2, True)
        for x in cands:  # each candidate setting, applied by hand, is bit-exact
            c.set_option(iac.OPT_PAIR_MODE, x["pair_mode"])
            c.set_option(iac.OPT_CELL_VOX, x["cell_vox"])
            c.set_option(iac.OPT_BOX_CAP, x["box_cap"])
            c.set_option(iac.OPT_FRAME_CHUNK, x["frame_chunk"])
            m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
            c.ac3d_sparse_batch(d_km, pix, cnt, off, int(data["frame_off"][-1]), shape, m,
                                interp1=interp1, interp2=interp2, double_map=True)
            assert np.array_equal(mesh_np(m), ref), x
    finally:
        c.close()


@pytest.mark.parametrize("rows,cols,dist,edge", [(128, 128, 2e5, 63), (60, 200, 1e5, 95), (210, 70, 3e5, 127),
                                                 (256, 256, 2e4, 61), (400, 64, 4e5, 191), (90, 90, 4e5, 21)])
@pytest.mark.parametrize("kind", ["ones", "counts", "heavy", "full", "large"])
def test_strips_vs_tiles(ctx, dev, rows, cols, dist, edge, kind):
    """Nearest-neighbour batches of frames with enough photons for strips, against the
    global-atomic tile kernel, equal in every voxel: wide and tall detectors, weights that fill a
    32-bit box after a few frames ("heavy") or within one ("full"), or are too large for it
    ("large"), frames that are empty, of one photon or of one corner, a zoom that cuts pairs, with
    a rotation per frame and without."""
    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    rng = np.random.default_rng(rows + 3 * edge)
    km, _, _, mq = iac.calc_kmap(iac.generate_pixel_map(rows, cols, 75.0, [0, 0, dist], (1, 0, 0), (0, 1, 0)))
    pix, cnt = [], []
    nf = 120
    for f in range(nf):
        n = [0, 1, 900][f] if f < 3 else int(rng.integers(1200, 3600)) * (3 if kind == "full" and f % 20 == 19 else 1)
        pix.append(np.sort(rng.integers(0, rows * cols if f != 2 else 16 * cols, n)))
        top = {"ones": 1, "heavy": 60, "full": 129}.get(kind, 5)
        cnt.append(np.full(n, top) if top > 5 else rng.integers(1, top + 1, n))
    if kind == "large":
        cnt[9][7] = 130
    off = np.concatenate([[0], np.cumsum([p.size for p in pix])])
    pix, cnt = np.concatenate(pix), np.concatenate(cnt)
    rots = W.random_rotations(nf, 5).astype(np.float32)
    rots[:60] = rots[0]
    rots[60:75] = np.eye(3, dtype=np.float32).reshape(9)
    for zoom, r in ((1.0, None), (1.8, None), (1.0, rots)):
        shape = iac.mesh_shape_big(mq, edge, zoom)
        got = []
        for kernel in (0, 1):
            ctx.set_option(iac.OPT_AC3D_KERNEL, kernel)
            try:
                before = ctx.dropped()
                m = mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off, shape, rots=r))
                got.append((m, ctx.dropped() - before))
            finally:
                ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
        assert np.array_equal(got[0][0], got[1][0]), (zoom, r is None)
        assert got[0][1] == got[1][1]


# Rows of bright patches on the edges of the detector's strips, as far apart as the distances that
# one task of the strips holds: each record meets two strips' records in one voxel of that task.
# "frames": 10,000 frames, a block adds nine of them; "frame": one fills the 32-bit box by itself.
BRIGHT_ROWS = {"frames": (512, 41, 10_000, (12, 13), [2, 6, 10, 14], 1.18919025, 90),
               "frame": (1024, 51, 400, (16, 16), [1, 5, 9, 13, 17, 21], 1.0, 129)}


def bright_rows(name):
    import incohautocorrelate_amd as iac

    n, edge, nf, (tall, wide), at, height, count = BRIGHT_ROWS[name]
    km, _, _, mq = iac.calc_kmap(iac.generate_pixel_map(n, n, 75.0, [0, 0, 5e5], (1, 0, 0), (0, 1, 0)))
    shape = iac.mesh_shape_big(mq, edge)
    k = km.reshape(n, n, 3)
    across = 1 if abs(k[0, -1, 1] - k[0, 0, 1]) > abs(k[-1, 0, 1] - k[0, 0, 1]) else 0  # the index y grows along
    line = k[n // 2, :, 1] if across else k[:, n // 2, 1]
    strip = (line - km[:, 1].min()) * shape.voxel_per_dq / height
    img = np.zeros((n, n), bool)
    for edge_at in at:
        c = int(np.argmin(abs(strip - edge_at)))
        y = slice(c - tall // 2, c - tall // 2 + tall)
        x = slice(n // 2 - wide // 2, n // 2 - wide // 2 + wide)
        img[(x, y) if across else (y, x)] = True
    pix = np.flatnonzero(img)
    return km, shape, pix, np.full(pix.size, count), nf


@pytest.mark.parametrize("name", list(BRIGHT_ROWS))
def test_strips_bright_rows(ctx, dev, name):
    """Equal frames whose fullest voxel passes 2^32 in a task of several strip distances: the mesh is
    that of one frame, by the tile kernel, times their number."""
    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    km, shape, pix, cnt, nf = bright_rows(name)
    off = np.arange(nf + 1) * pix.size
    m = mesh_np(gpu_batch(ctx, dev, km, np.tile(pix, nf), np.tile(cnt, nf), off, shape))
    ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
    try:
        one = mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off[:2], shape))
    finally:
        ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
    assert np.array_equal(m, one * np.uint64(nf))


def paths_of(ctx, call):
    """call()'s result, and the engine passes it took by the walk, by strips and by region tiles."""
    before = ctx.pair_paths()
    out = call()
    return out, tuple(b - a for a, b in zip(before, ctx.pair_paths()))


def many_frames(rows, cols, dist, edge, nf=800, mean=1000, seed=1):
    import incohautocorrelate_amd as iac

    rng = np.random.default_rng(seed)
    km, _, _, mq = iac.calc_kmap(iac.generate_pixel_map(rows, cols, 75.0, [0, 0, dist], (1, 0, 0), (0, 1, 0)))
    n = rng.integers(mean - 200, mean + 201, nf)
    n[3] = 0
    off = np.concatenate([[0], np.cumsum(n)])
    pix = rng.integers(0, rows * cols, off[-1])
    return km, iac.mesh_shape_big(mq, edge), pix, rng.integers(1, 5, off[-1]), off


@pytest.mark.parametrize("rows,cols,dist,edge", [(128, 128, 2e5, 63), (60, 200, 1e5, 95), (400, 64, 4e5, 191),
                                                 (700, 300, 5e5, 255), (512, 512, 5e5, 255)])
@pytest.mark.parametrize("rotated", [False, True])
def test_strips_of_several_distances(ctx, dev, rows, cols, dist, edge, rotated):
    """Runs whose tasks hold two to eight distances (one where the first detector is not rotated),
    strips along either axis, taken by strips and equal to the tile kernel in every voxel."""
    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    km, shape, pix, cnt, off = many_frames(rows, cols, dist, edge)
    rots = W.random_rotations(off.size - 1, 7).astype(np.float32) if rotated else None
    got, paths = paths_of(ctx, lambda: mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off, shape, rots=rots)))
    assert paths == (0, 1, 0)
    ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
    try:
        ref = mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off, shape, rots=rots))
    finally:
        ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
    assert np.array_equal(got, ref)


def test_strips_bright_rows_take_strips(ctx, dev):
    """The nine frames of a block still go by strips, in two flushes; the frame that fills the box
    alone goes by the walk."""
    from gpu_helpers import gpu_batch

    for name, want in (("frames", (0, 1, 0)), ("frame", (1, 0, 0))):
        km, shape, pix, cnt, nf = bright_rows(name)
        off = np.arange(nf + 1) * pix.size
        call = lambda: gpu_batch(ctx, dev, km, np.tile(pix, nf), np.tile(cnt, nf), off, shape)  # noqa: E731
        assert paths_of(ctx, call)[1] == want, name


def test_captured_strips_follow_the_counts(ctx, dev):
    """A captured batch on strips whose counts change between replays, with work in between: one
    too large for the strips sends that replay by the walk, the next goes by strips again."""
    import torch

    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    km, shape, pix, cnt, off = many_frames(60, 200, 1e5, 95)
    d_cnt = to_dev(cnt.astype(np.uint16), dev)
    batch = ctx.ac3d_batch(to_dev(km, dev), to_dev(pix.astype(np.uint32), dev), d_cnt,
                           to_dev(off.astype(np.uint64), dev), int(off[-1]), shape)
    m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
    try:
        batch.capture(m, zero_mesh=True)
        for top, want in ((4, (0, 1, 0)), (200, (1, 0, 0)), (4, (0, 1, 0)), (129, (0, 1, 0)), (130, (1, 0, 0))):
            c = cnt.copy()
            c[c.size // 3] = top
            d_cnt.copy_(to_dev(c.astype(np.uint16), dev))
            torch.cuda.synchronize()
            got, paths = paths_of(ctx, lambda: batch.launch(m, zero_mesh=True) or mesh_np(m))
            assert paths == want, top
            ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
            try:
                ref = mesh_np(gpu_batch(ctx, dev, km, pix, c, off, shape))
            finally:
                ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
            assert np.array_equal(got, ref), top
    finally:
        batch.destroy()


def test_batch_prepared_on_strips_follows_options_set_later(ctx, dev):
    """An engine option set between a batch's creation and its launch names the walk that takes it,
    and clearing it brings the strips back; the same mesh each time."""
    import torch

    import incohautocorrelate_amd as iac

    km, shape, pix, cnt, off = many_frames(60, 200, 1e5, 95)
    batch = ctx.ac3d_batch(to_dev(km, dev), to_dev(pix.astype(np.uint32), dev), to_dev(cnt.astype(np.uint16), dev),
                           to_dev(off.astype(np.uint64), dev), int(off[-1]), shape)
    m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
    ref = None
    try:
        for mode, want in ((0, (0, 1, 0)), (1, (1, 0, 0)), (2, (1, 0, 0)), (0, (0, 1, 0))):
            ctx.set_option(iac.OPT_PAIR_MODE, mode)
            got, paths = paths_of(ctx, lambda: batch.launch(m, zero_mesh=True) or mesh_np(m))
            ref = got if ref is None else ref
            assert paths == want, mode
            assert np.array_equal(got, ref), mode
    finally:
        ctx.set_option(iac.OPT_PAIR_MODE, 0)
        batch.destroy()


def test_strips_leave_the_run_to_the_walk_where_memory_is_short(dev):
    """A work buffer that holds the walk's records but not the strips' beside them: the same mesh by
    the walk, from one call and from a prepared batch; a buffer too small for either is an error,
    after which the context works on."""
    import torch

    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    km, shape, pix, cnt, off = many_frames(60, 200, 1e5, 95)
    n = int(off[-1])
    c = iac.Context(0)
    try:
        call = lambda: mesh_np(gpu_batch(c, dev, km, pix, cnt, off, shape))  # noqa: E731
        ref, paths = paths_of(c, call)
        assert paths == (0, 1, 0)
        c.close()
        c = iac.Context(0)
        c.set_option(iac.OPT_BUFFER_LIMIT, 24 * n)
        got, paths = paths_of(c, call)
        assert paths == (1, 0, 0) and np.array_equal(got, ref)
        m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
        c.set_option(iac.OPT_BUFFER_LIMIT, 24 * n + 8 * m.numel())  # a batch keeps its half mesh beside them
        batch = c.ac3d_batch(to_dev(km, dev), to_dev(pix.astype(np.uint32), dev), to_dev(cnt.astype(np.uint16), dev),
                             to_dev(off.astype(np.uint64), dev), n, shape)
        got, paths = paths_of(c, lambda: batch.launch(m) or mesh_np(m))
        batch.destroy()
        assert paths == (1, 0, 0) and np.array_equal(got, ref)
        c.close()
        c = iac.Context(0)
        c.set_option(iac.OPT_BUFFER_LIMIT, 17 * n // 2)
        with pytest.raises(iac.IACError):
            call()
        c.set_option(iac.OPT_BUFFER_LIMIT, 0)
        assert np.array_equal(call(), ref)
    finally:
        c.close()


def test_tuner_leaves_strips_and_tiles_reachable(dev):
    """A prefix too short for strips does not keep them from the whole batch, and settings tuned on
    AC_uw do not keep region tiles from C(q); an engine option set by the caller does both."""
    import torch

    import incohautocorrelate_amd as iac

    km, shape, pix, cnt, off = many_frames(60, 200, 1e5, 95)
    d_km, d_off = to_dev(km, dev), to_dev(off.astype(np.uint64), dev)
    d_pix, d_cnt = to_dev(pix.astype(np.uint32), dev), to_dev(cnt.astype(np.uint16), dev)
    small = iac.mesh_shape_small_cofq(iac.calc_kmap(iac.generate_pixel_map(60, 200, 75.0, [0, 0, 1e5], (1, 0, 0),
                                                                           (0, 1, 0)))[3], 31)
    img = to_dev(W.gamma_frames(60 * 200, 1, 1.0, 0.5, seed=2)[0], dev)
    m = torch.zeros(shape.size_ab ** 2 * shape.size_c, dtype=torch.int64, device=dev)
    cq = torch.zeros(small.size_ab ** 2 * small.size_c, dtype=torch.int64, device=dev)
    c = iac.Context(0)
    batch = lambda: c.ac3d_sparse_batch(d_km, d_pix, d_cnt, d_off, int(off[-1]), shape, m)  # noqa: E731
    image = lambda: c.cq_small(d_km, img, small, cq, 0, 1e6)  # noqa: E731
    try:
        c.ac3d_tune(d_km, d_pix, d_cnt, d_off, shape, 0, 0, True, prefix_frames=20)
        assert paths_of(c, batch)[1] == (0, 1, 0)
        c.ac3d_tune(d_km, d_pix, d_cnt, d_off, shape, 0, 0, True, prefix_frames=20)  # from the cache
        assert paths_of(c, batch)[1] == (0, 1, 0)
        c.ac3d_tune(d_km, d_pix, d_cnt, d_off, shape, 1, 1, True, prefix_frames=20)  # linear settings
        assert paths_of(c, image)[1] == (0, 0, 1)
        c.set_option(iac.OPT_CELL_VOX, 5)
        assert paths_of(c, batch)[1] == (1, 0, 0)
        assert paths_of(c, image)[1] == (1, 0, 0)
    finally:
        c.close()


def test_strips_with_a_distance_beyond_the_cut_between(ctx, dev):
    """Four panels, each within one strip of 2.18 voxels: the first and the third pair five strips
    apart, both with the second, three and two strips from it, only beyond Max_Q, and with the fourth
    likewise.  A task of up to seven distances must not hold those between."""
    import incohautocorrelate_amd as iac
    from gpu_helpers import gpu_batch

    mq = np.array([0.6, 0.8, 0.004], np.float32)
    shape = iac.mesh_shape_big(mq, 95, 2.0)
    vox, h, n = float(shape.voxel_per_dq), 2.1808762813, 24
    panels = []
    for y0, y1, x0 in ((0, 0.9 * h, 0), (3.05 * h, 3.9 * h, 60), (5.05 * h, 5.9 * h, 0), (0.8 * vox - 0.5, 0.8 * vox, 0)):
        y, x = np.meshgrid(np.linspace(y0, y1, n), np.linspace(x0, x0 + 6, n), indexing="ij")
        panels.append(np.stack([x.ravel(), y.ravel(), 0 * x.ravel()], 1))
    km = (np.concatenate(panels) / vox).astype(np.float32)
    rng = np.random.default_rng(3)
    off = np.arange(801) * 1000
    pix, cnt = rng.integers(0, len(km), off[-1]), rng.integers(1, 4, off[-1])
    rots = W.random_rotations(800, 9).astype(np.float32)
    got, paths = paths_of(ctx, lambda: mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off, shape, rots=rots)))
    assert paths == (0, 1, 0)
    ctx.set_option(iac.OPT_AC3D_KERNEL, 1)
    try:
        ref = mesh_np(gpu_batch(ctx, dev, km, pix, cnt, off, shape, rots=rots))
    finally:
        ctx.set_option(iac.OPT_AC3D_KERNEL, 0)
    assert np.array_equal(got, ref)
