"""Frame ingest at the edges of its kernels' work split: the frame sums are the reference's serial
float sums bit for bit, whatever the values do to the running sum's binade; the pixel averages at
the edges of the frames read ahead; the hit lists at the edges of slices and words."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def frames_of(kind, npix, rng):
    x = rng.random(npix).astype(np.float32)
    if kind == "analogue":  # grows through many binades, ties among the roundings
        v = x * 3 + 0.1
    elif kind == "ties":  # multiples of 1/8: a sum above 2^21 ties on every other value
        v = np.float32(2.0**21) * (np.arange(npix) == 0) + np.floor(x * 64) / 8
    elif kind == "sparse":
        v = np.where(x < 0.01, 1 + x * 20, 0)
    elif kind == "noise":  # wanders about zero: too many binades, the value-by-value rest
        v = rng.normal(0, 1, npix)
    elif kind == "offset_noise":  # negative values about a growing sum
        v = rng.normal(2, 20, npix)
    elif kind == "negative":
        v = -x * 100
    elif kind == "scales":  # values of every size
        v = np.exp2(rng.integers(-140, 100, npix)) * rng.choice([-1, 1], npix)
    elif kind == "cancel":  # back to exactly zero, then on
        v = np.where(np.arange(npix) % 2, -1, 1) * np.repeat(x[: npix // 2 + 1], 2)[:npix]
    elif kind == "inf":
        v = np.where(np.arange(npix) == npix // 2, np.inf, x)
    elif kind == "nan":
        v = np.where(np.arange(npix) == npix // 2, np.nan, x)
    else:  # powers: the sum sits on a binade's edge
        v = np.where(x < 0.5, 0, np.where(x < 0.75, -1, 1)) * 2.0**-24 + (np.arange(npix) == 0)
    return v.astype(np.float32)


KINDS = ["analogue", "ties", "sparse", "noise", "offset_noise", "negative", "scales", "cancel", "inf", "nan", "edge"]


@pytest.mark.parametrize("npix", [1, 15, 17, 1024, 16384, 16385, 50001])
def test_frame_sums_bit_exact(ctx, dev, npix):
    import torch

    rng = np.random.default_rng(npix)
    fr = np.stack([frames_of(k, npix, rng) for k in KINDS])
    with np.errstate(all="ignore"):
        ref = np.array([np.add.accumulate(f, dtype=np.float32)[-1] if npix > 1 else f[0] + np.float32(0) for f in fr])
        want = ref / np.float32(npix)
    got = torch.zeros(len(KINDS), device=dev)
    avg = torch.zeros(npix, device=dev)
    ctx.average_intensity(torch.from_numpy(fr).to(dev), None, -np.inf, 0.0, avg, got)
    got = got.cpu().numpy()
    same = (got.view(np.int32) == want.view(np.int32)) | (np.isnan(got) & np.isnan(want))
    assert same.all(), [(k, g, w) for k, g, w, s in zip(KINDS, got, want, same) if not s]


@pytest.mark.parametrize("nframes", [1, 7, 8, 9, 21])
@pytest.mark.parametrize("thr,step", [(0.2, 0.0), (0.5, 1.0)])
def test_average_over_frame_counts(ctx, dev, nframes, thr, step):
    """The pixel sequences at the edges of the frames read ahead, in one stack and in two."""
    import torch

    rng = np.random.default_rng(nframes)
    fr = (rng.poisson(0.7, (nframes, 333)) * rng.normal(1, 0.2, (nframes, 333))).astype(np.float32)
    ref, mi, pc = O.average_intensity(fr, thr, step, None)
    avg, g_mi = torch.zeros(333, device=dev), torch.zeros(nframes, device=dev)
    g_pc = torch.zeros(nframes, dtype=torch.int32, device=dev)
    ctx.average_intensity(torch.from_numpy(fr).to(dev), None, thr, step, avg, g_mi, g_pc if step > 0 else None)
    assert np.array_equal(avg.cpu().numpy().view(np.int32), ref.view(np.int32))
    assert np.array_equal(g_mi.cpu().numpy().view(np.int32), mi.view(np.int32))
    if step > 0:
        assert np.array_equal(g_pc.cpu().numpy(), pc)


@pytest.mark.parametrize("npix,nframes", [(1, 3), (63, 2), (65, 5), (2048, 3), (2049, 2), (33000, 2), (16385, 300)])
@pytest.mark.parametrize("fill", [0.0, 0.02, 1.0])
def test_hit_lists_at_slice_edges(ctx, dev, npix, nframes, fill):
    import torch

    rng = np.random.default_rng(npix + nframes)
    fr = np.where(rng.random((nframes, npix)) < fill, rng.random((nframes, npix)) * 5 + 0.6, -1).astype(np.float32)
    if fill > 0:
        fr[:, -1] = 2.5  # the last pixel
        fr[-1, 0] = 0.5  # the threshold itself
    km = rng.normal(size=(npix, 3)).astype(np.float32)
    mask = (rng.random(npix) > 0.1).astype(np.int32)
    rec = torch.zeros((nframes * npix, 4), device=dev)
    off = torch.zeros(nframes + 1, dtype=torch.int64, device=dev)
    for m in (None, mask):
        n = ctx.sparse_hit_list(torch.from_numpy(km).to(dev), torch.from_numpy(fr).to(dev),
                                None if m is None else torch.from_numpy(m).to(dev), 0.5, 0.7, rec, off)
        ref = [O.sparse_hit_list(f, km, 0.5, 0.7, np.ones(npix, np.int32) if m is None else m) for f in fr]
        assert n == sum(len(r) for r in ref)
        assert np.array_equal(off.cpu().numpy(), np.cumsum([0] + [len(r) for r in ref]))
        want = np.concatenate([np.asarray(r, np.float32).reshape(-1, 4) for r in ref])
        assert np.array_equal(rec[:n].cpu().numpy().view(np.int32), want.view(np.int32))


def test_frame_sum_near_2_32_pixels(ctx, dev):
    """The last chunk of a frame whose pixel positions end just below 2^32."""
    import torch

    npix = 2**32 - 300
    fr = torch.zeros(npix, device=dev)
    fr[0], fr[2**31 + 5], fr[-1] = 1.0, 4.0, 2.5
    avg, mean = torch.zeros(npix, device=dev), torch.zeros(1, device=dev)
    ctx.average_intensity(fr.reshape(1, npix), None, 0.0, 0.0, avg, mean)
    assert float(mean[0]) == float(np.float32(7.5) / np.float32(npix))
    assert [float(avg[i]) for i in (0, 2**31 + 5, npix - 1, 77)] == [1.0, 4.0, 2.5, 0.0]
    del fr, avg
    torch.cuda.empty_cache()


@pytest.mark.parametrize("npix", [63, 64, 65, 2560, 4095, 4096, 4097, 9000])
def test_frame_sums_bit_exact_about_the_short_frames(ctx, dev, npix):
    """One wave per frame up to 4,096 pixels, a block of partial chunks beyond."""
    test_frame_sums_bit_exact(ctx, dev, npix)


@pytest.mark.parametrize("rows,cols", [(8, 16), (32, 64), (33, 63), (80, 60)])
def test_photon_counts_of_corrected_frames(ctx, dev, rows, cols):
    """Gain-corrected frames, whose sums are no whole numbers: short frames and longer ones."""
    import torch

    npix, nf = rows * cols, 9
    rng = np.random.default_rng(npix)
    fr = (rng.random((nf, npix)) * 50).astype(np.float32)
    out = torch.zeros((nf, npix), device=dev)
    pc, mi = torch.zeros(nf, dtype=torch.int32, device=dev), torch.zeros(nf, device=dev)
    ctx.ppp_lap(torch.from_numpy(fr).to(dev), out, [], 37.0, gain_only=True, photon_count=pc, mean_intensity=mi)
    want = np.array([int(np.add.accumulate(f, dtype=np.float32)[-1]) for f in out.cpu().numpy()])
    assert np.array_equal(pc.cpu().numpy(), want)
    assert np.array_equal(mi.cpu().numpy(), want.astype(np.float32) / np.float32(npix))
