"""GPU checks of the measurement probes the bench reports beside the engine: every
atomic add reaches the mesh, in each address pattern."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,hot", [(0, 0), (1, 5000), (3, 0)])
def test_global_atomic_probe_counts_every_add(ctx, dev, mode, hot):
    import torch

    nvox = 65 ** 3
    m = torch.zeros(nvox, dtype=torch.int64, device=dev)
    ms = ctx.probe_atomics(m, 1 << 20, mode, hot)
    assert ms > 0
    assert int(m.sum()) == 1 << 20
    touched = int((m != 0).sum())
    if mode == 1:
        assert touched <= hot
    if mode == 3:
        # runs of 8 on whole 64-byte segments: nothing past the last whole segment
        assert int(m[nvox // 8 * 8:].abs().sum()) == 0


@pytest.mark.parametrize("mode", [2, 4])
def test_lds_atomic_probe_flushes_its_boxes(ctx, dev, mode):
    import torch

    nvox = 65 ** 3
    m = torch.zeros(nvox, dtype=torch.int64, device=dev)
    ctx.probe_atomics(m, 1 << 20, mode, 0)
    total = int(m.sum())
    assert 0 < total <= 1 << 20


def test_lds_probe_is_a_ceiling(ctx, dev):
    """The engine's own LDS adds stay below the probe's rate: AC1D's linear C(q) makes two uint64 adds
    per unordered pair, at random addresses too (2.2e12/s, where the probe hashed its addresses at 1.7e12/s)."""
    import torch

    import incohautocorrelate_amd as iac
    from gpu_helpers import to_dev
    from incohautocorrelate_amd import workloads as W

    m = torch.zeros(65 ** 3, dtype=torch.int64, device=dev)
    rate = max((1 << 32) / (ctx.probe_atomics(m, 1 << 32, 2, 0) * 1e-3) for _ in range(3))
    _, km, mq = W.detector(256)
    max_q, dq = iac.ac1d_shape(mq, 4096)
    img = to_dev(W.gamma_frames(256 * 256, 1, 1.0, 0.5, seed=3)[0], dev)
    d_km, h = to_dev(km, dev), torch.zeros(4096, dtype=torch.int64, device=dev)
    ctx.enable_timing(True)
    try:
        best = 0.0
        for _ in range(4):
            ctx.kernel_time(reset=True)
            ctx.ac1d_cq(d_km, img, 4096, max_q, dq, 1, 1e5, h)
            best = max(best, 2 * (65536 * 65537 / 2) / (ctx.kernel_time(reset=True)[0] * 1e-3))
    finally:
        ctx.enable_timing(False)
    assert best < rate, (best, rate)
