"""The phase times of vgc_stats: parts of the call's time, each moment counted
once."""
import numpy as np
import pytest

PHASES = ("t_build_ms", "t_knn_ms", "t_clip_ms", "t_pass_bc_ms", "t_compact_ms")


def _check(ctx, n, device, **kw):
    x = np.random.default_rng(6).random((n, 3))
    x[:20] = 0.5 + 1e-3 * x[:20]  # some cells for the passes after the first
    if device:
        import torch
        x = torch.from_numpy(x).cuda()
    for _ in range(3):  # the last one allocates nothing
        s = ctx.cells(x, **kw).stats
    assert all(s[p] >= 0 for p in PHASES)
    total, parts = s["t_total_ms"], sum(s[p] for p in PHASES)
    # (a microsecond of rounding; the rest of the call is bookkeeping)
    assert 0.8 * total <= parts <= total + 1e-3, {p: s[p] for p in PHASES + ("t_total_ms",)}
    return s


@pytest.mark.parametrize("k0", [0, 32])
def test_phases_add_up(emu_ctx, k0):
    s = _check(emu_ctx, 3000, False, k0=k0)
    assert s["t_build_ms"] > 0 and s["t_clip_ms"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("k0", [0, 32])
def test_phases_add_up_gpu(gpu_ctx, k0):
    s = _check(gpu_ctx, 300_000, True, k0=k0)
    # the events' times lie within the phases
    assert s["t_clip_ms"] >= 0.9 * s["t_clip_a_gpu_ms"] > 0
    assert s["t_pass_bc_ms"] >= 0.9 * s["t_redo_gpu_ms"]
    assert s["t_compact_ms"] > 0.02  # 60 MB of neighbours at 3 TB/s at least
    assert s["t_build_ms"] > 0.05    # a sort of 300k keys and the tree
