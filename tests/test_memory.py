"""The library's own memory and its caller's, on the CPU emulation, whose
"device" memory is the host's."""
import numpy as np

import geogram_amd as ga


def test_convex_levels_of_five_seeds():
    """Each buffer of a multilevel solve stays valid for as long as it is used:
    five seeds are fewer doubles than a bounding box has, so a buffer shared
    with the extent of the points would be replaced while the solve holds it."""
    rng = np.random.default_rng(3)
    x, nu = rng.random((5, 3)), np.full(5, 0.2)
    levels = np.array([0, 2, 5])
    ctx = ga.Context.emulated()
    ctx.lib.cdll.vgc_emu_watch_frees(ctx.ctx)
    w, sts = ctx.ot_solve_levels(x, nu, levels, tol=1e-6, convex=True)
    assert ctx.lib.cdll.vgc_emu_freed_writes(ctx.ctx) == 0
    assert all(s["converged"] for s in sts)
    vol = ctx.cells(x, weights=w).vol
    assert np.abs(vol - nu).max() <= 1e-6 * 0.2
    ctx.close()
