"""The library's own memory and its caller's, most of it on the CPU emulation, whose
"device" memory is the host's."""
import ctypes

import numpy as np
import pytest

import geogram_amd as ga
from geogram_amd._lib import (Stats, VGC_DEVICE_PTRS, VGC_ERR_CAPACITY, VGC_ERR_DEVICE,
                              VGC_NO_NEIGHBORS, VGC_OK)
from geogram_amd import _ptr


class _Arrays:
    """Output arrays of n cells for the C entry, filled with -7."""

    def __init__(self, n):
        self.vol, self.mg, self.farea = np.full(n, -7.0), np.full((n, 3), -7.0), np.full(24 * n, -7.0)
        self.ptr = np.full(n + 1, 7, dtype=np.uint64)
        self.nbr = np.full(24 * n, -7, dtype=np.int32)

    def untouched(self):
        return (np.all(self.vol == -7) and np.all(self.mg == -7) and np.all(self.ptr == 7)
                and self.no_neighbors())

    def no_neighbors(self):
        return bool(np.all(self.nbr == -7) and np.all(self.farea == -7))


def _cells(ctx, x, out, flags=0, mg=None):
    """vgc_cells on "device" arrays."""
    box, st = np.array([0.0, 0, 0, 1, 1, 1]), Stats()
    return ctx.lib.fn("cells")(ctx.ctx, _ptr(x), None, len(x), _ptr(box), 0, VGC_DEVICE_PTRS | flags,
                               _ptr(out.vol), _ptr(out.mg if mg is None else mg), _ptr(out.ptr),
                               _ptr(out.nbr), _ptr(out.farea), len(out.nbr), ctypes.byref(st))


def test_no_neighbors_leaves_the_arrays_alone():
    """A pass without neighbours writes none, also where an earlier pass on the
    same context had some."""
    x = np.random.default_rng(1).random((200, 3))
    ctx = ga.Context.emulated()
    a, b = _Arrays(200), _Arrays(200)
    assert _cells(ctx, x, a) == VGC_OK
    assert _cells(ctx, x, b, VGC_NO_NEIGHBORS) == VGC_OK
    assert np.array_equal(a.vol, b.vol)
    assert b.no_neighbors()
    ctx.close()


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


@pytest.mark.parametrize("flags", [0, VGC_NO_NEIGHBORS])
@pytest.mark.parametrize("copies", [True, False])
def test_a_failed_call_leaves_the_arrays_alone(flags, copies):
    """The caller's arrays are written when every pass has succeeded: whichever
    allocation of a call fails, they hold what they held."""
    x = np.random.default_rng(2).random((300, 3))
    if copies:
        x[:2] = x[2]  # cells for the passes after the first
    failures = 0
    while True:
        ctx, a = ga.Context.emulated(), _Arrays(300)
        ctx.lib.cdll.vgc_emu_fail_alloc(ctx.ctx, failures + 1)
        rc = _cells(ctx, x, a, flags)
        ctx.close()
        if rc == VGC_OK:
            break
        assert rc == VGC_ERR_DEVICE
        assert a.untouched(), f"allocation {failures + 1}"
        failures += 1
    assert failures > 10 and not a.untouched()


def test_outputs_over_inputs():
    """Centroids written over the seeds, as in a Lloyd step in place."""
    x = np.random.default_rng(4).random((500, 3))
    ctx, a, b = ga.Context.emulated(), _Arrays(500), _Arrays(500)
    assert _cells(ctx, x, a) == VGC_OK
    y = x.copy()
    assert _cells(ctx, y, b, mg=y) == VGC_OK
    assert np.array_equal(a.mg, y) and np.array_equal(a.vol, b.vol)
    assert np.array_equal(a.nbr, b.nbr) and np.array_equal(a.farea, b.farea)
    ctx.close()


# what a call may be given: arrays that hold the neighbours or are too small for
# them, only one of the two neighbour arrays, none of the others, arrays at
# addresses that are no multiple of their type
def _check_outputs(ctx, n, case, on_gpu):
    box, st = np.array([0.0, 0, 0, 1, 1, 1]), Stats()
    x = np.random.default_rng(9).random((n, 3))
    r = ctx.cells(x)
    nnz = int(r.nbr_ptr[-1])
    cap = nnz - 1 if case == "too small" else nnz
    off = 4 if case == "unaligned" else 0
    host = {k: np.full(m * s + off + 8, 0xA5, dtype=np.uint8)
            for k, m, s in (("vol", n, 8), ("mg", 3 * n, 8), ("ptr", n + 1, 8), ("nbr", nnz, 4),
                            ("farea", nnz, 8))}
    give = {"no areas": ("vol", "mg", "ptr", "nbr"), "no ids": ("vol", "mg", "ptr", "farea"),
            "areas only": ("farea",)}.get(case, tuple(host))
    xs = x
    if on_gpu:
        import torch
        host = {k: torch.from_numpy(v).cuda() for k, v in host.items()}
        xs = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
    addr = {k: ctypes.c_void_p(_ptr(v).value + off) if k in give else None for k, v in host.items()}
    rc = ctx.lib.fn("cells")(ctx.ctx, _ptr(xs), None, n, _ptr(box), 0, VGC_DEVICE_PTRS, addr["vol"],
                             addr["mg"], addr["ptr"], addr["nbr"], addr["farea"], cap,
                             ctypes.byref(st))
    assert rc == (VGC_ERR_CAPACITY if case == "too small" else VGC_OK)
    assert st.nb_neighbors == nnz
    want = {"vol": r.vol, "mg": r.mg, "ptr": r.nbr_ptr, "nbr": r.nbr, "farea": r.farea}
    for k, v in host.items():
        v = (v.cpu().numpy() if on_gpu else v)[off:]
        if k in give and not (case == "too small" and k in ("nbr", "farea")):
            w = np.ascontiguousarray(want[k]).tobytes()
            assert v[:len(w)].tobytes() == w and np.all(v[len(w):] == 0xA5), k
        else:
            assert np.all(v == 0xA5), k


OUTPUTS = [(n, c) for n in (1, 300) for c in
           ("all", "too small", "no areas", "no ids", "areas only", "unaligned")
           if not (n == 1 and c == "too small")]


@pytest.mark.parametrize("n,case", OUTPUTS)
def test_outputs(emu_ctx, n, case):
    _check_outputs(emu_ctx, n, case, False)


@pytest.mark.gpu
@pytest.mark.parametrize("n,case", [(n if n == 1 else 5001, c) for n, c in OUTPUTS if c != "unaligned"])
def test_outputs_gpu(gpu_ctx, n, case):
    _check_outputs(gpu_ctx, n, case, True)


def test_a_context_after_a_failed_allocation():
    """Buffers that could not grow are gone, not kept as freed ones: smaller
    calls on the same context go on as before, whichever growth failed."""
    rng = np.random.default_rng(6)
    small, large = rng.random((60, 3)), rng.random((900, 3))
    small[0] = small[1]
    ref = ga.Context.emulated()
    want = ref.cells(small)
    ref.close()
    k, failed = 0, True
    while failed:
        k += 1
        ctx = ga.Context.emulated()
        ctx.cells(small)
        ctx.lib.cdll.vgc_emu_watch_frees(ctx.ctx)
        ctx.lib.cdll.vgc_emu_fail_alloc(ctx.ctx, k)
        try:
            ctx.ot_solve(large, np.full(900, 1 / 900), tol=1e-2, max_newton=1)
            failed = False
        except ga.VgcError as e:
            assert e.code == VGC_ERR_DEVICE
        ctx.lib.cdll.vgc_emu_fail_alloc(ctx.ctx, 0)
        got = ctx.cells(small)
        assert np.array_equal(got.vol, want.vol) and np.array_equal(got.nbr, want.nbr)
        assert ctx.lib.cdll.vgc_emu_freed_writes(ctx.ctx) == 0, k
        ctx.close()
    assert k > 20
