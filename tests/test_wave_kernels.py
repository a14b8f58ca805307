"""The wavefront kernels at the edges of their sizes: the FP32 first pass
(1, 2, 4 or 8 cells per wavefront, in halves) against the FP64 first pass,
which writes the same bits; the exact kNN (up to 96 entries by a wavefront, 128
candidates) against brute force; device outputs against host outputs."""
import pathlib
import re

import numpy as np
import pytest

import geogram_amd as ga


def _same_cells(a, b):
    assert np.array_equal(a.vol, b.vol)
    assert np.array_equal(a.mg, b.mg)
    assert np.array_equal(a.nbr_ptr, b.nbr_ptr)
    m = int(a.nbr_ptr[-1])
    assert np.array_equal(a.nbr[:m], b.nbr[:m])
    assert np.array_equal(a.farea[:m], b.farea[:m])


def _seeds(n, kind, seed=3):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3))
    if kind == "clusters":  # cells of many rings beside dense clusters
        k = n // 2
        x[:k] = 0.5 + 0.004 * rng.standard_normal((k, 3))
    elif kind == "copies":  # pairs and triples of coincident seeds, any order
        x = np.concatenate([x[: n // 3], x[: n // 3], x])[:n]
        x = x[rng.permutation(n)]
    elif kind == "shell":  # the seed inside has more than 64 corners
        x = rng.standard_normal((n, 3))
        x = 0.5 + 0.4 * x / np.linalg.norm(x, axis=1)[:, None]
        x[n // 2] = 0.5
    return x


# Of coincident seeds only the one of smallest index has a cell; the first pass
# computes that one itself and leaves the others (the box, by the coincident-seed
# rule).
def _check_copies(ctx, n, weighted):
    x = _seeds(n, "copies")
    w = 0.3 * n ** (-2 / 3) * np.random.default_rng(5).random(n) if weighted else None
    a = ctx.cells(x, weights=w)
    _same_cells(a, ctx.cells(x, weights=w, fp64_first=True))
    copies = n - len(np.unique(x, axis=0))
    assert copies <= a.stats["nb_fp64_redo"] <= copies + n // 20
    assert a.stats["nb_disconnected"] == copies


@pytest.mark.parametrize("n,weighted", [(3, False), (900, False), (900, True), (4500, False)])
def test_first_pass_copies(emu_ctx, n, weighted):
    _check_copies(emu_ctx, n, weighted)


@pytest.mark.gpu
@pytest.mark.parametrize("n,weighted", [(900, True), (4500, False), (160_000, False),
                                        (160_000, True)])
def test_first_pass_copies_gpu(gpu_ctx, n, weighted):
    _check_copies(gpu_ctx, n, weighted)


def _check_first_pass(ctx, n, kind):
    x = _seeds(n, "uniform" if kind == "weighted" else kind)
    w = 3.0 * n ** (-2 / 3) * np.cos(5.0 * x[:, 0]) if kind == "weighted" else None
    a = ctx.cells(x, weights=w)
    b = ctx.cells(x, weights=w, fp64_first=True)
    _same_cells(a, b)
    assert a.stats["nb_failed"] == b.stats["nb_failed"] == 0


# one cell per wavefront up to 4096 cells, then two; trees of one leaf, of
# fewer and of more than 64 and 256 leaves
@pytest.mark.parametrize("n,kind", [
    (1, "uniform"), (2, "uniform"), (3, "weighted"), (17, "uniform"), (129, "shell"),
    (1025, "clusters"), (4096, "uniform"), (4097, "weighted"), (4099, "clusters")])
def test_first_pass_sizes(emu_ctx, n, kind):
    _check_first_pass(emu_ctx, n, kind)


# the lines to 2, 4 and 8 cells per wavefront, odd remainders
@pytest.mark.gpu
@pytest.mark.parametrize("n,kind", [
    (1, "weighted"), (129, "shell"), (4095, "clusters"), (4097, "uniform"), (149_999, "uniform"),
    (150_003, "clusters"), (150_001, "weighted"), (400_007, "uniform")])
def test_first_pass_sizes_gpu(gpu_ctx, n, kind):
    _check_first_pass(gpu_ctx, n, kind)


# instances that meet within a wavefront, of spacings far apart: it starts the
# cells of all of them from the first one's
def _check_batch(ctx, count, weighted, nmax=11):
    rng = np.random.default_rng(11)
    sizes = rng.integers(1, nmax + 1, count)
    scale = 10.0 ** rng.uniform(-4, 4, count)
    x = np.concatenate([s * rng.random((n, 3)) for n, s in zip(sizes, scale)])
    boxes = np.zeros((count, 6))
    boxes[:, 3:] = scale[:, None]
    w = np.repeat(0.05 * scale ** 2, sizes) * rng.random(len(x)) if weighted else None
    a = ctx.cells(x, weights=w, inst_n=sizes, boxes=boxes)
    b = ctx.cells(x, weights=w, inst_n=sizes, boxes=boxes, fp64_first=True)
    _same_cells(a, b)
    assert a.stats["nb_failed"] == 0
    # every instance fills its box
    vol = np.add.reduceat(a.vol, np.concatenate([[0], np.cumsum(sizes)[:-1]]))
    assert np.abs(vol / scale ** 3 - 1.0).max() < 1e-10


@pytest.mark.parametrize("count,weighted", [(100, False), (900, False), (900, True)])
def test_first_pass_batches(emu_ctx, count, weighted):
    _check_batch(emu_ctx, count, weighted)


def test_more_instances_than_16_bits(emu_ctx):
    _check_batch(emu_ctx, 66_000, False, nmax=2)


# 1, 2, 4 and 8 cells per wavefront
@pytest.mark.gpu
@pytest.mark.parametrize("count,weighted", [(100, False), (900, True), (30_000, False),
                                            (30_000, True), (70_000, False)])
def test_first_pass_batches_gpu(gpu_ctx, count, weighted):
    _check_batch(gpu_ctx, count, weighted)


def _check_knn(ctx, n, k, kind):
    x = _seeds(n, "clusters" if kind == "clusters" else "uniform")
    if kind == "lattice":  # ties, by index
        x = np.floor(x * 6) / 6 + 1 / 12
        x = np.unique(x, axis=0)
        n = len(x)
    d = ((x[:, None, :] - x[None, :, :]) ** 2)
    d = d[:, :, 0] + d[:, :, 1] + d[:, :, 2]  # the kernel's order of operations
    idx, d2 = ctx.knn(x, k)
    for i in range(n):
        o = np.lexsort((np.arange(n), d[i]))
        o = o[o != i][:k]
        assert np.array_equal(idx[i, :len(o)], o)
        assert np.array_equal(d2[i, :len(o)], d[i, o])
        assert np.all(idx[i, len(o):] == -1)


# 1 to 96 entries by wavefronts, more by lists; every other point
KNN = [(2, 1, "uniform"), (40, 39, "uniform"), (65, 64, "uniform"), (97, 95, "uniform"),
       (500, 1, "uniform"), (500, 63, "clusters"), (500, 64, "uniform"), (500, 95, "uniform"),
       (500, 96, "clusters"), (500, 16, "lattice")]


@pytest.mark.parametrize("n,k,kind", KNN)
def test_knn_sizes(emu_ctx, n, k, kind):
    _check_knn(emu_ctx, n, k, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,kind", KNN)
def test_knn_sizes_gpu(gpu_ctx, n, k, kind):
    _check_knn(gpu_ctx, n, k, kind)


# queries whose first radius holds far too few points: beside the points, and
# lone points around a dense cluster.  A wavefront finds the radius of each (the
# lists take a thousand times as long for such a query).
def _check_knn_far(ctx, left):
    rng = np.random.default_rng(8)
    u = rng.random((4000, 3))
    x = 0.5 + 0.02 * rng.standard_normal((20000, 3))
    x[:100] = rng.random((100, 3))
    for pts, q, k in [(u, 5.0 + rng.random((500, 3)), 8), (u, 3.0 * rng.random((500, 3)) - 1.0, 16),
                      (x, x[:100], 17), (x, rng.random((200, 3)), 1), (x, rng.random((200, 3)), 96)]:
        idx, d2 = ctx.knn_search(pts, q, k)
        for i in range(len(q)):
            d = (pts - q[i]) ** 2
            d = d[:, 0] + d[:, 1] + d[:, 2]
            o = np.argsort(d, kind="stable")[:k]
            assert np.array_equal(idx[i], o) and np.array_equal(d2[i], d[o])
    if left is not None:
        assert left() <= 5


def test_knn_far(emu_ctx):
    f, c = emu_ctx.lib.cdll.vgc_emu_knn_left, emu_ctx.ctx
    before = f(c)
    _check_knn_far(emu_ctx, lambda: f(c) - before)


@pytest.mark.gpu
def test_knn_far_gpu(gpu_ctx):
    _check_knn_far(gpu_ctx, None)


# outputs written straight into the caller's device arrays: not for a torus,
# and the neighbours only where they fit
@pytest.mark.gpu
@pytest.mark.parametrize("n,kw", [(1, {}), (5001, {}), (5001, {"periodic": True}),
                                  (5001, {"neighbors": False})])
def test_device_outputs(gpu_ctx, n, kw):
    import torch
    x = _seeds(n, "uniform")
    a = gpu_ctx.cells(x, **kw)
    b = gpu_ctx.cells(torch.from_numpy(x).cuda(), **kw)
    assert np.array_equal(a.vol, b.vol.cpu().numpy())
    assert np.array_equal(a.mg, b.mg.cpu().numpy())
    if kw.get("neighbors", True):
        m = int(a.nbr_ptr[-1])
        assert np.array_equal(a.nbr_ptr.astype(np.int64), b.nbr_ptr.cpu().numpy())
        assert np.array_equal(a.nbr[:m], b.nbr[:m].cpu().numpy())
        assert np.array_equal(a.farea[:m], b.farea[:m].cpu().numpy())


def test_tuner_times_the_launch_that_runs():
    """The work-group tuner's sample runs with the cells per wavefront of the
    whole pass (here 2; the sample alone would take 1)."""
    ctx = ga.Context.emulated()
    ctx.lib.cdll.vgc_emu_set_tune_run(ctx.ctx, 8)
    x = _seeds(4100, "uniform")
    a = ctx.cells(x, autotune=True)
    assert a.stats["tuned_waves"] in (1, 4)
    assert ctx.lib.cdll.vgc_emu_pair_groups(ctx.ctx) == 2
    _same_cells(a, ctx.cells(x))
    ctx.close()


def test_profiled_sources_are_all_kernel_sources():
    """The hash that dates a committed profile covers every file with device
    code."""
    from geogram_amd import profiling
    csrc = pathlib.Path(profiling._CSRC)
    device = {f.name for f in csrc.iterdir()
              if re.search(r"__global__|__device__|VGC_HD|VGC_SD", f.read_text())}
    device.discard("backend_emu.cpp")
    assert device <= set(profiling.KERNEL_SOURCES)
    assert set(profiling.KERNEL_SOURCES) <= {f.name for f in csrc.iterdir()}
