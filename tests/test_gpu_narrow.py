"""Plans: narrow kernels by regions at every width that a region size is
built for (steps of the walk, odd and even, the widest of a class), grids that
no region divides, the first and last slices of the table, widths mixed with
wider ones, FP16 storage and batches.  Taps are multiples of 1/4 and values
small integers, so every sum is exact and results equal the oracle's.  After them:
work items sized on the device, and the counters and scans of the plan's build."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tcv

pytestmark = pytest.mark.gpu


def job(seed, widths, nVis, gSize, os_=2):
    """Exact inputs with plane k of width widths[k]; the last visibilities lie on
    the table's first and last slices, at the grid's corners."""
    rng = np.random.default_rng(seed)
    w = np.asarray(widths, np.int32)
    size = w.astype(np.int64) ** 2 * os_ * os_
    start = np.concatenate([[0], np.cumsum(size)])
    plane = rng.integers(0, w.size, nVis).astype(np.int32)
    plane[-4:] = (0, 0, w.size - 1, w.size - 1)
    s = w[plane]
    cell = rng.integers(0, os_ * os_, nVis)
    cell[-4:] = (0, 0, os_ * os_ - 1, os_ * os_ - 1)
    co = (start[plane] + cell * s * s).astype(np.int32)
    half = s // 2
    u0 = (rng.random(nVis) * (gSize - s + 1)).astype(np.int32)
    v0 = (rng.random(nVis) * (gSize - s + 1)).astype(np.int32)
    u0[-4:], v0[-4:] = (0, gSize - s[-3], 0, gSize - s[-1]), (0, gSize - s[-3], gSize - s[-2], 0)
    cplx = lambda n, d: ((rng.integers(-4, 5, n) + 1j * rng.integers(-4, 5, n)) / d).astype(np.complex64)
    return dict(w=w, plane=plane, co=co, iu=u0 + half, iv=v0, C=cplx(int(start[-1]), 4),
                data=cplx(nVis, 1), grid=cplx(gSize * gSize, 1).reshape(gSize, gSize), gSize=gSize)


def visibilities(ctx, j):
    up = ctx.to_device
    return tcv.Visibilities(ctx, up(j["iu"]), up(j["iv"]), up(j["co"]), j["w"], j["gSize"], j["C"].size,
                            wPlane=up(j["plane"]))


def reference(j):
    pick = np.asarray([k for k in range(j["iu"].size) if j.get("ok") is None or j["ok"][k]])
    args = j["iu"][pick], j["iv"][pick], j["co"][pick], j["C"]
    g = O.grid(j["data"][pick], *args, j["gSize"], j["w"], wPlane=j["plane"][pick])
    o = np.zeros(j["iu"].size, np.complex64)
    o[pick] = O.degrid(j["grid"], *args, j["w"], wPlane=j["plane"][pick])
    return g, o


def run(ctx, plan, j):
    g = ctx.zeros((j["gSize"], j["gSize"]), np.complex64)
    plan.grid(ctx.to_device(j["data"]), ctx.to_device(j["C"]), g)
    out = ctx.empty(j["iu"].size, np.complex64)
    plan.degrid(ctx.to_device(j["grid"]), ctx.to_device(j["C"]), out)
    return g.download(), out.download()


@pytest.mark.parametrize("widths,nVis,gSize", [
    ([2], 700, 33), ([3, 4], 2000, 65), ([5], 1, 7), ([7, 9, 8], 3000, 257), ([10, 11], 1500, 64),
    ([12, 15], 2500, 127), ([16], 1025, 96), ([17, 18, 19], 4000, 200), ([19], 129, 19),
    ([20, 21], 600, 61), ([22, 23], 3000, 130), ([24, 27], 2000, 255), ([28, 31], 2500, 100), ([30], 65, 30),
    ([2, 9, 14, 19, 20, 31], 5000, 150), ([9, 19, 25, 40, 63], 4000, 201), ([7, 97], 2000, 300),
    ([21, 33], 1500, 128)])
def test_regions_equal_oracle(ctx, widths, nVis, gSize):
    j = job(sum(widths) + nVis, widths, max(nVis, 4) if nVis > 1 else 4, gSize)
    if nVis == 1:
        for k in ("plane", "co", "iu", "iv", "data"):
            j[k] = j[k][-1:]
    gref, oref = reference(j)
    plan = tcv.Plan(ctx, visibilities(ctx, j))
    for _ in range(2):
        g, o = run(ctx, plan, j)
        assert np.array_equal(g, gref)
        assert np.array_equal(o, oref)
        plan.build()
    # the same through tiles
    tiles = tcv.Plan(ctx, visibilities(ctx, j), slice_keys=16)
    g, o = run(ctx, tiles, j)
    assert np.array_equal(g, gref) and np.array_equal(o, oref)


@pytest.mark.parametrize("widths,nVis,near,regions", [
    ([27], 8192, (), 1), ([27], 8193, (), 0), ([27], 9000, (0,), 1), ([21], 30000, (), 0),
    ([9], 9000, (), 1), ([19, 18], 9000, (), 1),          # alone: never thin on so few regions
    ([9, 27], 20000, (), 0), ([9, 27], 20000, (0,), .5), ([9, 27], 20000, (0, 1), 1), ([9, 27], 20000, (1,), 1),
    ([17, 40], 20000, (), 0), ([17, 40], 20000, (0,), .5), ([5, 25, 63], 30000, (0, 2), 1 / 3)])
def test_thin_classes(ctx, widths, nVis, near, regions):
    """Classes whose visibilities lie thinly go to the tiles (`near`: widths whose
    visibilities lie close together); results are exact either way, and after other
    visibilities come into the plan."""
    gSize = 2048
    j = job(nVis + len(near), widths, nVis, gSize)
    rng = np.random.default_rng(nVis)
    for k in near:
        at = np.flatnonzero(j["plane"] == k)
        j["iu"][at], j["iv"][at] = rng.integers(200, 300, (2, at.size))
    gref, oref = reference(j)
    plan = tcv.Plan(ctx, visibilities(ctx, j))
    info = plan.info()
    g, o = run(ctx, plan, j)
    assert np.array_equal(g, gref) and np.array_equal(o, oref)
    # a visibility makes one entry by regions, and four or more of the widest by tiles
    w = j["w"][j["plane"]]
    order = sorted(set(widths))
    by = [w == x for x in order]
    share = {0: [], 1: order, .5: order[:1], 1 / 3: order[:1]}[regions]
    tile_w, tile_h = info["tile_w"], info["tile_h"]
    u0, v0 = j["iu"] - w // 2, j["iv"]
    tiles = ((u0 + w - 1) // tile_w - u0 // tile_w + 1) * ((v0 + w - 1) // tile_h - v0 // tile_h + 1)
    assert info["entries"] == sum(int(m.sum()) if x in share else int(tiles[m].sum()) for x, m in zip(order, by))
    j2 = dict(j, iu=np.ascontiguousarray(j["iu"][::-1]), iv=np.ascontiguousarray(j["iv"][::-1]),
              plane=np.ascontiguousarray(j["plane"][::-1]), co=np.ascontiguousarray(j["co"][::-1]))
    plan.build(visibilities(ctx, j2))
    gref, oref = reference(j2)
    g, o = run(ctx, plan, j2)
    assert np.array_equal(g, gref) and np.array_equal(o, oref)


@pytest.mark.parametrize("widths,nVis,gSize,want", [
    # tile_w, chunk, slice_keys, phases, grid_phases by the rules for tiles
    ([15], 30000, 300, (16, 512, 256, 1, 1)), ([27], 20000, 256, (32, 2048, 256, 1, 1)),
    ([9, 19, 40], 9000, 260, (32, 1024, 2048, 1, 1))])
def test_regions_report_their_tiles(ctx, widths, nVis, gSize, want):
    """info() of a plan with regions is the tuning of the tiles in their place: a plan
    made with it reports the same and computes the same."""
    j = job(nVis, widths, nVis, gSize, os_=16)
    plan = tcv.Plan(ctx, visibilities(ctx, j))
    info = plan.info()
    assert tuple(info[k] for k in ("tile_w", "chunk", "slice_keys", "phases", "grid_phases")) == want
    tuning = {k: v for k, v in info.items() if k not in ("entries", "items", "out_of_range")}
    given = tcv.Plan(ctx, visibilities(ctx, j), **tuning)
    again = given.info()
    assert {k: again[k] for k in tuning} == tuning and again["entries"] > info["entries"]
    gref, oref = reference(j)
    for p in (plan, given):
        g, o = run(ctx, p, j)
        assert np.array_equal(g, gref) and np.array_equal(o, oref)


def test_regions_out_of_range(ctx):
    j = job(5, [9, 25, 65], 900, 140)
    j["iu"][:3], j["iv"][3:6], j["co"][6:9] = 0, 139, j["C"].size
    j["ok"] = np.arange(900) >= 9
    plan = tcv.Plan(ctx, visibilities(ctx, j))
    g, o = run(ctx, plan, j)
    gref, oref = reference(j)
    assert np.array_equal(g, gref) and np.array_equal(o, oref)
    assert plan.info()["out_of_range"] == 9


def test_regions_half_storage(ctx):
    """FP16 holds these values exactly, up to the power-of-two scales."""
    j = job(6, [9, 18, 31, 33], 1200, 110, os_=2)
    starts = np.concatenate([[0], np.cumsum(j["w"].astype(np.int64) ** 2 * 4)])
    Ch = tcv.HalfTable(ctx, ctx.to_device(j["C"]), 4, 0, starts)
    dh = tcv.HalfVis(ctx, ctx.to_device(j["data"]))
    plan = tcv.Plan(ctx, visibilities(ctx, j), tap_bytes=4)
    gref, oref = reference(j)
    g = ctx.zeros((110, 110), np.complex64)
    plan.grid_half(dh, Ch, g)
    out = ctx.empty(1200, np.complex64)
    plan.degrid_half(ctx.to_device(j["grid"]), Ch, out)
    # a stored value is within 2^-12 of itself and FP32 sums add 1e-6: both cells
    # and results are sums whose terms' magnitudes bound the error
    bound = lambda x: 2.5 * 2.0 ** -12 * x + 1e-4
    mag = O.grid(np.full(1200, 8, np.complex64), j["iu"], j["iv"], j["co"],
                 np.full(j["C"].size, 2, np.complex64), 110, j["w"], wPlane=j["plane"]).real
    assert (np.abs(g.download() - gref) <= bound(mag)).all()
    assert (np.abs(out.download() - oref) <= bound(16.0 * j["w"][j["plane"]] ** 2)).all()


def test_regions_keep_non_finite_values_inside(ctx):
    """An infinite tap, value or cell shows in what it belongs to and nowhere else."""
    for s in (9, 25):
        j = job(7 + s, [s], 300, 90)
        n = s * s
        j["co"][:] = np.where(j["co"] == 3 * n, 2 * n, j["co"])   # nobody's slice: all infinite
        j["C"][3 * n:] = np.inf
        j["iu"] = np.minimum(j["iu"], 90 - s - 1 + s // 2)   # nor the last column of the grid
        j["grid"][:, 89] = np.nan
        gref, oref = reference(j)
        plan = tcv.Plan(ctx, visibilities(ctx, j))
        g, o = run(ctx, plan, j)
        assert np.array_equal(g, gref) and np.array_equal(o, oref)
        j["data"][0] = np.inf
        g, _ = run(ctx, plan, j)
        x, y = j["iu"][0] - s // 2, j["iv"][0]
        out = np.ones((90, 90), bool)
        out[y:y + s, x:x + s] = False
        assert np.array_equal(g[out], gref[out]) and not np.isfinite(g[~out]).any()


def test_regions_in_a_batch(ctx):
    """Automatic plans in a batch: jobs by regions, in part and by tiles alone; two
    of them share a grid."""
    from tcv.device import Batch
    jobs = [job(11, [17, 19], 1500, 120), job(12, [31, 16], 900, 120), job(13, [8, 12, 19], 700, 77),
            job(14, [15], 5000, 250)]
    jobs.append(job(15, [9, 40], 800, 130))
    plans = [tcv.Plan(ctx, visibilities(ctx, j), tile_w=16 if j is jobs[0] else 0) for j in jobs]
    with pytest.raises(tcv.TcvError):   # tile shapes differ, as for plans without regions
        Batch(ctx, [(p, ctx.to_device(j["data"]), ctx.to_device(j["C"]),
                     ctx.zeros((j["gSize"],) * 2, np.complex64), None) for p, j in zip(plans, jobs)])
    for pick in ([0, 2, 3], [1], [2, 3], [1, 4]):
        hold = []
        for k in pick:
            j = jobs[k]
            hold.append((plans[k], ctx.to_device(j["data"]), ctx.to_device(j["C"]),
                         ctx.zeros((j["gSize"],) * 2, np.complex64), ctx.empty(j["iu"].size, np.complex64)))
        b = Batch(ctx, hold)
        for _ in range(3):
            for h, k in zip(hold, pick):
                h[3].zero()
            b.run_graph(3)
            for h, k in zip(hold, pick):
                assert np.array_equal(h[3].download(), reference(jobs[k])[0]), k
        for h, k in zip(hold, pick):
            h[3].upload(jobs[k]["grid"])
        b.degrid()
        for h, k in zip(hold, pick):
            assert np.array_equal(h[4].download(), reference(jobs[k])[1]), k
        b.close()


@pytest.mark.parametrize("Sz,gSize,nVis,cluster,os_,planes", [
    (65, 200, 1, 0, 2, 2),            # one entry to a tile
    (65, 1500, 700, 0, 2, 3),         # fewer items than workgroups, one phase
    (129, 400, 2500, 60, 8, 5),       # few tiles: cut to chunks of 32
    (97, 700, 9000, 0, 8, 9),         # phases, one list of work items
    (63, 900, 70000, 0, 8, 33),       # two lists: finer phases for the degridder
    (63, 600, 120000, 12, 4, 4),      # hot tiles
    (49, 1100, 170000, 0, 4, 9)])     # many entries: 128 x 64 tiles below width 89
def test_adaptive_work_items(ctx, Sz, gSize, nVis, cluster, os_, planes):
    """Phases and chunks chosen on the device: exact results, and as many work items
    as a plan with the same numbers given makes."""
    from helpers import small_problem
    iu, iv, co, data, C = small_problem(Sz + nVis, nVis, gSize, Sz, os_=os_, nPlanes=planes, margin=1,
                                        cluster=cluster or None)
    rng = np.random.default_rng(nVis)
    C = ((rng.integers(-1, 2, C.size) + 1j * rng.integers(-1, 2, C.size)) / 4).astype(np.complex64)
    data = (rng.integers(-2, 3, nVis) + 1j * rng.integers(-2, 3, nVis)).astype(np.complex64)
    grid = (rng.integers(-2, 3, (gSize, gSize)) + 1j * rng.integers(-2, 3, (gSize, gSize))).astype(np.complex64)
    vis = tcv.Visibilities(ctx, iu, iv, co, [Sz], gSize, C.size)
    gref, oref = O.grid(data, iu, iv, co, C, gSize, Sz), O.degrid(grid, iu, iv, co, C, Sz)
    plan = tcv.Plan(ctx, vis)
    d_data, d_C, d_grid = ctx.to_device(data), ctx.to_device(C), ctx.to_device(grid)
    for _ in range(2):
        g = ctx.zeros((gSize, gSize), np.complex64)
        plan.grid(d_data, d_C, g)
        out = ctx.empty(nVis, np.complex64)
        plan.degrid(d_grid, d_C, out)
        assert np.array_equal(g.download(), gref)
        assert np.array_equal(out.download(), oref)
        plan.build()
    info = plan.info()
    assert info["tile_w"] == (128 if Sz > 88 or nVis == 170000 else 64)
    given = tcv.Plan(ctx, vis, **{k: info[k] for k in ("tile_w", "tile_h", "chunk", "slice_keys", "phases",
                                                       "grid_phases", "kernel", "degrid_kernel")}).info()
    assert (given["items"], given["entries"], given["phases"], given["chunk"]) == \
        (info["items"], info["entries"], info["phases"], info["chunk"])


def test_regions_in_the_kernel_statistics(ctx):
    """A batch's launches by regions count in its kernel families: two region sizes
    and tiles, of one job each."""
    from tcv.device import Batch
    jobs = [job(k, w, 300, 150) for k, w in enumerate([[15, 31], [31], [9, 40]])]
    hold = [(tcv.Plan(ctx, visibilities(ctx, j)), ctx.to_device(j["data"]), ctx.to_device(j["C"]),
             ctx.zeros((150, 150), np.complex64), ctx.empty(300, np.complex64)) for j in jobs]
    b = Batch(ctx, hold)
    ctx.set_profiling(True)
    try:
        ctx.reset_stats()
        b.grid()
        b.degrid()
        for family in ("grid_batch", "degrid_batch"):
            n, ms = ctx.kernel_stats(family)
            assert n == 3 and ms > 0, family
    finally:
        ctx.set_profiling(False)


@pytest.mark.parametrize("Sz,gSize,nVis,tile_w", [
    (49, 2048, 200000, 128), (71, 2048, 100000, 128), (71, 2816, 200000, 128), (71, 2944, 200000, 64), (49, 4096, 400000, 64),
    (72, 4096, 200000, 128), (72, 4096, 50000, 64), (65, 900, 200000, 64)])
def test_open_tile_shape(ctx, Sz, gSize, nVis, tile_w):
    """128 x 64 tiles from width 72 up, and from 48 up to 1024 of them (2816^2 has
    968, 2944^2 1058), for more than 262 144 entries on 128 and more of them.  A plan
    made for FP16 stays on 64 x 64."""
    rng = np.random.default_rng(Sz)
    iu = rng.integers(Sz, gSize - Sz, nVis).astype(np.int32)
    vis = tcv.Visibilities(ctx, iu, iu, np.zeros(nVis, np.int32), [Sz], gSize, Sz * Sz * 4)
    assert tcv.Plan(ctx, vis).info()["tile_w"] == tile_w
    assert tcv.Plan(ctx, vis, tap_bytes=4).info()["tile_w"] == 64


def test_widened_plans_in_a_batch(ctx):
    """Open plans of one width on either side of the size from which they take
    128 x 64 tiles, beside one given 64 x 64: one batch, two of the jobs on one
    grid.  Given 128 x 64 tiles stay refused."""
    from helpers import exact_problem
    from tcv.device import Batch
    Sz, hold, ref, plans = 49, [], [], []
    grids = {g: ctx.zeros((g, g), np.complex64) for g in (1100, 300)}
    sums = {g: np.zeros((g, g), np.complex64) for g in grids}
    for seed, (nVis, gSize, tuning) in enumerate([(3000, 1100, {}), (140000, 1100, {}), (2000, 300, dict(tile_w=64))]):
        iu, iv, co, data, C, grid = exact_problem(seed, nVis, gSize, Sz, cluster=None)
        plans.append(tcv.Plan(ctx, tcv.Visibilities(ctx, iu, iv, co, [Sz], gSize, C.size), **tuning))
        hold.append((plans[-1], ctx.to_device(data), ctx.to_device(C), grids[gSize], ctx.empty(nVis, np.complex64)))
        ref.append((iu, iv, co, C, grid, gSize))
        O.grid(data, iu, iv, co, C, gSize, Sz, out=sums[gSize])
    assert [p.info()["tile_w"] for p in plans] == [64, 128, 64]
    given = tcv.Plan(ctx, plans[1].vis, tile_w=128)
    for pair in ([(given,) + hold[1][1:], hold[0]], [hold[1], (given,) + hold[1][1:]]):
        with pytest.raises(tcv.TcvError, match="one tile shape"):
            Batch(ctx, pair)
    for pick in ([0, 1, 2], [2, 1, 0]):
        b = Batch(ctx, [hold[k] for k in pick])
        for rep in range(3):   # captured once, replayed
            for g in grids.values():
                g.zero()
            b.run_graph(3)
            for gSize, g in grids.items():
                assert np.array_equal(g.download(), sums[gSize]), (pick, rep)
        b.close()
    for gSize, g in grids.items():   # degridding one image into every job's output
        g.upload(ref[1 if gSize == 1100 else 2][4])
    want = [O.degrid(grids[gSize].download(), iu, iv, co, C, Sz) for iu, iv, co, C, _, gSize in ref]
    for pick in ([0, 1, 2], [1]):
        for h in hold:
            h[4].zero()
        b = Batch(ctx, [hold[k] for k in pick])
        b.rebuild()
        b.degrid()
        for k in pick:
            assert np.array_equal(hold[k][4].download(), want[k]), (pick, k)
        b.close()


@pytest.mark.parametrize("nVis,chunk", [(5000, 32), (100000, 72), (300000, 128)])
def test_adaptive_chunk_of_few_slots(ctx, nVis, chunk):
    """Work items of few tiles in one phase: 1 / 4096 of the entries, from 32 up to
    128 (2.97 entries a visibility here)."""
    from helpers import exact_problem
    Sz, gSize = 33, 300
    iu, iv, co, data, C, grid = exact_problem(nVis, nVis, gSize, Sz, cluster=None)
    vis = tcv.Visibilities(ctx, iu, iv, co, [Sz], gSize, C.size)
    plan = tcv.Plan(ctx, vis)
    info = plan.info()
    assert info["phases"] == info["grid_phases"] == 1
    assert info["chunk"] == chunk == max(32, min(2 * (info["entries"] // 8192), 128))
    g, out = ctx.zeros((gSize, gSize), np.complex64), ctx.empty(nVis, np.complex64)
    plan.grid(ctx.to_device(data), ctx.to_device(C), g)
    plan.degrid(ctx.to_device(grid), ctx.to_device(C), out)
    assert np.array_equal(g.download(), O.grid(data, iu, iv, co, C, gSize, Sz))
    assert np.array_equal(out.download(), O.degrid(grid, iu, iv, co, C, Sz))


def test_adaptive_plan_of_nothing(ctx):
    """Every visibility out of range: no items, cleared results."""
    vis = tcv.Visibilities(ctx, [1, 2], [0, 0], [0, 0], [65], 100, 65 * 65)
    plan = tcv.Plan(ctx, vis)
    info = plan.info()
    assert (info["items"], info["entries"], info["out_of_range"]) == (0, 0, 2)
    C = ctx.to_device(np.ones(65 * 65, np.complex64))
    g = ctx.zeros((100, 100), np.complex64)
    plan.grid(ctx.to_device(np.ones(2, np.complex64)), C, g)
    out = ctx.to_device(np.ones(2, np.complex64))
    plan.degrid(g, C, out)
    assert not g.download().any() and not out.download().any()


@pytest.mark.parametrize("keys,phases,nVis", [(256, 1, 5000), (64, 16, 5000), (16, 1, 300), (1, 1, 70000)])
def test_plan_of_many_counters(ctx, keys, phases, nVis):
    """65 536 tiles: counters and work-item slots beyond one block's scan, up to what
    the following blocks add up themselves, and beyond it."""
    j = job(keys + nVis, [9, 12], nVis, 4096, os_=8)
    gref, oref = reference(j)
    plan = tcv.Plan(ctx, visibilities(ctx, j), tile_w=8, tile_h=32, slice_keys=keys, phases=phases,
                    grid_phases=2 * phases if keys > 16 else phases)
    for _ in range(2):
        g, o = run(ctx, plan, j)
        assert np.array_equal(g, gref) and np.array_equal(o, oref)
        plan.build()


@pytest.mark.parametrize("gSize,keys,lone", [(1500, 3, 0), (1501, 1, 256), (1500, 7, 100)])
def test_plan_counter_remainders(ctx, gSize, keys, lone):
    """Counters in one level, more than a block of the scan and no multiple of a
    thread's 16; the two ends of the part of the table in use are one visibility's
    each, in different blocks of the kernel that notes the range."""
    j = job(gSize + keys, [9, 12], 513, gSize, os_=8)
    j["plane"][:] = 1   # width 12: the table's second part, 64 slices
    first = 9 * 9 * 64
    j["co"] = (first + np.random.default_rng(keys).integers(20, 40, 513) * 144).astype(np.int32)
    j["co"][lone], j["co"][512] = first, first + 63 * 144
    j["iu"], j["iv"] = np.clip(j["iu"], 6, gSize - 6), np.minimum(j["iv"], gSize - 12)
    gref, oref = reference(j)
    plan = tcv.Plan(ctx, visibilities(ctx, j), tile_w=8, tile_h=32, slice_keys=keys, phases=min(keys, 4),
                    grid_phases=min(keys, 4))
    for _ in range(2):
        g, o = run(ctx, plan, j)
        assert np.array_equal(g, gref) and np.array_equal(o, oref)
        plan.build()
