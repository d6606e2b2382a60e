"""Major-cycle pieces on the device (current/tMajorACC/tMajorACC.cc) against
the oracle: the shifted FFT and fftFix (FP32 transform vs numpy's FP64 one,
max|d|/max|ref| <= 1e-5), findPeak and Hogbom CLEAN (bit-exact: same float
operations in the same order per pixel), the visibility subtraction
(bit-exact), PSF gridding (<= 1e-5) and one small end-to-end cycle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
import tcv
from helpers import rel_err, small_problem
from tcv import major as M

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _img(rng, g, real=False):
    a = rng.standard_normal((g, g))
    if not real:
        a = a + 1j * rng.standard_normal((g, g))
    return a.astype(np.complex64)


@pytest.mark.parametrize("g", [8, 256, 4096])
@pytest.mark.parametrize("forward", [True, False])
def test_fft_exec_vs_oracle(ctx, g, forward):
    rng = np.random.default_rng(g + forward)
    x = _img(rng, g)
    d = ctx.to_device(x)
    M.fftExec(ctx, d, g, forward)
    assert rel_err(d.download(), O.fft_exec(x, forward)) <= TOL


def test_fft_exec_fix_and_fix_alone(ctx):
    g = 512
    rng = np.random.default_rng(9)
    x = _img(rng, g)
    scale = 1.0 / 12345.0
    want = O.fft_fix(O.fft_exec(x, False).astype(np.complex64), scale)
    d = ctx.to_device(x)
    M.fftExecFix(ctx, d, g, False, scale)
    got = d.download()
    assert np.all(got.imag == 0)
    assert rel_err(got, want) <= TOL
    d2 = ctx.to_device(x)
    M.fftFix(ctx, d2, scale)
    assert np.array_equal(d2.download(), O.fft_fix(x, scale))


def test_fft_rejects_odd_size(ctx):
    d = ctx.zeros((7, 7), np.complex64)
    with pytest.raises(tcv.TcvError):
        M.fftExec(ctx, d, 7, True)


def test_find_peak_bitexact(ctx):
    rng = np.random.default_rng(10)
    for g in (1, 33, 1024):
        x = _img(rng, g)
        assert M.findPeak(ctx, ctx.to_device(x)) == O.find_peak(x)
    z = np.zeros((64, 64), np.complex64)
    assert M.findPeak(ctx, ctx.to_device(z)) == (0.0, 0)
    z.flat[100] = -3.0
    z.flat[2000] = 3.0
    z.flat[4000] = 2.0 + 9j
    assert M.findPeak(ctx, ctx.to_device(z)) == O.find_peak(z) == (-3.0, 100)


def _dirty_and_psf(seed, g, nSrc=30):
    """A dirty image and PSF with realistic structure: point sources convolved
    with a PSF that has sidelobes, peak at the centre."""
    rng = np.random.default_rng(seed)
    yy, xx = np.mgrid[0:g, 0:g]
    c = g // 2
    r2 = ((xx - c) ** 2 + (yy - c) ** 2) / (g / 16) ** 2
    psf = (np.exp(-r2) + 0.2 * np.cos(0.9 * (xx - c)) * np.exp(-r2 / 9)).astype(np.float32)
    psf /= psf[c, c]
    sky = np.zeros((g, g), np.float32)
    for _ in range(nSrc):
        sky[rng.integers(g), rng.integers(g)] += rng.uniform(-1, 2)
    dirty = np.real(np.fft.ifft2(np.fft.fft2(sky) * np.fft.fft2(np.fft.ifftshift(psf))))
    return dirty.astype(np.complex64), psf.astype(np.complex64)


@pytest.mark.parametrize("g,niters", [(64, 50), (512, 200)])
def test_hogbom_bitexact(ctx, g, niters):
    dirty, psf = _dirty_and_psf(g, g)
    model0 = np.zeros_like(dirty)
    model0[3, 4] = 0.5 + 0.25j                       # the model accumulates
    r_ref, m_ref, (pv, pp), (dv, dp) = O.deconvolve(dirty, psf, model0, niters, 0.1)
    d_res, d_psf, d_model = ctx.to_device(dirty), ctx.to_device(psf), ctx.to_device(model0)
    (gpv, gpp), (gdv, gdp) = M.deconvolve(ctx, d_res, g, d_psf, g, d_model, niters, 0.1)
    assert (gpv, gpp) == (pv, pp)
    assert (gdv, gdp) == (dv, dp)
    assert np.array_equal(d_res.download(), r_ref)
    assert np.array_equal(d_model.download(), m_ref)


@pytest.mark.parametrize("g,pw", [(96, 40), (101, 37)])
def test_hogbom_small_psf_and_off_diagonal_peak(ctx, g, pw):
    """PSF narrower than the image, with its peak off the diagonal: the
    reference's row offset (ry - px) is reproduced, rows it would read outside
    the PSF are skipped, exactly as the oracle does.  Widths that are a
    multiple of four take the four-pixel path, others the one-pixel path."""
    rng = np.random.default_rng(12 + g)
    dirty = _img(rng, g, real=True)
    psf = (0.1 * _img(rng, pw, real=True)).astype(np.complex64)
    psf[9, 23] = 5.0                                   # peak at px=23, py=9
    r_ref, m_ref, pk_ref, dk_ref = O.deconvolve(dirty, psf, None, 60, 0.1)
    d_res, d_psf, d_model = ctx.to_device(dirty), ctx.to_device(psf), ctx.zeros((g, g), np.complex64)
    pk, dk = M.deconvolve(ctx, d_res, g, d_psf, pw, d_model, 60, 0.1)
    assert (pk, dk) == (pk_ref, dk_ref)
    assert np.array_equal(d_res.download(), r_ref)
    assert np.array_equal(d_model.download(), m_ref)


@pytest.mark.parametrize("g,niters", [(64, 1024), (64, 1025), (37, 2100), (300, 0)])
@pytest.mark.parametrize("peaks", [True, False])
def test_hogbom_many_iterations(ctx, g, niters, peaks):
    """Up to and beyond the iterations of one launch, most of them at pixels that
    earlier ones cleaned; and none."""
    dirty, psf = _dirty_and_psf(g + niters, g, nSrc=5)
    model0 = np.full_like(dirty, 0.125 - 1j)
    r_ref, m_ref, pk_ref, _ = O.deconvolve(dirty, psf, model0, niters, 0.1)
    dk_ref = O.find_peak(dirty)   # (the oracle's loop notes it in its first iteration)
    d_res, d_psf, d_model = ctx.to_device(dirty), ctx.to_device(psf), ctx.to_device(model0)
    got = M.deconvolve(ctx, d_res, g, d_psf, g, d_model, niters, 0.1, peaks=peaks)
    assert got == ((pk_ref, dk_ref) if peaks else None)
    assert np.array_equal(d_res.download(), r_ref)
    assert np.array_equal(d_model.download(), m_ref)


@pytest.mark.parametrize("g,niters", [(64, 50), (101, 1500)])
def test_hogbom_wait_limit(g, niters):
    """A loop whose workgroups may not wait for each other at all: a call that asks
    for the peaks finishes by one launch an iteration, one that doesn't reports it
    at the next waiting call and leaves residual and model alone."""
    dirty, psf = _dirty_and_psf(g, g)
    model0 = np.full_like(dirty, 0.5)
    r_ref, m_ref, pk_ref, dk_ref = O.deconvolve(dirty, psf, model0, niters, 0.1)
    with tcv.Context(0) as c:
        d_psf = c.to_device(psf)
        c.set_wait_limit(0)
        d_res, d_model = c.to_device(dirty), c.to_device(model0)
        assert M.deconvolve(c, d_res, g, d_psf, g, d_model, niters, 0.1) == (pk_ref, dk_ref)
        assert np.array_equal(d_res.download(), r_ref)
        assert np.array_equal(d_model.download(), m_ref)
        for waiting in (c.sync, lambda: d_res.download(), lambda: M.findPeak(c, d_psf)):
            d_res, d_model = c.to_device(dirty), c.to_device(model0)
            M.deconvolve(c, d_res, g, d_psf, g, d_model, niters, 0.1, peaks=False)
            with pytest.raises(tcv.TcvError, match="hogbom"):
                waiting()
            c.sync()   # reported once
            assert np.array_equal(d_res.download(), dirty)
            assert np.array_equal(d_model.download(), model0)
        c.set_wait_limit(1 << 24)
        M.deconvolve(c, d_res, g, d_psf, g, d_model, niters, 0.1, peaks=False)
        assert np.array_equal(d_res.download(), r_ref)
        assert np.array_equal(d_model.download(), m_ref)


def test_hogbom_twice_reuses_workspace(ctx):
    dirty, psf = _dirty_and_psf(5, 128)
    for niters in (30, 7):
        r_ref, m_ref, _, _ = O.deconvolve(dirty, psf, None, niters, 0.1)
        d_res = ctx.to_device(dirty)
        d_model = ctx.zeros((128, 128), np.complex64)
        M.deconvolve(ctx, d_res, 128, ctx.to_device(psf), 128, d_model, niters, 0.1, peaks=False)
        assert np.array_equal(d_res.download(), r_ref)
        assert np.array_equal(d_model.download(), m_ref)


def test_vis_subtract_bitexact(ctx):
    rng = np.random.default_rng(13)
    for n in (1, 1000, 1 << 20):
        a = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
        b = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
        d = ctx.to_device(a)
        M.subtractVis(ctx, d, ctx.to_device(b))
        assert np.array_equal(d.download(), O.vis_subtract(a, b))


def test_psf_gridding_vs_oracle(ctx):
    Sz, gSize = 65, 384
    iu, iv, co, _, C = small_problem(14, 3000, gSize, Sz)
    vis = tcv.Visibilities(ctx, iu, iv, co, [Sz], gSize, C.size)
    plan = tcv.Plan(ctx, vis)
    g = ctx.zeros((gSize, gSize), np.complex64)
    M.gridKernel(ctx, plan, None, ctx.to_device(C), g, isPSF=True)
    ones = np.ones(iu.size, np.complex64)
    assert rel_err(g.download(), O.grid(ones, iu, iv, co, C, gSize, Sz)) <= TOL


def test_major_cycle_small_vs_oracle(ctx):
    """Two cycles of tMajorACC's loop at a small size, every stage compared
    with the oracle chain started from the same visibilities."""
    mc = M.MajorCycle(ctx, nSamples=3000, wSize=9, nChan=1, cellSize=5.0, gSize=512,
                      baseline=200, nMajor=2, nMinor=20, nSources=25)
    s = 2 * mc.support + 1
    iu, iv, co = mc.vis.iu.download(), mc.vis.iv.download(), mc.vis.cOffset.download()
    C = mc.C.download()
    data = mc.data.download()
    # the visibilities are the degridded FFT of the true sky
    sky_grid = O.fft_exec(mc.sky, True).astype(np.complex64)
    assert rel_err(data, O.degrid(sky_grid, iu, iv, co, C, s)) <= 1e-4
    scale = np.float32(1.0 / float(mc.nVis))
    psf_img = O.fft_fix(O.fft_exec(O.grid(np.ones_like(data), iu, iv, co, C, 512, s), False)
                        .astype(np.complex64), scale)
    d = data.copy()
    for it in range(2):
        mc.cycle(it)
        if it == 0:
            assert rel_err(mc.psf.download(), psf_img) <= TOL
        img = O.fft_fix(O.fft_exec(O.grid(d, iu, iv, co, C, 512, s), False).astype(np.complex64),
                        scale)
        _, model, _, _ = O.deconvolve(img, psf_img, None, 20, 0.1)
        mg = O.fft_exec(model, True).astype(np.complex64)
        mvis = O.degrid(mg, iu, iv, co, C, s)
        d = O.vis_subtract(d, mvis)
        # same clean components, values within the FFT's rounding
        got_model_vis = mc.model_vis.download()
        assert rel_err(got_model_vis, mvis) <= 1e-4, it
        assert rel_err(mc.data.download(), d) <= 1e-4, it


@pytest.mark.parametrize("g", [256, 512, 1024, 2048])
@pytest.mark.parametrize("forward", [True, False])
def test_fft_power_of_two_passes(ctx, g, forward):
    """Every length of the two-pass transform, and its fftFix output.  FP32
    rounding of about 2 log2(g) butterfly levels, each within 2^-23 of values
    that grow with the transform, stays below 40 x 2^-23 = 4.8e-6 of the maximum."""
    rng = np.random.default_rng(2 * g + forward)
    x = _img(rng, g)
    want = O.fft_exec(x, forward)
    d = ctx.to_device(x)
    M.fftExec(ctx, d, g, forward)
    assert rel_err(d.download(), want) <= 4.8e-6
    d = ctx.to_device(x)
    M.fftExecFix(ctx, d, g, forward, 1.0 / g)
    got = d.download()
    assert np.all(got.imag == 0)
    assert np.abs(got.real - want.real / g).max() <= 4.8e-6 * np.abs(want).max() / g


@pytest.mark.parametrize("g,pw", [(1, 1), (5, 5), (7, 1), (255, 2), (257, 300), (1024, 1024), (1500, 90),
                                  (2051, 2051), (4096, 513), (4099, 64)])
def test_hogbom_image_sizes(ctx, g, pw):
    """The loop kernel's groupings (one, four and 16 rows a thread, rows that are
    no multiple of four, one workgroup and all of them), PSFs of a few pixels,
    wider than the image and off its edge, and an image beyond the loop
    kernel; two pixels tie for the first peak."""
    rng = np.random.default_rng(g + pw)
    dirty = rng.standard_normal((g, g)).astype(np.float32).astype(np.complex64)
    dirty.imag = 2.0
    if g > 4:
        dirty[g - 1, g - 2] = -9.0
        dirty[g // 2, 1] = 9.0
    psf = (0.05 * rng.standard_normal((pw, pw))).astype(np.complex64)
    psf[pw // 3, pw // 2] = 2.0
    niters = 6 if g > 1000 else 300
    r_ref, m_ref, pk_ref, dk_ref = O.deconvolve(dirty, psf, None, niters, 0.1)
    d_res, d_psf, d_model = ctx.to_device(dirty), ctx.to_device(psf), ctx.zeros((g, g), np.complex64)
    pk, dk = M.deconvolve(ctx, d_res, g, d_psf, pw, d_model, niters, 0.1)
    assert (pk, dk) == (pk_ref, dk_ref)
    assert np.array_equal(d_res.download(), r_ref)
    assert np.array_equal(d_model.download(), m_ref)
    assert M.findPeak(ctx, d_res) == O.find_peak(r_ref)


@pytest.mark.parametrize("nSamples,nChan,wSize", [(1, 1, 33), (255, 3, 9000), (70001, 5, 129), (300000, 2, 33)])
def test_offsets_histogram_over_strides(ctx, nSamples, nChan, wSize):
    """Index set-up with fewer and more visibilities than one stride of the
    grid, and more planes than the LDS histogram holds: the offsets, the plane
    counts and the out-of-range count equal the oracle's."""
    rng = np.random.default_rng(nSamples)
    u, v, w = (rng.uniform(-900, 900, nSamples) for _ in range(3))
    freq = (1.4e9 - 2.0e5 * np.arange(nChan) / nChan) / 2.998e8
    cell, wcs, g, os_, s = 5.0, 2.0 * 1000 * freq[0] / wSize, 1024, 8, 9
    du, dv, dw = (ctx.to_device(a) for a in (u, v, w))
    iu, iv, wp, co, npp, bad = tcv.init_offsets(ctx, du, dv, dw, freq, cell, wcs, wSize, g, os_, [s], None,
                                                want_wplane=True, allow_out_of_range=True)
    f = np.tile(freq, nSamples)
    us, vs, ws = (f * np.repeat(a, nChan) / c for a, c in ((u, cell), (v, cell), (w, wcs)))
    a, b = np.floor(us).astype(np.int64), np.floor(vs).astype(np.int64)
    plane = wSize // 2 + np.trunc(ws).astype(np.int64)
    fu, fv = (os_ * (us - a)).astype(np.int64), (os_ * (vs - b)).astype(np.int64)
    iu_r, iv_r = a + g // 2, b + g // 2
    assert np.array_equal(iu.download(), iu_r) and np.array_equal(iv.download(), iv_r)
    assert np.array_equal(wp.download(), plane)
    assert np.array_equal(co.download(), (s * s * (fu + os_ * (fv + os_ * plane))).astype(np.int32))
    ok = (plane >= 0) & (plane < wSize)
    out = ~ok | (iu_r - s // 2 < 0) | (iv_r < 0) | (iu_r - s // 2 + s > g) | (iv_r + s > g)
    assert np.array_equal(npp, np.bincount(plane[ok], minlength=wSize)) and bad == out.sum()
