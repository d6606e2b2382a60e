"""Work that a user of tcv has it do, as timed cases over the public entry points.

Kinds of case
  job      one gridding job (uniform kernel width): optionally re-bin the
           visibilities, clear the grid, grid, degrid; FP32 or FP16 storage
  current  a run of the current tConvolve generation (ASKAP layout, per-plane
           kernel widths), gridded and degridded
  batch    many uneven jobs in one captured launch (re-bin, grid, degrid)
  fft      the shifted 2-D transform of an image and back, with fftFix
  clean    a Hogbom minor cycle and the residual's peak after it
  offsets  the index set-up of a new snapshot's u, v, w
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "askap-benchmarks_amd"))
import tcv                                     # noqa: E402
from tcv import setup                          # noqa: E402
from tcv.gridder import BatchJobs, init_offsets  # noqa: E402
from tcv.major import deconvolve, fftExec, fftExecFix, findPeak  # noqa: E402

OS = 8                    # oversampling of every uniform table here
F0 = 1.4e9 / 2.998e8      # inverse wavelength of the lowest channel (1/m)
EXACT_POINTS = 4.0e9      # grid points up to which the 64-bit values take seconds


def listed():
    return [
        # a snapshot of a few thousand visibilities with narrow kernels: launches and latency
        dict(name="snapshot_narrow", kind="job", nVis=2000, nChan=1, width=15, planes=9, gSize=512,
             spread=0.9, wfrac=1.0, real=False, half=False, rebin=True),
        # the smallest job with the widest kernels (the smoke test's size)
        dict(name="snapshot_wide", kind="job", nVis=2000, nChan=1, width=129, planes=4, gSize=512,
             spread=1.0, wfrac=1.0, real=False, half=False, rebin=True),
        # mid-sized job of the uneven mix, re-binned for new u, v, w (odd grid)
        dict(name="mid_63", kind="job", nVis=100003, nChan=1, width=63, planes=65, gSize=2047,
             spread=1.0, wfrac=1.0, real=False, half=False, rebin=True),
        # the attic generation's constants: 160 000 visibilities, width 129, 4096^2, 33 planes of
        # which the generator uses the middle half; the plan is kept as Benchmark keeps it
        dict(name="attic", kind="job", nVis=160000, nChan=1, width=129, planes=33, gSize=4096,
             spread=0.49, wfrac=0.5, real=True, half=False, rebin=False),
        # the same with FP16 storage
        dict(name="attic_half", kind="job", nVis=160000, nChan=1, width=129, planes=33, gSize=4096,
             spread=0.49, wfrac=0.5, real=True, half=True, rebin=False),
        # spectral scale: 8 channels, 8.4 M visibilities, re-binned
        dict(name="spectral", kind="job", nVis=8388608, nChan=8, width=129, planes=129, gSize=4096,
             spread=0.97, wfrac=1.0, real=True, half=False, rebin=True),
        # current generation, continuum (widths 7-121) and spectral line (widths 7-19)
        dict(name="current_continuum", kind="current", runType=0, nVis=5443200, rebin=False),
        dict(name="current_line", kind="current", runType=1, nVis=3827520, rebin=True),
        # independent jobs of uneven size in one launch
        dict(name="batch_16", kind="batch", nJobs=16, mix=3, visMin=10000, visMax=500000),
        # the major cycle's neighbours of the gridder
        dict(name="fft_4096", kind="fft", gSize=4096),
        dict(name="clean_4096", kind="clean", width=4096, niter=100),
        # index set-up of 1 M samples x 8 channels
        dict(name="offsets", kind="offsets", nSamples=1048576, nChan=8, planes=129, gSize=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["job", "job", "job", "job", "job", "current", "current", "batch", "fft", "clean",
                       "offsets"])
    if kind == "job":
        width = _log(rng, 3, 65) * 2 + 1
        g = max(_log(rng, 256, 4096), 2 * width + 16 + rng.randrange(64))
        planes = min(rng.choice([1, 5, 9, 33, 65, 129]), int(1.1e9 / (8 * OS * OS * width * width)))
        nChan = rng.choice([1, 1, 1, 3, 8])
        samples = _log(rng, 1000, min(2.0e6, 3.0e10 / width ** 2) / nChan)
        return dict(kind="job", nVis=samples * nChan, nChan=nChan, width=width, planes=planes, gSize=g,
                    spread=rng.choice([0.3, 0.5, 0.9, 1.0]), wfrac=rng.choice([0.5, 1.0]),
                    real=rng.random() < 0.4, half=rng.random() < 0.2, rebin=rng.random() < 0.6)
    if kind == "current":
        rt = rng.choice([0, 0, 1, 1, 3, 4])
        return dict(kind="current", runType=rt, nVis=_log(rng, 20000, 600000 if rt == 4 else 3827520),
                    rebin=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind="batch", nJobs=rng.randrange(2, 25), mix=rng.randrange(1, 1000), visMin=5000,
                    visMax=_log(rng, 20000, 500000))
    if kind == "fft":
        # powers of two, and any other even size
        g = rng.choice([256, 512, 1024, 2048, 4096]) if rng.random() < 0.6 else 2 * _log(rng, 100, 2048)
        return dict(kind="fft", gSize=g)
    if kind == "clean":
        return dict(kind="clean", width=rng.choice([512, 1024, 2048, 4096, _log(rng, 200, 4096)]),
                    niter=_log(rng, 10, 100))
    nChan = rng.choice([1, 4, 8])
    return dict(kind="offsets", nSamples=_log(rng, 1000, 8388608 / nChan), nChan=nChan,
                planes=rng.choice([33, 65, 129]), gSize=rng.choice([1024, 2048, 4096]))


# ---- buffers ------------------------------------------------------------------

@functools.lru_cache(None)
def _ctx():
    return tcv.Context(0)


_TYPE = {np.dtype(np.complex64): "<c8", np.dtype(np.int32): "<i4", np.dtype(np.float64): "<f8"}


class _Interface:
    def __init__(self, a):
        self.a = a   # keeps the buffer alive while the tensor is
        self.__cuda_array_interface__ = dict(shape=tuple(int(n) for n in a.shape), typestr=_TYPE[a.dtype],
                                             data=(a.ptr.value, False), version=2, strides=None)


def _tensor(a):
    """The device buffer as a torch tensor (no copy)."""
    return torch.as_tensor(_Interface(a), device="cuda")


def _device(t):
    """A tensor's values in a device buffer of the library."""
    kind = {torch.complex64: np.complex64, torch.int32: np.int32, torch.float64: np.float64}[t.dtype]
    a = _ctx().empty(tuple(t.shape), kind)
    _tensor(a).copy_(t)
    torch.cuda.synchronize()
    return a


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _gauss(gen, *shape):
    """Complex Gaussian values with E|d|^2 = 1."""
    return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, device="cuda") * math.sqrt(0.5))


# ---- jobs ----------------------------------------------------------------------

def _table(case):
    """C(w) in the attic layout [plane][osj][osi][j][i]: cos (real) or Fresnel
    chirp (complex) per w-plane, a Gaussian on the middle plane."""
    s, planes = case["width"], case["planes"]
    c = (s - 1) // 2
    off = torch.arange(OS, device="cuda", dtype=torch.float64) / OS
    tap = torch.arange(s, device="cuda", dtype=torch.float64) - c
    x = tap.view(1, s) + off.view(OS, 1)                                     # [os][tap]
    r2 = (x ** 2).view(OS, 1, s, 1) + (x ** 2).view(1, OS, 1, s)             # [osj][osi][j][i]
    C = torch.empty((planes, OS, OS, s, s), dtype=torch.complex64, device="cuda")
    for k in range(planes):
        w = k - planes // 2
        if w == 0:
            v = torch.exp(-r2).to(torch.complex128)
        else:
            ph = r2 / (w * math.sqrt(abs(w)) * max(1.0, c / 3.0) / math.sqrt(max(1.0, planes / 2.0)))
            v = torch.cos(ph).to(torch.complex128) if case["real"] else torch.polar(
                torch.exp(-r2 / (0.6 * s) ** 2), ph)
        C[k] = (v * (OS * OS / v.abs().sum())).to(torch.complex64)
    return C.reshape(-1)


def _job_inputs(case, seed):
    g, s, n = case["gSize"], case["width"], case["nVis"]
    gen = _gen(seed)
    samples, chans = n // case["nChan"], case["nChan"]
    uvw = torch.rand(3, samples, 1, generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    f = (1.4e9 + 1.0e6 * torch.arange(chans, device="cuda", dtype=torch.float64)) / 1.4e9
    f = f / f.max()
    R = case["spread"] * (g // 2 - s - 2)
    x = (uvw[0] * f).reshape(-1) * R
    y = (uvw[1] * f).reshape(-1) * R
    w = (uvw[2] * f).reshape(-1) * case["wfrac"]
    iu, iv = torch.floor(x), torch.floor(y)
    fu, fv = (((a - b) * OS).to(torch.int64).clamp(0, OS - 1) for a, b in ((x, iu), (y, iv)))
    plane = torch.floor((w + 1) / 2 * case["planes"]).to(torch.int64).clamp(0, case["planes"] - 1)
    co = s * s * (fu + OS * (fv + OS * plane))
    return ((iu + g // 2).to(torch.int32), (iv + g // 2).to(torch.int32), co.to(torch.int32),
            _gauss(gen, n))


class _Job:
    pass


def _prepare_job(case, seed):
    st, ctx = _Job(), _ctx()
    iu, iv, co, data = _job_inputs(case, seed)
    st.C, st.data = _device(_table(case)), _device(data)
    st.vis = tcv.Visibilities(ctx, _device(iu), _device(iv), _device(co), [case["width"]], case["gSize"],
                              st.C.size)
    st.plan = tcv.Plan(ctx, st.vis, tap_bytes=4) if case["half"] else tcv.Plan(ctx, st.vis)
    if case["half"]:
        st.Ch = tcv.HalfTable(ctx, st.C, case["planes"], case["width"] ** 2 * OS * OS)
        st.dh = tcv.HalfVis(ctx, st.data)
    st.grid = ctx.zeros((case["gSize"],) * 2, np.complex64)
    st.out = ctx.zeros(case["nVis"], np.complex64)
    return st


def _run_job(case, st):
    if case["rebin"]:
        st.plan.build()
    st.grid.zero()
    if case.get("half"):
        st.plan.grid_half(st.dh, st.Ch, st.grid)
        st.plan.degrid_half(st.grid, st.Ch, st.out)
    else:
        st.plan.grid(st.data, st.C, st.grid)
        st.plan.degrid(st.grid, st.C, st.out)


def _grid_degrid64(iu, iv, co, s, data, C, g):
    """Gridding, then degridding of that grid, in complex128; widths s per visibility."""
    u0, v0 = iu.long() - s // 2, iv.long()
    inside = (u0 >= 0) & (v0 >= 0) & (u0 + s <= g) & (v0 + s <= g) & (co >= 0) & (co.long() + s.long() ** 2 <= C.numel())
    if not bool(inside.all()):
        raise ValueError("a footprint or slice lies outside the grid or the table")
    grid = torch.zeros((g * g, 2), dtype=torch.float64, device="cuda")
    out = torch.zeros(iu.numel(), dtype=torch.complex128, device="cuda")
    for fwd in (True, False):
        for width in torch.unique(s).tolist():
            at = torch.nonzero(s == width).reshape(-1)
            t = torch.arange(width, device="cuda")
            cell = (t.view(-1, 1) * g + t.view(1, -1)).reshape(1, -1)
            tap = torch.arange(width * width, device="cuda").view(1, -1)
            step = max(1, int(2.0e7 / width ** 2))
            for b in range(0, at.numel(), step):
                k = at[b:b + step]
                to = ((iv[k].long() * g + iu[k].long() - width // 2).view(-1, 1) + cell).reshape(-1)
                c = C[(co[k].long().view(-1, 1) + tap).reshape(-1)].to(torch.complex128)
                if fwd:
                    v = data[k].to(torch.complex128).view(-1, 1) * c.view(k.numel(), -1)
                    grid.index_add_(0, to, torch.view_as_real(v.reshape(-1)))
                else:
                    v = torch.view_as_complex(grid[to]) * c
                    out[k] = v.view(k.numel(), -1).sum(1)
    return torch.view_as_complex(grid).view(g, g), out


def _halved(v, planes):
    """FP16 storage of complex values: half pairs scaled by their plane's largest component."""
    r = torch.view_as_real(v).reshape(planes, -1)
    scale = r.abs().amax(1, keepdim=True)
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    r = (r / scale).half().double() * scale.double()
    return torch.view_as_complex(r.reshape(-1, 2))


def _exact_job(case, seed):
    if case["nVis"] * case["width"] ** 2 > EXACT_POINTS:
        return None
    iu, iv, co, data = _job_inputs(case, seed)
    C = _table(case)
    if case["half"]:
        C, data = _halved(C, case["planes"]), _halved(data, 1)
    grid, out = _grid_degrid64(iu, iv, co, torch.full_like(iu, case["width"]), data, C, case["gSize"])
    return dict(grid=grid, out=out)


# ---- the current generation -----------------------------------------------------

@functools.lru_cache(None)
def _current_table(rt):
    p = setup.current_params(rt)
    return (p,) + setup.current_initC(p["uvCellSize"], p["wSize"], p["support"], p["overSample"],
                                      p["wCellSize"])


def _current_inputs(case, seed):
    p, sSize, cOffset0, C = _current_table(case["runType"])
    u, v, w = setup.current_uvw(p["baseline"], setup.LCG(1 + int(seed)))
    n = min(case["nVis"], u.size)
    return p, sSize, cOffset0, C, [np.ascontiguousarray(a[:n]) for a in (u, v, w)]


def _prepare_current(case, seed):
    st, ctx = _Job(), _ctx()
    p, sSize, cOffset0, C, uvw = _current_inputs(case, seed)
    d = [ctx.to_device(a) for a in uvw]
    iu, iv, wp, co, _, _ = init_offsets(ctx, *d, setup.current_wavenumber(1), p["uvCellSize"],
                                        p["wCellSize"], p["wSize"], p["gSize"], p["overSample"], sSize,
                                        cOffset0, allow_out_of_range=True)
    st.C = ctx.to_device(C)
    st.data = _device(_gauss(_gen(seed), uvw[0].size))
    st.vis = tcv.Visibilities(ctx, iu, iv, co, sSize, p["gSize"], C.size, wPlane=wp)
    st.plan = tcv.Plan(ctx, st.vis)
    st.grid = ctx.zeros((p["gSize"],) * 2, np.complex64)
    st.out = ctx.zeros(uvw[0].size, np.complex64)
    return st


def _offsets64(u, v, w, f, cell, wCell, wSize, g, over):
    """initCOffset's positions, fractions and planes in FP64."""
    us, vs = f * u / cell, f * v / cell
    a, b = np.floor(us), np.floor(vs)
    plane = wSize // 2 + np.trunc(f * w / wCell).astype(np.int64) if wCell > 0 else np.zeros(u.size, np.int64)
    return (a.astype(np.int64) + g // 2, b.astype(np.int64) + g // 2, (over * (us - a)).astype(np.int64),
            (over * (vs - b)).astype(np.int64), plane)


def _current_points(case):
    # mean taps per visibility of the generator's runs
    return case["nVis"] * {0: 380.0, 1: 86.0, 3: 49.0, 4: 7569.0}[case["runType"]]


def _exact_current(case, seed):
    if _current_points(case) > EXACT_POINTS:
        return None
    p, sSize, cOffset0, C, (u, v, w) = _current_inputs(case, seed)
    f = float(setup.current_wavenumber(1)[0])
    iu, iv, fu, fv, plane = _offsets64(u, v, w, f, p["uvCellSize"], p["wCellSize"], p["wSize"], p["gSize"],
                                       p["overSample"])
    s = sSize.astype(np.int64)[plane]
    co = s * s * (fu + p["overSample"] * fv) + cOffset0[plane]
    g = p["gSize"]
    t = [torch.from_numpy(a).cuda() for a in (iu, iv, co, s)]
    grid, out = _grid_degrid64(*t, _gauss(_gen(seed), u.size), torch.from_numpy(C).cuda(), g)
    return dict(grid=grid, out=out)


# ---- batches --------------------------------------------------------------------

@functools.lru_cache(8)
def _mix(nJobs, mix, lo, hi):
    specs = setup.uneven_batch(nJobs, seed=mix, vis_min=lo, vis_max=hi)
    for sp in specs:
        for k in ("u", "v", "w", "data"):
            del sp[k]   # the sizes are the case's; the values come from the seed
    return specs


def _specs(case):
    return [dict(sp) for sp in _mix(case["nJobs"], case["mix"], case["visMin"], case["visMax"])]


def _prepare_batch(case, seed):
    st = _Job()
    rng = np.random.default_rng(int(seed))
    specs = _specs(case)
    for sp in specs:
        n, B = sp["nVis"], sp["baseline"]
        sp["u"], sp["v"], sp["w"] = (rng.uniform(-B, B, n) for _ in range(3))
        sp["data"] = ((rng.standard_normal(n) + 1j * rng.standard_normal(n)) * math.sqrt(0.5)).astype(np.complex64)
    st.jobs = BatchJobs(_ctx(), specs)
    st.views = [dict(grid=_tensor(j["grid"]), out=_tensor(j["out"])) for j in st.jobs.jobs]
    return st


# ---- image plane ----------------------------------------------------------------

def _prepare_fft(case, seed):
    st = _Job()
    st.img = _device(_gauss(_gen(seed), case["gSize"], case["gSize"]))
    return st


def _clean_inputs(case, seed):
    """A PSF with decaying rings, and the dirty image of 40 sources plus noise."""
    W, gen = case["width"], _gen(seed)
    x = torch.arange(W, device="cuda", dtype=torch.float64) - W // 2
    r = torch.sqrt(x.view(-1, 1) ** 2 + x.view(1, -1) ** 2)
    psf = 0.8 * torch.exp(-(r / 3.0) ** 2) + 0.15 * torch.cos(r / 5.0) * torch.exp(-r / (W / 10.0)) * (r > 0)
    psf[W // 2, W // 2] = 1.0
    sky = torch.zeros((W, W), dtype=torch.float64, device="cuda")
    at = torch.randint(W // 8, W - W // 8, (40, 2), generator=gen, device="cuda")
    sky[at[:, 0], at[:, 1]] = torch.rand(40, generator=gen, device="cuda", dtype=torch.float64) + 0.2
    img = torch.fft.ifft2(torch.fft.fft2(sky) * torch.fft.fft2(torch.roll(psf, (-(W // 2),) * 2, (0, 1)))).real
    img = img + 2e-3 * torch.randn(W, W, generator=gen, device="cuda", dtype=torch.float64)
    return img.to(torch.complex64), psf.to(torch.complex64)


def _prepare_clean(case, seed):
    st = _Job()
    img, psf = _clean_inputs(case, seed)
    st.res, st.psf, st.model = _device(img), _device(psf), _device(torch.zeros_like(img))
    return st


def _exact_clean(case, seed):
    img, psf = _clean_inputs(case, seed)
    W = case["width"]
    res, p = img.real.double(), psf.real.double()
    model = torch.zeros_like(res)
    pk = int(p.abs().argmax())
    px, py = pk % W, pk // W
    first = int(res.abs().argmax())
    peaks = [float(p.view(-1)[pk]), pk, float(res.view(-1)[first]), first]
    gain = float(np.float32(0.1))
    for _ in range(case["niter"]):
        at = int(res.abs().argmax())
        rx, ry = at % W, at // W
        v = gain * float(res.view(-1)[at])
        model.view(-1)[at] += v
        x0, x1 = max(0, rx - px), min(W, rx + W - px)
        y0, y1 = max(0, ry - py), min(W, ry + W - py)
        res[y0:y1, x0:x1] -= v * p[y0 - ry + px:y1 - ry + px, x0 - rx + px:x1 - rx + px]
    at = int(res.abs().argmax())
    z = torch.zeros_like(res)
    return dict(residual=torch.complex(res, z), model=torch.complex(model, z), peaks=peaks,
                peak=[float(res.view(-1)[at]), at])


# ---- index set-up ---------------------------------------------------------------

def _offset_args(case):
    B = 2000
    cell = setup.tightest_cell(B, case["gSize"])
    freq = (1.4e9 - 1.0e6 * np.arange(case["nChan"], dtype=np.float64)) / 2.998e8
    support, wCell, _ = setup.attic_initC(float(freq[0]), cell, case["planes"], B, OS, table=False)
    return B, cell, freq, wCell, 2 * support + 1


def _uvw(case, seed):
    B = _offset_args(case)[0]
    return (torch.rand(3, case["nSamples"], generator=_gen(seed), device="cuda", dtype=torch.float64) * 2 - 1) * B


def _prepare_offsets(case, seed):
    st = _Job()
    st.uvw = [_device(a.contiguous()) for a in _uvw(case, seed)]
    st.args = _offset_args(case)
    return st


# ---- the interface --------------------------------------------------------------

def prepare(case, seed):
    st = dict(job=_prepare_job, current=_prepare_current, batch=_prepare_batch, fft=_prepare_fft,
              clean=_prepare_clean, offsets=_prepare_offsets)[case["kind"]](case, seed)
    st.case = case
    if case["kind"] in ("job", "current"):
        st.views = dict(grid=_tensor(st.grid), out=_tensor(st.out))
    elif case["kind"] == "fft":
        st.views = _tensor(st.img)
    elif case["kind"] == "clean":
        st.views = dict(residual=_tensor(st.res), model=_tensor(st.model))
    return st


def run(st):
    case, ctx = st.case, _ctx()
    kind = case["kind"]
    if kind in ("job", "current"):
        _run_job(case, st)
        return st.views
    if kind == "batch":
        st.jobs.zero_grids()
        st.jobs.run_batched(graph=True)
        return st.views
    if kind == "fft":
        g = case["gSize"]
        fftExec(ctx, st.img, g, True)
        fftExecFix(ctx, st.img, g, False, 1.0 / (float(g) * g))
        return st.views
    if kind == "clean":
        W = case["width"]
        (pv, pp), (dv, dp) = deconvolve(ctx, st.res, W, st.psf, W, st.model, case["niter"], 0.1)
        v, p = findPeak(ctx, st.res)
        return dict(st.views, peaks=[pv, pp, dv, dp], peak=[v, p])
    B, cell, freq, wCell, s = st.args
    iu, iv, _, co, per, bad = init_offsets(ctx, *st.uvw, freq, cell, wCell, case["planes"], case["gSize"],
                                           OS, [s], None, want_wplane=False)
    return dict(iu=_tensor(iu), iv=_tensor(iv), cOffset=_tensor(co), perPlane=per, bad=bad)


def work(case):
    kind = case["kind"]
    if kind == "job":
        pts = float(case["nVis"]) * case["width"] ** 2
        slices = case["planes"] * case["wfrac"] * OS * OS
        table = min(slices, case["nVis"]) * case["width"] ** 2 * (4 if case["half"] else 8)
        return dict(flops=16 * pts, bytes=2 * table + 24.0 * case["gSize"] ** 2 +
                    case["nVis"] * (24 if case["half"] else 40))
    if kind == "current":
        p = setup.current_params(case["runType"])
        table = {0: 311e6, 1: 12e6, 3: 6.4e6, 4: 3.9e6}[case["runType"]]
        return dict(flops=16 * _current_points(case),
                    bytes=2 * table + 24.0 * p["gSize"] ** 2 + case["nVis"] * 48)
    if kind == "batch":
        sp = _specs(case)
        return dict(flops=16.0 * sum(j["nVis"] * j["sSize"] ** 2 for j in sp),
                    bytes=sum(2.0 * min(j["wSize"] * OS * OS, j["nVis"]) * j["sSize"] ** 2 * 8 +
                              24.0 * j["gSize"] ** 2 + 52.0 * j["nVis"] for j in sp))
    if kind == "fft":
        n = float(case["gSize"]) ** 2
        return dict(flops=20 * n * math.log2(case["gSize"]), bytes=32 * n)
    if kind == "clean":
        n = float(case["width"]) ** 2
        return dict(flops=2 * n * case["niter"], bytes=(12 * case["niter"] + 32) * n)
    n = float(case["nSamples"])
    return dict(flops=20 * n * case["nChan"], bytes=24 * n + 12 * n * case["nChan"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "job":
        return _exact_job(case, seed)
    if kind == "current":
        return _exact_current(case, seed)
    if kind == "fft":
        x = _gauss(_gen(seed), case["gSize"], case["gSize"])
        return torch.complex(x.real.double(), torch.zeros_like(x.real, dtype=torch.float64))
    if kind == "clean":
        return _exact_clean(case, seed)
    return None   # batches would take minutes; the index set-up's outputs are whole numbers
