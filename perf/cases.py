"""Performance cases: the work that a simulation program gives this library.

Three kinds of case, each through the package's public entry points:

  sh   steps of a Shack-Hartmann WFS engine (engine.WfsGrad): queue the step,
       fetch the gradients (and the pixel intensities or the long-exposure
       sums where the program reads them)
  evl  steps of the science evaluation (engine.Evl): trace, wavefront error of
       every step, long-exposure PSFs at the end
  py   steps of a pyramid WFS (engine.PywfsEngine): queue the step, fetch the
       gradients and the intensities

A program uploads its turbulence screens once and then steps through them, so
the screens belong to the case; the seed gives what differs between programs:
where in the frozen flow the steps lie, the guide stars, the static surfaces,
the tip/tilt and deformable-mirror commands.
"""
import math

import numpy as np
import torch

from maos_amd import _lib, engine
from maos_amd.powfs import (AS2RAD, PTYPE_COG, PTYPE_MF, AperCfg, AtmCfg, LltCfg, Powfs, PowfsCfg, SimCfg,
                            SodiumCfg, genatm)
from maos_amd.pywfs import Pywfs, PywfsCfg

DT = 1.0 / 800
HT = [0.0, 500.0, 1000.0, 2000.0, 4000.0, 8000.0, 16000.0]
WT = [0.45, 0.15, 0.10, 0.10, 0.08, 0.07, 0.05]
WS = [9.0, 7.5, 12.0, 14.0, 18.0, 11.0, 6.0]
WD = [10.0, 250.0, 75.0, 160.0, 310.0, 40.0, 120.0]


def _sh(name, **kw):
    c = dict(name=name, kind="sh", d=8.0, din=1.2, order=16, dsa=0.5, dxinv=32, embfac=2, notf=0, nwvl=1, wvl=0.7e-6,
             pixpsa=8, pixtheta=0.5, llt=0.0, mf=False, nwfs=1, fov=0.0, nx=2048, nlayer=1, nreal=1, dm=0,
             variant="auto", frames=1, out="grad")
    c.update(kw)
    return c


def _lgs(name, order, **kw):
    d = dict(d=0.5 * order, din=0.06 * order, order=order, dxinv=64, wvl=0.589e-6, pixpsa=6, pixtheta=1.0, llt=0.4,
             mf=True, nwfs=6, fov=35.0, nx=1024, nlayer=7)
    d.update(kw)
    return _sh(name, **d)


def _evl(name, **kw):
    c = dict(name=name, kind="evl", d=8.0, din=1.2, dxinv=32, n=1024, psfsize=256, nwvl=2, wvl=1.25e-6, ndir=4,
             fov=30.0, nx=1024, nlayer=7, dm=0, frames=10)
    c.update(kw)
    return c


def _py(name, **kw):
    c = dict(name=name, kind="py", d=8.0, din=1.2, order=16, dxinv=32, nside=4, modulate=5.0, modulpos=32, nx=1024,
             nlayer=7)
    c.update(kw)
    return c


def listed():
    return [
        # the closed loop of an 8 m telescope's NGS sensor, a deformable mirror's new shape before every step: the
        # smallest call, where latency counts
        _sh("ngs8m_closed_loop", dm=1),
        # one step of six LGS sensors of a 10 m telescope, the intensities read as well (telemetry)
        _lgs("lgs10m_ints", 20, out="ints"),
        # the 30 m telescope's six LGS sensors, one step of the control loop
        _lgs("lgs30m_step", 60, nx=4096),
        # matched-filter calibration: the long-exposure images of 20 steps, four realisations in one engine
        _lgs("lgs15m_x4_i0", 30, nreal=4, frames=20, out="i0"),
        # a 20 m telescope's LGS sensors in the FP32 form, for a program that wants FP32 images
        _lgs("lgs20m_fp32", 40, variant="fft32", nx=2048),
        # LGS sensors with fields padded to 128^2 (OTF at twice Nyquist)
        _lgs("lgs10m_pad128", 20, embfac=4),
        # three low-order NGS sensors of 2 x 2 subapertures on the 30 m pupil, two wavelengths
        _sh("ngs_lo_step", d=30.0, din=3.6, order=2, dsa=15.0, dxinv=16, notf=512, nwvl=2, wvl=1.25e-6, pixpsa=16,
            pixtheta=0.008, nwfs=3, fov=60.0, nx=4096, nlayer=7),
        # the tip-tilt sensor of the 30 m pupil: one subaperture, one large field
        _sh("ngs_tt_step", d=30.0, din=3.6, order=1, dsa=30.0, dxinv=16, notf=1024, wvl=2.2e-6, pixpsa=16,
            pixtheta=0.008, fov=25.0, nx=4096, nlayer=7),
        # science evaluation of an 8 m telescope: four directions, two wavelengths, small PSF windows
        _evl("evl8m", dm=1),
        # science evaluation of the 30 m telescope at 1/64 m: 4096^2 transforms at three wavelengths
        _evl("evl30m", d=30.0, din=3.6, dxinv=64, n=4096, psfsize=1024, nwvl=3, ndir=1, nx=4096, frames=16),
        # pyramid sensors of an 8 m (784^2 grid) and of the 30 m telescope (2916^2 grid)
        _py("pywfs8m_step"),
        _py("pywfs30m_step", d=30.0, din=3.6, order=60, nx=4096),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """Another case of the ranges above: NGS, LGS, padded LGS, low-order NGS,
    science evaluation or pyramid, with other sizes and options."""
    k = rng.choice(["ngs", "ngs64", "lgs", "lgs", "pad", "lf", "lf", "evl", "evl", "py", "py"])
    nl = rng.choice([1, 2, 3, 5, 7])
    if k == "ngs":
        order = int(_log(rng, 6, 33))
        c = _sh(k, d=0.5 * order, din=0.07 * order, order=order, notf=32, pixpsa=rng.choice([4, 6, 7, 8]),
                nwfs=rng.randint(1, 4), fov=rng.uniform(5, 60), nx=1024, nlayer=nl, dm=rng.choice([0, 1, 2]),
                out=rng.choice(["grad", "ints"]))
    elif k == "ngs64":
        order = int(_log(rng, 5, 40))
        c = _sh(k, d=0.5 * order, din=0.07 * order, order=order, dxinv=64, notf=64, nwvl=rng.randint(1, 2),
                pixpsa=rng.choice([4, 6]), pixtheta=rng.uniform(0.25, 0.4), nwfs=rng.randint(1, 3),
                fov=rng.uniform(5, 60), nx=1024, nlayer=nl, variant=rng.choice(["auto", "fft32"]))
    elif k == "lgs":
        npix = rng.choice([4, 5, 6, 8])
        c = _lgs(k, int(_log(rng, 8, 56)), nwfs=rng.randint(1, 6), fov=rng.uniform(20, 60), nlayer=nl,
                 pixpsa=npix, pixtheta=6.0 / npix * rng.uniform(0.8, 1.05), variant=rng.choice(["auto", "auto", "fft32"]),
                 frames=rng.choice([1, 1, 8]))
        c["out"] = "i0" if c["frames"] > 1 else rng.choice(["grad", "ints"])
    elif k == "pad":
        c = _lgs(k, int(_log(rng, 8, 22)), nwfs=rng.randint(1, 6), fov=rng.uniform(20, 60), nlayer=nl, embfac=4)
    elif k == "lf":
        # (nxsa, notf, subapertures across, 1/dx)
        nxsa, notf, order, dxinv = rng.choice([(48, 120, 2, 24), (240, 512, 2, 16), (480, 1024, 1, 16), (64, 128, 3, 16),
                                               (96, 192, 2, 16), (240, 480, 2, 16), (320, 640, 1, 16), (144, 300, 2, 24)])
        d = nxsa / dxinv * order
        c = _sh(k, d=d, din=0.12 * d, order=order, dsa=nxsa / dxinv, dxinv=dxinv, notf=notf, nwvl=rng.randint(1, 2),
                wvl=rng.choice([1.25e-6, 1.65e-6, 2.2e-6]), pixpsa=rng.choice([8, 11, 16]), nwfs=rng.randint(1, 3),
                fov=rng.uniform(20, 60), nx=2048, nlayer=nl)
        c["pixtheta"] = 0.5 * c["wvl"] / c["dsa"] / AS2RAD
    elif k == "evl":
        n = rng.choice([256, 512, 1024, 2048])
        dxinv = rng.choice([16, 32])
        d = round(n * rng.uniform(0.3, 0.49) / dxinv, 2)
        c = _evl(k, d=d, din=round(0.12 * d, 2), dxinv=dxinv, n=n, psfsize=rng.choice([64, 100, 128, 250]),
                 nwvl=rng.randint(1, 3), ndir=rng.randint(1, 9 if n < 2048 else 3), fov=rng.uniform(5, 60), nlayer=nl,
                 dm=rng.choice([0, 1]), frames=rng.randint(3, 12))
    else:
        order = int(_log(rng, 8, 36))
        c = _py(k, d=0.5 * order, din=0.07 * order, order=order, dxinv=rng.choice([16, 32]),
                nside=rng.choice([4, 4, 3]), modulate=rng.choice([3.0, 4.0, 5.0]),
                modulpos=rng.choice([8, 12, 16, 32]), nlayer=nl)
    del c["name"]
    return c


# ------------------------------------------------------------------ the tables and screens of a case
_tables = {}
_uploaded = [None]


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _once(key, make):
    if key not in _tables:
        if len(_tables) > 8:
            _tables.clear()
        _tables[key] = make()
    return _tables[key]


def _layers(case):
    """The screens of each realisation."""
    n = case["nlayer"]
    wt = [w / sum(WT[:n]) for w in WT[:n]]

    def make():
        return [genatm(AtmCfg(r0=0.186, L0=30.0, ht=HT[:n], wt=wt, ws=WS[:n], wddeg=WD[:n], dx=1.0 / 64,
                              nx=case["nx"], seeds=[1 + i + 10 * r for i in range(n)]))
                for r in range(case.get("nreal", 1))]
    return _once(("atm", case["nx"], n, case.get("nreal", 1)), make)


def _upload(case):
    key = ("atm", case["nx"], case["nlayer"], case.get("nreal", 1))
    if _uploaded[0] != key:
        engine.init(0)
        for r, layers in enumerate(_layers(case)):
            engine.atm2gpu(layers, ireal=r)
        _uploaded[0] = key
    engine.dm2gpu([])


def _wvl(case):
    return [case["wvl"] * (1 + 0.32 * i) for i in range(case["nwvl"])]


def _powfs(case):
    def make():
        n = case["nwvl"]
        p = Powfs(AperCfg(d=case["d"], din=case["din"]),
                  PowfsCfg(order=case["order"], dsa=case["dsa"], dx=1.0 / case["dxinv"], saat=0.3,
                           hs=90e3 if case["llt"] else math.inf, embfac=case["embfac"], wvl=_wvl(case),
                           wvlwts=[1.0 / n] * n, pixpsa=case["pixpsa"], pixtheta=case["pixtheta"], pixblur=0.3,
                           notf=case["notf"], phytype=PTYPE_MF if case["mf"] else PTYPE_COG, sigmatch=1, siglev=960.0,
                           llt=LltCfg(d=case["llt"], widthp=0.6) if case["llt"] else None,
                           sodium=SodiumCfg(center=90e3, fwhm=10e3, hmin=70e3, hmax=110e3, dh=20.0)), SimCfg(dt=DT))
        ref = p.mtch(*p.i0_model(0.186, 30.0))[:2] if case["mf"] else None
        return p, ref
    return _once(("powfs", _key(case)), make)


def _aperture(case):
    def make():
        dx = 1.0 / case["dxinv"]
        n = int(round(case["d"] / dx)) + 1
        c = (np.arange(n) - (n - 1) / 2) * dx
        X, Y = np.meshgrid(c, c)
        r = np.hypot(X, Y)
        m = (r <= case["d"] / 2 + 1e-9) & (r >= case["din"] / 2)
        x, y = X[m].copy(), Y[m].copy()
        emb, N = engine.loc_embed(x, y, dx, nembed=case["n"])
        return x, y, np.full(len(x), 1.0 / len(x)), emb
    return _once(("aper", _key(case)), make)


def _pyramid(case):
    def make():
        pw = Pywfs(PywfsCfg(D=case["d"], din=case["din"], order=case["order"], dx=1.0 / case["dxinv"],
                            nside=case["nside"], modulate=case["modulate"], modulpos=case["modulpos"]))
        # the calibration's images come from the plain 64-bit imaging below, so that every program has the same tables
        return pw.calibrate(lambda p: (lambda opd: [a.cpu().numpy() for a in _py_image(p, _t(opd))]))
    return _once(("py", _key(case)), make)


# ------------------------------------------------------------------ what the seed gives
def _drawn_inputs(case, seed):
    r = np.random.RandomState(seed % (1 << 31))
    s = {"isim": int(r.randint(100, 30000))}
    n = case.get("nwfs", case.get("ndir", 1))
    a0 = r.uniform(0, 2 * math.pi)
    f = case.get("fov", 0.0) * AS2RAD
    ang = a0 + 2 * math.pi * np.arange(n) / max(1, n - 1)
    rad = np.where(np.arange(n) == 0, 0.1 if n > 1 else 1.0, 1.0) * f
    s["theta"] = np.stack([rad * np.cos(ang), rad * np.sin(ang)], axis=1)
    # mirror commands: smooth shapes on a 0.5 m actuator grid that is wider than the pupil and its footprints
    s["dm"] = []
    for i in range(case.get("dm", 0)):
        ht = 8000.0 * i
        m = int(case["d"] / 2 + 2 * f * ht + 3) * 4 + 1
        c = (np.arange(m) - m // 2) * 0.5
        X, Y = np.meshgrid(c, c)
        p = sum(r.normal() * 6e-8 * np.cos(r.uniform(0.2, 1.5) * X + r.uniform(0.2, 1.5) * Y + r.uniform(0, 6))
                for _ in range(6))
        s["dm"].append((p, 0.5, -(m // 2) * 0.5, -(m // 2) * 0.5, ht))
    if case["kind"] == "sh":
        s["ptt"] = r.normal(size=(n, 3)) * np.array([1e-7, 1e-7, 1e-7])
        w = r.uniform(0.2, 1.2, size=(4, 3))
        s["surf"] = lambda x, y: sum(2e-8 * np.sin(w[j, 0] * x + w[j, 1] * y + 6 * w[j, 2]) for j in range(4))
    return s


def _points(p):
    """Coordinates of the subaperture points [nsa, nxsa, nxsa], x fastest."""
    g = np.arange(p.nxsa) * p.dx
    shape = (p.nsa, p.nxsa, p.nxsa)
    return (np.broadcast_to(p.ptsx[:, None, None] + g[None, None, :], shape),
            np.broadcast_to(p.ptsy[:, None, None] + g[None, :, None], shape))


def prepare(case, seed):
    _upload(case)
    s = dict(case=case, **_drawn_inputs(case, seed))
    if case["kind"] == "sh":
        p, ref = _powfs(case)
        wfs = [engine.WfsSpec(thetax=t[0], thetay=t[1], hs=p.cfg.hs, sigsim=p.sigsim, wvlwts=p.wvlwts)
               for t in s["theta"]]
        e = engine.WfsGrad(p, wfs, nreal=case["nreal"])
        if case["variant"] == "fft32":
            e.set_variant(_lib.VARIANT_FFT32)
        e.set_graph(True)
        if ref is not None:
            e.update_ref(*ref)
        e.set_opdadd(s.pop("surf")(*_points(p)))
        for i in range(e.nwfs):
            e.set_ptt(s["ptt"][i % len(wfs)], i)
        s["engine"] = e
    elif case["kind"] == "evl":
        x, y, amp, emb = _aperture(case)
        n = case["nwvl"]
        s["engine"] = engine.Evl(amp, _wvl(case), [case["n"]] * n, [case["psfsize"]] * n, np.tile(emb, n), locx=x,
                                 locy=y, dirs=[(t[0], t[1], 0.0) for t in s["theta"]])
    else:
        s["engine"] = engine.PywfsEngine(_pyramid(case))
    return s


def run(state):
    case, e, isim = state["case"], state["engine"], state["isim"]
    if state["dm"]:
        engine.dm2gpu(state["dm"])
    if case["kind"] == "sh":
        if case["out"] == "i0":
            e.i0_control(True, reset=True)
        for k in range(case["frames"]):
            e.queue(isim + k, DT)
        if case["out"] == "i0":
            return [e.i0_get(i)[0] for i in range(e.nwfs)]
        got = [e.sync(i, want_ints=case["out"] == "ints") for i in range(e.nwfs)]
        return got if case["out"] == "ints" else [g for g, _ in got]
    if case["kind"] == "evl":
        e.reset()
        wfe = []
        for k in range(case["frames"]):
            e.trace(isim + k, DT)
            wfe.append(e.wfe())
        return [np.stack([w[0] for w in wfe]), np.stack([w[1] for w in wfe]),
                [e.psf(d, w)[0] for d in range(e.ndir) for w in range(e.nwvl)]]
    e.queue(isim, DT)
    return list(e.sync())


# ------------------------------------------------------------------ plain 64-bit results
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=_dev())


def _interp(scr, x, y, wrap):
    """Bilinear values of map scr [ny, nx] at x, y (samples); without wrap,
    points off the map give zero."""
    ny, nx = scr.shape
    ok = 1.0
    if wrap:
        x, y = torch.remainder(x, nx), torch.remainder(y, ny)
    else:
        ok = ((x >= 0) & (x < nx - 1) & (y >= 0) & (y <= ny - 1)).double()
    ix, iy = torch.floor(x), torch.floor(y)
    fx, fy = x - ix, y - iy
    ix, iy = ix.long() % nx, iy.long() % ny
    jx, jy = (ix + 1) % nx, (iy + 1) % ny
    return ok * ((1 - fy) * ((1 - fx) * scr[iy, ix] + fx * scr[iy, jx]) +
                 fy * ((1 - fx) * scr[jy, ix] + fx * scr[jy, jx]))


def _screens(case):
    return [[(_t(L.p), L) for L in r] for r in _layers(case)]


def _trace(screens, x, y, theta, hs, isim):
    """Frozen-flow OPD at points x, y (m)."""
    o = torch.zeros_like(x)
    for scr, L in screens:
        sc = 1.0 - L.ht / hs if math.isfinite(hs) else 1.0
        dx, dy = L.ht * theta[0] - L.vx * DT * isim, L.ht * theta[1] - L.vy * DT * isim
        o += _interp(scr, x / L.dx * sc + (dx - L.ox) / L.dx, y / L.dx * sc + (dy - L.oy) / L.dx, True)
    return o


def _mirrors(s, x, y, theta, hs):
    o = torch.zeros_like(x)
    for p, dx, ox, oy, ht in s["dm"]:
        sc = 1.0 - ht / hs if math.isfinite(hs) else 1.0
        o -= _interp(_t(p), (x * sc + ht * theta[0] - ox) / dx, (y * sc + ht * theta[1] - oy) / dx, False)
    return o


def _field(opd, amp, wvl, n):
    """amp exp(2 pi i opd / wvl) in the middle of an n^2 grid."""
    k = (n - opd.shape[-1]) // 2
    f = torch.polar(amp.expand_as(opd).contiguous(), 2 * math.pi / wvl * opd)
    return torch.nn.functional.pad(f, (k, n - k - opd.shape[-1], k, n - k - opd.shape[-1]))


def _sh_frame(p, s, screens, xy, surf, theta, ptt, isim):
    """Intensities [nsa, npix] of one step of one WFS."""
    x, y = xy
    hs, N, nw = p.cfg.hs, p.notf, p.nxsa * p.cfg.embfac
    opd = _trace(screens, x, y, theta, hs, isim) + _mirrors(s, x, y, theta, hs)
    opd += surf + ptt[0] + ptt[1] * x + ptt[2] * y
    amp = _t(p.amp).reshape(opd.shape)
    ints = torch.zeros(p.nsa, p.npix, dtype=torch.float64, device=opd.device)
    norm = p.areascale / (p.nxsa * nw) ** 2 * p.sigsim / N ** 2
    for iw, wvl in enumerate(p.wvl):
        up = None
        if p.llt is not None:
            g = torch.arange(p.llt_nx, dtype=torch.float64, device=opd.device) * p.dx + p.llt_origin
            ly, lx = torch.meshgrid(g, g, indexing="ij")
            lo = _trace(screens, lx, ly, theta, hs, isim)
            lf = torch.fft.fft2(_field(lo, _t(p.llt_amp).reshape(lo.shape), wvl, nw)).abs() ** 2 / nw ** 2
            up = torch.fft.fft2(lf).conj()
        pp = p.si_pp[iw]
        col = _t(np.repeat(np.arange(N * N), np.diff(pp)))
        nz = int(pp[-1])
        pix, wt = _t(p.si_pi[iw][:nz]), _t(p.si_px[iw][:nz])
        step = max(1, (1 << 24) // (N * N))
        for a in range(0, p.nsa, step):
            b = min(p.nsa, a + step)
            f = torch.fft.fft2(_field(opd[a:b], amp[a:b], wvl, nw))
            f = f.real ** 2 + f.imag ** 2
            if nw < N:
                h, q = nw // 2, f.new_zeros(b - a, N, N)
                q[:, :h, :h], q[:, :h, -h:], q[:, -h:, :h], q[:, -h:, -h:] = (f[:, :h, :h], f[:, :h, -h:],
                                                                              f[:, -h:, :h], f[:, -h:, -h:])
                f = q
            o = torch.fft.fft2(f)
            if up is not None:
                o *= up
                o *= _t(p.etf[iw].reshape(p.nsa, N * N * 2)[a:b].view(np.complex128)).reshape(o.shape)
            else:
                o *= _t(p.nominal[iw]).reshape(N, N)
            im = torch.fft.ifft2(o).real.reshape(b - a, N * N)[:, col] * (N * N) * wt
            ints[a:b].index_add_(1, pix, im, alpha=float(p.wvlwts[iw]) * norm)
    return ints


def _sh_grad(p, ref, ints):
    if ref is not None:
        m, i0sum = _t(ref[0]).reshape(p.nsa, p.npix, 2), _t(ref[1])
        sc = i0sum / ints.sum(1)
        sc = torch.where((sc <= 0) | (sc > 10) | ~torch.isfinite(sc), torch.ones_like(sc), sc)
        return torch.einsum("spk,sp->ks", m, ints * sc[:, None]).reshape(-1)
    w = ints * (ints > 0)
    ii = torch.arange(p.npix, device=ints.device, dtype=torch.float64)
    n = p.pixpsax
    gx = ((w * (ii % n)).sum(1) / w.sum(1) - (n - 1) / 2) * p.pixthetax
    gy = ((w * torch.div(ii, n, rounding_mode="floor")).sum(1) / w.sum(1) - (n - 1) / 2) * p.pixthetay
    return torch.cat([gx, gy])


def _py_image(pw, opd, siglev=None):
    """(ints [nside, nsa], gradients) of a pupil OPD."""
    c, N = pw.cfg, pw.N
    h = N // 2
    siglev = c.siglev if siglev is None else siglev
    pup = torch.zeros(N, N, dtype=torch.float64, device=opd.device)
    amp, emb = _t(pw.amp), _t(pw.embed)
    for iw, wvl in enumerate(pw.wvl):
        f = torch.zeros(N * N, dtype=torch.complex128, device=opd.device)
        f[emb] = torch.polar(amp, 2 * math.pi / wvl * opd)
        f = torch.fft.fftshift(torch.fft.fft2(f.reshape(N, N))) / (amp.square().sum().sqrt() * N)
        mask = torch.view_as_complex(_t(pw.mask[iw]).reshape(N, N, 2))
        for ip in range(c.modulpos):
            th = 2 * math.pi * ip / c.modulpos
            dth = wvl / (c.dx * N)
            ox, oy = (int(math.floor(abs(v) + 0.5)) * (1 if v >= 0 else -1) for v in
                      (math.cos(th) * pw.modulate / dth, math.sin(th) * pw.modulate / dth))
            o = torch.zeros_like(f)
            ya, yb, xa, xb = max(0, -oy), N - max(0, oy), max(0, -ox), N - max(0, ox)
            o[ya:yb, xa:xb] = f[ya + oy:yb + oy, xa + ox:xb + ox] * mask[ya:yb, xa:xb]
            o = torch.fft.ifft2(o) * (N * N)
            pup += (o.real ** 2 + o.imag ** 2) * (float(pw.wvlwts[iw]) / (N * N * c.modulpos))
    pup = (torch.fft.ifft2(torch.fft.fft2(pup) * _t(pw.nominal).reshape(N, N)) * (N * N)).real
    sx, sy = _t(pw.salocx), _t(pw.salocy)
    ints = []
    for k in range(c.nside):
        x = sx / c.dx + pw.sioff[2 * k] * h + h - 0.5
        y = sy / c.dx + pw.sioff[2 * k + 1] * h + h - 0.5
        ix, iy = torch.floor(x), torch.floor(y)
        v = torch.zeros_like(x)
        for a in (0, 1):
            for b in (0, 1):
                w = (x - ix if b else 1 - (x - ix)) * (y - iy if a else 1 - (y - iy))
                px, py = ix.long() + b, iy.long() + a
                ok = (w > 1e-15) & (px >= 0) & (px < N) & (py >= 0) & (py < N)
                v += torch.where(ok, w * pup[py.clamp(0, N - 1), px.clamp(0, N - 1)], torch.zeros_like(w))
        ints.append(v * (pw.nsa * siglev / (N * N)))
    I = torch.stack(ints)
    a = pw.gain / (I.sum() / pw.nsa * _t(pw.saa))
    if c.nside == 3:
        g = torch.cat([(I[1] - I[2]) * a * math.sqrt(3.0) * 0.5, (I[0] - 0.5 * (I[1] + I[2])) * a])
    else:
        g = torch.cat([(I[0] - I[1] + I[2] - I[3]) * a, (I[0] + I[1] - I[2] - I[3]) * a])
    if pw.gradoff is not None:
        g = g - _t(pw.gradoff)
    return I, g


def exact(case, seed):
    s = _drawn_inputs(case, seed)
    screens = _screens(case)
    if case["kind"] == "sh":
        p, ref = _powfs(case)
        px, py = _points(p)
        surf, xy = _t(s["surf"](px, py)), (_t(px), _t(py))
        out = []
        for r in range(case["nreal"]):
            for th, ptt in zip(s["theta"], s["ptt"]):
                tot = 0
                for k in range(case["frames"]):
                    tot = tot + _sh_frame(p, s, screens[r], xy, surf, th, ptt, s["isim"] + k)
                if case["out"] == "i0":
                    out.append(tot.cpu().numpy())
                else:
                    g = _sh_grad(p, ref, tot).cpu().numpy()
                    out.append((g, tot.cpu().numpy()) if case["out"] == "ints" else g)
        return out
    if case["kind"] == "py":
        pw = _pyramid(case)
        x, y = _t(pw.locx), _t(pw.locy)
        return [a.cpu().numpy() for a in _py_image(pw, _trace(screens[0], x, y, (0.0, 0.0), math.inf, s["isim"]))]
    x, y, amp, emb = (_t(a) for a in _aperture(case))
    n, h = case["n"], case["psfsize"] // 2
    v = torch.stack([torch.ones_like(x), x, y])
    mcc = (v * amp) @ v.T
    rms, coeff = [], []
    psf = [[0 for _ in range(case["nwvl"])] for _ in s["theta"]]
    win = torch.arange(-h, h, device=x.device) % n
    for k in range(case["frames"]):
        for d, th in enumerate(s["theta"]):
            o = _trace(screens[0], x, y, th, math.inf, s["isim"] + k) + _mirrors(s, x, y, th, math.inf)
            c = v @ (amp * o)
            q = torch.linalg.solve(mcc, c)
            tot, pis, ptt = (amp * o * o).sum(), c[0] ** 2 / mcc[0, 0], (c * q).sum()
            rms.append(torch.stack([tot - pis, ptt - pis, tot - ptt]))
            coeff.append(q)
            for w, wvl in enumerate(_wvl(case)):
                f = torch.zeros(n * n, dtype=torch.complex128, device=x.device)
                f[emb] = torch.polar(amp, 2 * math.pi / wvl * o)
                f = torch.fft.fft2(f.reshape(n, n))[win][:, win]
                psf[d][w] = psf[d][w] + f.real ** 2 + f.imag ** 2
    shape = (case["frames"], len(s["theta"]), 3)
    a2 = float(amp.sum()) ** 2 * case["frames"]
    return [torch.stack(rms).reshape(shape).cpu().numpy(), torch.stack(coeff).reshape(shape).cpu().numpy(),
            [(a / a2).cpu().numpy() for d in psf for a in d]]


# ------------------------------------------------------------------ the work of one pass
def _fft2(n):
    return 5.0 * n * n * math.log2(n * n)


def work(case):
    nl, fr, d = case["nlayer"], case["frames"] if "frames" in case else 1, case["d"]
    if case["kind"] == "sh":
        nxsa = int(round(case["dsa"] * case["dxinv"]))
        nw = nxsa * case["embfac"]
        N, nw2 = case["notf"] or nw, case["nwvl"]
        nsa = max(1.0, math.pi / 4 * (d ** 2 - case["din"] ** 2) / case["dsa"] ** 2) if case["order"] > 2 else case["order"] ** 2
        wfs, npix = case["nwfs"] * case["nreal"], case["pixpsa"] ** 2
        scr = 4.0 * nl * case["nreal"] * min((64 * d) ** 2, case["nx"] ** 2)  # the pupil's part of each screen
        tab = 4.0 * nsa * nxsa ** 2 * 2 + (4.0 * nsa * N * N * nw2 if case["llt"] else 4.0 * N * N * nw2)
        per = 8.0 * npix if case["out"] != "grad" else 0.0
        by = fr * (scr + tab + wfs * nsa * (16.0 + per + (8.0 * npix if case["mf"] else 0.0)))
        fl = fr * wfs * nsa * (8.0 * nl * nxsa ** 2 + nw2 * (_fft2(nw) + 2 * _fft2(N) + 15.0 * N * N))
        return {"bytes": by, "flops": fl}
    npts = math.pi / 4 * (d ** 2 - case["din"] ** 2) * case["dxinv"] ** 2
    if case["kind"] == "py":
        N = 3.0 * d * case["dxinv"]
        by = 4.0 * nl * npts + 12.0 * npts + 12.0 * N * N
        return {"bytes": by, "flops": 8.0 * nl * npts + (case["modulpos"] + 3) * _fft2(N)}
    P, n, many = case["psfsize"], case["n"], case["ndir"] * case["nwvl"]
    band = d * case["dxinv"]
    by = fr * (4.0 * nl * npts * case["ndir"] + 12.0 * npts + 8.0 * P * P * many)
    fl = fr * case["ndir"] * (8.0 * nl * npts + 10.0 * npts) + fr * many * 5.0 * n * math.log2(n) * (band + P)
    return {"bytes": by, "flops": fl}
