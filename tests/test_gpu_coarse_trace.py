"""The ray trace of grids coarser than a screen: an engine of enough WFS to go
by tiles gives the very numbers that engines of one WFS, one point per thread,
give, with static surfaces, tip/tilt and mirrors, for one layer and for the
remainders of four, a layer above the source and the uplink's grids; and a case
of each against the oracle."""
import math

import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _powfs(order, nxsa, llt):
    from maos_amd.powfs import (PTYPE_COG, AS2RAD, AperCfg, LltCfg, Powfs, PowfsCfg, SimCfg, SodiumCfg)
    wvl = 0.589e-6
    dsa = nxsa / 32
    # (16^2 and 32^2 points at twice Nyquist, larger grids in the large-field form)
    pcfg = PowfsCfg(order=order, dsa=dsa, dx=1 / 32, saat=0.3, hs=90e3 if llt else math.inf, embfac=2, wvl=[wvl], wvlwts=[1.0],
                    pixpsa=4, pixtheta=0.6 * wvl / dsa / AS2RAD, pixblur=0.3, notf=2 * nxsa, phytype=PTYPE_COG,
                    sigmatch=1, siglev=1000.0, llt=LltCfg(d=1.0, widthp=0.6) if llt else None,
                    sodium=SodiumCfg(center=90e3, fwhm=10e3, hmin=70e3, hmax=110e3, dh=50.0))
    return Powfs(AperCfg(order * dsa, 0.1 * order * dsa), pcfg, SimCfg(dt=1 / 800))


# order, points, WFS: at least 1024 tiles together (of 16^2, of 32^2, 9 of 16^2
# and 4 of 32^2 a grid), fewer in one WFS; layers; mirrors; with a launch telescope
@pytest.mark.parametrize("order,nxsa,nwfs,nps,ndm,llt", [
    (16, 16, 6, 1, 0, False), (16, 16, 6, 5, 2, False), (16, 16, 6, 3, 1, True), (16, 32, 6, 1, 1, False),
    (16, 32, 6, 6, 2, False), (16, 32, 6, 3, 0, True), (8, 48, 3, 2, 1, False), (8, 64, 6, 7, 0, False)])
def test_tiles_match_points(order, nxsa, nwfs, nps, ndm, llt):
    import oracle
    from maos_amd import engine
    from maos_amd.powfs import AtmCfg, genatm
    print("case: %d^2 points, %d WFS, %d layers, %d mirrors, llt %d" % (nxsa, nwfs, nps, ndm, llt), flush=True)
    p = _powfs(order, nxsa, llt)
    side = 32 if nxsa % 32 == 0 else 16
    tiles = p.nsa * (nxsa // side) ** 2
    assert tiles * nwfs >= 1024 > tiles
    ht = [0.0, 500.0, 1000.0, 2000.0, 4000.0, 8000.0, 16000.0][:nps]
    if llt:
        ht[-1] = 95e3  # above the laser guide star
    layers = genatm(AtmCfg(r0=0.186, L0=30.0, ht=ht, wt=[1 / nps] * nps, ws=[8.0 + i for i in range(nps)],
                           wddeg=[50.0 * i for i in range(nps)], dx=1 / 64, nx=512, seeds=list(range(1, nps + 1))))
    rs = np.random.RandomState(7)
    engine.init(0)
    engine.atm2gpu(layers)
    engine.dm2gpu([(1e-7 * rs.standard_normal((61, 61)), 0.5, -15.0, -15.0, 5000.0 * i) for i in range(ndm)])
    wfs = [engine.WfsSpec(thetax=3e-5 * i, thetay=-2e-5 * i, hs=p.cfg.hs, sigsim=p.sigsim, wvlwts=p.wvlwts,
                          misregx=0.01 * i) for i in range(nwfs)]
    surf = 5e-8 * rs.standard_normal((nwfs, p.nsa * nxsa * nxsa))
    ptt = 1e-7 * rs.standard_normal((nwfs, 3))

    def make(which):
        e = engine.WfsGrad(p, [wfs[i] for i in which])
        if ndm != 1:  # (one case each without the inputs)
            for k, i in enumerate(which):
                e.set_opdadd(surf[i], iwfs=k)
                e.set_ptt(ptt[i], iwfs=k)
        e.queue(23, 1 / 800)
        e.wait()
        return e
    many = make(range(nwfs))
    for i in (0, nwfs - 1):
        one = make([i])
        assert np.array_equal(many.debug_opd(i), one.debug_opd(0))
        if llt:
            assert np.array_equal(many.debug_lotf(i), one.debug_lotf(0))
        one.close()
    if ndm == 0 and not llt:
        many.set_opdadd(None)
        many.set_ptt(None)
        many.queue(23, 1 / 800)
        o = oracle.Oracle(p)
        o.atm(layers)
        ri = o.step(wfs[nwfs - 1], 23, 1 / 800)[0]
        e_int = rel_l2(many.sync(nwfs - 1)[1], ri)
        print("ints %.2e" % e_int, flush=True)
        assert e_int <= 2e-5  # the parity bar of the forms
    many.close()
    engine.dm2gpu([])
