"""The large-field form with detectors that sample many rows of the image, up
to all of it (more than 128 sampled rows or columns keep the whole image),
against the oracle: either side of the line between the directly summed rows
and the transformed columns, odd numbers of columns, short and long columns,
wavelengths of which only one keeps the whole image, and more outputs than one
thread each of a launch can count (260 chains of 512^2)."""
import math

import numpy as np
import pytest

from conftest import RAD2MAS, rel_l2

pytestmark = pytest.mark.gpu

INTS_TOL = 2e-5  # the parity bars of the forms
GRAD_TOL_MAS = 0.1


# spacing: samples of the image between pixels (2: two rows a pixel; 1: pixpsa + 1 rows)
@pytest.mark.parametrize("nxsa,embfac,notf,pixpsa,spacing,wvls,order,nwfs", [
    (64, 2, 128, 16, 2.1, (1.25e-6,), 2, 2),    # 32 rows
    (64, 2, 128, 17, 2.1, (1.25e-6,), 2, 2),    # 34
    (64, 2, 270, 17, 2.1, (1.25e-6,), 2, 2),    # long columns
    (96, 2, 210, 34, 1.0, (1.25e-6,), 1, 2),    # 35: the last column alone
    (64, 2, 140, 66, 2.1, (1.25e-6,), 1, 2),    # the whole image, short columns
    (64, 2, 256, 70, 2.1, (1.25e-6,), 1, 2),
    (64, 2, 270, 70, 2.1, (1.25e-6,), 2, 2),    # and long ones
    (240, 2, 500, 66, 2.1, (1.25e-6,), 1, 1),
    (64, 2, 256, 70, 2.1, (1.25e-6, 3e-6), 2, 2),  # the second wavelength: about 60 rows
    (64, 2, 256, 70, 0.9, (3e-6, 1.25e-6), 2, 1),  # the first
    (16, 2, 512, 66, 2.1, (1.25e-6,), 8, 5),
])
def test_wide_detectors(nxsa, embfac, notf, pixpsa, spacing, wvls, order, nwfs):
    import oracle
    from maos_amd import configs, engine
    from maos_amd.powfs import PTYPE_COG, AS2RAD, AperCfg, AtmCfg, Powfs, PowfsCfg, SimCfg, genatm
    print("case: nxsa %d notf %d, %d pixels %g samples apart, %d wavelengths, order %d, %d WFS"
          % (nxsa, notf, pixpsa, spacing, len(wvls), order, nwfs), flush=True)
    dsa = 1.0
    pcfg = PowfsCfg(order=order, dsa=dsa, dx=dsa / nxsa, saat=0.3, hs=math.inf, embfac=embfac, wvl=list(wvls),
                    wvlwts=[1.0 / len(wvls)] * len(wvls), pixpsa=pixpsa,
                    pixtheta=spacing * wvls[0] * nxsa / (dsa * notf) / AS2RAD, pixblur=0.3, notf=notf,
                    phytype=PTYPE_COG, sigmatch=1, siglev=1000.0)
    sim = SimCfg(dt=1.0 / 800)
    atm = AtmCfg(r0=0.15, L0=30.0, ht=[0.0, 5000.0], wt=[0.7, 0.3], ws=[8.0, 12.0], wddeg=[30.0, 200.0],
                 dx=1.0 / 64, nx=256, seeds=[3, 4])
    p = Powfs(AperCfg(float(order), 0.1 * order), pcfg, sim)
    layers = genatm(atm)
    cfg = dict(powfs=pcfg, wfs=[dict(thetax=4e-5 * i, thetay=-2e-5 * i) for i in range(nwfs)])
    engine.init(0)
    engine.dm2gpu([])
    engine.atm2gpu(layers)
    wfs = configs.wfs_specs(cfg, p)
    eng = engine.WfsGrad(p, wfs)
    assert order < 8 or p.nsa * nwfs >= 256
    o = oracle.Oracle(p)
    o.atm(layers)
    eng.queue(19, sim.dt)
    for i in {0, nwfs - 1}:
        g, ints = eng.sync(i)
        ri, rg, _, _ = o.step(wfs[i], 19, sim.dt)
        e_int, e_g = rel_l2(ints, ri), np.abs(g - rg).max() * RAD2MAS
        print("wfs %d ints %.2e grad %.2e mas" % (i, e_int, e_g), flush=True)
        assert e_int <= INTS_TOL and e_g <= GRAD_TOL_MAS
    eng.close()


@pytest.mark.parametrize("notf", [128, 270])
def test_detector_tables_change_between_graph_steps(notf):
    """An engine that steps as a graph and is given the tables of a wider
    detector (18 sampled rows, then 34, transformed instead of summed) gives
    what an engine made for that detector gives."""
    from maos_amd import _lib, configs, engine
    from maos_amd._lib import check, dptr, lptr
    from maos_amd.powfs import PTYPE_COG, AS2RAD, AperCfg, AtmCfg, Powfs, PowfsCfg, SimCfg, genatm
    print("case: OTF %d, detector tables replaced" % notf, flush=True)
    nxsa, dsa, wvl = 64, 1.0, 1.25e-6

    def powfs(spacing):
        pcfg = PowfsCfg(order=2, dsa=dsa, dx=dsa / nxsa, saat=0.3, hs=math.inf, embfac=2, wvl=[wvl], wvlwts=[1.0],
                        pixpsa=17, pixtheta=spacing * wvl * nxsa / (dsa * notf) / AS2RAD, pixblur=0.3, notf=notf,
                        phytype=PTYPE_COG, sigmatch=1, siglev=1000.0)
        return Powfs(AperCfg(2.0, 0.2), pcfg, SimCfg(dt=1.0 / 800))
    near, far = powfs(1.0), powfs(2.1)
    engine.init(0)
    engine.dm2gpu([])
    engine.atm2gpu(genatm(AtmCfg(r0=0.15, L0=30.0, ht=[0.0], wt=[1.0], ws=[8.0], wddeg=[30.0], dx=1.0 / 64, nx=256,
                                 seeds=[3])))
    wfs = configs.wfs_specs(dict(powfs=near.cfg, wfs=[dict(thetax=4e-5, thetay=0.0)]), near)
    eng, ref = engine.WfsGrad(near, wfs), engine.WfsGrad(far, wfs)
    eng.set_graph(True)
    for i in range(3):
        eng.queue(i, 1.0 / 800)
    before = eng.sync(0)[1]
    check(_lib.hip().mx_wfsgrad_set_dtf(eng.h, 0, dptr(far.nominal[0]), far.npix, notf * notf, lptr(far.si_pp[0]),
                                        lptr(far.si_pi[0]), dptr(far.si_px[0])))
    for i in (7, 8):
        eng.queue(i, 1.0 / 800)
        ref.queue(i, 1.0 / 800)
        got, want = eng.sync(0)[1], ref.sync(0)[1]
        assert np.array_equal(got, want)
    assert not np.array_equal(before, want)
    eng.close()
    ref.close()
