"""The large-field form over line lengths of many plans (odd and composite
radices, one short stage and four, padded and equal field and OTF sizes, short
and long sampled columns) against the oracle."""
import math

import numpy as np
import pytest

from conftest import RAD2MAS, rel_l2

pytestmark = pytest.mark.gpu

INTS_TOL = 2e-5  # the parity bars of the forms
GRAD_TOL_MAS = 0.1


# nxsa, embfac, notf: 16 = 4 4 and 18 = 6 3 (one radix, split); 48 = 8 6; 70 = 10 7;
# 80 = 16 5; 84 = 12 7; 96 = 16 6 in 210 = 7 6 5, in 250 = 10 5 5 and in 256 = 16 16
# (columns of 129 points, the longest of the staged sums); 128 = 16 8 in 270 = 9 6 5
# (columns of 136, summed by waves); 432 = 9 8 6 in 486 = 9 9 6; 480 = 16 6 5 in
# 1000 = 10 10 10; 448 = 8 8 7
@pytest.mark.parametrize("nxsa,embfac,notf", [(16, 1, 16), (16, 1, 18), (16, 3, 48), (16, 3, 70), (16, 5, 84), (48, 2, 210), (48, 2, 250),
                                              (48, 2, 256), (64, 2, 270), (144, 3, 486), (240, 2, 1000),
                                              (224, 2, 448)])
@pytest.mark.parametrize("nwvl", [1, 2])
def test_large_field_sizes(nxsa, embfac, notf, nwvl):
    import oracle
    from maos_amd import configs, engine
    from maos_amd.powfs import PTYPE_COG, AS2RAD, AperCfg, AtmCfg, Powfs, PowfsCfg, SimCfg, genatm
    print("case: nxsa %d embfac %d notf %d, %d wavelengths" % (nxsa, embfac, notf, nwvl), flush=True)
    dsa = 1.0
    wvl = [1.25e-6 * (1 + 0.3 * i) for i in range(nwvl)]
    pcfg = PowfsCfg(order=2, dsa=dsa, dx=dsa / nxsa, saat=0.3, hs=math.inf, embfac=embfac, wvl=wvl,
                    wvlwts=[1.0 / nwvl] * nwvl, pixpsa=6, pixtheta=0.6 * wvl[0] / dsa / AS2RAD, pixblur=0.3,
                    notf=notf, phytype=PTYPE_COG, sigmatch=1, siglev=1000.0)
    sim = SimCfg(dt=1.0 / 800)
    atm = AtmCfg(r0=0.15, L0=30.0, ht=[0.0, 5000.0], wt=[0.7, 0.3], ws=[8.0, 12.0], wddeg=[30.0, 200.0],
                 dx=1.0 / 64, nx=256, seeds=[3, 4])
    p = Powfs(AperCfg(2.0, 0.3), pcfg, sim)
    layers = genatm(atm)
    cfg = dict(powfs=pcfg, wfs=[dict(thetax=0.0, thetay=0.0), dict(thetax=4e-5, thetay=-2e-5)])
    engine.init(0)
    engine.atm2gpu(layers)
    wfs = configs.wfs_specs(cfg, p)
    eng = engine.WfsGrad(p, wfs)
    o = oracle.Oracle(p)
    o.atm(layers)
    eng.queue(19, sim.dt)
    for i, w in enumerate(wfs):
        g, ints = eng.sync(i)
        ri, rg, _, _ = o.step(w, 19, sim.dt)
        e_int, e_g = rel_l2(ints, ri), np.abs(g - rg).max() * RAD2MAS
        print("wfs %d ints %.2e grad %.2e mas" % (i, e_int, e_g), flush=True)
        assert e_int <= INTS_TOL and e_g <= GRAD_TOL_MAS
    eng.close()
