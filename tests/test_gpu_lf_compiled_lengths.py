"""The large-field passes of the lengths that kernels are compiled for: each of
them with its own partner and with another one (a compiled pass beside the
general ones), for every block size that the autotuner tries, against the
oracle."""
import math

import numpy as np
import pytest

from conftest import RAD2MAS, rel_l2

pytestmark = pytest.mark.gpu

INTS_TOL = 2e-5  # the parity bars of the forms
GRAD_TOL_MAS = 0.1


# fields of 96, 128, 480 and 960 points; OTFs of 120, 128, 512 and 1024
@pytest.mark.parametrize("nxsa,embfac,notf,pixpsa", [(48, 2, 120, 6), (32, 4, 128, 6), (64, 2, 128, 6), (240, 2, 512, 6),
                                                     (480, 2, 1024, 6), (48, 2, 128, 6), (64, 2, 512, 6), (48, 2, 1024, 6),
                                                     (240, 2, 500, 6), (480, 2, 960, 6), (16, 5, 120, 6),
                                                     (32, 3, 120, 40), (48, 2, 512, 40)])
def test_compiled_lengths(nxsa, embfac, notf, pixpsa):
    import oracle
    from maos_amd import configs, engine
    from maos_amd.powfs import PTYPE_COG, AS2RAD, AperCfg, AtmCfg, Powfs, PowfsCfg, SimCfg, genatm
    print("case: nxsa %d embfac %d notf %d, %d pixels" % (nxsa, embfac, notf, pixpsa), flush=True)
    dsa, wvl = 1.0, 1.25e-6
    pcfg = PowfsCfg(order=2, dsa=dsa, dx=dsa / nxsa, saat=0.3, hs=math.inf, embfac=embfac, wvl=[wvl], wvlwts=[1.0],
                    pixpsa=pixpsa, pixtheta=min(0.6, 1.5 * nxsa / notf) * wvl / dsa / AS2RAD, pixblur=0.3, notf=notf,
                    phytype=PTYPE_COG, sigmatch=1, siglev=1000.0)
    sim = SimCfg(dt=1.0 / 800)
    atm = AtmCfg(r0=0.15, L0=30.0, ht=[0.0, 5000.0], wt=[0.7, 0.3], ws=[8.0, 12.0], wddeg=[30.0, 200.0],
                 dx=1.0 / 64, nx=256, seeds=[3, 4])
    p = Powfs(AperCfg(2.0, 0.3), pcfg, sim)
    layers = genatm(atm)
    engine.init(0)
    engine.dm2gpu([])
    engine.atm2gpu(layers)
    wfs = configs.wfs_specs(dict(powfs=pcfg, wfs=[dict(thetax=4e-5, thetay=-2e-5)]), p)
    o = oracle.Oracle(p)
    o.atm(layers)
    ri, rg, _, _ = o.step(wfs[0], 19, sim.dt)
    for tuned in (False, True):
        eng = engine.WfsGrad(p, wfs)
        if tuned:
            eng.autotune(3, sim.dt, nrep=2)  # (steps of 128, 256 and 512 threads)
        eng.queue(19, sim.dt)
        g, ints = eng.sync(0)
        eng.close()
        e_int, e_g = rel_l2(ints, ri), np.abs(g - rg).max() * RAD2MAS
        print("tuned %d ints %.2e grad %.2e mas" % (tuned, e_int, e_g), flush=True)
        assert e_int <= INTS_TOL and e_g <= GRAD_TOL_MAS
