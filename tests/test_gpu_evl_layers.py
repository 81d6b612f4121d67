"""The trace of the science evaluation for every remainder of four layers, with
layers above a direction's source, against the oracle."""
import numpy as np
import pytest

from test_gpu_evl import _oracle_opd, annulus

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nps", [0, 1, 2, 3, 4, 5, 9])
def test_trace_layer_counts(nps):
    from maos_amd import engine
    from maos_amd.powfs import AtmCfg, genatm
    print("case: evl trace, %d layers" % nps, flush=True)
    ht = [0.0, 12e3, 400.0, 11e3, 2000.0, 500.0, 13e3, 8000.0, 16e3][:nps]
    layers = genatm(AtmCfg(r0=0.186, L0=30.0, ht=ht, wt=[1 / nps] * nps, ws=[8.0 + i for i in range(nps)],
                           wddeg=[50.0 * i for i in range(nps)], dx=1 / 64, nx=256,
                           seeds=list(range(1, nps + 1)))) if nps else []
    locx, locy = annulus(3.0, 0.4, 1 / 32)
    emb, N = engine.loc_embed(locx, locy, 1 / 32, nembed=256)
    dirs = [(0.0, 0.0, 0.0), (3e-5, -2e-5, 10e3), (1e-5, 1e-5, 90e3)]
    engine.init(0)
    engine.dm2gpu([])
    engine.atm2gpu(layers, atmscale=1.1)
    ev = engine.Evl(np.full(len(locx), 1.0 / len(locx)), [1.65e-6], [N], [1], emb, locx=locx, locy=locy, dirs=dirs)
    ev.trace(23, 1 / 800, add_psf=False)
    got = ev.opd()
    ev.close()
    want = np.stack([_oracle_opd(layers, [], locx, locy, d, 23, 1 / 800, 1.1) for d in dirs])
    # FP32 screens and sums: nps + 4 roundings of 2^-24 of the largest partial sum
    tol = (nps + 4) * 2.0 ** -24 * 1.1 * sum(np.abs(L.p).max() for L in layers)
    assert np.abs(got - want).max() <= tol
    assert nps == 0 or np.abs(want[1]).max() > 0
