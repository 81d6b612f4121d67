"""Pyramid handles of several grid sizes alive at once: a handle whose line FFTs
need more LDS than a later one's gives the same results after the later one is
made and stepped."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pywfs(D, dx):
    from maos_amd.pywfs import Pywfs, PywfsCfg
    return Pywfs(PywfsCfg(D=D, din=0.2, order=6, dx=dx, saat=0.3, modulpos=2, modulate=3.0, wvl=[0.7e-6], wvlwts=[1.0]))


# 3888^2: two columns of a block take more LDS than a launch may without asking; 100^2: a third of that
def test_large_grid_after_small(D=40.0):
    from maos_amd import engine
    pw = _pywfs(D, 1 / 32)
    assert pw.N == 3888
    print("case: pyramid of %d^2, then one of 100^2" % pw.N, flush=True)
    big = engine.PywfsEngine(pw)
    opd = 1e-7 * np.random.default_rng(3).normal(size=pw.nloc)
    want = big.image(opd)
    ps = _pywfs(2.0, 1 / 16)
    assert ps.N == 100
    small = engine.PywfsEngine(ps)
    small.image(np.zeros(ps.nloc))
    got = big.image(opd)
    small.close()
    last = big.image(opd)
    big.close()
    assert np.isfinite(want[0]).all() and np.abs(want[0]).max() > 0
    for r in (got, last):
        assert np.array_equal(r[0], want[0]) and np.array_equal(r[1], want[1])
