"""Pyramid WFS on the GPU over batches of modulation positions, splits of a
batch, line lengths of several plans and groups of columns that the grid does
not fill, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from conftest import RAD2MAS, rel_l2

pytestmark = pytest.mark.gpu

INTS_TOL = 2e-5  # the parity bars of the pyramid
GRAD_TOL_MAS = 0.1


# positions: one; fewer than the splits; one batch exactly (32); one more than
# a batch; two rings (17 + 34 positions) and two wavelengths, whose weights differ
@pytest.mark.parametrize("pos,ring,nwvl", [(1, 1, 1), (5, 1, 1), (32, 1, 1), (33, 1, 1), (34, 2, 1), (6, 2, 2)])
# grids of 100 = 10 10, 126 = 18 7 (126 columns in groups of 16), 196 = 7 7 4 and 486 = 9 9 6
@pytest.mark.parametrize("D,dx,N", [(2.0, 1 / 16, 100), (2.56, 1 / 16, 126), (4.0, 1 / 16, 196), (5.0, 1 / 32, 486)])
def test_pywfs_batches(D, dx, N, pos, ring, nwvl):
    from maos_amd import engine
    from maos_amd.pywfs import Pywfs, PywfsCfg
    pw = Pywfs(PywfsCfg(D=D, din=0.2, order=6, dx=dx, saat=0.3, modulpos=pos, modulring=ring, modulate=3.0,
                        wvl=[0.7e-6 * (1 + 0.2 * i) for i in range(nwvl)], wvlwts=[0.7, 0.3][:nwvl] if nwvl > 1 else [1.0]))
    print("case: pyramid N=%d (%d), %d positions, %d rings, %d wavelengths" % (pw.N, N, pos, ring, nwvl), flush=True)
    eng = engine.PywfsEngine(pw)
    rng = np.random.default_rng(7)
    for scale in (1e-7, 3e-6):  # the second: several wavelengths
        opd = scale * (rng.normal() * pw.locx + rng.normal() * pw.locy ** 2 + 0.1 * rng.normal(size=pw.nloc))
        gi, gg = eng.image(opd)
        ri, rg = oracle.pywfs_image(pw, opd)
        e_i, e_g = rel_l2(gi, ri), np.abs(gg - rg).max() * RAD2MAS * pw.modulate
        print("ints %.2e grad %.2e mas" % (e_i, e_g), flush=True)
        assert e_i <= INTS_TOL and e_g <= GRAD_TOL_MAS
    eng.close()
