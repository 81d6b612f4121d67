"""The static surface and piston/tip/tilt inputs of the WFS OPD on the GPU, in
every form of the kernel that writes the OPD last: the staged ray trace (32-
and 16-point tiles), the direct one (a grid coarser than the screens) and the
deformable-mirror pass; with one surface for all WFS and one for each."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndm", [0, 1, 2])
@pytest.mark.parametrize("case", ["ngs_two_wvl", "ngs_small", "lf_mixed"])
def test_opd_inputs_add_to_the_traced_opd(case, ndm, request):
    from maos_amd import configs, engine
    cfg, p, layers = request.getfixturevalue(case)
    print("case: opd inputs %s, %d DMs" % (case, ndm), flush=True)
    engine.init(0)
    engine.atm2gpu(layers)
    rs = np.random.RandomState(5)
    engine.dm2gpu([(1e-7 * rs.standard_normal((41, 41)), 0.5, -10.0, -10.0, 1000.0 * i) for i in range(ndm)])
    wfs = configs.wfs_specs(cfg, p)
    eng = engine.WfsGrad(p, wfs)
    eng.set_geom(1)  # the OPD is what is looked at: no detector tables needed
    n, nw = p.nxsa, len(wfs)
    g = np.arange(n) * p.dx
    X = (p.ptsx[:, None, None] + g[None, None, :] + 0 * g[None, :, None]).reshape(-1)
    Y = (p.ptsy[:, None, None] + g[None, :, None] + 0 * g[None, None, :]).reshape(-1)
    surf = 5e-8 * rs.standard_normal((nw + 1, p.nsa * n * n))
    ptt = rs.normal(size=(nw, 3)) * 1e-7
    isim, dt = 31, cfg["sim"].dt

    def opds():
        eng.queue(isim, dt)
        eng.wait()
        return [eng.debug_opd(i) for i in range(nw)]
    base = opds()
    # each sum rounds to FP32 (relative 2^-24 of the largest partial sum): the
    # surface, the tilt, and the surface's own conversion
    def check(s):
        for i, o in enumerate(opds()):
            want = base[i] + s[i] + ptt[i][0] + ptt[i][1] * X + ptt[i][2] * Y
            tol = 4 * 2.0 ** -24 * (np.abs(base[i]).max() + np.abs(s[i]).max() + np.abs(want).max())
            assert np.abs(o - want).max() <= tol
    for i in range(nw):
        eng.set_ptt(ptt[i], iwfs=i)
    check(np.zeros((nw, 1)))
    eng.set_opdadd(surf[nw])  # one for all
    check([surf[nw]] * nw)
    eng.set_opdadd(surf[0], iwfs=0)  # then another for the first
    check([surf[0]] + [surf[nw]] * (nw - 1))
    for i in range(nw):
        eng.set_opdadd(surf[i], iwfs=i)
    check(surf)
    eng.close()
    engine.dm2gpu([])
