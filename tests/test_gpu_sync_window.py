"""Results of a step fetched in windows of consecutive WFS: every order of the
calls, a window that ends inside the WFS list, a step queued between two calls,
and gradients without intensities give what a fresh engine gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_sync_orders_and_windows(lgs_small):
    from maos_amd import configs, engine
    cfg, p, layers = lgs_small
    engine.init(0)
    for r in range(4):
        engine.atm2gpu(layers[r:] + layers[:r], ireal=r)  # the layer order changes the rounding only a little, the wind much
    wfs = configs.wfs_specs(cfg, p)
    i0 = np.ones((p.nsa, p.npix)) + np.arange(p.npix) % 7
    m, s, _ = p.mtch(i0)

    def make():
        e = engine.WfsGrad(p, wfs, nreal=4)  # 24 WFS of 11,808 pixels: a window holds 22
        e.update_ref(m, s)
        return e
    eng, one = make(), make()
    dt = cfg["sim"].dt
    n = eng.nwfs
    print("case: 24 WFS, windows of 22", flush=True)
    want = {}
    for isim in (5, 6):
        one.queue(isim, dt)
        one.wait()
        want[isim] = [one.sync(i) for i in range(n)]
    assert not np.array_equal(want[5][0][0], want[6][0][0])

    def same(isim, i, got):
        assert np.array_equal(got[0], want[isim][i][0])
        assert got[1] is None or np.array_equal(got[1], want[isim][i][1])
    eng.queue(5, dt)
    for i in list(range(n)) + [23, 0, 22, 21, 1]:
        same(5, i, eng.sync(i))
    eng.queue(6, dt)
    for i in (20, 3, 23):
        same(6, i, eng.sync(i, want_ints=False))
    for i in (20, 3, 23):
        same(6, i, eng.sync(i))
    eng.queue(5, dt)
    same(5, 7, eng.sync(7))
    eng.queue(6, dt)
    same(6, 8, eng.sync(8))
    same(6, 7, eng.sync(7))
    eng.close()
    one.close()


def test_dm_shapes_and_geometry_change(ngs_small):
    """New shapes on the same mirrors, other mirrors, fewer and none: the OPD
    follows each upload."""
    from maos_amd import configs, engine
    cfg, p, layers = ngs_small
    engine.init(0)
    engine.atm2gpu(layers)
    wfs = configs.wfs_specs(cfg, p)
    eng = engine.WfsGrad(p, wfs)
    dt = cfg["sim"].dt

    def opd():
        eng.queue(3, dt)
        eng.wait()
        return eng.debug_opd(0)
    engine.dm2gpu([])
    base = opd()
    tol = 4 * 2.0 ** -24 * (np.abs(base).max() + 4e-6)  # FP32 sums of the OPD and flat mirrors
    for values, n, dx in [((1e-6,), 41, 0.5), ((2e-6,), 41, 0.5), ((2e-6, -5e-7), 41, 0.5), ((3e-6,), 81, 0.25),
                          ((1e-6,), 41, 0.5), ((), 0, 0)]:
        engine.dm2gpu([(np.full((n, n), v), dx, -(n // 2) * dx, -(n // 2) * dx, 0.0) for v in values])
        assert np.abs(opd() - (base - sum(values))).max() <= tol
    eng.close()
