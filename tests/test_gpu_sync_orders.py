"""Results of a step fetched in any order: one WFS of each step, then others of
the same step, all in descending and in mixed orders give what an engine read
in ascending order gives, and the order costs little."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine(ngs_small, nreal):
    from maos_amd import configs, engine
    cfg, p, layers = ngs_small
    engine.init(0)
    engine.dm2gpu([])
    for r in range(nreal):
        engine.atm2gpu(layers[r % len(layers):] + layers[:r % len(layers)], ireal=r)
    wfs = configs.wfs_specs(cfg, p) * 3
    for i, w in enumerate(wfs):
        wfs[i] = type(w)(thetax=1e-5 * i, thetay=-1e-5 * i, hs=w.hs, sigsim=w.sigsim, wvlwts=w.wvlwts)
    return engine.WfsGrad(p, wfs, nreal=nreal), cfg["sim"].dt


def test_orders_give_the_same(ngs_small):
    eng, dt = _engine(ngs_small, 8)
    ref, _ = _engine(ngs_small, 8)
    n = eng.nwfs
    print("case: %d WFS of %d pixels" % (n, eng.nsa * eng.npix), flush=True)
    assert n >= 24
    rs = np.random.RandomState(2)
    orders = [[5], [5], [7], [n - 1], list(range(n)), [3], [3, 4, n - 1, 0], list(range(n - 1, -1, -1)), [0, 0], [1, 1, 0],
              list(rs.permutation(n)), [n - 1], list(range(n - 1, -1, -1))]
    for step, order in enumerate(orders):
        eng.queue(step, dt)
        ref.queue(step, dt)
        want = [ref.sync(i) for i in range(n)]
        for k, i in enumerate(order):
            g, v = eng.sync(i, want_ints=(step + k) % 3 != 0)
            assert np.array_equal(g, want[i][0]), (step, i)
            assert v is None or np.array_equal(v, want[i][1]), (step, i)
    eng.close()
    ref.close()


def test_descending_reads_cost_as_ascending(ngs_small):
    """Each window once in either order (from the WFS asked for, descending
    reads copied 1, 2, 3, .. WFS: four times the ascending ones' time)."""
    eng, dt = _engine(ngs_small, 16)
    n = eng.nwfs
    print("case: %d WFS, both orders timed" % n, flush=True)

    def best(order):
        t = []
        for r in range(12):
            eng.queue(r, dt)
            eng.wait()
            t0 = time.perf_counter()
            for i in order:
                eng.sync(i)
            t.append(time.perf_counter() - t0)
        return min(t)
    up, down = best(range(n)), best(range(n - 1, -1, -1))
    print("ascending %.0f us, descending %.0f us" % (up * 1e6, down * 1e6), flush=True)
    eng.close()
    assert down <= 2 * up
