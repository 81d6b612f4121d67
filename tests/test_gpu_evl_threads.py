"""Several threads read the PSFs and the wavefront error of one handle that no
call steps: each gets what a single reader gets."""
import threading

import numpy as np
import pytest

from test_gpu_evl import annulus

pytestmark = pytest.mark.gpu


def test_reads_from_several_threads():
    from maos_amd import engine
    print("case: 8 threads reading windows of 64^2, 250^2 and 1024^2", flush=True)
    x, y = annulus(3.0, 0.4, 1 / 32)
    N, sizes = [256, 256, 1024], [64, 250, 1024]
    emb = np.concatenate([engine.loc_embed(x, y, 1 / 32, nembed=n)[0] for n in N])
    ndir = 4
    opd = np.random.default_rng(6).normal(size=(ndir, len(x))) * 1e-7
    ev = engine.Evl(np.full(len(x), 1.0 / len(x)), [1e-6, 1.2e-6, 1.4e-6], N, sizes, emb, locx=x, locy=y,
                    dirs=[(0, 0, 0)] * ndir)
    ev.psf_add(opd)
    keys = [(d, w) for d in range(ndir) for w in range(3)]
    want = {k: ev.psf(*k)[0] for k in keys}
    wfe = ev.wfe()
    bad = []

    def read(t):
        for r in range(12):
            k = keys[(5 * t + 7 * r) % len(keys)]
            if not np.array_equal(ev.psf(*k)[0], want[k]):
                bad.append((t, k))
            if r % 4 == 0 and not all(np.array_equal(a, b) for a, b in zip(ev.wfe(), wfe)):
                bad.append((t, "wfe"))
    th = [threading.Thread(target=read, args=(t,)) for t in range(8)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    ev.close()
    assert not bad
