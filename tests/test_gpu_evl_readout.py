"""Read-out of the science evaluation on the GPU: the mean PSF in strips of
rows (windows of more than 2^21 values take several), and the
piston/tip/tilt sums over one slice of points and over many."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(n):
    c = (np.arange(n) - (n - 1) / 2) / 16
    X, Y = np.meshgrid(c, c)
    m = np.hypot(X, Y) <= c[-1] + 1e-9
    return X[m].copy(), Y[m].copy()


# P = 2 and 34: less than a tile and its remainder; 512: the widest window that
# is written to host memory (2^18 values), 514 the first that is copied; 1448: the
# widest of one strip (1448^2 < 2^21); 1450: the first of two; 2050: three, the
# last short
@pytest.mark.parametrize("N,P", [(64, 2), (64, 34), (512, 512), (1024, 514), (2048, 1448), (2048, 1450), (4096, 2050)])
def test_psf_readout_strips(N, P):
    from maos_amd import engine
    x, y = _points(25)
    print("case: PSF %d of %d^2" % (P, N), flush=True)
    emb, _ = engine.loc_embed(x, y, 1 / 16, nembed=N)
    amp = np.full(len(x), 1.0 / len(x))
    opd = np.random.default_rng(3).normal(size=len(x)) * 1e-7
    ev = engine.Evl(amp, [1e-6], [N], [P], emb)
    ev.psf_add(opd)
    got, n = ev.psf(0, 0)
    ev.close()
    f = np.zeros(N * N, dtype=complex)
    f[emb] = amp * np.exp(2j * np.pi * 1e6 * opd)
    f = np.fft.fftshift(np.fft.fft2(f.reshape(N, N)))
    h = N // 2
    want = np.abs(f[h - P // 2:h + P // 2, h - P // 2:h + P // 2]) ** 2
    # FP32 transforms: log2(N^2) <= 24 butterfly levels of 2^-24 relative to the field, twice for |.|^2
    assert n == 1 and np.linalg.norm(got - want) <= 2 * 24 * 2.0 ** -24 * np.linalg.norm(want)


# points on a 3, 65 and 301 wide disk: 9, 3,281 and 70,781, i.e. one slice of
# less than 1024, four slices and 70 (64 directions: 64)
@pytest.mark.parametrize("n,ndir", [(3, 1), (65, 3), (301, 1), (301, 64)])
def test_wavefront_error_slices(n, ndir):
    from maos_amd import engine
    x, y = _points(n)
    print("case: wavefront error, %d points, %d directions" % (len(x), ndir), flush=True)
    amp = np.linspace(1, 2, len(x))
    amp /= amp.sum()
    rng = np.random.default_rng(4)
    opd = (rng.normal(size=(ndir, 1)) * 1e-7 * x + rng.normal(size=(ndir, len(x))) * 1e-7).astype(np.float32)
    emb, _ = engine.loc_embed(x, y, 1 / 16, nembed=512)
    ev = engine.Evl(amp, [1e-6], [512], [1], emb, locx=x, locy=y, dirs=[(0, 0, 0)] * ndir)
    ev.psf_add(opd)
    rms, coeff = ev.wfe()
    ev.close()
    v = np.stack([np.ones_like(x), x, y])
    mcc = (v * amp) @ v.T
    for d in range(ndir):
        o = opd[d].astype(np.float64)
        c = v @ (amp * o)
        q = np.linalg.solve(mcc, c)
        tot, pis, ptt = (amp * o * o).sum(), c[0] ** 2 / mcc[0, 0], c @ q
        # FP64 sums: nloc roundings of 2^-53 relative to sums of the same sign, with the inverse's condition (< 1e3)
        tol = 1e3 * len(x) * 2.0 ** -53
        assert np.abs(rms[d] - [tot - pis, ptt - pis, tot - ptt]).max() <= tol * tot
        assert np.abs(coeff[d] - q).max() <= tol * np.abs(o).max() * max(1, 1 / np.abs(x).max())


def test_wavelengths_of_several_sizes():
    """Wavelengths that share a launch (the same sizes, other bands), that do
    not, a Strehl-only one between them, and scratch for one at a time (134 MB
    each of two directions) give what handles of one wavelength give."""
    from maos_amd import engine
    x, y = _points(9)
    amp = np.linspace(1, 2, len(x))
    opd = np.random.default_rng(5).normal(size=(2, len(x))) * 2e-7
    dirs = [(0, 0, 0)] * 2
    ix, iy = np.round((x - x.min()) * 16).astype(int), np.round((y - y.min()) * 16).astype(int)

    def emb(N, sy, oy):  # rows sy apart from row oy on
        return (ix + 3) + (iy * sy + oy) * N
    for spec in ([(64, 32, 1, 5), (64, 32, 5, 2), (64, 1, 1, 0), (128, 32, 3, 0)],
                 [(64, 32, 1, 5), (128, 128, 15, 0), (64, 32, 2, 5), (64, 32, 5, 2)],
                 [(4096, 2048, 500, 0), (4096, 2048, 511, 1), (4096, 2048, 300, 9)]):
        print("case: wavelengths of sizes %s" % (spec,), flush=True)
        wvl = [1e-6 * (1 + 0.1 * k) for k in range(len(spec))]
        e = [emb(N, sy, oy) for N, P, sy, oy in spec]
        ev = engine.Evl(amp, wvl, [s[0] for s in spec], [s[1] for s in spec], np.concatenate(e), dirs=dirs)
        ev.psf_add(opd)
        ev.psf_add(0.5 * opd)
        for k, (N, P, _, _) in enumerate(spec):
            one = engine.Evl(amp, [wvl[k]], [N], [P], e[k], dirs=dirs)
            one.psf_add(opd)
            one.psf_add(0.5 * opd)
            for d in range(2):
                assert np.array_equal(ev.psf(d, k)[0], one.psf(d, 0)[0])
            one.close()
        ev.close()
