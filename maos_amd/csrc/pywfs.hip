// Pyramid WFS imaging on the GPU (included by shwfs.hip).
//
// One step of a pyramid WFS (pywfs_ints and pywfs_grad, lib/pywfs.c:370-522;
// the reference's GPU form is cuda/sim/pywfs.cu:160-280):
//   field   amp exp(i 2 pi opd / wvl) on the pupil points, embedded in an
//           N x N grid, forward 2-D FFT, centred and scaled so that the PSF
//           sums to one;
//   modul.  for each modulation position: the centred PSF shifted by the
//           position (rounded to a sample) times the pyramid phase mask,
//           inverse 2-D FFT, |.|^2 added to the pupil intensity;
//   DTF     pupil intensity -> FFT -> x detector transfer function ->
//           inverse FFT;
//   sample  bilinear at every subaperture centre of each pupil image;
//   grads   the quad-cell (or three-facet) combination, flux-normalised.
// Every 2-D transform is a row pass and a column pass of line FFTs in LDS
// (linefft.hip): rows are read and written whole, columns L adjacent ones at
// a time.  Layouts are [row][column] with the column contiguous;
// "transposed" arrays hold [x][y].
//
// The modulation positions go through in batches: one launch transforms the
// rows of a batch's masked PSFs into a scratch plane each, one launch takes
// the columns of those planes and sums |.|^2 over its positions in registers,
// so the pupil intensity is read and written once for a batch and a small
// grid still fills the chip (its positions shared out to splits, each with a
// sum of its own that the detector's first pass adds up).  One position at a
// time, with a transpose between the passes, the three launches of a 784^2
// grid took 26 us a position, mostly latency (196 blocks), and those of a
// 2916^2 grid 191 us, a seventh of them in the transpose.  In batches a step of
// the 784^2 grid (32 positions) takes 295 us with its read-out against 960, one
// of the 2916^2 grid 3.8 ms against 6.6.  Three positions of 2916^2: the rows 121
// us (131 MB read, 189 MB written: 2.6 TB/s; VALU issue 62%, waits 46% of the
// wave cycles), the columns 197 us (239 MB read where the planes hold 204, 37 MB
// written: 1.3 TB/s; VALU issue 33%): not the bytes, but the chain of each
// position's loads, stages and barriers at the three blocks of six waves a CU
// that its lines leave.
constexpr int MX_PY_MAXN = 4096;
constexpr int MX_PY_MAXSIDE = 4;
constexpr int MX_PY_LDS = 96 * 1024;        // most LDS of a block's lines (71,216 bytes for two columns of 4050 points)
constexpr int MX_PY_MAXB = 32;              // most positions of a batch
// bytes of scratch planes that a batch aims at (at least one plane): the
// rows' mask and PSF reads and the sum's update are shared by a batch.  Queued
// steps in us: 784^2: 32 MB 321, 64 MB 264, 140 MB 246, 205 MB and more (all 32
// positions) 227; 2916^2: one plane 3,940, two to four (140, 205, 280 MB) 3,690,
// 3,710 and 3,650, eight (560 MB) 3,360: kept at what one sensor may hold, not at
// the fastest
constexpr long MX_PY_SCRATCH = 256L << 20;
constexpr int MX_PY_MAXSPLIT = 8;           // most partial pupil intensities

enum PyMode { PY_EMBED = 0, PY_PSF, PY_MOD, PY_ACC, PY_REAL, PY_DTF, PY_IMG };

struct PyArgs {
    LinePlan plan;            // line length n
    int n, L, lgL, nlines;    // lines per block, lines of the pass
    // PY_EMBED: CSR of the band rows: (x, point) entries, duplicates resolved
    const int *rowp;
    const int2 *ent;
    const float *opd, *amp;
    double inv_wvl;
    const float2 *in;         // input (all modes but PY_EMBED, PY_REAL)
    const float *inr;         // PY_REAL: the nsplit pupil intensities
    float2 *out;
    float *outr;              // PY_ACC: pupil intensities [nsplit][n][n]; PY_IMG: image
    const float2 *mask;       // PY_MOD: pyramid mask, transposed [ux][uy]
    int y0, y1;               // PY_PSF: rows of the input that hold the field
    int npos, nsplit, first;  // PY_MOD, PY_ACC: positions of the batch, splits; first: ACC stores, else adds
    int ox[MX_PY_MAXB], oy[MX_PY_MAXB]; // PY_MOD: modulation offset (samples) of the window in the PSF
    float wt[MX_PY_MAXB];     // PY_ACC: weight of |.|^2
    float scale;              // PY_PSF: PSF normalisation
    const float *nomt;        // PY_DTF: detector transfer function, transposed [kx][ky]
};
extern __shared__ float2 pyl[];

// (the 18 points a thread holds and their twiddles: five to seven waves a SIMD;
// PY_REAL, once a step, four, with the splits' loads all in flight)
template <int MODE>
__global__ __launch_bounds__(1024) void k_py_rows(PyArgs a) {
    const int n = a.n, L = a.L, S = a.plan.S, tid = threadIdx.x;
    const LxLines ln{L, a.lgL};
    const LxPlan plan = LX_PLAN(PyArgs, plan);
    const int u = xcd_unit((int)blockIdx.x, (int)gridDim.x);
    if constexpr (MODE == PY_EMBED) {
        const int r0 = u * L;
        for (int i = tid; i < L * S; i += blockDim.x) pyl[i] = make_float2(0.f, 0.f);
        __syncthreads(); // the zeroed lines before the scatter
        for (int l = 0; l < L && r0 + l < a.nlines; l++)
            for (int k = a.rowp[r0 + l] + tid; k < a.rowp[r0 + l + 1]; k += blockDim.x) {
                const int2 en = a.ent[k];
                // the phase in revolutions, reduced in FP64
                double rev = (double)a.opd[en.y] * a.inv_wvl;
                rev -= rint(rev);
                float sn, cs;
                sincospif(2.f * (float)rev, &sn, &cs);
                const float A = a.amp[en.y];
                pyl[l * S + en.x] = make_float2(A * cs, A * sn);
            }
        __syncthreads();
        float2 *out = a.out + (long)r0 * n;
        const int nl = a.nlines - r0;
        lx_fft<false, LX_ROW, LX_ROW, true>(
            pyl, plan, ln, [&](int l, int j, int off) LX_INLINE { return pyl[__mul24(l, S) + j + off]; },
            [&](int l, int d, int off, float2 v, int) LX_INLINE {
                if (l < nl) lx_at(out + off, __mul24(l, n) + d) = v;
            });
    } else if constexpr (MODE == PY_MOD) {
        // row ux of the window: PSF row ux + ox (x), columns uy + oy (y); the
        // positions of one row group are neighbours, since they share the mask
        const int pos = u % a.npos, r0 = u / a.npos * L, ox = a.ox[pos], oy = a.oy[pos];
        const float2 *in = a.in, *mask = a.mask + (long)r0 * n;
        float2 *out = a.out + (long)pos * n * n + (long)r0 * n;
        const int nl = a.nlines - r0;
        lx_fft<true, LX_ROW, LX_ROW, false>(
            pyl, plan, ln,
            [&](int l, int j, int off) LX_INLINE {
                const int sx = r0 + l + ox, sy = j + off + oy;
                const bool ok = l < nl && sx >= 0 && sx < n && sy >= 0 && sy < n;
                const float2 p = lx_at(in, ok ? __mul24(sx, n) + sy : 0), m = lx_at(mask, ok ? __mul24(l, n) + j + off : 0);
                return lx_sel(ok, cmul(p, m));
            },
            [&](int l, int d, int off, float2 v, int) LX_INLINE {
                if (l < nl) lx_at(out + off, __mul24(l, n) + d) = v;
            });
    } else { // PY_REAL, PY_IMG
        const int r0 = u * L, nl = a.nlines - r0;
        const float2 *in = MODE == PY_IMG ? a.in + (long)r0 * n : nullptr;
        const float *inr = MODE == PY_REAL ? a.inr + (long)r0 * n : nullptr;
        const int nsplit = a.nsplit;
        const long nn = (long)n * n;
        auto store = [&](int l, int d, int off, float2 v, int) LX_INLINE {
            if (l >= nl) return;
            const int i = __mul24(l, n) + d;
            if constexpr (MODE == PY_IMG) lx_at(a.outr + (long)r0 * n + off, i) = v.x;
            else lx_at(a.out + (long)r0 * n + off, i) = v;
        };
        if (MODE == PY_IMG || nsplit == 1) {
            lx_fft<MODE == PY_IMG, LX_ROW, LX_ROW, false>(
                pyl, plan, ln,
                [&](int l, int j, int off) LX_INLINE {
                    const bool ok = l < nl;
                    const int i = ok ? __mul24(l, n) + j + off : 0;
                    if constexpr (MODE == PY_IMG) return lx_sel(ok, lx_at(in, i));
                    else return lx_sel(ok, make_float2(lx_at(inr, i), 0.f));
                },
                store);
        } else if constexpr (MODE == PY_REAL) {
            lx_fft<false, LX_ROW, LX_ROW, false>(
                pyl, plan, ln,
                [&](int l, int j, int off) LX_INLINE {
                    const bool ok = l < nl;
                    const int i = ok ? __mul24(l, n) + j + off : 0;
                    float v = 0.f;
#pragma unroll
                    for (int q = 0; q < MX_PY_MAXSPLIT; q++) { // (loads of all at once, past the last split the first again)
                        const float t = lx_at(inr + (q < nsplit ? q * nn : 0), i);
                        v += q < nsplit ? t : 0.f;
                    }
                    return make_float2(ok ? v : 0.f, 0.f);
                },
                store);
        }
    }
}

// columns c0 .. c0 + L - 1
template <int MODE>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(5))) void k_py_cols(PyArgs a) {
    const int n = a.n, L = a.L, S = a.plan.S;
    const LxLines ln{L, a.lgL};
    const LxPlan plan = LX_PLAN(PyArgs, plan);
    const int u = xcd_unit((int)blockIdx.x, (int)gridDim.x);
    const int n2 = n / 2;
    if constexpr (MODE == PY_PSF) {
        // centred (cfftshift) and scaled: column kx -> row (kx + n/2) % n of
        // the transposed PSF, ky -> (ky + n/2) % n
        const int c0 = u * L, nl = n - c0, y0 = a.y0, y1 = a.y1;
        const float2 *in = a.in + c0;
        float2 *out = a.out;
        const float sc = a.scale;
        lx_fft<false, LX_COL, LX_ROW, false>(
            pyl, plan, ln,
            [&](int l, int j, int off) LX_INLINE {
                const int e = j + off;
                const bool ok = l < nl && e >= y0 && e < y1;
                return lx_sel(ok, lx_at(in, ok ? __mul24(e, n) + l : 0));
            },
            [&](int l, int d, int off, float2 v, int) LX_INLINE {
                if (l >= nl) return;
                const int x = c0 + l, ky = d + off;
                lx_at(out, __mul24(x < n2 ? x + n2 : x - n2, n) + (ky < n2 ? ky + n2 : ky - n2)) =
                    make_float2(v.x * sc, v.y * sc);
            });
    } else if constexpr (MODE == PY_ACC) {
        // |.|^2 of this split's positions, in registers (slot: the thread's
        // point of the last stage, the same one for every position)
        const int split = u % a.nsplit, c0 = u / a.nsplit * L, nl = n - c0;
        const long nn = (long)n * n;
        float acc[LX_E];
#pragma unroll
        for (int k = 0; k < LX_E; k++) acc[k] = 0.f;
        for (int pos = split; pos < a.npos; pos += a.nsplit) {
            const float2 *in = a.in + pos * nn + c0;
            const float wt = a.wt[pos];
            __syncthreads(); // the previous position's last reads of the lines
            lx_fft<true, LX_COL, LX_ROW, false>(
                pyl, plan, ln,
                [&](int l, int j, int off) LX_INLINE {
                    const bool ok = l < nl;
                    return lx_sel(ok, lx_at(in, ok ? __mul24(j + off, n) + l : 0));
                },
                [&](int, int, int, float2 v, int slot) LX_INLINE { acc[slot] += wt * (v.x * v.x + v.y * v.y); });
        }
        float *out = a.outr + split * nn + (long)c0 * n;
        const bool first = a.first != 0;
        lx_outputs<LX_ROW>(plan, ln, [&](int l, int d, int off, int slot) LX_INLINE {
            if (l >= nl) return;
            float &o = lx_at(out + off, __mul24(l, n) + d);
            o = first ? acc[slot] : o + acc[slot];
        });
    } else { // PY_DTF: along ky, times the transfer function, then back to y
        const int c0 = u * L, nl = n - c0;
        const float2 *in = a.in + c0;
        const float *nm = a.nomt + (long)c0 * n;
        float2 *out = a.out + c0;
        lx_fft<false, LX_COL, LX_ROW, false>(
            pyl, plan, ln,
            [&](int l, int j, int off) LX_INLINE {
                const bool ok = l < nl;
                return lx_sel(ok, lx_at(in, ok ? __mul24(j + off, n) + l : 0));
            },
            [&](int l, int d, int off, float2 v, int) LX_INLINE {
                const float f = lx_at(nm + off, l < nl ? __mul24(l, n) + d : 0);
                pyl[__mul24(l, S) + d + off] = make_float2(v.x * f, v.y * f);
            });
        __syncthreads();
        lx_fft<true, LX_ROW, LX_COL, true>(
            pyl, plan, ln, [&](int l, int j, int off) LX_INLINE { return pyl[__mul24(l, S) + j + off]; },
            [&](int l, int d, int off, float2 v, int) LX_INLINE {
                if (l < nl) lx_at(out + (long)off * n, __mul24(d, n) + l) = v;
            });
    }
}

// ints[side][isa] = alpha * (bilinear sample of the image at the
// subaperture centre of that pupil image), with mkht's rules (weights <=
// 1e-15 and points off the grid dropped, no renormalisation)
struct PySampleArgs {
    const float *img;
    int n, nsa, nside;
    const double *sax, *say;        // subaperture centres (m)
    double inv_dx;                  // 1 / pupil-image sampling
    double offx[MX_PY_MAXSIDE], offy[MX_PY_MAXSIDE]; // image centre of each side (samples), minus 1/2
    double alpha;
    float *ints;
};
__global__ __launch_bounds__(256) void k_py_sample(PySampleArgs a) {
    const int i = (int)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.nsa * a.nside) return;
    const int side = i / a.nsa, isa = i - side * a.nsa;
    const double fx = a.sax[isa] * a.inv_dx + a.offx[side], fy = a.say[isa] * a.inv_dx + a.offy[side];
    const double ix = floor(fx), iy = floor(fy);
    const double wx[2] = {1. - (fx - ix), fx - ix}, wy[2] = {1. - (fy - iy), fy - iy};
    double s = 0;
    for (int q = 0; q < 4; q++) {
        const long x = (long)ix + (q & 1), y = (long)iy + (q >> 1);
        const double w = wx[q & 1] * wy[q >> 1];
        if (w > 1e-15 && x >= 0 && x < a.n && y >= 0 && y < a.n) s += w * a.img[y * a.n + x];
    }
    a.ints[i] = (float)(a.alpha * s);
}

// gradients (pywfs_grad, lib/pywfs.c:457-522), one block
struct PyGradArgs {
    const float *ints;
    int nsa, nside, sigmatch, raw;
    double gain, siglev;
    const float *saa, *gradoff; // gradoff may be null
    float *grad;
};
__global__ __launch_bounds__(256) void k_py_grad(PyGradArgs a) {
    __shared__ double red[256];
    const int tid = threadIdx.x, nsa = a.nsa;
    double s = 0;
    if (a.sigmatch == 2)
        for (int i = tid; i < nsa * a.nside; i += 256) s += (double)a.ints[i];
    red[tid] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) red[tid] += red[tid + k];
        __syncthreads();
    }
    const double imean = red[0] / nsa;
    const bool raw = a.raw || a.nside < 3;
    const int ng = raw ? a.nside : 2;
    for (int isa = tid; isa < nsa; isa += 256) {
        const float *I = a.ints + isa;
        double g[MX_PY_MAXSIDE] = {};
        if (raw) {
            for (int sd = 0; sd < a.nside; sd++) g[sd] = (double)I[sd * nsa] * (a.gain / a.siglev);
        } else {
            double isum = 0;
            if (a.sigmatch == 0) isum = a.siglev * a.saa[isa];
            else if (a.sigmatch == 1)
                for (int sd = 0; sd < a.nside; sd++) isum += I[sd * nsa];
            else isum = imean * a.saa[isa];
            const double al = a.gain / isum;
            if (a.nside == 3) {
                g[0] = ((double)I[nsa] - I[2 * nsa]) * al * 0.86602540378443865;
                g[1] = ((double)I[0] - 0.5 * ((double)I[nsa] + I[2 * nsa])) * al;
            } else {
                g[0] = ((double)I[0] - I[nsa] + I[2 * nsa] - I[3 * nsa]) * al;
                g[1] = ((double)I[0] + I[nsa] - I[2 * nsa] - I[3 * nsa]) * al;
            }
        }
        for (int k = 0; k < ng; k++) a.grad[isa + k * nsa] = (float)(g[k] - (a.gradoff ? a.gradoff[isa + k * nsa] : 0.f));
    }
}

struct mx_pywfs_s {
    int device = 0;
    hipStream_t stream = nullptr;
    long nloc = 0, n = 0, nsa = 0;
    int nwvl = 0, nside = 4, ng = 2, sigmatch = 2, raw = 0;
    double dx = 0, siglev = 1, gain = 1, thetax = 0, thetay = 0, hs = 0;
    double wvl[MX_MAXWVL] = {}, wvlwts[MX_MAXWVL] = {};
    double ampnorm = 0;
    double modulate = 0;
    int modulpos = 0, modulring = 1;
    double sioff[2 * MX_PY_MAXSIDE] = {};
    int ylo = 0, nband = 0;  // grid rows holding points
    int ireal = 0;
    LinePlan plan{};
    int nbatch = 1, nsplit = 1; // scratch planes, partial pupil intensities
    float2 *d_tw = nullptr;
    int *d_rowp = nullptr;
    int2 *d_ent = nullptr;
    double *d_locx = nullptr, *d_locy = nullptr, *d_sax = nullptr, *d_say = nullptr;
    float *d_amp = nullptr, *d_opd = nullptr, *d_saa = nullptr, *d_gradoff = nullptr;
    float2 *d_mask = nullptr;   // [nwvl][n][n] transposed
    float *d_nomt = nullptr;    // [n][n] transposed
    float2 *d_A = nullptr, *d_B = nullptr, *d_P = nullptr; // work, scratch [nbatch], centred PSF [nwvl] (transposed)
    float *d_pup = nullptr, *d_img = nullptr; // pupil intensity [nsplit], image
    float *d_ints = nullptr, *d_grad = nullptr;
    bool have_gradoff = false;
    bool timing = false;
    hipEvent_t ev[2] = {nullptr, nullptr};
    long t_n = 0;
    double t_ms = 0;
    std::vector<float> hbuf;
};

namespace {
void pywfs_release(mx_pywfs_t *h) {
    if (!h) return;
    hipSetDevice(h->device);
    if (h->stream) hipStreamSynchronize(h->stream);
    void *ptrs[] = {h->d_tw, h->d_rowp, h->d_ent, h->d_locx, h->d_locy, h->d_sax, h->d_say, h->d_amp, h->d_opd,
                    h->d_saa, h->d_gradoff, h->d_mask, h->d_nomt, h->d_A, h->d_B, h->d_P, h->d_pup, h->d_img,
                    h->d_ints, h->d_grad};
    for (void *p : ptrs)
        if (p) hipFree(p);
    for (hipEvent_t e : h->ev)
        if (e) hipEventDestroy(e);
    if (h->stream) hipStreamDestroy(h->stream);
    delete h;
}

// Lines per block: as many as 4096 points hold (a power of two, at most 16), so
// that a block has about 256 threads and a CU several blocks; columns at least
// two, since a run of L columns is what the pass reads of a row.  (Queued steps
// of 784^2: 2 columns 252 us, 4 227, 8 243, 16 257; of 2916^2: 1 column 3,810, 2
// 3,690, 4 4,360.)
int py_row_lines(long n) {
    int L = 16;
    while (L > 1 && L * n > 4096) L /= 2;
    return L;
}
int py_col_lines(long n) {
    int L = 16;
    while (L > 2 && L * n > 4096) L /= 2;
    return L;
}

int py_pass(mx_pywfs_t *h, int mode, PyArgs a, int nlines) {
    const bool cols = mode == PY_PSF || mode == PY_ACC || mode == PY_DTF;
    a.plan = h->plan;
    a.plan.tw = h->d_tw;
    a.n = (int)h->n;
    a.L = cols ? py_col_lines(h->n) : py_row_lines(h->n);
    a.lgL = ilog2c(a.L);
    a.nlines = nlines;
    const int many = mode == PY_MOD ? a.npos : mode == PY_ACC ? a.nsplit : 1;
    const dim3 grid((unsigned)((nlines + a.L - 1) / a.L * many)), block((unsigned)lx_threads(a.plan, a.L));
    const size_t lds = sizeof(float2) * (size_t)a.L * a.plan.S; // (at most MX_PY_LDS)
    switch (mode) {
    case PY_EMBED: k_py_rows<PY_EMBED><<<grid, block, lds, h->stream>>>(a); break;
    case PY_PSF: k_py_cols<PY_PSF><<<grid, block, lds, h->stream>>>(a); break;
    case PY_MOD: k_py_rows<PY_MOD><<<grid, block, lds, h->stream>>>(a); break;
    case PY_ACC: k_py_cols<PY_ACC><<<grid, block, lds, h->stream>>>(a); break;
    case PY_REAL: k_py_rows<PY_REAL><<<grid, block, lds, h->stream>>>(a); break;
    case PY_DTF: k_py_cols<PY_DTF><<<grid, block, lds, h->stream>>>(a); break;
    default: k_py_rows<PY_IMG><<<grid, block, lds, h->stream>>>(a); break;
    }
    return MX_OK;
}

// pywfs_ints and pywfs_grad on the OPD in d_opd (queued on the stream)
int py_image(mx_pywfs_t *h, double siglev) {
    const long n = h->n, nn = n * n;
    const int n2 = (int)(n / 2);
    if (h->timing) HIPCHK(hipEventRecord(h->ev[0], h->stream));
    // The PSF's normalisation is applied as the power of two next to it and
    // the weights relative to the first one's, both exact (the latter for one
    // ring and wavelength); the rest goes into the samples' FP64 factor, so
    // that no rounding of a factor scales every intensity alike.
    const double psfnorm = 1. / (std::sqrt(h->ampnorm) * (double)n), psf2 = std::exp2(std::rint(std::log2(psfnorm)));
    bool first = true;
    double wt0 = 0;
    for (int iw = 0; iw < h->nwvl; iw++) {
        float2 *P = h->d_P + (size_t)iw * nn;
        // field rows (band only) along x -> A [y][kx]; columns along y,
        // centred and scaled -> P [kx][ky]
        PyArgs e{};
        e.rowp = h->d_rowp;
        e.ent = h->d_ent;
        e.opd = h->d_opd;
        e.amp = h->d_amp;
        e.inv_wvl = 1. / h->wvl[iw];
        e.out = h->d_A + (size_t)h->ylo * n;
        py_pass(h, PY_EMBED, e, h->nband);
        PyArgs f{};
        f.in = h->d_A;
        f.out = P;
        f.y0 = h->ylo;
        f.y1 = h->ylo + h->nband;
        f.scale = (float)psf2;
        py_pass(h, PY_PSF, f, (int)n);
        // modulation positions (lib/pywfs.c:390-430), in batches: rows ux of
        // the window along uy -> scratch [position][ux][y]; columns along ux,
        // |.|^2 -> pup [split][y][x]
        const double dtheta = h->wvl[iw] / (h->dx * (double)n);
        PyArgs m{};
        m.in = P;
        m.mask = h->d_mask + (size_t)iw * nn;
        m.out = h->d_B;
        m.nsplit = h->nsplit;
        auto flush = [&]() {
            if (!m.npos) return;
            py_pass(h, PY_MOD, m, (int)n);
            PyArgs c = m;
            c.in = h->d_B;
            c.outr = h->d_pup;
            c.first = first;
            py_pass(h, PY_ACC, c, (int)n);
            first = false;
            m.npos = 0;
        };
        for (int ir = 0; ir < h->modulring; ir++) {
            const double ri = h->modulate * (ir + 1) / h->modulring;
            const int npos = h->modulpos * (ir + 1) / h->modulring;
            for (int ip = 0; ip < npos; ip++) {
                const double th = 2. * M_PI * ((double)ip / npos);
                m.ox[m.npos] = (int)std::lround(std::cos(th) * ri / dtheta);
                m.oy[m.npos] = (int)std::lround(std::sin(th) * ri / dtheta);
                const double wt = h->wvlwts[iw] / ((double)nn * npos * h->modulring);
                if (wt0 == 0) wt0 = wt;
                m.wt[m.npos] = wt0 != 0 ? (float)(wt / wt0) : 0.f;
                if (++m.npos == h->nbatch) flush();
            }
        }
        flush();
    }
    // detector transfer function: rows of the pupil intensity along x, columns
    // along y x DTF and back, rows back
    PyArgs r1{};
    r1.inr = h->d_pup;
    r1.nsplit = h->nsplit;
    r1.out = h->d_A;
    py_pass(h, PY_REAL, r1, (int)n);
    PyArgs r2{};
    r2.in = h->d_A;
    r2.nomt = h->d_nomt;
    r2.out = h->d_B;
    py_pass(h, PY_DTF, r2, (int)n);
    PyArgs r3{};
    r3.in = h->d_B;
    r3.outr = h->d_img;
    py_pass(h, PY_IMG, r3, (int)n);
    // samples and gradients
    PySampleArgs s{};
    s.img = h->d_img;
    s.n = (int)n;
    s.nsa = (int)h->nsa;
    s.nside = h->nside;
    s.sax = h->d_sax;
    s.say = h->d_say;
    s.inv_dx = 1. / h->dx;
    for (int k = 0; k < h->nside; k++) {
        s.offx[k] = h->sioff[2 * k] * n2 + n2 - 0.5;
        s.offy[k] = h->sioff[2 * k + 1] * n2 + n2 - 0.5;
    }
    s.alpha = (double)h->nsa * siglev / (double)nn * wt0 * (psfnorm / psf2) * (psfnorm / psf2);
    s.ints = h->d_ints;
    k_py_sample<<<dim3((unsigned)((h->nsa * h->nside + 255) / 256)), dim3(256), 0, h->stream>>>(s);
    PyGradArgs g{h->d_ints, (int)h->nsa, h->nside, h->sigmatch, h->raw, h->gain, h->siglev,
                 h->d_saa, h->have_gradoff ? h->d_gradoff : nullptr, h->d_grad};
    k_py_grad<<<dim3(1), dim3(256), 0, h->stream>>>(g);
    HIPCHK(hipGetLastError());
    if (h->timing) {
        HIPCHK(hipEventRecord(h->ev[1], h->stream));
        HIPCHK(hipEventSynchronize(h->ev[1]));
        float ms = 0;
        HIPCHK(hipEventElapsedTime(&ms, h->ev[0], h->ev[1]));
        h->t_ms += ms;
        h->t_n++;
    }
    return MX_OK;
}
} // namespace

#define PYCHK(call)                                                                   \
    do {                                                                              \
        hipError_t e_ = (call);                                                       \
        if (e_ != hipSuccess)                                                         \
            return fail(set_err(MX_EHIP, "%s failed: %s", #call, hipGetErrorString(e_))); \
    } while (0)

extern "C" {

int mx_pywfs_init(mx_pywfs_t **out, const mx_pywfs_cfg_t *c) {
    if (!out || !c) return set_err(MX_EINVAL, "mx_pywfs_init: null argument");
    *out = nullptr;
    const long n = c->nembed, nn = n * n;
    if (c->nloc < 1 || !c->amp || !c->embed) return set_err(MX_EINVAL, "mx_pywfs_init: no pupil points");
    if (c->nwvl < 1 || c->nwvl > MX_MAXWVL || !c->wvl) return set_err(MX_EINVAL, "mx_pywfs_init: nwvl=%d", c->nwvl);
    if (c->nside < 2 || c->nside > 4)
        return set_err(MX_EINVAL, "mx_pywfs_init: nside=%d (2, 3 or 4 pupil images)", c->nside);
    if (n % 2)
        return set_err(MX_EINVAL, "mx_pywfs_init: the FFT grid side %ld must be even", n);
    LinePlan plan;
    if (n > MX_PY_MAXN || !lx_plan(n, plan))
        return set_err(MX_EINVAL, "mx_pywfs_init: FFT grid side %ld is not a product of 2, 3, 5 and 7 up to %d", n,
                       MX_PY_MAXN);
    if (c->nsa < 1 || !c->salocx || !c->salocy || !c->sioff || !c->mask || !c->nominal)
        return set_err(MX_EINVAL, "mx_pywfs_init: missing tables");
    if (!(c->dx > 0) || c->modulpos < 1 || c->modulring < 1 || c->modulate < 0)
        return set_err(MX_EINVAL, "mx_pywfs_init: bad sampling or modulation");
    for (long i = 0; i < c->nloc; i++)
        if (c->embed[i] < 0 || c->embed[i] >= nn)
            return set_err(MX_EINVAL, "mx_pywfs_init: embed[%ld]=%ld outside the %ld^2 grid", i, c->embed[i], n);
    mx_pywfs_t *h = new mx_pywfs_t();
    auto fail = [h](int rc) {
        pywfs_release(h);
        return rc;
    };
    h->device = g_device;
    h->nloc = c->nloc;
    h->n = n;
    h->nsa = c->nsa;
    h->nwvl = c->nwvl;
    h->nside = c->nside;
    h->raw = c->raw;
    h->ng = (c->raw || c->nside < 3) ? c->nside : 2;
    h->sigmatch = c->sigmatch;
    h->dx = c->dx;
    h->siglev = c->siglev;
    h->gain = 1.;
    h->modulate = c->modulate;
    h->modulpos = c->modulpos;
    h->modulring = c->modulring;
    h->thetax = c->thetax;
    h->thetay = c->thetay;
    h->hs = std::isfinite(c->hs) ? c->hs : 0.;
    for (int iw = 0; iw < c->nwvl; iw++) {
        h->wvl[iw] = c->wvl[iw];
        h->wvlwts[iw] = c->wvlwts ? c->wvlwts[iw] : 1. / c->nwvl;
    }
    for (int k = 0; k < 2 * c->nside; k++) h->sioff[k] = c->sioff[k];
    for (long i = 0; i < c->nloc; i++) h->ampnorm += c->amp[i] * c->amp[i];
    h->plan = plan;
    PYCHK(hipSetDevice(h->device));
    {
        // the lines of a block may exceed the default dynamic LDS limit; the
        // limit belongs to the kernel, not to this handle, so it is the one that
        // every grid side fits
        const void *k[] = {reinterpret_cast<const void *>(&k_py_rows<PY_EMBED>),
                           reinterpret_cast<const void *>(&k_py_cols<PY_PSF>),
                           reinterpret_cast<const void *>(&k_py_rows<PY_MOD>),
                           reinterpret_cast<const void *>(&k_py_cols<PY_ACC>),
                           reinterpret_cast<const void *>(&k_py_rows<PY_REAL>),
                           reinterpret_cast<const void *>(&k_py_cols<PY_DTF>),
                           reinterpret_cast<const void *>(&k_py_rows<PY_IMG>)};
        for (const void *f : k) PYCHK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, MX_PY_LDS));
    }
    PYCHK(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    PYCHK(hipEventCreate(&h->ev[0]));
    PYCHK(hipEventCreate(&h->ev[1]));
    // band rows and their entries; a later point at one index replaces the
    // earlier one (locfft_psf's sequential embedding)
    long ylo = n, yhi = -1;
    for (long i = 0; i < c->nloc; i++) {
        ylo = std::min(ylo, c->embed[i] / n);
        yhi = std::max(yhi, c->embed[i] / n);
    }
    h->ylo = (int)ylo;
    h->nband = (int)(yhi - ylo + 1);
    std::vector<std::vector<std::pair<int, int>>> rows(h->nband);
    {
        // points sorted by grid index, the last of a run of equal indices kept
        std::vector<std::pair<long, long>> idx(c->nloc);
        for (long i = 0; i < c->nloc; i++) idx[i] = {c->embed[i], i};
        std::stable_sort(idx.begin(), idx.end(), [](const std::pair<long, long> &a, const std::pair<long, long> &b) {
            return a.first < b.first;
        });
        for (size_t k = 0; k < idx.size(); k++) {
            if (k + 1 < idx.size() && idx[k + 1].first == idx[k].first) continue; // a later point follows
            const long e = idx[k].first;
            rows[e / n - ylo].push_back({(int)(e % n), (int)idx[k].second});
        }
    }
    std::vector<int> rowp(h->nband + 1, 0);
    std::vector<int2> ent;
    for (int r = 0; r < h->nband; r++) {
        for (auto &p : rows[r]) ent.push_back(make_int2(p.first, p.second));
        rowp[r + 1] = (int)ent.size();
    }
    std::vector<float2> tw;
    lx_twiddles(n, tw);
    std::vector<float> amp(c->nloc);
    for (long i = 0; i < c->nloc; i++) amp[i] = (float)c->amp[i];
    std::vector<float2> mt((size_t)c->nwvl * nn);
    for (int iw = 0; iw < c->nwvl; iw++)
        for (long y = 0; y < n; y++)
            for (long x = 0; x < n; x++) {
                const double *m = c->mask + 2 * ((size_t)iw * nn + x + y * n);
                mt[(size_t)iw * nn + x * n + y] = make_float2((float)m[0], (float)m[1]);
            }
    std::vector<float> nt(nn);
    for (long y = 0; y < n; y++)
        for (long x = 0; x < n; x++) nt[x * n + y] = (float)c->nominal[x + y * n];
    auto up = [&](auto **d, const auto *src, size_t cnt) -> hipError_t {
        hipError_t e = hipMalloc((void **)d, sizeof(**d) * cnt + 16);
        if (e == hipSuccess && src) e = hipMemcpy(*d, src, sizeof(**d) * cnt, hipMemcpyHostToDevice);
        return e;
    };
    PYCHK(up(&h->d_tw, tw.data(), tw.size()));
    PYCHK(up(&h->d_rowp, rowp.data(), rowp.size()));
    PYCHK(up(&h->d_ent, ent.data(), std::max<size_t>(ent.size(), 1)));
    PYCHK(up(&h->d_amp, amp.data(), amp.size()));
    PYCHK(up(&h->d_mask, mt.data(), mt.size()));
    PYCHK(up(&h->d_nomt, nt.data(), nt.size()));
    PYCHK(up(&h->d_sax, c->salocx, (size_t)c->nsa));
    PYCHK(up(&h->d_say, c->salocy, (size_t)c->nsa));
    if (c->locx && c->locy) {
        PYCHK(up(&h->d_locx, c->locx, (size_t)c->nloc));
        PYCHK(up(&h->d_locy, c->locy, (size_t)c->nloc));
    }
    std::vector<float> ones(c->nsa, 1.f);
    PYCHK(up(&h->d_saa, ones.data(), ones.size()));
    PYCHK(up(&h->d_gradoff, (const float *)nullptr, (size_t)h->ng * c->nsa));
    PYCHK(up(&h->d_opd, (const float *)nullptr, (size_t)c->nloc));
    PYCHK(up(&h->d_A, (const float2 *)nullptr, (size_t)nn));
    {
        // positions per batch, evened out; splits of a batch's positions so
        // that the column pass has four blocks for each CU
        int npos = 0;
        for (int ir = 0; ir < h->modulring; ir++) npos += h->modulpos * (ir + 1) / h->modulring;
        npos = std::max(npos, 1);
        const int most = (int)std::max(1L, std::min({MX_PY_SCRATCH / (8 * nn), (long)MX_PY_MAXB, (long)npos}));
        const int nlaunch = (npos + most - 1) / most;
        h->nbatch = (npos + nlaunch - 1) / nlaunch;
        const int groups = (int)((n + py_col_lines(n) - 1) / py_col_lines(n));
        h->nsplit = std::max(1, std::min({h->nbatch, MX_PY_MAXSPLIT, (1024 + groups - 1) / groups}));
    }
    PYCHK(up(&h->d_B, (const float2 *)nullptr, (size_t)nn * h->nbatch));
    PYCHK(up(&h->d_P, (const float2 *)nullptr, (size_t)nn * c->nwvl));
    PYCHK(up(&h->d_pup, (const float *)nullptr, (size_t)nn * h->nsplit));
    PYCHK(up(&h->d_img, (const float *)nullptr, (size_t)nn));
    PYCHK(up(&h->d_ints, (const float *)nullptr, (size_t)c->nsa * c->nside));
    PYCHK(up(&h->d_grad, (const float *)nullptr, (size_t)h->ng * c->nsa));
    *out = h;
    return MX_OK;
}

int mx_pywfs_free(mx_pywfs_t *h) {
    pywfs_release(h);
    return MX_OK;
}

int mx_pywfs_set_calib(mx_pywfs_t *h, double gain, const double *saa, const double *gradoff) {
    if (!h || !(gain > 0)) return set_err(MX_EINVAL, "mx_pywfs_set_calib: bad argument");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream)); // a queued step may still read the tables replaced here
    h->gain = gain;
    std::vector<float> t((size_t)h->ng * h->nsa);
    if (saa) {
        for (long i = 0; i < h->nsa; i++) t[i] = (float)saa[i];
        HIPCHK(hipMemcpy(h->d_saa, t.data(), sizeof(float) * h->nsa, hipMemcpyHostToDevice));
    }
    h->have_gradoff = gradoff != nullptr;
    if (gradoff) {
        for (size_t i = 0; i < t.size(); i++) t[i] = (float)gradoff[i];
        HIPCHK(hipMemcpy(h->d_gradoff, t.data(), sizeof(float) * t.size(), hipMemcpyHostToDevice));
    }
    return MX_OK;
}

int mx_pywfs_ints_opd(mx_pywfs_t *h, const double *opd, double siglev) {
    if (!h || !opd) return set_err(MX_EINVAL, "mx_pywfs_ints_opd: bad argument");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    h->hbuf.resize(h->nloc);
    for (long i = 0; i < h->nloc; i++) h->hbuf[i] = (float)opd[i];
    HIPCHK(hipMemcpy(h->d_opd, h->hbuf.data(), sizeof(float) * h->nloc, hipMemcpyHostToDevice));
    return py_image(h, siglev);
}

int mx_pywfs_queue(mx_pywfs_t *h, long isim, double dt, double siglev) {
    if (!h) return set_err(MX_EINVAL, "mx_pywfs_queue: null handle");
    if (!h->d_locx) return set_err(MX_ESTATE, "mx_pywfs_queue: the handle was made without point coordinates");
    const int r = h->ireal;
    if (g_atm[r].nps < 0) return set_err(MX_ESTATE, "mx_pywfs_queue: no screens uploaded for realisation %d", r);
    HIPCHK(hipSetDevice(h->device));
    EvlOpdArgs a{};
    a.layers = g_dlayers + (size_t)r * MX_MAXLAYER;
    a.dms = g_dm[r].ndm ? g_ddms + (size_t)r * MX_MAXDM : nullptr;
    a.locx = h->d_locx;
    a.locy = h->d_locy;
    a.opd = h->d_opd;
    a.nloc = h->nloc;
    a.isim = isim;
    a.dt = dt;
    a.atmscale = g_atm[r].atmscale;
    a.nps = g_atm[r].nps;
    a.ndm = g_dm[r].ndm;
    a.thetax[0] = h->thetax;
    a.thetay[0] = h->thetay;
    a.hs[0] = h->hs;
    k_evl_opd<<<dim3((unsigned)((h->nloc + 255) / 256), 1), dim3(256), 0, h->stream>>>(a);
    HIPCHK(hipGetLastError());
    return py_image(h, siglev);
}

int mx_pywfs_sync(mx_pywfs_t *h, double *grad, double *ints) {
    if (!h) return set_err(MX_EINVAL, "mx_pywfs_sync: null handle");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    if (grad) {
        const size_t m = (size_t)h->ng * h->nsa;
        h->hbuf.resize(m);
        HIPCHK(hipMemcpy(h->hbuf.data(), h->d_grad, sizeof(float) * m, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < m; i++) grad[i] = h->hbuf[i];
    }
    if (ints) {
        const size_t m = (size_t)h->nside * h->nsa;
        h->hbuf.resize(m);
        HIPCHK(hipMemcpy(h->hbuf.data(), h->d_ints, sizeof(float) * m, hipMemcpyDeviceToHost));
        for (size_t i = 0; i < m; i++) ints[i] = h->hbuf[i];
    }
    return MX_OK;
}

int mx_pywfs_opd_get(mx_pywfs_t *h, double *opd) {
    if (!h || !opd) return set_err(MX_EINVAL, "mx_pywfs_opd_get: bad argument");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    h->hbuf.resize(h->nloc);
    HIPCHK(hipMemcpy(h->hbuf.data(), h->d_opd, sizeof(float) * h->nloc, hipMemcpyDeviceToHost));
    for (long i = 0; i < h->nloc; i++) opd[i] = h->hbuf[i];
    return MX_OK;
}

int mx_pywfs_set_real(mx_pywfs_t *h, int ireal) {
    if (!h || ireal < 0 || ireal >= MX_MAXREAL) return set_err(MX_EINVAL, "mx_pywfs_set_real: bad argument");
    h->ireal = ireal;
    return MX_OK;
}

int mx_pywfs_timing_enable(mx_pywfs_t *h, int enable) {
    if (!h) return set_err(MX_EINVAL, "null handle");
    h->timing = enable != 0;
    h->t_n = 0;
    h->t_ms = 0;
    return MX_OK;
}

int mx_pywfs_timing(mx_pywfs_t *h, long *nstep, double *ms) {
    if (!h) return set_err(MX_EINVAL, "null handle");
    if (nstep) *nstep = h->t_n;
    if (ms) *ms = h->t_ms;
    return MX_OK;
}

int mx_pywfs_wait(mx_pywfs_t *h) {
    if (!h) return set_err(MX_EINVAL, "null handle");
    HIPCHK(hipSetDevice(h->device));
    HIPCHK(hipStreamSynchronize(h->stream));
    return MX_OK;
}

} // extern "C"
