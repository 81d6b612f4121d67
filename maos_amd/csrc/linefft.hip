// Line FFTs in LDS (included by shwfs.hip): L lines of n points transformed
// in place by one block, for the large-field Shack-Hartmann passes and the
// pyramid WFS.
//
// The transform is a Stockham autosort over few, large radices (2 to 10, 12,
// 16 and 18; at most four stages up to 4096 points where the length allows).
// What bounds such a pass is the chain of its stages: an LDS round trip, the
// twiddle loads and barriers each.  So
//  - the radices are large (512 = 8 8 8, 480 = 16 6 5, 2916 = 18 18 9 rather
//    than 4 3 3 3 3 3 3; as 9 9 9 4 a pyramid step of that grid took 4.13 ms
//    against 3.85), a thread holding up to LX_E points in registers;
//  - the first stage reads its points through a functor (from global memory,
//    or computed) and the last one hands its points to a functor, so a
//    transform of s stages makes s - 1 LDS round trips and touches no LDS
//    before and after;
//  - the lines are transformed in place (a stage holds all its points across
//    the barrier between its reads and writes), which halves the LDS of a
//    ping-pong pair and doubles the blocks a CU holds;
//  - every twiddle is a table entry rounded from FP64 (products of a few of
//    them cost no less time and 1.2 to 1.5 times the error of the images).
//  - the index arithmetic is per butterfly, not per point: between stages a
//    line is padded by pad elements after every Ns R of them (one chunk that
//    the stage writes), so that a butterfly's points are a uniform step apart
//    both where they are written (Ns) and where the next stage reads them
//    (rstep), and the pad is chosen on the host for the fewest bank conflicts.
constexpr int LX_MAXST = 12; // most stages
constexpr int LX_E = 18;     // most points a thread holds in a stage
struct LinePlan {
    int n, nst, cap;         // cap: fewest points per thread of any stage
    int S;                   // LDS stride of a line (odd): its most padded form
    // of stage i: radix, n / radix, n / (span radix); pad of its output and
    // the step between the points of a butterfly of its input in LDS
    int rad[LX_MAXST], nb[LX_MAXST], ts[LX_MAXST], pad[LX_MAXST], rstep[LX_MAXST];
    const float2 *tw;        // exp(-2 pi i t / n), t < n
};

// butterflies of radix R that a thread holds
__host__ __device__ constexpr int lx_per(int R) { return LX_E / R; }
// LDS cycles of the 64 lanes (8 bytes each, 64 banks of 4) that reach the
// elements at(lane): the most lanes on one pair of banks, counted per 32
template <class F>
constexpr int lx_conflicts(int lanes, F at) {
    int worst = 0, cnt[32] = {};
    for (int i = 0; i < lanes; i++) {
        const int c = ++cnt[at(i) % 32];
        worst = c > worst ? c : worst;
    }
    return worst;
}
constexpr int lx_min(int a, int b) { return a < b ? a : b; }
// the plan of the radices rad[0 .. nst)
constexpr void lx_fill(LinePlan &P, const int *rad, int nst) {
    int n = 1;
    for (int i = 0; i < nst; i++) n *= rad[i];
    P.n = n;
    P.nst = nst;
    P.cap = LX_E;
    int Ns = 1, S = n;
    for (int i = 0; i < nst; i++) {
        const int R = rad[i];
        P.rad[i] = R;
        P.nb[i] = n / R;
        P.ts[i] = n / (Ns * R);
        P.cap = lx_min(P.cap, R * lx_per(R));
        if (i > 0) P.rstep[i] = P.nb[i] + P.pad[i - 1] * (P.nb[i] / Ns);
        if (i + 1 < nst) {
            // the pad with the fewest conflicts of the stage's writes and the
            // next one's reads (lanes at consecutive butterflies)
            const int Nx = Ns * R, nbx = n / rad[i + 1];
            int least = 1 << 30;
            for (int p = 0; p <= 17; p++) {
                const int c =
                    lx_conflicts(lx_min(64, P.nb[i]), [=](int j) { return j / Ns * (Nx + p) + j % Ns; }) +
                    lx_conflicts(lx_min(64, nbx), [=](int j) { return j + j / Nx * p; });
                if (c < least) {
                    least = c;
                    P.pad[i] = p;
                }
            }
            const int padded = n + P.pad[i] * (n / Nx);
            S = padded > S ? padded : S;
        }
        Ns *= R;
    }
    P.S = S | 1;
}

// a plan in constant memory: its run-time indexed arrays are scalar loads
typedef const __attribute__((address_space(4))) LinePlan *LxPlan;
// the member of that type of a kernel's only argument, a struct
#define LX_PLAN(ARGS, MEMBER)                                                                             \
    ((LxPlan)((const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr() +    \
              offsetof(ARGS, MEMBER)))

// element i of a uniform base (32-bit offset, the base in scalar registers)
template <class T>
__device__ __forceinline__ const T &lx_at(const T *base, int i) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + (size_t)((unsigned)i * (unsigned)sizeof(T)));
}
template <class T>
__device__ __forceinline__ T &lx_at(T *base, int i) {
    return *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + (size_t)((unsigned)i * (unsigned)sizeof(T)));
}

// v, or zero: the load of v is issued either way, and its address is the
// caller's to keep in range (a branch around each load of a butterfly would
// put the loads one after another)
__device__ __forceinline__ float2 lx_sel(bool ok, float2 v) { return make_float2(ok ? v.x : 0.f, ok ? v.y : 0.f); }

// a / b for 0 <= a < 2^22 from a rounded reciprocal rb of b, corrected
__device__ __forceinline__ int qdiv(int a, int b, float rb) {
    int q = (int)((float)a * rb);
    const int r = a - __mul24(q, b);
    q += r >= b ? 1 : (r < 0 ? -1 : 0);
    return q;
}

// x k for a constant k, as if k were not rounded to FP32: the rounding of a
// root of unity shifts the gain of every transform alike (the radix-3 sine by
// 2e-8 a stage, 5e-7 of an intensity after the 24 stages of a pyramid's 2916^2
// grid), where everything else is random
__device__ __forceinline__ float mulk(float x, double k) {
    return fmaf(x, (float)k, x * (float)(k - (double)(float)k));
}
__device__ __forceinline__ float2 mulk2(float2 z, double k) { return make_float2(mulk(z.x, k), mulk(z.y, k)); }
__device__ __forceinline__ float2 mul_ti(float2 z, float t) { return make_float2(-t * z.y, t * z.x); }
// v[q] <- sum_r v[r] exp(t 2 pi i r q / R), t = +-1
template <int R>
__device__ __forceinline__ void small_dft(float2 (&v)[R], float t) {
    if constexpr (R == 2) {
        const float2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        const float2 s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const float2 s13 = cadd(v[1], v[3]), d13 = mul_ti(csub(v[1], v[3]), t);
        v[0] = cadd(s02, s13);
        v[2] = csub(s02, s13);
        v[1] = cadd(d02, d13);
        v[3] = csub(d02, d13);
    } else if constexpr (R == 8) {
        // even and odd halves by 4-point transforms, then w8^q = exp(t 2 pi i q / 8)
        // on the odd half: w8 = (1 + t i) / sqrt 2, w8^2 = t i, w8^3 = (-1 + t i) / sqrt 2
        const double h = 0.70710678118654752440;
        float2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        small_dft<4>(e, t);
        small_dft<4>(o, t);
        const float2 o1 = mul_ti(o[1], t), o3 = mul_ti(o[3], t);
        o[1] = mulk2(cadd(o[1], o1), h);
        o[2] = mul_ti(o[2], t);
        o[3] = mulk2(csub(o3, o[3]), h);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            v[q] = cadd(e[q], o[q]);
            v[q + 4] = csub(e[q], o[q]);
        }
    } else if constexpr (R == 3) {
        const double h = 0.86602540378443864676; // sqrt(3)/2
        const float2 s = cadd(v[1], v[2]), d = csub(v[1], v[2]);
        const float2 m = make_float2(v[0].x - 0.5f * s.x, v[0].y - 0.5f * s.y);
        const float2 r = mul_ti(mulk2(d, h), t);
        v[0] = cadd(v[0], s);
        v[1] = cadd(m, r);
        v[2] = csub(m, r);
    } else if constexpr (R == 7) {
        // pairs r, 7 - r: v[k] = v0 + sum_r cos(2 pi r k / 7) (v[r] + v[7-r])
        //                      + t i sum_r sin(2 pi r k / 7) (v[r] - v[7-r])
        constexpr double c[4] = {1., 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
        constexpr double sn[4] = {0., 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
        float2 a[4], b[4];
#pragma unroll
        for (int r = 1; r <= 3; r++) {
            a[r] = cadd(v[r], v[7 - r]);
            b[r] = csub(v[r], v[7 - r]);
        }
        const float2 v0 = v[0];
#pragma unroll
        for (int k = 1; k <= 3; k++) {
            float2 p = v0, q = make_float2(0.f, 0.f);
#pragma unroll
            for (int r = 1; r <= 3; r++) {
                const int m = (r * k) % 7; // cos(2 pi m / 7), sin of it with the sign of m <= 3
                const double cm = c[m <= 3 ? m : 7 - m], sm = m <= 3 ? sn[m] : -sn[7 - m];
                p = cadd(p, mulk2(a[r], cm));
                q = cadd(q, mulk2(b[r], sm));
            }
            q = mul_ti(q, t);
            v[k] = cadd(p, q);
            v[7 - k] = csub(p, q);
        }
        v[0] = cadd(v0, cadd(a[1], cadd(a[2], a[3])));
    } else { // 5: cos and sin of 2 pi/5 and 4 pi/5
        const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
        const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
        const float2 a1 = cadd(v[1], v[4]), a2 = cadd(v[2], v[3]);
        const float2 b1 = csub(v[1], v[4]), b2 = csub(v[2], v[3]);
        const float2 p1 = cadd(v[0], cadd(mulk2(a1, c1), mulk2(a2, c2)));
        const float2 p2 = cadd(v[0], cadd(mulk2(a1, c2), mulk2(a2, c1)));
        const float2 q1 = mul_ti(cadd(mulk2(b1, s1), mulk2(b2, s2)), t);
        const float2 q2 = mul_ti(csub(mulk2(b1, s2), mulk2(b2, s1)), t);
        v[0] = cadd(v[0], cadd(a1, a2));
        v[1] = cadd(p1, q1);
        v[4] = csub(p1, q1);
        v[2] = cadd(p2, q2);
        v[3] = csub(p2, q2);
    }
}

// sine and cosine of 2 pi m / R, m < R, at compile time (Taylor sums in FP64
// of the angle reduced to [-pi, pi])
template <int R>
struct LxRoots {
    double c[R], s[R];
    constexpr LxRoots() : c(), s() {
        for (int m = 0; m < R; m++) {
            const double x = 6.283185307179586476925 * (2 * m > R ? m - R : m) / R;
            double tc = 1, ts = x, sc = 1, ss = x;
            for (int k = 1; k < 16; k++) {
                tc *= -x * x / ((2 * k - 1) * (2 * k));
                ts *= -x * x / ((2 * k) * (2 * k + 1));
                sc += tc;
                ss += ts;
            }
            c[m] = sc;
            s[m] = ss;
        }
    }
};
// R1 R2 points as R2 transforms of R1 (points R2 n1 + n2), the twiddles
// w^(n2 k1) and R1 transforms of R2; output k1 + R1 k2
template <int R, bool INV>
__device__ __forceinline__ void lx_dft(float2 (&v)[R]);
template <int R1, int R2, bool INV>
__device__ __forceinline__ void comp_dft(float2 (&v)[R1 * R2]) {
    constexpr LxRoots<R1 * R2> W{};
    constexpr float t = INV ? 1.f : -1.f;
    float2 a[R2][R1];
#pragma unroll
    for (int n2 = 0; n2 < R2; n2++) {
        float2 u[R1];
#pragma unroll
        for (int n1 = 0; n1 < R1; n1++) u[n1] = v[R2 * n1 + n2];
        lx_dft<R1, INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < R1; k1++)
            if (n2 * k1) {
                const double c = W.c[(n2 * k1) % (R1 * R2)], s = t * W.s[(n2 * k1) % (R1 * R2)];
                a[n2][k1] = make_float2(mulk(u[k1].x, c) - mulk(u[k1].y, s), mulk(u[k1].x, s) + mulk(u[k1].y, c));
            } else {
                a[n2][k1] = u[k1];
            }
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; k1++) {
        float2 u[R2];
#pragma unroll
        for (int n2 = 0; n2 < R2; n2++) u[n2] = a[n2][k1];
        lx_dft<R2, INV>(u);
#pragma unroll
        for (int k2 = 0; k2 < R2; k2++) v[k1 + R1 * k2] = u[k2];
    }
}
template <int R, bool INV>
__device__ __forceinline__ void lx_dft(float2 (&v)[R]) {
    if constexpr (R == 6) comp_dft<2, 3, INV>(v);
    else if constexpr (R == 9) comp_dft<3, 3, INV>(v);
    else if constexpr (R == 10) comp_dft<2, 5, INV>(v);
    else if constexpr (R == 12) comp_dft<4, 3, INV>(v);
    else if constexpr (R == 16) comp_dft<4, 4, INV>(v);
    else if constexpr (R == 18) comp_dft<3, 6, INV>(v);
    else if constexpr (R > 1) small_dft<R>(v, INV ? 1.f : -1.f);
}
// which index of (line, butterfly) is fastest over the threads: the
// butterfly (LX_ROW: a line's points contiguous in memory) or the line
// (LX_COL: adjacent columns; L a power of two)
enum LxMap { LX_ROW = 0, LX_COL };
struct LxLines {
    int L, lgL; // lines, log2 L (LX_COL)
};
// a / b: by the compiler where b is a constant of the plan (CT), else from its
// reciprocal
template <bool CT>
__device__ __forceinline__ int lx_div(int a, int b, float rb) {
    if constexpr (CT) return (int)((unsigned)a / (unsigned)b);
    else return qdiv(a, b, rb);
}
template <int MAP, bool CT>
__device__ __forceinline__ void lx_item(int it, int nb, float rnb, const LxLines &g, int &l, int &j) {
    if constexpr (MAP == LX_COL) {
        l = it & (g.L - 1);
        j = it >> g.lgL;
    } else {
        l = lx_div<CT>(it, nb, rnb);
        j = it - __mul24(l, nb);
    }
}
// What a stage reads of its plan: at run time, stage i of span Ns ...
struct LxRtStage {
    LxPlan P;
    int i, Ns;
    static constexpr bool CT = false;
    __device__ int nb() const { return P->nb[i]; }
    __device__ int S() const { return P->S; }
    __device__ int pad() const { return P->pad[i]; }
    __device__ int prev_pad() const { return P->pad[i - 1]; }
    __device__ int rstep() const { return P->rstep[i]; }
    __device__ int ts() const { return P->ts[i]; }
    __device__ const float2 *tw() const { return P->tw; }
};
// ... or constants: the plan of radices R..., of a length that kernels are
// compiled for (tw: its twiddles)
template <int... R>
struct LxCt {
    static constexpr LinePlan make() {
        LinePlan P{};
        const int r[] = {R...};
        lx_fill(P, r, (int)sizeof...(R));
        return P;
    }
    static constexpr LinePlan P = make();
    const float2 *tw;
};
template <class CP, int I>
struct LxCtStage {
    static constexpr int span() {
        int s = 1;
        for (int i = 0; i < I; i++) s *= CP::P.rad[i];
        return s;
    }
    const float2 *tw_;
    static constexpr int Ns = span();
    static constexpr bool CT = true;
    __device__ static constexpr int nb() { return CP::P.nb[I]; }
    __device__ static constexpr int S() { return CP::P.S; }
    __device__ static constexpr int pad() { return CP::P.pad[I]; }
    __device__ static constexpr int prev_pad() { return CP::P.pad[I > 0 ? I - 1 : 0]; }
    __device__ static constexpr int rstep() { return CP::P.rstep[I]; }
    __device__ static constexpr int ts() { return CP::P.ts[I]; }
    __device__ const float2 *tw() const { return tw_; }
};
// Stage V (radix R, span Ns).  FIRST reads ld(l, j, off): point j + off of
// line l, off uniform; LAST hands st(l, d, off, v, slot) point d + off, off
// uniform (slot: the thread's register slot, a constant after unrolling); the
// others use the padded LDS lines s.  BAR: ld reads LDS that the stage
// overwrites.
template <int R, bool INV, bool FIRST, bool LAST, int MAP, bool BAR, class V, class LD, class ST>
__device__ __forceinline__ void lx_stage(float2 *s, const V P, const LxLines &g, LD &ld, ST &st) {
    constexpr int PER = lx_per(R);
    const int nb = P.nb(), Ns = P.Ns, total = g.L * nb, T = (int)blockDim.x;
    const float rnb = 1.f / (float)nb, rns = 1.f / (float)Ns;
    float2 v[PER][R];
#pragma unroll
    for (int p = 0; p < PER; p++) {
        const int it = (int)threadIdx.x + p * T;
        if (it < total) {
            int l, j;
            lx_item<MAP, V::CT>(it, nb, rnb, g, l, j);
            if constexpr (FIRST) {
#pragma unroll
                for (int r = 0; r < R; r++) v[p][r] = ld(l, j, r * nb);
            } else {
                const int q = lx_div<V::CT>(j, Ns, rns);
                const float2 *x = s + __mul24(l, P.S()) + j + __mul24(q, P.prev_pad());
#pragma unroll
                for (int r = 0; r < R; r++) v[p][r] = x[r * P.rstep()];
            }
        }
    }
    if (!FIRST || BAR) __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; p++) {
        const int it = (int)threadIdx.x + p * T;
        if (it < total) {
            int l, j;
            lx_item<MAP, V::CT>(it, nb, rnb, g, l, j);
            const int q = FIRST ? j : lx_div<V::CT>(j, Ns, rns), k = FIRST ? 0 : j - __mul24(q, Ns);
            if constexpr (!FIRST) {
                const int t = __mul24(k, P.ts());
                int tm = t;
#pragma unroll
                for (int m = 1; m < R; m++, tm += t) {
                    const float2 w = lx_at(P.tw(), tm);
                    v[p][m] = cmul(v[p][m], make_float2(w.x, INV ? -w.y : w.y));
                }
            }
            lx_dft<R, INV>(v[p]);
            if constexpr (LAST) {
#pragma unroll
                for (int r = 0; r < R; r++) st(l, __mul24(q, Ns * R) + k, r * Ns, v[p][r], p * R + r);
            } else {
                float2 *y = s + __mul24(l, P.S()) + __mul24(q, Ns * R + P.pad()) + k;
#pragma unroll
                for (int r = 0; r < R; r++) y[r * Ns] = v[p][r];
            }
        }
    }
    if (!LAST) __syncthreads();
}
// (the functors are called once per point of every radix: inlined, or the
// points would pass through memory)
#define LX_INLINE __attribute__((always_inline))
#define LX_RADIX(X)                                                                                                  \
    X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(12) X(16) X(18)
// FFT of the block's g.L lines (exp(-i ...); INV: exp(+i ...), not scaled):
// points come from ld by map MI and go to st by map MO; LDSIN: ld reads LDS.
//   Every thread of the block takes part, and
// blockDim.x plan.cap >= L n.  The LDS may be written again after the next
// barrier only.
template <bool INV, int MI, int MO, bool LDSIN, class LD, class ST>
__device__ __forceinline__ void lx_fft(float2 *s, LxPlan P, const LxLines &g, LD &&ld, ST &&st) {
#define LX_CASE(R) case R: lx_stage<R, INV, true, false, MI, LDSIN>(s, LxRtStage{P, 0, 1}, g, ld, st); break;
    switch (P->rad[0]) { LX_RADIX(LX_CASE) default: break; }
#undef LX_CASE
    int Ns = P->rad[0], i = 1;
    for (; i < P->nst - 1; i++) {
#define LX_CASE(R) case R: lx_stage<R, INV, false, false, LX_ROW, false>(s, LxRtStage{P, i, Ns}, g, ld, st); break;
        switch (P->rad[i]) { LX_RADIX(LX_CASE) default: break; }
#undef LX_CASE
        Ns *= P->rad[i];
    }
#define LX_CASE(R) case R: lx_stage<R, INV, false, true, MO, false>(s, LxRtStage{P, i, Ns}, g, ld, st); break;
    switch (P->rad[i]) { LX_CASE(1) LX_RADIX(LX_CASE) default: break; }
#undef LX_CASE
}

// the same for a plan of constants
template <bool INV, int MI, int MO, bool LDSIN, int I, class CP, class LD, class ST>
__device__ __forceinline__ void lx_stages(float2 *s, const CP &P, const LxLines &g, LD &ld, ST &st) {
    constexpr bool first = I == 0, last = I == CP::P.nst - 1;
    lx_stage<CP::P.rad[I], INV, first, last, first ? MI : last ? MO : LX_ROW, first && LDSIN>(
        s, LxCtStage<CP, I>{P.tw}, g, ld, st);
    if constexpr (!last) lx_stages<INV, MI, MO, LDSIN, I + 1>(s, P, g, ld, st);
}
template <bool INV, int MI, int MO, bool LDSIN, int... R, class LD, class ST>
__device__ __forceinline__ void lx_fft(float2 *s, const LxCt<R...> &P, const LxLines &g, LD &&ld, ST &&st) {
    lx_stages<INV, MI, MO, LDSIN, 0>(s, P, g, ld, st);
}
// a kernel's plan: constants (T an LxCt) or p
struct LxRt {};
template <class T>
__device__ __forceinline__ auto lx_pick(LxPlan p) {
    if constexpr (std::is_same<T, LxRt>::value) return p;
    else return T{p->tw};
}
// and its LDS stride of a line
template <class T>
__device__ __forceinline__ int lx_stride(const LinePlan &p) {
    if constexpr (std::is_same<T, LxRt>::value) return p.S;
    else return T::P.S;
}

// f(l, d, off, slot) for every point that lx_fft's last stage hands this
// thread by map MO (the last span is the line, so d is the butterfly)
template <int MO, class F>
__device__ __forceinline__ void lx_outputs(LxPlan P, const LxLines &g, F &&f) {
    const int i = P->nst - 1, nb = P->nb[i], total = g.L * nb;
    const float rnb = 1.f / (float)nb;
#define LX_CASE(R)                                                                                                   \
    case R:                                                                                                          \
        _Pragma("unroll") for (int p = 0; p < lx_per(R); p++) {                                                      \
            const int it = (int)threadIdx.x + p * (int)blockDim.x;                                                   \
            if (it < total) {                                                                                        \
                int l, j;                                                                                            \
                lx_item<MO, false>(it, nb, rnb, g, l, j);                                                            \
                _Pragma("unroll") for (int r = 0; r < R; r++) f(l, j, r * nb, p * R + r);                            \
            }                                                                                                        \
        }                                                                                                            \
        break;
    switch (P->rad[i]) { LX_CASE(1) LX_RADIX(LX_CASE) default: break; }
#undef LX_CASE
}

// The plan of length n (factors 2, 3, 5, 7): fewest stages, then most points
// per thread, then the smallest largest radix; the largest radix first.  There
// are always a first and a last stage: a length of one radix is split into its
// two closest factors (16 = 4 4: steps of one 16^2 field 40 -> 36 us against one
// point-heavy stage and one of radix 1), a prime has a stage of radix 1.  False
// if n does not factor so.
inline void lx_search(long n, int most, std::vector<int> &cur, std::vector<int> &best) {
    static const int rad[] = {18, 16, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    if (n == 1) {
        auto cap = [](const std::vector<int> &v) {
            int c = LX_E;
            for (int r : v) c = std::min(c, r * lx_per(r));
            return c;
        };
        if (best.empty() || cur.size() < best.size() ||
            (cur.size() == best.size() && (cap(cur) > cap(best) || (cap(cur) == cap(best) && cur[0] < best[0]))))
            best = cur;
        return;
    }
    if (!best.empty() && cur.size() >= best.size()) return;
    for (int r : rad)
        if (r <= most && n % r == 0) {
            cur.push_back(r);
            lx_search(n / r, r, cur, best);
            cur.pop_back();
        }
}
inline bool lx_plan(long n, LinePlan &P) {
    P = LinePlan{};
    if (n < 2) return false;
    std::vector<int> cur, best;
    lx_search(n, 18, cur, best);
    if (best.empty() || best.size() > (size_t)LX_MAXST - 1) return false;
    if (best.size() == 1) {
        int r = 1;
        for (int k = 2; k * k <= n; k++)
            if (n % k == 0) r = k;
        best = {(int)n / r, r};
    }
    lx_fill(P, best.data(), (int)best.size());
    return true;
}
inline void lx_twiddles(long n, std::vector<float2> &tw) {
    for (long t = 0; t < n; t++) {
        const double a = -2. * M_PI * (double)t / (double)n;
        tw.push_back(make_float2((float)std::cos(a), (float)std::sin(a)));
    }
}
// threads of a block of L lines: a multiple of 64 (8192 points, the most of a
// block, take 820 at the fewest points of any stage, 10), mul times as many if
// they fit a block
inline int lx_threads(const LinePlan &P, int L, int mul = 1) {
    return std::min(1024, mul * ((int)(((long)L * P.n + P.cap - 1) / P.cap + 63) / 64 * 64));
}
