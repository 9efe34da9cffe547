// Per-mode tridiagonal solves for gfx950 (the reference's "Middle stuff":
// 2D_Program/solver_functions/solver.c:71-86 with the factors of
// 2D_Program/main_functions/LU.c:3-46; 3D_Program/solver_functions/
// solver.c:356-369 / cuda_kernels.cu:208-249 with 3D_Program/main_functions/
// LU.c:4-81).
//
// Mode m owns the system  sub_q x_{q-1} + dia_q x_q + sup_q x_{q+1} = d_q,
// q = 0..n-1, along the last axis (y in 2D, z in 3D).  The bands are
// rebuilt on the fly from the O(n) stencil coefficient vectors and the
// closed-form eigenvalues 2cos(k pi/(N+1)); nothing of size N^2 or N^3 is
// stored (the reference streams 48 B/DOF of L, U, Up).
//
// Block = W neighbouring modes x P chunks.  Thread (w, c) owns rows
// [s, e] of mode w in registers (row-major layout is kept: lanes w are
// adjacent in memory, so each load instruction moves W*16-byte segments).
//   1. downward sweep: row q in the form  a~_q x_s + x_q + c~_q x_{q+1} = d~_q
//   2. upward sweep:   row q in the form  a^_q x_s + x_q + c^_q x_e = d^_q
//   3. the chunk's first and last rows give two rows of a reduced
//      tridiagonal system of size 2P in (x_s^0, x_e^0, x_s^1, ...), solved by
//      parallel cyclic reduction in LDS with normalised rows;
//   4. x_q = d^_q - a^_q x_s - c^_q x_e, store.
// HBM is read once and written once; the solve may run in place.
#include <type_traits>

#include "hh_common.h"
#include "hh_internal.h"

namespace hh {

// Helmholtz mode bands.  coef is an array of complex rows: 2D [q][6] =
// (bm, am, b, a, bp, ap) with sub = bm lam + am etc.; 3D [q][12] =
// (a, b, c, d, ap, bp, cp, dp, am, bm, cm, dm) with
// dia = a lx ly + b lx + c ly + d.
// With nop > 1 operators, right-hand side b uses the table at
// coef + (b % nop) * cstride (one operator per problem of a batch).
// One row of a tridiagonal system, returned by value (reference outputs
// written under branches defeat scalar replacement and land in scratch).
template <typename OT> struct Band {
    OT sub, dia, sup;
};

// Arithmetic on the operator's coefficients, OT = C2<T> (complex bands) or
// T (real bands: every stencil coefficient real, as for real k), and on
// complex right-hand sides scaled by them.  The real form needs a quarter
// of the multiplies of the complex one and half the registers and LDS.
template <typename T, typename OT> struct OpAr;
template <typename T> struct OpAr<T, C2<T>> {
    using O = C2<T>;
    static HH_DEV O zero() { return mk<T>(0, 0); }
    static HH_DEV O one() { return mk<T>(1, 0); }
    static HH_DEV O mul(O a, O b) { return cmul<T>(a, b); }
    static HH_DEV O neg(O a) { return cneg<T>(a); }
    static HH_DEV O fms(O a, O b, O c) { return cfms<T>(a, b, c); }      // c - a b
    static HH_DEV O rcp(O a) { return crcp<T>(a); }
    static HH_DEV C2<T> xmul(O a, C2<T> x) { return cmul<T>(a, x); }
    static HH_DEV C2<T> xfms(O a, C2<T> x, C2<T> y) { return cfms<T>(a, x, y); }   // y - a x
    // y - (a x + b z), c - (a b + d e): the products summed first
    static HH_DEV C2<T> xfms2(O a, C2<T> x, O b, C2<T> z, C2<T> y) {
        return csub<T>(y, cadd<T>(cmul<T>(a, x), cmul<T>(b, z)));
    }
    static HH_DEV O fms2(O a, O b, O d, O e, O c) { return csub<T>(c, cadd<T>(cmul<T>(a, b), cmul<T>(d, e))); }
};
// Real: the fused operations are written out and nothing else is contracted, so
// that both forms of the bands (one per mode, one per row) round alike.
HH_DEV double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
HH_DEV float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
#pragma clang fp contract(off)
template <typename T> struct OpAr<T, T> {
    using O = T;
    static HH_DEV O zero() { return (T)0; }
    static HH_DEV O one() { return (T)1; }
    static HH_DEV O mul(O a, O b) { return a * b; }
    static HH_DEV O neg(O a) { return -a; }
    static HH_DEV O fms(O a, O b, O c) { return fma_(-a, b, c); }
    // rcp_nr's Newton steps hold for either sign of a nonzero argument
    static HH_DEV O rcp(O a) { return rcp_nr(a); }
    static HH_DEV C2<T> xmul(O a, C2<T> x) { return mk<T>(a * x.x, a * x.y); }
    static HH_DEV C2<T> xfms(O a, C2<T> x, C2<T> y) { return mk<T>(fma_(-a, x.x, y.x), fma_(-a, x.y, y.y)); }
    static HH_DEV C2<T> xfms2(O a, C2<T> x, O b, C2<T> z, C2<T> y) { return xfms(b, z, xfms(a, x, y)); }
    static HH_DEV O fms2(O a, O b, O d, O e, O c) { return fms(d, e, fms(a, b, c)); }
};
#pragma clang fp contract(fast)

template <typename T, int DIM, bool REAL> struct HelmBands {
    using OT = typename std::conditional<REAL, T, C2<T>>::type;
    int n, Nx, nop;
    // complex table [q][6] / [q][12]; real table: the same coefficients'
    // real parts in pairs, [q][3] / [q][6] of (re c_{2i}, re c_{2i+1})
    const C2<T> *coef;
    long cstride;
    const double *lamx, *lamy;
    struct Mode { T l0, l1, l2; const C2<T> *cf; };
    HH_DEV Mode mode(long m, int bt) const {
        Mode md;
        md.cf = coef + (long)(bt % nop) * cstride;
        if constexpr (DIM == 2) {
            md.l0 = (T)lamx[m]; md.l1 = 0; md.l2 = 0;
        } else {
            long i = m % Nx, j = m / Nx;
            T lx = (T)lamx[i], ly = (T)lamy[j];
            md.l0 = lx * ly; md.l1 = lx; md.l2 = ly;
        }
        return md;
    }
    // Bands in the reference's operation order with no fused multiply-adds
    // (2D_Program/main_functions/LU.c:16-23, 3D_Program/main_functions/
    // LU.c:34-47): the FP64 bands equal the reference's to the last bit.
    // raw: from table row q, as if it had both neighbours.
    HH_DEV Band<OT> raw(const Mode &md, int q) const {
#pragma clang fp contract(off)
        Band<OT> r;
        if constexpr (REAL) {
            if constexpr (DIM == 2) {   // pairs (bm, am), (b, a), (bp, ap)
                const C2<T> *c = md.cf + 3 * (long)q;
                const T l = md.l0;
                const C2<T> c0 = c[0], c1 = c[1], c2 = c[2];
                r.sub = c0.x * l + c0.y;
                r.dia = c1.x * l + c1.y;
                r.sup = c2.x * l + c2.y;
            } else {   // pairs (a, b), (c, d), (ap, bp), (cp, dp), (am, bm), (cm, dm)
                const C2<T> *c = md.cf + 6 * (long)q;
                const T a = md.l0, b = md.l1, g = md.l2;
                const C2<T> c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3], c4 = c[4], c5 = c[5];
                r.dia = c0.x * a + c0.y * b + c1.x * g + c1.y;
                r.sup = c2.x * a + c2.y * b + c3.x * g + c3.y;
                r.sub = c4.x * a + c4.y * b + c5.x * g + c5.y;
            }
        } else if constexpr (DIM == 2) {
            const C2<T> *c = md.cf + 6 * (long)q;
            const T l = md.l0;
            r.sub = mk<T>(c[0].x * l + c[1].x, c[0].y * l + c[1].y);
            r.dia = mk<T>(c[2].x * l + c[3].x, c[2].y * l + c[3].y);
            r.sup = mk<T>(c[4].x * l + c[5].x, c[4].y * l + c[5].y);
        } else {
            const C2<T> *c = md.cf + 12 * (long)q;
            const T a = md.l0, b = md.l1, g = md.l2;
            r.dia = mk<T>(c[0].x * a + c[1].x * b + c[2].x * g + c[3].x, c[0].y * a + c[1].y * b + c[2].y * g + c[3].y);
            r.sup = mk<T>(c[4].x * a + c[5].x * b + c[6].x * g + c[7].x, c[4].y * a + c[5].y * b + c[6].y * g + c[7].y);
            r.sub = mk<T>(c[8].x * a + c[9].x * b + c[10].x * g + c[11].x,
                          c[8].y * a + c[9].y * b + c[10].y * g + c[11].y);
        }
        return r;
    }
    // the first row has no sub-, the last no superdiagonal
    HH_DEV Band<OT> ends(Band<OT> r, int q) const {
        const T ms = q > 0 ? (T)1 : (T)0, ps = q < n - 1 ? (T)1 : (T)0;
        if constexpr (REAL) {
            r.sub *= ms;
            r.sup *= ps;
        } else {
            r.sub = cscale<T>(r.sub, ms);
            r.sup = cscale<T>(r.sup, ps);
        }
        return r;
    }
};

// Helmholtz problem: bands from HelmBands, right-hand side and solution in
// the row-major field (element (b, m, q) at b*field + m + q*S), or, with
// tw > 0, the mode-tiled one the row DSTs write for it (tiles of tw
// neighbouring modes, tile t0 = m & ~(tw-1) holding its modes for all n rows
// contiguously: b*field + t0*n + q*w + (m - t0), w = min(tw, nmodes - t0)),
// where each thread's rows are whole w*16-byte segments one after another.
template <typename T_, typename Ti_, typename To_, int DIM_, bool REAL_> struct HelmProb {
    using T = T_;
    using Ti = Ti_;
    using To = To_;
    static constexpr int DIM = DIM_;
    static constexpr bool REAL = REAL_;
    using OT = typename HelmBands<T, DIM, REAL>::OT;
    HelmBands<T, DIM, REAL> bands;
    const C2<Ti> *in;
    C2<To> *out;
    long field, S, nmodes;
    int tw;
    const uint32_t *fbits;   // near-resonant modes, solved by chain_block: not stored by tri_block
    int fwords;
    const uint32_t *uni;     // per operator: every row of its table is the same
    struct Mode { typename HelmBands<T, DIM, REAL>::Mode bm; long off, step; };
    HH_DEV int n() const { return bands.n; }
    // where mode m's rows lie in a field
    HH_DEV void place(long m, long &off, long &step) const {
        if (tw == 0) {
            off = m;
            step = S;
        } else {
            const long t0 = m & ~(long)(tw - 1);
            step = min((long)tw, nmodes - t0);
            off = t0 * bands.n + (m - t0);
        }
    }
    HH_DEV Mode mode(long m, int bt) const {
        Mode md;
        md.bm = bands.mode(m, bt);
        place(m, md.off, md.step);
        return md;
    }
    HH_DEV Band<OT> raw(const Mode &md, int q) const { return bands.raw(md.bm, q); }
    HH_DEV Band<OT> ends(Band<OT> r, int q) const { return bands.ends(r, q); }
    HH_DEV bool uniform(int o) const { return uni[o] != 0; }
    HH_DEV C2<T> rhs(int b, const Mode &md, int q) const {
        return cconv<T, Ti>(in[b * field + md.off + (long)q * md.step]);
    }
    HH_DEV void store(int b, const Mode &md, int q, C2<T> x) const {
        out[b * field + md.off + (long)q * md.step] = cconv<To, T>(x);
    }
    HH_DEV bool skip(int o, long m) const { return fbits && ((fbits[(long)o * fwords + (m >> 5)] >> (m & 31)) & 1u); }
};

// Blocks are dealt round-robin to the 8 XCDs (block b runs on XCD b % 8).
// Neighbouring mode tiles share cache lines when W*sizeof(complex) < 128,
// so tiles are renumbered to run consecutively on one XCD and its L2.
HH_DEV long xcd_tile(long b, long G) {
    const long G8 = G & ~7L;
    if (b >= G8) return b;
    return (b & 7) * (G8 >> 3) + (b >> 3);
}

// NR right-hand sides that share the operator (indices o, o+nop, o+2 nop,
// ... of a batch) ride through one thread: the operator-only quantities
// (bands, pivots, the a~, c~ coefficients of the sweeps and the A, C of the
// reduced rows) are computed once for all of them, only the right-hand-side
// recurrences are repeated.  Block (mode tile, y): operator o = y % nop,
// right-hand sides o + nop (NR (y / nop) + r), r < NR, those past the batch
// are computed on a clamped index and not stored.
template <typename T, int MMAX, int NR, bool UNI, class Prob>
HH_DEV void tri_block(const Prob &prob, long nmodes, int W, int P, int batch, int nop, int g0, int by, int gy) {
    using OT = typename Prob::OT;
    using O = OpAr<T, OT>;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    // two buffers of the reduced rows, each [A | C | D_0 .. D_{NR-1}], rows x W;
    // A and C are operator values (OT), the D the right-hand sides (complex)
    const int RR = 2 * P;
    const int RW = RR * W;
    const int BUFB = RW * (int)(2 * sizeof(OT) + NR * sizeof(C2<T>));   // bytes per buffer (< 160 KiB)
    auto bufA = [&](int k) { return reinterpret_cast<OT *>(smem_raw + k * BUFB); };
    auto bufC = [&](int k) { return reinterpret_cast<OT *>(smem_raw + k * BUFB) + RW; };
    auto bufD = [&](int k) { return reinterpret_cast<C2<T> *>(reinterpret_cast<OT *>(smem_raw + k * BUFB) + 2 * RW); };
    const int n = prob.n();
    const int w = threadIdx.x % W, c = threadIdx.x / W;
    const long m = xcd_tile(blockIdx.x, gridDim.x) * W + w;
    const bool valid = (c < P) && (m < nmodes);
    // right-hand-side groups in reverse launch order: the row transform
    // before this pass wrote the last right-hand sides last, so they are the
    // ones still in the memory-side cache when the pass starts (and the
    // first ones this pass writes last, where the next row transform starts)
    const int ng = gy / nop;
    const int o = by % nop, jg = g0 + (ng - 1 - by / nop);
    int bidx[NR];
    bool bok[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int b = o + nop * (jg * NR + r);
        bok[r] = b < batch;
        bidx[r] = bok[r] ? b : (o < batch ? o : 0);
    }
    // Idle lanes (c >= P, padding modes) run the same code on a clamped
    // chunk and mode so that every load is in bounds and no branch splits
    // the sweeps; their results are discarded.
    const int cq = c < P ? c : P - 1;
    const int s = (int)(((long)cq * n) / P), e = (int)(((long)(cq + 1) * n) / P) - 1;
    const int len = e - s + 1;   // 2 <= len <= MMAX
    const auto md = prob.mode(m < nmodes ? m : nmodes - 1, bidx[0]);
    const bool skip = prob.skip(o, m < nmodes ? m : nmodes - 1);   // asked for early: the stores wait for it

    // 0. issue every right-hand-side load of the chunk up front (rows past
    //    e repeat row e), so that the HBM latency is paid once per chunk and
    //    not once per row of the recurrence
    C2<T> db[NR][MMAX];
    OT ab[MMAX], cb[MMAX];
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int t = 0; t < MMAX; t++) db[r][t] = prob.rhs(bidx[r], md, min(s + t, e));
    // An operator whose table rows are all equal (constant k) has one band per
    // mode: its 3 (2D) or 6 (3D) loads are made once, not per row.
    Band<OT> same;
    if constexpr (UNI) same = prob.raw(md, 0);
    auto band = [&](int q) {
        if constexpr (UNI) return prob.ends(same, q);
        else return prob.ends(prob.raw(md, q), q);
    };
    const Band<OT> bs = band(s);
    const OT sub_s = bs.sub, dia_s = bs.dia, sup_s = bs.sup;
    C2<T> d_s[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) d_s[r] = db[r][0];

    // 1. downward sweep over rows s+1..e: row s+t becomes
    //    ab[t] x_s + x_{s+t} + cb[t] x_{s+t+1} = db[t]
    OT pa = O::zero(), pc = O::zero();
    C2<T> pd[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) pd[r] = mk<T>(0, 0);
#pragma unroll
    for (int t = 1; t < MMAX; t++) {
        const Band<OT> bq = band(min(s + t, e));
        const OT a = bq.sub;
        const OT den = (t == 1) ? bq.dia : O::fms(a, pc, bq.dia);
        const OT rc = O::rcp(den);
        const OT na = (t == 1) ? O::mul(a, rc) : O::neg(O::mul(O::mul(a, pa), rc));
        const OT nc = O::mul(bq.sup, rc);
        C2<T> nd[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) nd[r] = (t == 1) ? O::xmul(rc, db[r][t]) : O::xmul(rc, O::xfms(a, pd[r], db[r][t]));
        if (t < len) {   // selects, not a branch
            ab[t] = na; cb[t] = nc;
            pa = na; pc = nc;
#pragma unroll
            for (int r = 0; r < NR; r++) { db[r][t] = nd[r]; pd[r] = nd[r]; }
        }
    }
    // reduced row 2c+1 (x_e): pa x_s + x_e + pc x_{e+1} = pd  (already normalised)
    OT A1 = pa, C1 = pc;
    C2<T> D1[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) D1[r] = pd[r];
    // 2. upward sweep over rows e-2..s+1 (row e-1 keeps its downward form):
    //    row s+t becomes ab[t] x_s + x_{s+t} + cb[t] x_e = db[t]
#pragma unroll
    for (int t = MMAX - 3; t >= 1; t--) {
        const OT cbt = cb[t];
        const OT na = O::fms(cbt, ab[t + 1], ab[t]);
        const OT nc = O::neg(O::mul(cbt, cb[t + 1]));
        C2<T> nd[NR];
#pragma unroll
        for (int r = 0; r < NR; r++) nd[r] = O::xfms(cbt, db[r][t + 1], db[r][t]);
        if (t <= len - 3) {
            ab[t] = na; cb[t] = nc;
#pragma unroll
            for (int r = 0; r < NR; r++) db[r][t] = nd[r];
        }
    }
    // reduced row 2c (x_s): sub_s x_{s-1} + B x_s + C x_e = D
    OT B0, C0;
    C2<T> D0[NR];
    if (len >= 3) {
        B0 = O::fms(sup_s, ab[1], dia_s);
        C0 = O::neg(O::mul(sup_s, cb[1]));
#pragma unroll
        for (int r = 0; r < NR; r++) D0[r] = O::xfms(sup_s, db[r][1], d_s[r]);
    } else {
        B0 = dia_s; C0 = sup_s;
#pragma unroll
        for (int r = 0; r < NR; r++) D0[r] = d_s[r];
    }
    OT A0;
    {
        const OT rc = O::rcp(B0);
        A0 = O::mul(sub_s, rc);
        C0 = O::mul(C0, rc);
#pragma unroll
        for (int r = 0; r < NR; r++) D0[r] = O::xmul(rc, D0[r]);
    }
    if (!valid) {  // identity rows for idle threads and padding modes
        A0 = C0 = A1 = C1 = O::zero();
#pragma unroll
        for (int r = 0; r < NR; r++) D0[r] = D1[r] = mk<T>(0, 0);
    }
    // 3. PCR on the reduced system, rows r0 = 2c, r1 = 2c+1, layout [row][W].
    //    Two LDS buffers: step i reads buffer i%2 and writes the other, so
    //    one barrier per step suffices.
    // state of the thread's two reduced rows q = 2c + h, h = 0 (x_s), 1 (x_e),
    // row q at LDS slot q W + w.  (Slots (q & 1) P + (q >> 1), free of the
    // two-way bank conflicts of this layout, measured 7% slower: 872 against
    // 811 us at N=1023 x 64 right-hand sides.)
    auto slot = [&](int q) { return q * W + w; };
    OT PA[2] = {A0, A1}, PC[2] = {C0, C1};
    C2<T> PD[2][NR];
#pragma unroll
    for (int r = 0; r < NR; r++) { PD[0][r] = D0[r]; PD[1][r] = D1[r]; }
    if (c < P) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int q = 2 * c + h;
            bufA(0)[slot(q)] = PA[h];
            bufC(0)[slot(q)] = PC[h];
#pragma unroll
            for (int r = 0; r < NR; r++) bufD(0)[r * RW + slot(q)] = PD[h][r];
        }
    }
    int cur = 0;
    for (int dd = 1; dd < RR; dd <<= 1) {
        __syncthreads();
        const OT *sA = bufA(cur), *sC = bufC(cur);
        const C2<T> *sD = bufD(cur);
        OT *tA = bufA(cur ^ 1), *tC = bufC(cur ^ 1);
        C2<T> *tD = bufD(cur ^ 1);
        if (c < P) {
            // row q: A x_{q-d} + x_q + C x_{q+d} = D, eliminated against rows q-d and q+d
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int q = 2 * c + h;
                // neighbours outside the system read the row itself and are zeroed
                const int qL = q - dd, qU = q + dd;
                const bool hL = qL >= 0, hU = qU < RR;
                const int iL = slot(hL ? qL : q), iU = slot(hU ? qU : q);
                OT aL = sA[iL], cL = sC[iL], aU = sA[iU], cU = sC[iU];
                C2<T> dL[NR], dU[NR];
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    dL[r] = sD[r * RW + iL];
                    dU[r] = sD[r * RW + iU];
                }
                if (!hL) {
                    aL = cL = O::zero();
#pragma unroll
                    for (int r = 0; r < NR; r++) dL[r] = mk<T>(0, 0);
                }
                if (!hU) {
                    aU = cU = O::zero();
#pragma unroll
                    for (int r = 0; r < NR; r++) dU[r] = mk<T>(0, 0);
                }
                const OT A = PA[h], C = PC[h];
                const OT bb = O::fms2(A, cL, C, aU, O::one());
                const OT ib = O::rcp(bb);
#pragma unroll
                for (int r = 0; r < NR; r++) {
                    PD[h][r] = O::xmul(ib, O::xfms2(A, dL[r], C, dU[r], PD[h][r]));
                    tD[r * RW + slot(q)] = PD[h][r];
                }
                PA[h] = O::neg(O::mul(O::mul(A, aL), ib));
                PC[h] = O::neg(O::mul(O::mul(C, cU), ib));
                tA[slot(q)] = PA[h];
                tC[slot(q)] = PC[h];
            }
        }
        cur ^= 1;
    }
#pragma unroll
    for (int r = 0; r < NR; r++) { D0[r] = PD[0][r]; D1[r] = PD[1][r]; }
    if (!valid || skip) return;
    // 4. back-substitution of the interior and store
#pragma unroll
    for (int r = 0; r < NR; r++) {
        if (!bok[r]) continue;
        const C2<T> xs = D0[r], xe = D1[r];
        const int b = bidx[r];
        prob.store(b, md, s, xs);
#pragma unroll
        for (int t = 1; t < MMAX - 1; t++) {
            if (t < len - 1) {
                const C2<T> x = O::xfms2(ab[t], xs, cb[t], xe, db[r][t]);
                prob.store(b, md, s + t, x);
            }
        }
        prob.store(b, md, e, xe);
    }
}

// Near-resonant modes: the reference's substitution (2D_Program/
// solver_functions/solver.c:71-86, 3D_Program/solver_functions/
// solver.c:356-369) in its own operation order, with the factors the host
// computed in the order of its LU():
//   y_0 = d_0,  y_q = d_q - L_q y_{q-1};
//   2D: x_q = (y_q - Up_q x_{q+1}) / U_q;   3D: x_q = (y_q - Up_q x_{q+1}) U_q,
// FP64 with no fused operations, whatever the storage type, so that for
// real operators every operation rounds as the reference's does and the
// result differs from the reference's only through its input (the
// transforms' rounding).  The 2D quotient is the correctly rounded one:
// q0 = a r, q = q0 + (a - p q0) r with r = RN(1/p) from the host and the
// residual exact by a fused multiply-add (Markstein).
//
// The recurrences are sequential, so the parallelism is across chains.  A chain
// is one near-resonant mode of one right-hand side, or, with real factors, one
// part of it: the real and imaginary parts follow independent recurrences, and
// apart they have half the instructions per row on the walk's critical path.
template <typename OT, typename V> struct SeqOps;
template <> struct SeqOps<double, double> {   // real factors, one part of the right-hand side
    static HH_DEV double fms(double a, double x, double y) {   // y - a x
#pragma clang fp contract(off)
        return y - a * x;
    }
    static HH_DEV double mul(double a, double x) { return a * x; }
    static HH_DEV double div(double a, double p, double r) {
        const double q0 = a * r;
        return __builtin_fma(__builtin_fma(-p, q0, a), r, q0);
    }
};
template <> struct SeqOps<double, double2> {   // both parts
    using P = SeqOps<double, double>;
    static HH_DEV double2 fms(double a, double2 x, double2 y) { return mk<double>(P::fms(a, x.x, y.x), P::fms(a, x.y, y.y)); }
    static HH_DEV double2 mul(double a, double2 x) { return mk<double>(a * x.x, a * x.y); }
    static HH_DEV double2 div(double2 a, double p, double r) { return mk<double>(P::div(a.x, p, r), P::div(a.y, p, r)); }
};
template <> struct SeqOps<double2, double2> {   // complex factors: C99 products, quotients through the reciprocal
    static HH_DEV double2 mul(double2 a, double2 x) {
#pragma clang fp contract(off)
        return mk<double>(a.x * x.x - a.y * x.y, a.x * x.y + a.y * x.x);
    }
    static HH_DEV double2 fms(double2 a, double2 x, double2 y) {
#pragma clang fp contract(off)
        const double2 p = mul(a, x);
        return mk<double>(y.x - p.x, y.y - p.y);
    }
    static HH_DEV double2 div(double2 a, double2, double2 r) { return mul(r, a); }
};
HH_DEV double real_of(double v, double) { return v; }
HH_DEV double2 real_of(double v, double2) { return mk<double>(v, 0); }   // a real as either type
// a or b by value (a conditional between named vectors selects an address and puts them in scratch)
HH_DEV double pick(bool c, double a, double b) { return c ? a : b; }
HH_DEV double2 pick(bool c, double2 a, double2 b) { return mk<double>(c ? a.x : b.x, c ? a.y : b.y); }
HH_DEV double shift(double v, int k, bool up) { return up ? __shfl_up(v, k, 64) : __shfl_down(v, k, 64); }
HH_DEV double2 shift(double2 v, int k, bool up) { return mk<double>(shift(v.x, k, up), shift(v.y, k, up)); }

// The chains of a launch: `blocks` blocks of C chains each (a power of two),
// in the first `rows` grid rows.  Chain = parts (b nfx + x) + part (parts: 2 where the real and imaginary part
// are chains of their own, else 1): right-hand side b, its operator's near-resonant entry x, at ent[o nfx + x] = (mode, factors'
// index) or (-1, 0) where the operator has fewer.
struct Chains {
    const int2 *ent;
    const void *fac;   // [row][index](L, P, R, Up)
    long nent, blocks;
    int nfx, C, rows;
};

// One block of chains.  Lane l holds chain l % C and, at position l / C of its
// wave, R consecutive rows in registers (all loads issued up front).  A chain's
// positions are walked in order: the C lanes of one position run their rows
// while the others wait, then hand the carried value to the next position by a
// lane shuffle, and from wave to wave through LDS.
template <int R, bool SPLIT, class Prob>
HH_DEV void chain_block(const Prob &prob, const Chains &ch, long block, int batch, int nop) {
    using OT = typename std::conditional<Prob::REAL, double, double2>::type;
    using V = typename std::conditional<SPLIT, double, double2>::type;
    using S = SeqOps<OT, V>;
    constexpr int parts = SPLIT ? 2 : 1;
    const V zero = real_of(0.0, V());
    const OT fzero = real_of(0.0, OT()), fone = real_of(1.0, OT());
    extern __shared__ __align__(16) unsigned char smem_raw[];
    V *carry = reinterpret_cast<V *>(smem_raw);   // C values
    const int n = prob.n(), C = ch.C, PW = 64 / C;   // positions per wave
    const int G = (n + R - 1) / R, NW = (G + PW - 1) / PW;   // positions and waves with rows
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if (wave >= NW && NW == 1) return;   // one wave walks alone, without barriers
    const int c = lane & (C - 1), pw = lane / C;
    const int s = (wave * PW + pw) * R;   // first row of this lane
    const long chain = block * C + c, item = chain / parts;
    const int part = (int)(chain % parts);
    int b, x;
    if (item <= 0x7fffffff) {   // as 32-bit division: a chain's latency counts
        b = (int)((unsigned)item / (unsigned)ch.nfx);
        x = (int)((unsigned)item - (unsigned)b * (unsigned)ch.nfx);
    } else {
        b = (int)(item / ch.nfx);
        x = (int)(item % ch.nfx);
    }
    // idle chains of the last block and of shorter operators run on a valid entry and store nothing
    const bool in = b < batch;
    const int bb = in ? b : 0;
    const int2 en = ch.ent[(long)(bb % nop) * ch.nfx + (in ? x : 0)];
    const bool live = in && en.x >= 0;
    long off, step;
    prob.place(live ? en.x : 0, off, step);
    off += bb * prob.field;
    const OT *fac = reinterpret_cast<const OT *>(ch.fac) + (long)en.y * 4;
    // Rows past n (the tail of the last position) become identity rows
    // (d = 0, L = 0, P = R = 1, Up = 0): the forward walk ends on them with a
    // carry nobody reads, the backward walk leaves them with 0, as it starts,
    // so every real row keeps its bits, and the walks need no per-row branch.
    V d[R];
    OT L[R], Pv[R], Rv[R], Up[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
        const int q = min(s + i, n - 1);
        const bool pad = s + i >= n;
        const auto *src = prob.in + off + q * step;
        V v;
        if constexpr (SPLIT) v = (double)reinterpret_cast<const typename Prob::Ti *>(src)[part];
        else v = mk<double>((double)src->x, (double)src->y);
        const OT *f = fac + (long)q * ch.nent * 4;
        const OT f0 = f[0], f1 = f[1], f2 = f[2], f3 = f[3];
        d[i] = pick(pad, zero, v);
        L[i] = pick(pad, fzero, f0);
        Pv[i] = pick(pad, fone, f1);
        Rv[i] = pick(pad, fone, f2);
        Up[i] = pick(pad, fzero, f3);
    }
    // forward: y_q = d_q - L_q y_{q-1} (L_0 = 0); backward: x_q = (y_q - Up_q
    // x_{q+1}) / U_q (2D) or * U_q (3D) (Up_{n-1} = 0).  cnt: the positions of a
    // wave that hold rows.  A last wave with fewer than PW has loops of its own
    // (255 x 520: 34 -> 19 us; one loop for both costs the full ones 5%).
    V cy = zero;
    auto forward = [&](int cnt, bool hand) {
        for (int pp = 0; pp < cnt; pp++) {
            if (pw == pp) {
#pragma unroll
                for (int i = 0; i < R; i++) {
                    d[i] = S::fms(L[i], cy, d[i]);
                    cy = d[i];
                }
                if (hand && pp == cnt - 1) carry[c] = cy;
            }
            if (pp < cnt - 1) cy = shift(cy, C, true);
        }
    };
    auto backward = [&](int cnt) {
        for (int pp = cnt - 1; pp >= 0; pp--) {
            if (pw == pp) {
#pragma unroll
                for (int i = R - 1; i >= 0; i--) {
                    const V a = S::fms(Up[i], cy, d[i]);
                    if constexpr (Prob::DIM == 2) d[i] = S::div(a, Pv[i], Rv[i]);
                    else d[i] = S::mul(Rv[i], a);
                    cy = d[i];
                }
                if (pp == 0) carry[c] = cy;
            }
            if (pp > 0) cy = shift(cy, C, false);
        }
    };
    const int last = G - (NW - 1) * PW;
    for (int w = 0; w < NW; w++) {
        if (wave == w) {
            if (w > 0) cy = carry[c];
            if (w == NW - 1 && last < PW) forward(last, false);
            else forward(PW, true);
        }
        if (NW > 1) __syncthreads();
    }
    cy = zero;
    for (int w = NW - 1; w >= 0; w--) {
        if (wave == w) {
            if (w < NW - 1) cy = carry[c];
            if (w == NW - 1 && last < PW) backward(last);
            else backward(PW);
        }
        if (NW > 1) __syncthreads();
    }
    if (!live) return;
#pragma unroll
    for (int i = 0; i < R; i++) {
        if (s + i >= n) break;
        auto *dst = prob.out + off + (s + i) * step;
        using To = typename Prob::To;
        if constexpr (SPLIT) reinterpret_cast<To *>(dst)[part] = (To)d[i];
        else *dst = mk<To>((To)d[i].x, (To)d[i].y);
    }
}

// Many chains: a launch of their own, both parts of a value in a lane and as
// many neighbouring modes side by side as 512 threads hold (whole cache lines a
// row).  64 x 1023^2, 1152 modes: 60 us before the elimination's 551; beside it
// as half as wide blocks of split chains the two took 618.
template <int R, class Prob>
__global__ __launch_bounds__(512) void k_chains(Prob prob, int batch, int nop, Chains ch) {
    chain_block<R, false>(prob, ch, blockIdx.x, batch, nop);
}

// Rows per lane of a chain: as many as a thread of the elimination holds, 8
// where that would set the kernel's registers (complex factors, FP32 storage).
template <typename T, int MMAX, class Prob> constexpr int chain_rows() {
    return MMAX > 8 && !(Prob::REAL && sizeof(T) == 8) ? 8 : MMAX;
}

// The mode solves of a right-hand-side slice.  The first grid rows hold the
// near-resonant modes' chains (up to one block per CU), the others the
// partitioned elimination of the rest: the two touch disjoint outputs (tri_block
// reads the near-resonant rows, which chain_block rewrites, but does not store
// what it makes of them), so the chains' latency runs beside the elimination
// instead of before it: one right-hand side at n = 100: 8.3 + 7.4 -> 7.2 us;
// 6 x 1023^2: 37 + 53 -> 59; 6 x 2047^2: 64 + 263 -> 273; complex, 12 x 511 x 640:
// 50 + 74 -> 73.
//
// Real operators whose table rows are all equal (constant k) take one band per
// mode, others one per row; which, is read from the device beside the tables,
// so that recorded work follows operators replaced later.  Both forms give the
// same bits.  Loads per row were what the pass waited for: 64 x 1023^2 599 ->
// 551 us, 2047^2 x 6 308 -> 263, 255^3 156 -> 103 to 125 (4.2 to 5.1 TB/s), 125^3
// 24.0 -> 19.2.
template <typename T, int MMAX, int NR, int NT, class Prob>
__global__ __launch_bounds__(NT) void k_tri(Prob prob, long nmodes, int W, int P, int batch, int nop, int g0, Chains ch) {
    const int by = (int)blockIdx.y - ch.rows, gy = (int)gridDim.y - ch.rows;
    if (by < 0) {
        const long id = (long)blockIdx.y * gridDim.x + blockIdx.x;
        if (id < ch.blocks) chain_block<chain_rows<T, MMAX, Prob>(), Prob::REAL>(prob, ch, id, batch, nop);
        return;
    }
    if constexpr (Prob::REAL) {
        if (prob.uniform(by % nop)) {
            tri_block<T, MMAX, NR, true>(prob, nmodes, W, P, batch, nop, g0, by, gy);
            return;
        }
    }
    tri_block<T, MMAX, NR, false>(prob, nmodes, W, P, batch, nop, g0, by, gy);
}

// Most chains, a power of two up to 64, whose g positions each fit a block of `threads` threads.
static int chains_in(int g, int threads) {
    int C = 64;
    while (C > 1 && (g + 64 / C - 1) / (64 / C) * 64 > threads) C /= 2;
    return C;
}

// 16 rows per lane with real factors; 8 with complex ones (twice the
// registers), except above n = 4096 where 512 threads need 16
template <int R, class Prob> static hipError_t launch_chains(const Prob &pb, Chains ch, long items, int batch, hipStream_t st) {
    const int g = (pb.bands.n + R - 1) / R;
    ch.C = chains_in(g, 512);
    ch.blocks = (items + ch.C - 1) / ch.C;
    if (ch.blocks > 0x7fffffffL) return hipErrorInvalidValue;
    const int threads = (g + 64 / ch.C - 1) / (64 / ch.C) * 64;
    if (threads > 512) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_chains<R, Prob>), dim3((unsigned)ch.blocks), dim3(threads), 64 * sizeof(double2), st, pb, batch,
                       pb.bands.nop, ch);
    return hipGetLastError();
}

template <typename T, int MM, int NR, class Prob>
static hipError_t launch_tri_nr(const Prob &pb, const TriHelm &t, hipStream_t st) {
    const int n = pb.bands.n, W = t.W, P = t.P, batch = t.batch, nop = pb.bands.nop;
    const long nmodes = pb.nmodes;
    if (n < 2 || batch < 1 || nop < 1) return hipErrorInvalidValue;
    // every chunk needs at least two rows, at most MM rows
    if (P < 1 || P > n / 2 || (n + P - 1) / P > MM || W * P > 1024) return hipErrorInvalidValue;
    int threads = ((W * P + 63) / 64) * 64;
    size_t shm = tri_lds_bytes(sizeof(typename Prob::OT), sizeof(C2<T>), P, W, NR);
    if (shm > 160 * 1024) return hipErrorInvalidValue;
    if (nop > 65535) return hipErrorInvalidValue;
    const int per_op = (batch + nop - 1) / nop;
    const int groups = (per_op + NR - 1) / NR;
    // grid y holds at most 65535 blocks: launch the right-hand-side groups in
    // slices, the last slice first (the kernel walks its groups backwards too)
    const int gmax = 65535 / nop;
    const int g_first = ((groups - 1) / gmax) * gmax;
    const unsigned gx = (unsigned)((nmodes + W - 1) / W);
    Chains ch{};
    if (t.nfx > 0) {
        if (!t.ent || !t.fac) return hipErrorInvalidValue;
        ch.ent = t.ent;
        ch.fac = t.fac;
        ch.nent = t.nent;
        ch.nfx = t.nfx;
        const long items = (long)t.nfx * batch;
        // Beside the elimination where one block per CU holds the chains: alone
        // in a wave (no barrier in the walk) if the blocks suffice, else as many
        // as the block's waves hold.  More take a launch of their own.
        constexpr int R = chain_rows<T, MM, Prob>();
        const int g = (n + R - 1) / R;   // positions of one chain
        const int wide = threads < g ? (g + 63) / 64 * 64 : threads;
        const long chains = items * (Prob::REAL ? 2 : 1);
        ch.C = chains_in(g, 64);
        if (g > 64 || (chains + ch.C - 1) / ch.C > 256) ch.C = chains_in(g, wide);
        ch.blocks = (chains + ch.C - 1) / ch.C;
        if (ch.blocks <= 256 && wide <= 1024 && nop * (groups - g_first) + (ch.blocks + gx - 1) / gx <= 65535) {
            ch.rows = (int)((ch.blocks + gx - 1) / gx);
            threads = wide;
            if (shm < 64 * sizeof(double2)) shm = 64 * sizeof(double2);
        } else {
            hipError_t e;
            if constexpr (Prob::REAL) e = launch_chains<16>(pb, ch, items, batch, st);
            else e = n > 4096 ? launch_chains<16>(pb, ch, items, batch, st) : launch_chains<8>(pb, ch, items, batch, st);
            if (e != hipSuccess) return e;
        }
    }
    // 512-thread bound: at most 256 VGPRs per lane and two waves per SIMD.
    // (16 FP64 rows spill a few registers there; measured faster than the
    // spill-free 256-thread bound, which leaves one wave per SIMD.)
    auto kfn = threads <= 512 ? k_tri<T, MM, NR, 512, Prob> : k_tri<T, MM, NR, 1024, Prob>;
    if (shm > 65536) {
        hipError_t e = hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        if (e != hipSuccess) return e;
    }
    for (int g0 = g_first; g0 >= 0; g0 -= gmax) {
        const int ng = groups - g0 < gmax ? groups - g0 : gmax;
        hipLaunchKernelGGL(kfn, dim3(gx, (unsigned)(ch.rows + nop * ng)), dim3(threads), shm, st, pb, nmodes, W, P, batch, nop,
                           g0, ch);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        ch.rows = 0;   // the chains ride with the first slice
    }
    return hipSuccess;
}

template <typename T, int MM, class Prob>
static hipError_t launch_tri_prob(const Prob &pb, const TriHelm &t, hipStream_t st) {
    if (t.nr == 1) return launch_tri_nr<T, MM, 1>(pb, t, st);
    if constexpr (sizeof(T) == 8) {   // several right-hand sides per thread: FP64 elimination only
        if (t.nr == 2) return launch_tri_nr<T, MM, 2>(pb, t, st);
        if (t.nr == 4) return launch_tri_nr<T, MM, 4>(pb, t, st);
    }
    return hipErrorInvalidValue;
}

void tri_shape(int n, long nmodes, int *W, int *P, int *mmax) {
    // Measured on MI355X (FP64, k = 50 compact operators, row-major field):
    // 256-thread blocks win at every length tried; 16 rows per thread above
    // n = 512 (fewer chunks, a shallower reduced system), 8 below.  n = 1023,
    // 64 x 1023 modes: W = 4 x 16 rows 809 us against 899 us for W = 2 x 8
    // rows and 917 us for W = 8 x 16; n = 255, 255^2 modes: W = 8 x 8 rows
    // 207 us against 283 us for 16 x 8.
    int mm = n > 512 ? 16 : 8;
    if (n <= 16) mm = 4;
    tri_shape_rows(n, nmodes, mm, W, P);
    *mmax = mm;
}

void tri_shape_rows(int n, long nmodes, int mm, int *W, int *P) {
    int p = (n + mm - 1) / mm;
    if (p > n / 2) p = n / 2;
    if (p < 1) p = 1;
    int w = 256 / p;
    if (w > 16) w = 16;
    if (w < 1) w = 1;
    int pw = 1;
    while (pw * 2 <= w) pw *= 2;
    w = pw;
    while (w > 1 && w / 2 >= nmodes) w /= 2;
    *W = w; *P = p;
}

template <typename T, typename Ti, typename To, int MM, int DIM, bool REAL>
static hipError_t launch_tri_r(const TriHelm &t, const void *in, void *out, hipStream_t st);

template <typename T, typename Ti, typename To, int MM, int DIM>
static hipError_t launch_tri_d(const TriHelm &t, const void *in, void *out, hipStream_t st) {
    if (t.real) return launch_tri_r<T, Ti, To, MM, DIM, true>(t, in, out, st);
    return launch_tri_r<T, Ti, To, MM, DIM, false>(t, in, out, st);
}

template <typename T, typename Ti, typename To, int MM, int DIM, bool REAL>
static hipError_t launch_tri_r(const TriHelm &t, const void *in, void *out, hipStream_t st) {
    HelmProb<T, Ti, To, DIM, REAL> pb;
    pb.bands.Nx = t.Nx;
    // the real table holds the coefficients' real parts in pairs: half the entries
    pb.bands.coef = (const C2<T> *)(REAL ? t.coefr : t.coef);
    pb.bands.nop = t.nop > 0 ? t.nop : 1;
    pb.bands.cstride = REAL ? t.cstride / 2 : t.cstride;
    pb.bands.lamx = t.lamx;
    pb.bands.lamy = t.lamy;
    pb.in = (const C2<Ti> *)in;
    pb.out = (C2<To> *)out;
    pb.field = t.field;
    long nmodes;
    if (t.dim == 2) { pb.bands.n = t.Ny; nmodes = t.Nx; pb.S = t.Nx; }
    else { pb.bands.n = t.Nz; nmodes = (long)t.Nx * t.Ny; pb.S = (long)t.Nx * t.Ny; }
    pb.nmodes = nmodes;
    // tiles are powers of two holding whole blocks of W modes
    pb.tw = t.tiled;
    pb.fbits = t.fbits;
    pb.fwords = t.fwords;
    pb.uni = t.uni;
    if (t.tiled && ((t.tiled & (t.tiled - 1)) || t.tiled % t.W)) return hipErrorInvalidValue;
    return launch_tri_prob<T, MM>(pb, t, st);
}

template <typename T, typename Ti, typename To, int MM>
static hipError_t launch_tri_t(const TriHelm &t, const void *in, void *out, hipStream_t st) {
    if (t.dim == 2) return launch_tri_d<T, Ti, To, MM, 2>(t, in, out, st);
    return launch_tri_d<T, Ti, To, MM, 3>(t, in, out, st);
}

template <typename T, typename Ti, typename To>
static hipError_t launch_tri_mm(const TriHelm &t, const void *in, void *out, hipStream_t st) {
    switch (t.mmax) {
    case 4: return launch_tri_t<T, Ti, To, 4>(t, in, out, st);
    case 8: return launch_tri_t<T, Ti, To, 8>(t, in, out, st);
    case 16: return launch_tri_t<T, Ti, To, 16>(t, in, out, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_tri_helm(const TriHelm &t, DstTypes ty, const void *in, void *out, hipStream_t st) {
    if (ty.comp == 0 && ty.in == 0 && ty.out == 0) return launch_tri_mm<double, double, double>(t, in, out, st);
    if (ty.comp == 1 && ty.in == 1 && ty.out == 1) return launch_tri_mm<float, float, float>(t, in, out, st);
    return hipErrorInvalidValue;
}

}  // namespace hh
