// Sixth-order right-hand sides for gfx950: the compact fourth-order
// derivatives and the combination of rhs.c in two passes (2D) or three (3D).
//   2D_Program/main_functions/rhs.c:78-86,126-148 with
//   2D_Program/partial_derivatives/4th_order_*.c
//   3D_Program/main_functions/rhs.c:150-174 with
//   3D_Program/partial_derivatives/4th_order_partials.c:94-294
//
// A compact derivative is one system (1, diag, 1) s = d per grid line, with
//   second derivative (diag 10): d = 12 (f_{q+1} - 2 f_q + f_{q-1}) / h^2
//   first derivative  (diag 4):  d = 3 (f_{q+1} - f_{q-1}) / h
// and the known boundary value moved to the right-hand side of the first and
// last row.  The second difference of such an s along its own line needs no
// neighbours: s_{q-1} - 2 s_q + s_{q+1} = 12 (delta^2 f_q / h^2 - s_q), so the
// pass along a direction adds everything of that direction to the sum at once:
//   2D   x lines: write f_xx;  y lines: read f_xx and f, write F
//   3D   x lines: write f_xx;  y lines: write f_xx + f_yy and the terms of x
//        and y;  z lines: read both and f, write F
// Each pass reads and writes every line once; f_xx (2D) and the partial sum
// (3D) live in F's own storage, which the last pass rewrites in place.
//
// What bounds it: memory, 5 (2D) and 10 (3D) fields moved, where derivative
// fields on the extended grid, their zeroing and a separate combination took
// 14 and 24.  8 x 1023^2: x 75 us (3.6 TB/s), y 150 us (2.7 TB/s: 128-byte
// segments 16 KB apart), before 478 us in five kernels; 200^3: x 65, y 125, z 112
// us (4.6 TB/s), before 615 us in six.
#include <algorithm>

#include "hh_closure.h"
#include "hh_common.h"
#include "hh_internal.h"

namespace hh {

namespace {

typedef double2 z2;

HH_DEV z2 za(z2 a, z2 b) { return cadd<double>(a, b); }
HH_DEV z2 zd(z2 a, z2 b) { return csub<double>(a, b); }
HH_DEV z2 zs(z2 a, double s) { return cscale<double>(a, s); }
HH_DEV z2 zm(z2 a, z2 b) { return cmul<double>(a, b); }
// b or zero, by value (a conditional between two named vectors selects an address and puts them in scratch)
HH_DEV z2 zsel(bool c, z2 b) { return mk<double>(c ? b.x : 0.0, c ? b.y : 0.0); }
// a + s b
HH_DEV z2 zf(z2 a, double s, z2 b) { return mk<double>(__builtin_fma(s, b.x, a.x), __builtin_fma(s, b.y, a.y)); }

// Thread (w, c) of a block holds rows c MM .. c MM + MM - 1 of line w.  The
// reciprocal pivots R_0 = 1/diag, R_q = 1/(diag - R_{q-1}) reach their limit
// to the last bit within 16 rows for both diagonals; they are constants (17
// divisions, one after the other, kept each block's first loads waiting).
constexpr int CPIV = 16;
struct Pivots { double r[CPIV + 1]; };
constexpr Pivots pivots(double diag) {
    Pivots p{};
    double r = 1.0 / diag;
    for (int q = 0; q <= CPIV; q++) { p.r[q] = r; r = 1.0 / (diag - r); }
    return p;
}
__constant__ const Pivots PIVOTS[2] = {pivots(10.0), pivots(4.0)};
template <int DIAG> HH_DEV void pivot_table(double *R) {
    if (threadIdx.x <= CPIV) R[threadIdx.x] = PIVOTS[DIAG == 4].r[threadIdx.x];
}
HH_DEV double pivot(const double *R, int q) { return R[q < CPIV ? q : CPIV]; }

// A line is eliminated and substituted by chunks: each chunk runs its
// recurrence from zero, the value carried into it is assembled from the LV
// chunks before it (after it, for the substitution) and then propagated
// through the chunk.  A carry shrinks by 0.27 (diag 4) or 0.10 (diag 10) per
// row, so what lies LV chunks away is below 1e-18 of the value it would join.
template <int MM, int DIAG> struct Levels {
    static constexpr int LV = MM >= 16 ? 2 : DIAG == 4 ? 4 : 3;
};
// carry into chunk c from the chunks c + step, c + 2 step, ..: end values and
// products of their recurrences in LDS, [chunk][W]
template <int LV> HH_DEV z2 carried(const z2 *end, const double *prod, int c, int step, int P, int W, int w) {
    z2 acc = mk<double>(0, 0);
#pragma unroll
    for (int k = LV; k >= 1; k--) {
        const int cc = c + step * k;
        if (cc >= 0 && cc < P) acc = zf(end[cc * W + w], prod[cc * W + w], acc);
    }
    return acc;
}

template <int MM> HH_DEV void eliminate(z2 *v, const double *R, int q0, int n, z2 *end, double *prod) {
    double p = 1.0;
#pragma unroll
    for (int t = 0; t < MM; t++) {   // y_q = d_q - R_{q-1} y_{q-1}; rows past n stay zero
        const double L = q0 + t > 0 ? pivot(R, q0 + t - 1) : 0.0;
        if (t > 0) v[t] = zf(v[t], q0 + t < n ? -L : 0.0, v[t - 1]);
        p *= -L;
    }
    *end = v[MM - 1];
    *prod = p;
}
template <int MM> HH_DEV void eliminate_carry(z2 *v, const double *R, int q0, int n, z2 carry) {
    double p = 1.0;
#pragma unroll
    for (int t = 0; t < MM; t++) {
        p *= q0 + t > 0 && q0 + t < n ? -pivot(R, q0 + t - 1) : 0.0;
        v[t] = zf(v[t], p, carry);
    }
}
template <int MM> HH_DEV void substitute(z2 *v, const double *R, int q0, z2 *end, double *prod) {
    double p = 1.0;
#pragma unroll
    for (int t = MM - 1; t >= 0; t--) {   // x_q = (y_q - x_{q+1}) R_q
        const double r = pivot(R, q0 + t);
        v[t] = zs(t < MM - 1 ? zd(v[t], v[t + 1]) : v[t], r);
        p *= -r;
    }
    *end = v[0];
    *prod = p;
}
template <int MM> HH_DEV void substitute_carry(z2 *v, const double *R, int q0, z2 carry) {
    double p = 1.0;
#pragma unroll
    for (int t = MM - 1; t >= 0; t--) {
        p *= -pivot(R, q0 + t);
        v[t] = zf(v[t], p, carry);
    }
}

template <int MM> HH_DEV void subtract_last(z2 *v, int t, z2 x) {   // row t of the chunk, known at run time
#pragma unroll
    for (int k = 0; k < MM; k++)
        v[k] = zd(v[k], zsel(k == t, x));
}

// LDS of one system per line: pivots, end values and products of both sweeps
struct Exchange {
    double *R;
    z2 *ye, *xe;
    double *yp, *xp;
    static constexpr size_t bytes(int P, int W) { return ((CPIV + 2) + 6 * (size_t)P * W) * sizeof(double); }
    HH_DEV Exchange(unsigned char *m, int P, int W) {
        ye = reinterpret_cast<z2 *>(m);
        xe = ye + P * W;
        yp = reinterpret_cast<double *>(xe + P * W);
        xp = yp + P * W;
        R = xp + P * W;
    }
};

// Neighbouring tiles run on one XCD (blocks go round-robin to the 8 XCDs):
// they share cache lines at their edges and the rows of f beside them.
HH_DEV long xcd_order(long b, long G) {
    const long G8 = G & ~7L;
    return b >= G8 ? b : (b & 7) * (G8 >> 3) + (b >> 3);
}

// Second derivative along contiguous lines.  Line l of right-hand side b reads
// f at b fB + (l / nA) fO + (l % nA + 1) (n + 2) + fC (its first ghost) and
// writes n values at b oB + l n; the boundary values sit at b eB + e0 + (l %
// nA) + (l / nA) eA.
struct XLines {
    int n, W, P;
    int nlines, nA;
    long fB, fO, fC, oB, eB, e0, eA;
    const z2 *f, *lo, *hi;
    z2 *out;
    double rh2;   // 12 / h^2
};

constexpr int line_pad(int i) { return i + (i >> 3); }

// STAGE: lines pass through LDS so that both transfers are coalesced (a
// thread's rows are 128 contiguous bytes); without it lines longer than the
// LDS are read directly.
template <int MM, bool STAGE>
__global__ __launch_bounds__(1024) void k_compact_x(XLines a, int b0) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = a.n, P = a.P, W = a.W, nt = blockDim.x;
    Exchange ex(smem, P, W);
    z2 *line = reinterpret_cast<z2 *>(smem + (Exchange::bytes(P, W) + 15) / 16 * 16);
    const int LS = line_pad(n + 2) + 1;
    const int t = threadIdx.x;
    const int b = b0 + blockIdx.y;
    const int l0 = blockIdx.x * W;
    const int nl = min(a.nlines - l0, W);
    // this thread's line: its first ghost in f and its boundary values, asked for first
    const int w = min(t / P, W - 1), c = t - w * P;
    const bool live = c < P && w < nl;
    const int q0 = live ? c * MM : 0;
    const int l = l0 + (live ? w : 0), outer = (unsigned)l / (unsigned)a.nA, inner = l - outer * a.nA;
    const long fbase = b * a.fB + outer * a.fO + (inner + 1) * (long)(n + 2) + a.fC;
    const long eo = b * a.eB + a.e0 + inner + outer * a.eA;
    const z2 lo = a.lo[eo], hi = a.hi[eo];
    pivot_table<10>(ex.R);
    if constexpr (STAGE) {
        long *base = reinterpret_cast<long *>(ex.ye);
        if (live && c == 0) base[w] = fbase;
        __syncthreads();
        const int total = nl * (n + 2);   // eight loads in flight per thread
        // e / (n + 2) by a reciprocal, exact below 2^21 elements (the tile fits the LDS)
        const float inv = 1.0f / (float)(n + 2);
        for (int e0 = t; e0 < total; e0 += 8 * nt) {
            z2 g[8];
            int pos[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int e = min(e0 + k * nt, total - 1), w = (int)(((float)e + 0.5f) * inv), i = e - w * (n + 2);
                pos[k] = w * LS + line_pad(i);
                g[k] = a.f[base[w] + i];
            }
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (e0 + k * nt < total) line[pos[k]] = g[k];
        }
    }
    __syncthreads();
    z2 v[MM];
    {
        z2 g[MM + 2];
        const long src = STAGE ? (live ? w : 0) * LS : fbase;
#pragma unroll
        for (int k = 0; k < MM + 2; k++) {
            const int i = min(q0 + k, n + 1);
            if constexpr (STAGE) g[k] = line[src + line_pad(i)];
            else g[k] = a.f[src + i];
        }
#pragma unroll
        for (int k = 0; k < MM; k++) {
            v[k] = zsel(q0 + k < n, zs(za(zd(g[k], zs(g[k + 1], 2.0)), g[k + 2]), a.rh2));
        }
        if (q0 == 0) v[0] = zd(v[0], lo);
        if (q0 + MM >= n) subtract_last<MM>(v, n - 1 - q0, hi);
    }
    constexpr int LV = Levels<MM, 10>::LV;
    z2 end;
    double prod;
    eliminate<MM>(v, ex.R, q0, n, &end, &prod);
    if (live) { ex.ye[c * W + w] = end; ex.yp[c * W + w] = prod; }
    __syncthreads();
    if (live) eliminate_carry<MM>(v, ex.R, q0, n, carried<LV>(ex.ye, ex.yp, c, -1, P, W, w));
    substitute<MM>(v, ex.R, q0, &end, &prod);
    if (live) { ex.xe[c * W + w] = end; ex.xp[c * W + w] = prod; }
    __syncthreads();
    if (live) {
        substitute_carry<MM>(v, ex.R, q0, carried<LV>(ex.xe, ex.xp, c, 1, P, W, w));
#pragma unroll
        for (int k = 0; k < MM; k++) {
            if (q0 + k >= n) continue;
            if constexpr (STAGE) line[w * LS + line_pad(q0 + k)] = v[k];
            else a.out[b * a.oB + l * (long)n + q0 + k] = v[k];
        }
    }
    if constexpr (STAGE) {
        __syncthreads();
        z2 *dst = a.out + b * a.oB + l0 * (long)n;
        for (int w2 = 0; w2 < nl; w2++)
            for (int i = t; i < n; i += nt) dst[(long)w2 * n + i] = line[w2 * LS + line_pad(i)];
    }
}

// A value finished here: without it the compiler moves its arithmetic to where
// it is used, behind the exchanges, keeps every operand alive until then and
// spills (600 to 1000 bytes a thread).
HH_DEV void settle(z2 &v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
// Rows whose loads are in flight together in a strided pass.
constexpr int GRP = 4;

// Strided passes: lane w of a block owns column i = tile W + w (neighbours in
// memory), its chunk of rows is read and written in W * 16-byte segments.
// Every load is issued before the first exchange and every store follows the
// last, so a pass may rewrite its input in place (a block owns whole lines).
struct Strided {
    int n, W, P;
    int Nx;
};
HH_DEV void strided_thread(const Strided &s, int &w, int &c, int &i, bool &live) {
    w = threadIdx.x % s.W;
    c = threadIdx.x / s.W;
    i = (int)xcd_order(blockIdx.x, gridDim.x) * s.W + w;
    live = c < s.P && i < s.Nx;
    if (!live) { c = min(c, s.P - 1); i = min(i, s.Nx - 1); }
}

struct Y2D {
    Strided s;
    double hx, hy;
    const z2 *f_e, *u_e, *fy_b, *fxx_b, *fyy_b, *k2c, *k2y, *coef;
    int nop;
    z2 *F;   // holds f_xx on entry
};

// 2D, along y: f_yy and f_y of a line and the whole right-hand side
//   F / hy^2 = (1 - k^2 hy^2/20) f + hy^2/12 (f_xx + f_yy) + hy^4/360 (f_xxxx + f_yyyy)
//            + hy^4/90 f_xxyy + hy^4/60 (k^2)_y f_y                    (rhs.c:78-86)
// FY: with f_y.  Where k does not vary, its weight (k^2)_y is zero in every
// row and the line holds two arrays instead of three, which is what lets 1024
// threads a block (128-byte segments at n = 1023) keep them in registers.
template <int MM, bool FY> __global__ __launch_bounds__(FY ? 512 : 1024) void k_rhs2d_6(Y2D a, int b0) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = a.s.n, P = a.s.P, W = a.s.W, Nx = a.s.Nx, X = Nx + 2;
    Exchange e2(smem, P, W), e1(smem + (Exchange::bytes(P, W) + 15) / 16 * 16, P, W);
    pivot_table<10>(e2.R);
    if constexpr (FY) pivot_table<4>(e1.R);
    int w, c, i;
    bool live;
    strided_thread(a.s, w, c, i, live);
    const int b = b0 + blockIdx.y, o = b % a.nop;
    const int q0 = c * MM;
    const long XY = (long)X * (n + 2), Nxy = (long)Nx * n;
    const int nring = 2 * X + 2 * (n + 2);
    const double h2 = a.hy * a.hy, rx2 = 1.0 / (a.hx * a.hx), ry2 = 1.0 / h2;
    const z2 *f = a.f_e + b * XY + i + 1;
    z2 *F = a.F + b * Nxy + i;
    const z2 *rxx = a.fxx_b + (long)b * nring + 1 + i, *ryy = a.fyy_b + (long)b * nring + 1 + i;
    z2 G[MM], B[MM], D[FY ? MM : 1];   // sum so far, f_yy and f_y
    {
        z2 fm = f[(long)q0 * X], fc = f[(long)(q0 + 1) * X];
        z2 am = *(q0 == 0 ? rxx : F + (long)(q0 - 1) * Nx), ac = F[(long)q0 * Nx];
        const z2 top = rxx[X];
#pragma unroll
        for (int t = 0; t < MM; t++) {
            const int q = min(q0 + t, n - 1);   // rows past the end repeat the last one and are dropped below
            const z2 *fr = f + (long)(q + 1) * X;
            const z2 fp = fr[X], fl = fr[-1], fn = fr[1];
            z2 ap = F[(long)min(q + 1, n - 1) * Nx];
            ap = mk<double>(q == n - 1 ? top.x : ap.x, q == n - 1 ? top.y : ap.y);
            const z2 k2 = a.k2c[(long)o * n + q];
            const z2 dxx = zs(za(zd(fl, zs(fc, 2.0)), fn), rx2), dyy = zs(za(zd(fm, zs(fc, 2.0)), fp), ry2);
            z2 g = zd(fc, zs(zm(k2, fc), h2 / 20.0));
            g = zf(g, h2 / 12.0, ac);
            g = zf(g, h2 * h2 / 30.0 * rx2, zd(dxx, ac));
            g = zf(g, h2 / 30.0, dyy);
            G[t] = zf(g, h2 / 90.0, za(zd(am, zs(ac, 2.0)), ap));
            B[t] = zsel(q0 + t < n, zs(dyy, 12.0));
            if constexpr (FY) D[t] = zsel(q0 + t < n, zs(zd(fp, fm), 3.0 / a.hy));
            fm = fc; fc = fp;
            am = ac; ac = ap;
            settle(G[t]); settle(B[t]);
            if constexpr (FY) settle(D[t]);
            if (t % GRP == GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
        if (q0 == 0) B[0] = zd(B[0], ryy[0]);
        if (q0 + MM >= n) subtract_last<MM>(B, n - 1 - q0, ryy[X]);
        if constexpr (FY) {
            const z2 *fy = a.fy_b + (long)b * 2 * Nx + i;
            if (q0 == 0) D[0] = zd(D[0], fy[0]);
            if (q0 + MM >= n) subtract_last<MM>(D, n - 1 - q0, fy[Nx]);
        }
    }
    __syncthreads();   // pivots
    constexpr int L2 = Levels<MM, 10>::LV, L1 = Levels<MM, 4>::LV;
    const int slot = c * W + w;
    z2 ve, ue;
    double vp, up;
    eliminate<MM>(B, e2.R, q0, n, &ve, &vp);
    if constexpr (FY) eliminate<MM>(D, e1.R, q0, n, &ue, &up);
    if (live) {
        e2.ye[slot] = ve; e2.yp[slot] = vp;
        if constexpr (FY) { e1.ye[slot] = ue; e1.yp[slot] = up; }
    }
    __syncthreads();
    eliminate_carry<MM>(B, e2.R, q0, n, carried<L2>(e2.ye, e2.yp, c, -1, P, W, w));
    if constexpr (FY) eliminate_carry<MM>(D, e1.R, q0, n, carried<L1>(e1.ye, e1.yp, c, -1, P, W, w));
    substitute<MM>(B, e2.R, q0, &ve, &vp);
    if constexpr (FY) substitute<MM>(D, e1.R, q0, &ue, &up);
    if (live) {
        e2.xe[slot] = ve; e2.xp[slot] = vp;
        if constexpr (FY) { e1.xe[slot] = ue; e1.xp[slot] = up; }
    }
    __syncthreads();
    if (!live) return;
    substitute_carry<MM>(B, e2.R, q0, carried<L2>(e2.xe, e2.xp, c, 1, P, W, w));
    if constexpr (FY) substitute_carry<MM>(D, e1.R, q0, carried<L1>(e1.xe, e1.xp, c, 1, P, W, w));
#pragma unroll
    for (int t = 0; t < MM; t++) {
        const int q = q0 + t;
        if (q >= n) break;
        z2 v = zf(G[t], h2 / 12.0 - h2 / 30.0, B[t]);
        if constexpr (FY) v = zf(v, h2 * h2 / 60.0, zm(a.k2y[(long)o * n + q], D[t]));
        F[(long)q * Nx] = zs(v, h2);
    }
    // the closure, by the threads that hold boundary points (kept out of the
    // loop above: unrolled there, its loads cost every thread registers)
    const bool side = i == 0 || i == Nx - 1;
    if (!side && q0 > 0 && q0 + MM < n) return;
#pragma unroll 1
    for (int q = q0; q < min(q0 + MM, n); q++)
        if (side || q == 0 || q == n - 1)
            F[(long)q * Nx] = dirichlet2d(F[(long)q * Nx], Nx, n, i, q, a.coef + 6 * ((long)o * n + q), a.u_e + b * XY);
}

struct Y3D {
    Strided s;
    int Nz;
    double hx, hy, hz;
    const z2 *f_e, *fyy_f, *k2e;
    int nop;
    z2 *A;   // f_xx on entry, f_xx + f_yy on return
    z2 *F;   // the terms of x and y
};

// 3D, along y (rows of one z layer; blockIdx.y = layer, blockIdx.z = right-hand side)
template <int MM> __global__ __launch_bounds__(1024) void k_rhs3d_6y(Y3D a, int b0, int lay0) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = a.s.n, P = a.s.P, W = a.s.W, Nx = a.s.Nx;
    Exchange ex(smem, P, W);
    pivot_table<10>(ex.R);
    int w, c, i;
    bool live;
    strided_thread(a.s, w, c, i, live);
    const int lay = lay0 + blockIdx.y, b = b0 + blockIdx.z, q0 = c * MM;
    const long X = Nx + 2, XY = X * (n + 2), Z = a.Nz + 2;
    const double h2 = a.hz * a.hz, rx2 = 1.0 / (a.hx * a.hx), ry2 = 1.0 / (a.hy * a.hy);
    const z2 *f = a.f_e + (b * Z + lay + 1) * XY + i + 1;
    const long own = ((long)b * a.Nz + lay) * n * Nx + i;
    z2 *A = a.A + own, *F = a.F + own;
    const z2 k2 = a.k2e[(long)(b % a.nop) * Z + lay + 1];
    const z2 wt = mk<double>(1.0 - h2 / 20.0 * k2.x, -h2 / 20.0 * k2.y);
    z2 G[MM], B[MM];
    {
        z2 fm = f[(long)q0 * X], fc = f[(long)(q0 + 1) * X];
        z2 am = A[(long)max(q0 - 1, 0) * Nx], ac = A[(long)q0 * Nx];
        am = zsel(q0 > 0, am);   // f_xx is zero on the y faces
#pragma unroll
        for (int t = 0; t < MM; t++) {
            const int q = min(q0 + t, n - 1);
            const z2 *fr = f + (long)(q + 1) * X;
            const z2 fp = fr[X], fl = fr[-1], fn = fr[1];
            z2 ap = A[(long)min(q + 1, n - 1) * Nx];
            ap = zsel(q < n - 1, ap);
            const z2 dxx = zs(za(zd(fl, zs(fc, 2.0)), fn), rx2), dyy = zs(za(zd(fm, zs(fc, 2.0)), fp), ry2);
            z2 g = zf(zm(wt, fc), h2 / 12.0, ac);
            g = zf(g, h2 * h2 / 30.0 * rx2, zd(dxx, ac));
            g = zf(g, h2 * h2 / 30.0 * ry2, dyy);
            G[t] = zf(g, h2 * h2 / 90.0 * ry2, za(zd(am, zs(ac, 2.0)), ap));
            B[t] = zsel(q0 + t < n, zs(dyy, 12.0));
            fm = fc; fc = fp;
            am = ac; ac = ap;
            settle(G[t]); settle(B[t]);
            if (t % GRP == GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
        const z2 *face = a.fyy_f + (long)b * 2 * X * Z + (lay + 1) * X + 1 + i;
        if (q0 == 0) B[0] = zd(B[0], face[0]);
        if (q0 + MM >= n) subtract_last<MM>(B, n - 1 - q0, face[X * Z]);
    }
    __syncthreads();   // pivots
    constexpr int LV = Levels<MM, 10>::LV;
    const int slot = c * W + w;
    z2 end;
    double prod;
    eliminate<MM>(B, ex.R, q0, n, &end, &prod);
    if (live) { ex.ye[slot] = end; ex.yp[slot] = prod; }
    __syncthreads();
    eliminate_carry<MM>(B, ex.R, q0, n, carried<LV>(ex.ye, ex.yp, c, -1, P, W, w));
    substitute<MM>(B, ex.R, q0, &end, &prod);
    if (live) { ex.xe[slot] = end; ex.xp[slot] = prod; }
    __syncthreads();
    if (!live) return;
    substitute_carry<MM>(B, ex.R, q0, carried<LV>(ex.xe, ex.xp, c, 1, P, W, w));
#pragma unroll
    for (int t = 0; t < MM; t++) {
        const int q = q0 + t;
        if (q >= n) break;
        F[(long)q * Nx] = zf(G[t], h2 / 12.0 - h2 * h2 / 30.0 * ry2, B[t]);
        A[(long)q * Nx] = za(A[(long)q * Nx], B[t]);   // read again: kept, it would not fit the registers
    }
}

struct Z3D {
    Strided s;   // Nx: columns of a layer (Nx Ny)
    int NX, NY;
    double hz;
    const z2 *f_e, *u_e, *fzz_f, *kz, *coef;
    int nop;
    const z2 *A;   // f_xx + f_yy
    z2 *F;         // the terms of x and y on entry
};

// 3D, along z: f_zz, its terms, the cross terms with x and y and the closure (rhs.c:150-174)
template <int MM> __global__ __launch_bounds__(1024) void k_rhs3d_6z(Z3D a, int b0) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int n = a.s.n, P = a.s.P, W = a.s.W, Nx = a.NX, Ny = a.NY;
    Exchange ex(smem, P, W);
    pivot_table<10>(ex.R);
    int w, c, m;
    bool live;
    strided_thread(a.s, w, c, m, live);
    const int b = b0 + blockIdx.y, o = b % a.nop, q0 = c * MM;
    const int i = m % Nx, j = m / Nx;
    const long X = Nx + 2, XY = X * (Ny + 2), E = XY * (n + 2), L = (long)Nx * Ny;
    const double h2 = a.hz * a.hz, r2 = 1.0 / h2;
    const long g0 = (i + 1) + (j + 1) * X;
    const z2 *f = a.f_e + b * E + g0;
    const z2 *A = a.A + (long)b * n * L + m;
    z2 *F = a.F + (long)b * n * L + m;
    z2 G[MM], C[MM];
    {
        z2 fm = f[(long)q0 * XY], fc = f[(long)(q0 + 1) * XY];
        z2 am = A[(long)max(q0 - 1, 0) * L], ac = A[(long)q0 * L];
        am = zsel(q0 > 0, am);   // f_xx and f_yy are zero on the z faces
#pragma unroll
        for (int t = 0; t < MM; t++) {
            const int q = min(q0 + t, n - 1);
            const z2 fp = f[(long)(q + 2) * XY];
            z2 ap = A[(long)min(q + 1, n - 1) * L];
            ap = zsel(q < n - 1, ap);
            const z2 dzz = zs(za(zd(fm, zs(fc, 2.0)), fp), r2);
            z2 g = zf(F[(long)q * L], h2 / 30.0, dzz);
            g = zf(g, h2 / 90.0, za(zd(am, zs(ac, 2.0)), ap));
            G[t] = za(g, zs(zm(a.kz[(long)o * n + q], zd(fp, fm)), h2 * a.hz / 120.0));
            C[t] = zsel(q0 + t < n, zs(dzz, 12.0));
            fm = fc; fc = fp;
            am = ac; ac = ap;
            settle(G[t]); settle(C[t]);
            if (t % GRP == GRP - 1) __builtin_amdgcn_sched_barrier(0);
        }
        const z2 *face = a.fzz_f + (long)b * 2 * XY + g0;
        if (q0 == 0) C[0] = zd(C[0], face[0]);
        if (q0 + MM >= n) subtract_last<MM>(C, n - 1 - q0, face[XY]);
    }
    __syncthreads();   // pivots
    constexpr int LV = Levels<MM, 10>::LV;
    const int slot = c * W + w;
    z2 end;
    double prod;
    eliminate<MM>(C, ex.R, q0, n, &end, &prod);
    if (live) { ex.ye[slot] = end; ex.yp[slot] = prod; }
    __syncthreads();
    eliminate_carry<MM>(C, ex.R, q0, n, carried<LV>(ex.ye, ex.yp, c, -1, P, W, w));
    substitute<MM>(C, ex.R, q0, &end, &prod);
    if (live) { ex.xe[slot] = end; ex.xp[slot] = prod; }
    __syncthreads();
    if (!live) return;
    substitute_carry<MM>(C, ex.R, q0, carried<LV>(ex.xe, ex.xp, c, 1, P, W, w));
#pragma unroll
    for (int t = 0; t < MM; t++) {
        const int q = q0 + t;
        if (q >= n) break;
        F[(long)q * L] = zf(G[t], h2 / 12.0 - h2 / 30.0, C[t]);
    }
#pragma unroll 1
    for (int s = 0; s < 2; s++) {   // the closure of the first and the last layer, as in k_rhs2d_6
        const int q = s == 0 ? 0 : n - 1;
        if (q >= q0 && q < q0 + MM)
            F[(long)q * L] = dirichlet3d(F[(long)q * L], X, XY, n, q, g0, a.coef + 12 * (long)o * n, a.u_e + b * E);
    }
}

// Rows per thread: 8, or 16 where 1024 threads would not span the line.
int chunk_rows(int n) { return n > 8192 ? 16 : 8; }

// Columns per block: at least 8 (128-byte segments) and up to 512 threads where that fits 1024.
void strided_shape(Strided &s, int n, int ncols, int mm, int most = 1024) {
    s.n = n;
    s.Nx = ncols;
    s.P = (n + mm - 1) / mm;
    int w = 1;
    while (w < 64 && 2 * w * s.P <= (w < 8 ? most : 512)) w *= 2;
    while (w > 1 && w / 2 >= ncols) w /= 2;
    s.W = w;
}

template <class K> hipError_t with_lds(K kfn, size_t shm) {
    if (shm <= 65536) return hipSuccess;
    return hipFuncSetAttribute((const void *)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
}

hipError_t launch_x(XLines a, int batch, hipStream_t st) {
    const size_t per_line = (size_t)(line_pad(a.n + 2) + 1) * 16;
    auto lds = [&](int P, int W) { return (Exchange::bytes(P, W) + 15) / 16 * 16 + W * per_line; };
    const int mm = chunk_rows(a.n);
    a.P = (a.n + mm - 1) / mm;
    if (a.P > 1024) return hipErrorInvalidValue;
    const bool stage = mm == 8 && lds(a.P, 1) <= 160 * 1024 - 1024;
    // one wave per block where lines are short: its barriers wait for no other
    // (200^3: 65 us, 74 with 256 threads; 8 x 1023^2, 128 threads a line: 75 and 74;
    // 16 rows per thread, one wave a line there: 100)
    a.W = std::max(1, 64 / a.P);
    if (a.W > a.nlines) a.W = a.nlines;
    const size_t shm = stage ? lds(a.P, a.W) : Exchange::bytes(a.P, a.W);
    auto kfn = !stage ? (mm == 8 ? k_compact_x<8, false> : k_compact_x<16, false>) : k_compact_x<8, true>;
    hipError_t e = with_lds(kfn, shm);
    if (e != hipSuccess) return e;
    const long tiles = ((long)a.nlines + a.W - 1) / a.W;
    const int threads = (a.W * a.P + 63) / 64 * 64;
    for (int b0 = 0; b0 < batch; b0 += 65535) {
        const int nb = batch - b0 < 65535 ? batch - b0 : 65535;
        hipLaunchKernelGGL(kfn, dim3((unsigned)tiles, (unsigned)nb), dim3(threads), shm, st, a, b0);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rhs2d_6(const Rhs2D &r, void *F, hipStream_t st) {
    const int Nx = r.Nx, Ny = r.Ny, X = Nx + 2, Y = Ny + 2;
    XLines x{};
    x.n = Nx; x.nlines = Ny; x.nA = Ny;
    x.f = (const z2 *)r.f_e; x.fB = (long)X * Y; x.fO = 0; x.fC = 0;
    x.out = (z2 *)F; x.oB = (long)Nx * Ny;
    x.lo = (const z2 *)r.fxx_b + 2 * X; x.hi = x.lo + Y; x.eB = 2 * X + 2 * Y; x.e0 = 1; x.eA = 0;
    x.rh2 = 12.0 / (r.hx * r.hx);
    hipError_t e = launch_x(x, r.batch, st);
    if (e != hipSuccess) return e;
    Y2D a{};
    const bool fy = r.k2y_nonzero != 0;
    const int mm = fy && Ny > 4096 ? 16 : 8;   // Ny <= 8192: 512 threads with f_y, 1024 without
    strided_shape(a.s, Ny, Nx, mm, fy ? 512 : 1024);
    if (a.s.P > (fy ? 512 : 1024)) return hipErrorInvalidValue;
    a.hx = r.hx; a.hy = r.hy;
    a.f_e = (const z2 *)r.f_e; a.u_e = (const z2 *)r.u_e;
    a.fy_b = (const z2 *)r.fy_b; a.fxx_b = (const z2 *)r.fxx_b; a.fyy_b = (const z2 *)r.fyy_b;
    a.k2c = (const z2 *)r.k2c; a.k2y = (const z2 *)r.k2y; a.coef = (const z2 *)r.coef; a.nop = r.nop > 0 ? r.nop : 1;
    a.F = (z2 *)F;
    const size_t shm = 2 * ((Exchange::bytes(a.s.P, a.s.W) + 15) / 16 * 16);
    auto kfn = !fy ? k_rhs2d_6<8, false> : mm == 8 ? k_rhs2d_6<8, true> : k_rhs2d_6<16, true>;
    if ((e = with_lds(kfn, shm)) != hipSuccess) return e;
    const int threads = (a.s.W * a.s.P + 63) / 64 * 64;
    for (int b0 = 0; b0 < r.batch; b0 += 65535) {
        const int nb = r.batch - b0 < 65535 ? r.batch - b0 : 65535;
        hipLaunchKernelGGL(kfn, dim3((unsigned)((Nx + a.s.W - 1) / a.s.W), (unsigned)nb), dim3(threads), shm, st, a, b0);
    }
    return hipGetLastError();
}

hipError_t launch_rhs3d_6(const Rhs3D &r, void *F, hipStream_t st) {
    const int Nx = r.Nx, Ny = r.Ny, Nz = r.Nz;
    const long X = Nx + 2, Y = Ny + 2, Z = Nz + 2, XY = X * Y;
    const int nop = r.nop > 0 ? r.nop : 1;
    XLines x{};
    if ((long)Ny * Nz > 0x7fffffffL) return hipErrorInvalidValue;
    x.n = Nx; x.nlines = Ny * Nz; x.nA = Ny;
    x.f = (const z2 *)r.f_e; x.fB = XY * Z; x.fO = XY; x.fC = XY;
    x.out = (z2 *)r.work; x.oB = (long)Nx * Ny * Nz;
    x.lo = (const z2 *)r.fxx_f; x.hi = x.lo + Y * Z; x.eB = 2 * Y * Z; x.e0 = 1 + Y; x.eA = Y;
    x.rh2 = 12.0 / (r.hx * r.hx);
    hipError_t e = launch_x(x, r.batch, st);
    if (e != hipSuccess) return e;
    Y3D y{};
    const int mm = chunk_rows(Ny);
    strided_shape(y.s, Ny, Nx, mm);
    if (y.s.P > 1024) return hipErrorInvalidValue;
    y.Nz = Nz; y.hx = r.hx; y.hy = r.hy; y.hz = r.hz;
    y.f_e = (const z2 *)r.f_e; y.fyy_f = (const z2 *)r.fyy_f; y.k2e = (const z2 *)r.k2e; y.nop = nop;
    y.A = (z2 *)r.work; y.F = (z2 *)F;
    size_t shm = Exchange::bytes(y.s.P, y.s.W);
    auto ky = mm == 8 ? k_rhs3d_6y<8> : k_rhs3d_6y<16>;
    if ((e = with_lds(ky, shm)) != hipSuccess) return e;
    int threads = (y.s.W * y.s.P + 63) / 64 * 64;
    for (int b0 = 0; b0 < r.batch; b0 += 65535)
        for (int l0 = 0; l0 < Nz; l0 += 65535) {
            const int nb = r.batch - b0 < 65535 ? r.batch - b0 : 65535, nl = Nz - l0 < 65535 ? Nz - l0 : 65535;
            hipLaunchKernelGGL(ky, dim3((unsigned)((Nx + y.s.W - 1) / y.s.W), (unsigned)nl, (unsigned)nb), dim3(threads),
                               shm, st, y, b0, l0);
        }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    Z3D z{};
    if ((long)Nx * Ny > 0x7fffffffL) return hipErrorInvalidValue;
    strided_shape(z.s, Nz, Nx * Ny, 8);   // Nz <= 8192
    if (z.s.P > 1024) return hipErrorInvalidValue;
    z.NX = Nx; z.NY = Ny; z.hz = r.hz;
    z.f_e = (const z2 *)r.f_e; z.u_e = (const z2 *)r.u_e; z.fzz_f = (const z2 *)r.fzz_f;
    z.kz = (const z2 *)r.kz; z.coef = (const z2 *)r.coef; z.nop = nop;
    z.A = (const z2 *)r.work; z.F = (z2 *)F;
    shm = Exchange::bytes(z.s.P, z.s.W);
    auto kz = k_rhs3d_6z<8>;
    if ((e = with_lds(kz, shm)) != hipSuccess) return e;
    threads = (z.s.W * z.s.P + 63) / 64 * 64;
    for (int b0 = 0; b0 < r.batch; b0 += 65535) {
        const int nb = r.batch - b0 < 65535 ? r.batch - b0 : 65535;
        hipLaunchKernelGGL(kz, dim3((unsigned)((Nx * Ny + z.s.W - 1) / z.s.W), (unsigned)nb), dim3(threads), shm, st, z, b0);
    }
    return hipGetLastError();
}

}  // namespace hh
