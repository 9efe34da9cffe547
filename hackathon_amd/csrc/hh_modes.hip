// Host-side classification of the per-mode tridiagonal systems and the
// reference-order factors of the ill-conditioned ones.
//
// Every mode m of an operator o owns a tridiagonal system T (sub, dia, sup
// along y in 2D, z in 3D).  The partitioned elimination of the device kernel
// (hh_tri.hip) restarts the pivot recurrence at every 16-row chunk and
// combines the chunks through a reduced system; its relative error on a mode
// grows like c eps kappa(T) with c <= 0.05 measured over the C2/C4 operators
// (FP64, white-noise right-hand sides, against 40-digit solutions), which is
// up to 10x the error of the reference's sequential Thomas elimination on
// the nearly singular low modes.  Modes are therefore split:
//
//  * well separated: strictly diagonally dominant with Varah's bound
//      kappa_inf(T) <= max_q (|sub|+|dia|+|sup|) / min_q (|dia|-|sub|-|sup|)
//    at most kappa_flag (default 4096): partitioned elimination on the
//    device (relative error <= ~2e-14 in FP64; FP32 in the mixed path);
//  * near-resonant (everything else, including every indefinite mode with
//    |lambda_j - k^2| small): the factors of the reference's LU() are
//    computed here in its operation order (2D_Program/main_functions/
//    LU.c:16-40, divide form; 3D_Program/main_functions/LU.c:34-72,
//    reciprocal form), with contraction off, so they are bit-identical to
//    the reference's for real operators, and the device runs the
//    reference's substitution (2D_Program/solver_functions/solver.c:71-86,
//    3D_Program/solver_functions/solver.c:356-369) in sequential order with
//    the same operations, so these modes differ from the reference's only
//    through their input.  (An exact double-double substitution, evaluated
//    as a parallel scan, was measured too: more accurate than the
//    reference, it disagreed with it by up to 1.3e-12 on a manufactured
//    solution at N = 511, k = 39, where the reference's own FP64
//    substitution loses 4e-13 to pivots of 4e-3; the sequential order stays
//    within 3e-14 there.)
//
// A near-resonant mode whose estimated condition number exceeds
// HH_SINGULAR_KAPPA (or whose pivot is zero or not finite) makes its
// operator singular to working precision: the plan reports HH_ERR_SINGULAR
// for solves that use it.  The reference divides by such pivots unchecked
// (2D LU.c:36, 3D LU.c:68).
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdint>
#include <vector>

#include "hh_internal.h"

namespace hh {

using cd = std::complex<double>;

namespace {

// Bands of row q of mode (lx, ly) in the reference's operation order:
// 2D  sub = bm lam + am, dia = b lam + a, sup = bp lam + ap  (LU.c:16-23),
// 3D  e3 = a lxy + b lx + c ly + d, and the P / M variants  (LU.c:34-47),
// complex coefficient times real eigenvalue componentwise.  Table rows:
// 2D (bm, am, b, a, bp, ap); 3D (a, b, c, d, ap, bp, cp, dp, am, bm, cm, dm).
struct RowBands {
    cd sub, dia, sup;
};

#pragma clang fp contract(off)
inline cd cr(cd a, double s) { return cd(a.real() * s, a.imag() * s); }
inline cd add(cd a, cd b) { return cd(a.real() + b.real(), a.imag() + b.imag()); }

inline RowBands row_bands(int dim, const cd *row, double lx, double ly, double lxy) {
    RowBands r;
    if (dim == 2) {
        r.sub = add(cr(row[0], lx), row[1]);
        r.dia = add(cr(row[2], lx), row[3]);
        r.sup = add(cr(row[4], lx), row[5]);
    } else {
        auto e = [&](const cd *c) { return add(add(add(cr(c[0], lxy), cr(c[1], lx)), cr(c[2], ly)), c[3]); };
        r.dia = e(row);
        r.sup = e(row + 4);
        r.sub = e(row + 8);
    }
    return r;
}

// Real-operator factors of G modes, reference order, FP64 with no fused operations.
// out rows: (L_q, P_q, R_q, Up_q).  2D: the reference divides by its pivot
// U_q; P_q = U_q and R_q = RN(1/U_q), with which the device reproduces the
// correctly rounded quotient (one fused correction step, Markstein).  3D:
// the reference multiplies by its stored reciprocal pivot U_q; R_q = U_q and
// P_q = 1/U_q (unused).  ok: no pivot is zero or not finite.
// Each mode is a serial chain of divisions; G of them side by side keep the
// divider busy, and one mode's operations do not change (1023 rows, 11 modes
// with their condition estimates: 309 us one by one, 92 in groups of 4, on the
// host while a serving loop's GPU waits).
constexpr int GROUP = 4;
template <int DIM>
void factors_real(int n, const cd *tab, const double *lx, const double *ly, double *const *out, bool *ok) {
    constexpr int NC = DIM == 2 ? 6 : 12;
    double Uprev[GROUP] = {}, Upprev[GROUP] = {}, bad[GROUP] = {}, lxy[GROUP];
    for (int g = 0; g < GROUP; g++) lxy[g] = lx[g] * ly[g];
    for (int q = 0; q < n; q++) {
        const cd *row = tab + (long)q * NC;
        double L[GROUP], U[GROUP], R[GROUP], P[GROUP], sup[GROUP];
        for (int g = 0; g < GROUP; g++) {
            double sub, dia;
            if constexpr (DIM == 2) {
                sub = row[0].real() * lx[g] + row[1].real();
                dia = row[2].real() * lx[g] + row[3].real();
                sup[g] = row[4].real() * lx[g] + row[5].real();
                // LU.c:32-40: L = sub / U_{q-1}, U = dia - L Up_{q-1}
                L[g] = q == 0 ? 0.0 : sub / Uprev[g];
                U[g] = q == 0 ? dia : dia - L[g] * Upprev[g];
                R[g] = 1.0 / U[g];
                P[g] = U[g];
            } else {
                auto e = [&](const cd *c) {
                    return ((c[0].real() * lxy[g] + c[1].real() * lx[g]) + c[2].real() * ly[g]) + c[3].real();
                };
                dia = e(row);
                sup[g] = e(row + 4);
                sub = e(row + 8);
                // LU.c:61-72: L = sub U_{q-1} (U reciprocal), U = 1 / (dia - Up_{q-1} L)
                L[g] = q == 0 ? 0.0 : sub * Uprev[g];
                U[g] = q == 0 ? 1.0 / dia : 1.0 / (dia - Upprev[g] * L[g]);
                R[g] = U[g];
                P[g] = 1.0 / U[g];
            }
            bad[g] += (L[g] - L[g]) + (R[g] - R[g]) + (P[g] - P[g]);   // zero, or NaN once a value is not finite
            Uprev[g] = U[g];
            Upprev[g] = sup[g];
        }
        for (int g = 0; g < GROUP; g++) {
            double *o = out[g] + 4 * (long)q;
            o[0] = L[g];
            o[1] = P[g];
            o[2] = R[g];
            o[3] = q == n - 1 ? 0.0 : sup[g];   // the last row has no superdiagonal
        }
    }
    for (int g = 0; g < GROUP; g++) ok[g] = bad[g] == 0.0;
}

bool factors_complex(int dim, int n, const cd *tab, int nc, double lx, double ly, double lxy, cd *out) {
    bool ok = true;
    cd Uprev = 0, Upprev = 0;
    for (int q = 0; q < n; q++) {
        const RowBands b = row_bands(dim, tab + (long)q * nc, lx, ly, lxy);
        cd L, U, R, P;
        if (dim == 2) {
            L = q == 0 ? cd(0) : b.sub / Uprev;
            U = q == 0 ? b.dia : b.dia - L * Upprev;
            R = cd(1) / U;
            P = U;
        } else {
            L = q == 0 ? cd(0) : b.sub * Uprev;
            U = q == 0 ? cd(1) / b.dia : cd(1) / (b.dia - Upprev * L);
            R = U;
            P = cd(1) / U;
        }
        Uprev = U;
        if (!std::isfinite(std::abs(L)) || !std::isfinite(std::abs(R)) || U == cd(0)) ok = false;
        Upprev = b.sup;
        out[4 * q] = L;
        out[4 * q + 1] = P;
        out[4 * q + 2] = R;
        out[4 * q + 3] = q == n - 1 ? cd(0) : b.sup;
    }
    return ok;
}
#pragma clang fp contract(on)

// Varah margin min (|dia| - |sub| - |sup|) and row sum max (|dia| + |sub| +
// |sup|) of G modes over rows qbeg .. qend - 1.  Magnitudes as sqrt(re^2 +
// im^2): the bands are far from overflow, std::abs's hypot costs several times more.
template <int DIM, bool REAL>
void mode_bounds(int n, const cd *tab, int qbeg, int qend, const double *lx, const double *ly, double *margin,
                 double *rowsum) {
    constexpr int NC = DIM == 2 ? 6 : 12;
    double mn[GROUP], mx[GROUP], lxy[GROUP];
    for (int g = 0; g < GROUP; g++) { mn[g] = INFINITY; mx[g] = 0; lxy[g] = lx[g] * ly[g]; }
    for (int q = qbeg; q < qend; q++) {
        const cd *c = tab + (long)q * NC;
        double s[GROUP], d[GROUP], u[GROUP];
        auto part = [&](auto at, double *out) {   // |band| of the coefficients at(i), componentwise
            double re[GROUP], im[GROUP];
            for (int g = 0; g < GROUP; g++) {
                if constexpr (DIM == 2) {
                    re[g] = at(0).real() * lx[g] + at(1).real();
                    im[g] = REAL ? 0.0 : at(0).imag() * lx[g] + at(1).imag();
                } else {
                    re[g] = at(0).real() * lxy[g] + at(1).real() * lx[g] + at(2).real() * ly[g] + at(3).real();
                    im[g] = REAL ? 0.0 : at(0).imag() * lxy[g] + at(1).imag() * lx[g] + at(2).imag() * ly[g] + at(3).imag();
                }
            }
            for (int g = 0; g < GROUP; g++)
                out[g] = REAL ? std::fabs(re[g]) : __builtin_sqrt(re[g] * re[g] + im[g] * im[g]);
        };
        if constexpr (DIM == 2) {   // (bm, am, b, a, bp, ap)
            part([&](int i) { return c[i]; }, s);
            part([&](int i) { return c[2 + i]; }, d);
            part([&](int i) { return c[4 + i]; }, u);
        } else {   // (a..d, ap..dp, am..dm)
            part([&](int i) { return c[i]; }, d);
            part([&](int i) { return c[4 + i]; }, u);
            part([&](int i) { return c[8 + i]; }, s);
        }
        for (int g = 0; g < GROUP; g++) {
            const double sg = q == 0 ? 0.0 : s[g], ug = q == n - 1 ? 0.0 : u[g];
            const double a = d[g] - sg - ug, b = d[g] + sg + ug;
            mn[g] = a < mn[g] ? a : mn[g];
            mx[g] = mx[g] < b ? b : mx[g];
        }
    }
    for (int g = 0; g < GROUP; g++) { margin[g] = mn[g]; rowsum[g] = mx[g]; }
}

// ||T^{-1} e||_inf for e = all ones and e = a fixed +-1 pattern, with the
// factors (L, P, R, Up) of the reference substitution, for G systems; y: 2 n G values.
template <typename V, int G> void inv_norm_est(int n, const V *const *f, std::vector<V> &y, double *inv) {
    y.resize(2 * (size_t)n * G);
    V last[2 * G] = {};
    uint32_t s = 0x9e3779b9u;
    for (int q = 0; q < n; q++) {
        s = s * 1664525u + 1013904223u;
        const double e[2] = {1.0, (s >> 31) ? 1.0 : -1.0};
        V *yq = y.data() + 2 * (size_t)G * q;
        for (int g = 0; g < G; g++) {
            const V L = f[g][4 * (long)q];
            for (int k = 0; k < 2; k++) yq[2 * g + k] = last[2 * g + k] = q == 0 ? V(e[k]) : V(e[k]) - L * last[2 * g + k];
        }
    }
    V x[2 * G] = {};
    double mx[2 * G] = {};
    for (int q = n - 1; q >= 0; q--) {
        const V *yq = y.data() + 2 * (size_t)G * q;
        for (int g = 0; g < G; g++) {
            const V R = f[g][4 * (long)q + 2], up = f[g][4 * (long)q + 3];
            for (int k = 0; k < 2; k++) {
                const int i = 2 * g + k;
                x[i] = q == n - 1 ? yq[i] * R : (yq[i] - up * x[i]) * R;
                mx[i] = std::max(mx[i], std::abs(x[i]));
            }
        }
    }
    for (int g = 0; g < G; g++) inv[g] = std::max(std::max(0.0, mx[2 * g]), mx[2 * g + 1]);
}

}  // namespace

void classify_modes(int dim, int Nx, int Ny, int Nz, int nop, const cd *hcoef, const double *lamx,
                    const double *lamy, bool real, double kappa_flag, ModeSet &ms) {
    const int n = dim == 2 ? Ny : Nz;
    const int nc = dim == 2 ? 6 : 12;
    const long nmodes = dim == 2 ? Nx : (long)Nx * Ny;
    ms.n = n;
    ms.nmodes = nmodes;
    ms.nop = nop;
    ms.words = (int)((nmodes + 31) / 32);
    ms.foff.assign(nop + 1, 0);
    ms.fmode.clear();
    ms.bits.assign((size_t)nop * (1 + ms.words), 0u);
    ms.facc.clear();
    ms.facr.clear();
    ms.singular.assign(nop, 0);
    ms.kappa_worst.assign(nop, 0.0);
    ms.nfx = 0;
    std::vector<double> yr, sums;
    std::vector<cd> yc;
    for (int o = 0; o < nop; o++) {
        const cd *tab = hcoef + (size_t)o * n * nc;
        // a table whose rows are all equal (constant k) gives every interior
        // row the same bands: one row decides the mode
        bool uniform = true;
        for (int q = 1; q < n && uniform; q++)
            for (int t = 0; t < nc; t++)
                if (tab[(long)q * nc + t] != tab[t]) { uniform = false; break; }
        ms.bits[o] = uniform;
        ms.foff[o] = (int)ms.fmode.size();
        // equal rows: an inner one has the smallest margin and the largest sum
        const int qbeg = uniform && n > 2 ? 1 : 0, qend = uniform ? std::min(n, 2) : n;
        auto bounds = dim == 2 ? (real ? mode_bounds<2, true> : mode_bounds<2, false>)
                               : (real ? mode_bounds<3, true> : mode_bounds<3, false>);
        double margins[GROUP], rowsums[GROUP];
        for (long m = 0; m < nmodes; m++) {
            const int g = (int)(m % GROUP);
            if (g == 0) {
                double lx[GROUP], ly[GROUP];
                for (int i = 0; i < GROUP; i++) {
                    const long mm = std::min(m + i, nmodes - 1);
                    lx[i] = dim == 2 ? lamx[mm] : lamx[mm % Nx];
                    ly[i] = dim == 2 ? 0.0 : lamy[mm / Nx];
                }
                bounds(n, tab, qbeg, qend, lx, ly, margins, rowsums);
            }
            const double margin = margins[g], rowsum = rowsums[g];
            const bool flag = !(margin > 0) || rowsum > kappa_flag * margin;
            if (!flag) continue;
            ms.fmode.push_back((int)m);
            ms.bits[nop + (size_t)o * ms.words + m / 32] |= 1u << (m % 32);
            sums.push_back(rowsum);
        }
        // factors and condition estimates of the operator's flagged modes
        const size_t e0 = ms.foff[o], e1 = ms.fmode.size(), len = 4 * (size_t)n;
        if (real) ms.facr.resize(e1 * len);
        else ms.facc.resize(e1 * len);
        for (size_t e = e0; e < e1; e += real ? GROUP : 1) {
            bool ok[GROUP];
            double lx[GROUP], ly[GROUP], inv[GROUP];
            const int ng = real ? (int)std::min<size_t>(GROUP, e1 - e) : 1;
            for (int g = 0; g < GROUP; g++) {   // a last group repeats its last mode
                const long m = ms.fmode[e + std::min(g, ng - 1)];
                lx[g] = dim == 2 ? lamx[m] : lamx[m % Nx];
                ly[g] = dim == 2 ? 0.0 : lamy[m / Nx];
            }
            if (real) {
                double *out[GROUP];
                for (int g = 0; g < GROUP; g++) out[g] = ms.facr.data() + (e + std::min(g, ng - 1)) * len;
                if (dim == 2) factors_real<2>(n, tab, lx, ly, out, ok);
                else factors_real<3>(n, tab, lx, ly, out, ok);
                inv_norm_est<double, GROUP>(n, out, yr, inv);
            } else {
                cd *out = ms.facc.data() + e * len;
                ok[0] = factors_complex(dim, n, tab, nc, lx[0], ly[0], lx[0] * ly[0], out);
                inv_norm_est<cd, 1>(n, &out, yc, inv);
            }
            for (int g = 0; g < ng; g++) {
                const double kap = sums[e + g] * (ok[g] ? inv[g] : INFINITY);
                if (!ok[g] || !std::isfinite(kap) || kap > HH_SINGULAR_KAPPA) ms.singular[o] = 1;
                if (!(kap <= ms.kappa_worst[o])) ms.kappa_worst[o] = kap;
            }
        }
        const int cnt = (int)ms.fmode.size() - ms.foff[o];
        if (cnt > ms.nfx) ms.nfx = cnt;
    }
    ms.foff[nop] = (int)ms.fmode.size();
}

// Device tables of a plan's operators from their host form: one launch for
// what took up to eight copies of pageable memory (a serving loop's batch of
// three 1023-row operators: 150 us of copies that queued behind its
// right-hand sides on the copy engine).  The sources are read once, over the
// link when they are in host memory; the FP32 and real forms of the bands,
// the complex form of real factors and the factors' device order
// [row][entry](L, P, R, Up), in which the lanes of neighbouring entries read
// neighbouring records, are made here and do not cross it.
__global__ __launch_bounds__(256) void k_operator_tables(OperatorTables t) {
    const long id = (long)blockIdx.x * 256 + threadIdx.x, step = (long)gridDim.x * 256;
    for (long i = id; i < t.ncoef; i += step) {
        const double2 v = t.coef[i];
        t.coef64[i] = v;
        t.coef32[i] = make_float2((float)v.x, (float)v.y);
        t.coefr64[i] = v.x;
        t.coefr32[i] = (float)v.x;
    }
    const long per = 4L * t.n;   // values of one entry
    for (long i = id; i < t.nfac; i += step) {
        const long g = t.fac0 + i, e = g / per, r = g - e * per, q = r >> 2, to = (q * t.nent + e) * 4 + (r & 3);
        if (t.facr) {
            const double v = t.facr[i];
            t.outr[to] = v;
            t.outc[to] = make_double2(v, 0.0);
        } else {
            t.outc[to] = t.facc[i];
        }
    }
    for (long i = id; i < t.nslot; i += step) t.outent[i] = t.ent[i];
    for (long i = id; i < t.nbits; i += step) t.outbits[i] = t.bits[i];
}

hipError_t launch_operator_tables(const OperatorTables &t, hipStream_t st) {
    const long work = std::max(std::max(t.ncoef, t.nfac), std::max(t.nslot, t.nbits));
    const long blocks = std::min(1024L, (work + 255) / 256);
    hipLaunchKernelGGL(k_operator_tables, dim3((unsigned)std::max(1L, blocks)), dim3(256), 0, st, t);
    return hipGetLastError();
}

}  // namespace hh
