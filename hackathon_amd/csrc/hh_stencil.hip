// Stencil kernels for gfx950: compact right-hand-side assembly, the FP64
// compact-operator residual, norms and small field operations.
//
// Right-hand side (kernel set "c"):
//   2D_Program/main_functions/rhs.c:4-150 with 2D_Program/partial_derivatives
//   3D_Program/main_functions/rhs.c:13-294 with 3D_Program/partial_derivatives
// Orders 2 and 4 are pointwise differences, combined with the Dirichlet closure
// in one pass; the sixth order with its compact derivatives is hh_compact.hip.
// Residual: 2D_Program/main_functions/residual.c:3-34 (9-point),
//           3D_Program/main_functions/residual.c:42-96 (27-point).
#include <type_traits>

#include "hh_closure.h"
#include "hh_common.h"
#include "hh_internal.h"

namespace hh {

typedef double2 z2;

HH_DEV z2 zr(double r) { return mk<double>(r, 0); }
HH_DEV z2 zs(z2 a, double s) { return cscale<double>(a, s); }
HH_DEV z2 za(z2 a, z2 b) { return cadd<double>(a, b); }
HH_DEV z2 zd(z2 a, z2 b) { return csub<double>(a, b); }
HH_DEV z2 zm(z2 a, z2 b) { return cmul<double>(a, b); }

// ---------------------------------------------------------------- 2D RHS
struct Rhs2DArgs {
    int order, Nx, Ny;
    double hx, hy;
    const z2 *f_e, *u_e, *coef;
    int nop;
};

__global__ void k_rhs2d_combine(Rhs2DArgs a, long total, z2 *F) {
    long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const int Nx = a.Nx, Ny = a.Ny, X = Nx + 2;
    const long Nxy = (long)Nx * Ny, XY = (long)X * (Ny + 2);
    const int b = (int)(id / Nxy);
    const long p = id % Nxy;
    const int i = (int)(p % Nx), j = (int)(p / Nx);
    const z2 *f = a.f_e + b * XY;
    const long c0 = (i + 1) + (long)(j + 1) * X;
    const double hy2 = a.hy * a.hy;
    z2 v;
    if (a.order == 4) {                                    // rhs.c:21-38
        z2 s4 = za(za(za(f[c0 - X], f[c0 + X]), f[c0 - 1]), f[c0 + 1]);
        v = zs(za(zs(f[c0], 2.0 / 3.0), zs(s4, 1.0 / 12.0)), hy2);
    } else {                                                      // rhs.c:4-19
        v = zs(f[c0], hy2);
    }
    // Dirichlet closure rhs.c:126-148: subtract the stencil weight times u
    // for every neighbour that lies on the boundary
    if (i == 0 || i == Nx - 1 || j == 0 || j == Ny - 1)
        v = dirichlet2d(v, Nx, Ny, i, j, a.coef + 6 * ((long)(b % a.nop) * Ny + j), a.u_e + b * XY);
    F[id] = v;
}

hipError_t launch_rhs2d(const Rhs2D &r, void *F, hipStream_t st) {
    if (r.order == 6) return launch_rhs2d_6(r, F, st);
    const int Nx = r.Nx, Ny = r.Ny;
    Rhs2DArgs a;
    a.order = r.order; a.Nx = Nx; a.Ny = Ny; a.hx = r.hx; a.hy = r.hy;
    a.f_e = (const z2 *)r.f_e; a.u_e = (const z2 *)r.u_e;
    a.coef = (const z2 *)r.coef; a.nop = r.nop > 0 ? r.nop : 1;
    long total = (long)Nx * Ny * r.batch;
    hipLaunchKernelGGL(k_rhs2d_combine, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a, total, (z2 *)F);
    return hipGetLastError();
}

// ---------------------------------------------------------------- 3D RHS
struct Rhs3DArgs {
    int order, Nx, Ny, Nz;
    double hx, hy, hz;
    const z2 *f_e, *u_e, *coef;
    int nop;
};

__global__ void k_rhs3d_combine(Rhs3DArgs a, long total, z2 *F) {
    long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const long Nx = a.Nx, Ny = a.Ny, Nz = a.Nz, X = Nx + 2, XY = X * (Ny + 2), E = XY * (Nz + 2);
    const long N3 = Nx * Ny * Nz;
    const int b = (int)(id / N3);
    const long p = id % N3;
    const long i = p % Nx, j = (p / Nx) % Ny, l = p / (Nx * Ny);
    const z2 *f = a.f_e + b * E;
    const long c0 = (i + 1) + (j + 1) * X + (l + 1) * XY;
    z2 v;
    if (a.order == 4) {                                    // rhs.c:34-53
        z2 s6 = za(za(za(za(za(f[c0 - 1], f[c0 + 1]), f[c0 - X]), f[c0 + X]), f[c0 - XY]), f[c0 + XY]);
        v = za(f[c0], zs(zd(s6, zs(f[c0], 6.0)), 1.0 / 12.0));
    } else {                                                      // rhs.c:13-32
        v = f[c0];
    }
    // z-face closure (rhs.c:24-29, 55-62)
    if (l == 0 || l == Nz - 1) {
        const z2 *u = a.u_e + b * E;
        const long g = (i + 1) + (j + 1) * X;
        if (a.order == 2) {
            if (l == 0) v = zd(v, u[g]);
            if (l == Nz - 1) v = zd(v, u[g + (Nz + 1) * XY]);
        } else {
            v = dirichlet3d(v, X, XY, (int)Nz, (int)l, g, a.coef + 12 * (long)(b % a.nop) * Nz, u);
        }
    }
    F[id] = v;
}

hipError_t launch_rhs3d(const Rhs3D &r, void *F, hipStream_t st) {
    if (r.order == 6) return launch_rhs3d_6(r, F, st);
    const long Nx = r.Nx, Ny = r.Ny, Nz = r.Nz;
    Rhs3DArgs a;
    a.order = r.order; a.Nx = r.Nx; a.Ny = r.Ny; a.Nz = r.Nz; a.hx = r.hx; a.hy = r.hy; a.hz = r.hz;
    a.f_e = (const z2 *)r.f_e; a.u_e = (const z2 *)r.u_e;
    a.coef = (const z2 *)r.coef; a.nop = r.nop > 0 ? r.nop : 1;
    long total = Nx * Ny * Nz * r.batch;
    hipLaunchKernelGGL(k_rhs3d_combine, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a, total, (z2 *)F);
    return hipGetLastError();
}

// ---------------------------------------------------------------- residual
// res = A u - F with the ghosts of u zero (2D_Program/main_functions/
// residual.c:3-34, 3D_Program/main_functions/residual.c:42-96).  Each thread
// marches along the last axis over a chunk of rows (2D) or layers (3D),
// keeping the 3 x 3 (x 3) neighbourhood in registers so that every value of
// u is loaded about once per thread row; the coefficient row of a step is
// the same for the whole block and comes through scalar loads (__restrict__: the
// result never overlaps the table); as vector loads each row's coefficients were
// waited for behind the row's own.  The sums keep the order of the reference.
// 64 x 1023^2: 689 -> 599 us (5.4 TB/s), 8 x 1023^2: 93 -> 74 us.
constexpr int RES_ROWS = 4;   // rows per thread in 2D (8 rows: 618 and 79 us; 16: 663 and 92)

// NORM: the maxima of |res|^2 (as stored) and |F|^2 go to `norms` as well, one
// atomic maximum of each per block (the bits of a nonnegative double order as
// an integer, so the result does not depend on the order).  A refinement
// sweep's norm then costs no pass of its own: 127 x 255 x 200 in FP32, 11 us a
// sweep, and 17 us for the norm of F.
template <int NT> HH_DEV void block_norms(double r2, double f2, unsigned long long *norms, unsigned block) {
    constexpr int NW = NT / 64;
    __shared__ double part[2 * NW];
    const int t = threadIdx.y * blockDim.x + threadIdx.x;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        r2 = fmax(r2, __shfl_xor(r2, s));
        f2 = fmax(f2, __shfl_xor(f2, s));
    }
    if (t % 64 == 0) { part[t / 64] = r2; part[NW + t / 64] = f2; }
    __syncthreads();
    if (t < 2) {
        double m = part[t * NW];
#pragma unroll
        for (int k = 1; k < NW; k++) m = fmax(m, part[t * NW + k]);
        atomicMax(norms + t * NORM_SLOTS + block % NORM_SLOTS, (unsigned long long)__double_as_longlong(m));
    }
}

template <typename To, bool NORM>
__global__ __launch_bounds__(256) void k_residual2d(int Nx, int Ny, const z2 *__restrict__ coef, int nop, const z2 *u,
                                                    const z2 *F, C2<To> *res, int b0, unsigned long long *norms) {
    int i = blockIdx.x * 256 + threadIdx.x;
    const int j0 = blockIdx.y * RES_ROWS;
    const int b = b0 + (int)blockIdx.z;
    double r2 = 0, f2 = 0;
    if constexpr (NORM) i = min(i, Nx - 1);   // idle lanes repeat the last column
    else if (i >= Nx) return;
    const long Nxy = (long)Nx * Ny;
    const z2 *ub = u + b * Nxy;
    const z2 *cb = coef + 6L * (b % nop) * Ny;   // per row: bm, am, b, a, bp, ap
    auto row = [&](int jj, z2 &l, z2 &c, z2 &r) {
        if (jj < 0 || jj >= Ny) { l = c = r = zr(0.0); return; }
        const z2 *p = ub + (long)jj * Nx;
        c = p[i];
        l = i > 0 ? p[i - 1] : zr(0.0);
        r = i + 1 < Nx ? p[i + 1] : zr(0.0);
    };
    z2 lm, cm, rm, l0, c0, r0, lp, cp, rp;
    row(j0 - 1, lm, cm, rm);
    row(j0, l0, c0, r0);
    const int j1 = min(j0 + RES_ROWS, Ny);
    for (int j = j0; j < j1; j++) {
        row(j + 1, lp, cp, rp);
        const z2 *cq = cb + 6L * j;
        const z2 top = za(za(zm(cq[4], lp), zm(cq[5], cp)), zm(cq[4], rp));
        const z2 mid = za(za(zm(cq[2], l0), zm(cq[3], c0)), zm(cq[2], r0));
        const z2 bot = za(za(zm(cq[0], lm), zm(cq[1], cm)), zm(cq[0], rm));
        const long id = b * Nxy + (long)j * Nx + i;
        const z2 f = F[id];
        const C2<To> r = cconv<To, double>(zd(za(za(top, mid), bot), f));
        res[id] = r;
        if constexpr (NORM) {
            r2 = fmax(r2, cabs2<double>(cconv<double, To>(r)));
            f2 = fmax(f2, cabs2<double>(f));
        }
        lm = l0; cm = c0; rm = r0;
        l0 = lp; c0 = cp; r0 = rp;
    }
    if constexpr (NORM) block_norms<256>(r2, f2, norms, blockIdx.y + blockIdx.z * gridDim.y);
}


// Tile of the 3D residual: RX x RY points of a layer per block, marching
// RZ layers along z.  Each layer's tile with its one-point halo goes
// through LDS once, loaded coalesced (three layer buffers in rotation); a
// thread reads the new layer's nine values from LDS per step and keeps, for
// each of its three layers, the four sums the stencil weights.  The loads are software-
// pipelined: a step stores the layer fetched during the previous step and
// issues the fetch of the next one (and of the next F value) before its
// barrier, so HBM latency is not paid once per layer.  The coefficients come
// through scalar loads (__restrict__: the result never overlaps the table): as
// vector loads they sat behind the prefetches in the in-order load counter, and
// every step waited for the next layer it had just asked for.  255^3: 242 ->
// 165 us (4.8 TB/s), 127 x 255 x 200: 105 -> 71 us; two and three layers ahead
// measured the same.  Tiles are 64 points wide, 32 where that covers Nx with
// fewer idle lanes (200^3: 89 against 95 us; 255^3: 178 against 168).
constexpr int RY = 8, RZ = 16;

template <typename To, int RX, bool NORM>
__global__ __launch_bounds__(RX * RY) void k_residual3d(int Nx, int Ny, int Nz, int nchunk, const z2 *__restrict__ coef, int nop,
                                                       const z2 *u, const z2 *F, C2<To> *res, int b0,
                                                       unsigned long long *norms) {
    constexpr int HX = RX + 2, HY = RY + 2, HE = HX * HY, NT = RX * RY;
    static_assert(HE <= 2 * NT, "a layer tile with halo takes at most two loads per thread");
    __shared__ z2 lay[3][HE];
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * RX + tx;
    const int i0 = blockIdx.x * RX, j0 = blockIdx.y * RY;
    const int i = i0 + tx, j = j0 + ty;
    const int zc = (int)blockIdx.z % nchunk;
    const int b = b0 + (int)blockIdx.z / nchunk;
    const long Nxy = (long)Nx * Ny, N3 = Nxy * Nz;
    const z2 *ub = u + b * N3;
    // the (at most two) halo-tile elements this thread loads; points outside
    // the grid read zero (the reference's zero ghosts)
    const int e1 = tid + NT;
    const bool has1 = e1 < HE;
    auto src = [&](int e, int ll, bool &in) -> long {
        const int hy = e / HX, hx = e - hy * HX;
        const int ii = i0 + hx - 1, jj = j0 + hy - 1;
        in = ll >= 0 && ll < Nz && ii >= 0 && ii < Nx && jj >= 0 && jj < Ny;
        return in ? ii + (long)jj * Nx + (long)ll * Nxy : 0;
    };
    z2 n0, n1, fn;   // the next layer's elements and right-hand side, in flight during a step
    auto zsel = [](bool c, z2 v) { return mk<double>(c ? v.x : 0.0, c ? v.y : 0.0); };
    auto fetch = [&](int ll) {
        bool in0, in1;
        const long s0 = src(tid, ll, in0), s1 = src(has1 ? e1 : tid, ll, in1);
        n0 = ub[s0];
        n1 = ub[s1];
    };
    auto stash = [&](int slot, int ll) {
        bool in0, in1;
        src(tid, ll, in0);
        src(has1 ? e1 : tid, ll, in1);
        lay[slot][tid] = zsel(in0, n0);
        if (has1) lay[slot][e1] = zsel(in1, n1);
    };
    // a layer's 3 x 3 neighbourhood enters only through four coefficient-free
    // sums (corners, x and y neighbours, centre), kept instead of the nine values
    struct Part { z2 corner, xn, yn, ctr; };
    auto plane = [&](int slot, Part &p) {
        const z2 *q = &lay[slot][(ty + 1) * HX + tx + 1];
        p.corner = za(za(za(q[HX + 1], q[HX - 1]), q[-HX + 1]), q[-HX - 1]);
        p.xn = za(q[1], q[-1]);
        p.yn = za(q[HX], q[-HX]);
        p.ctr = q[0];
    };
    // one layer's contribution, coefficients c = (a, b, c, d) of that layer set
    auto layer = [&](const Part &p, const z2 *c) -> z2 {
        return za(za(za(zm(c[3], p.ctr), zm(c[0], p.corner)), zm(c[1], p.xn)), zm(c[2], p.yn));
    };
    const int l0 = zc * RZ, l1 = min(l0 + RZ, Nz);
    const bool out = i < Nx && j < Ny;
    const long id0 = b * N3 + (long)(out ? j : 0) * Nx + (out ? i : 0);
    fetch(l0 - 1);
    stash(0, l0 - 1);
    fetch(l0);
    stash(1, l0);
    fetch(l0 + 1);
    fn = F[id0 + (long)l0 * Nxy];
    __syncthreads();
    Part pm, pc, pp;
    plane(0, pm);
    plane(1, pc);
    double r2 = 0, f2 = 0;
    int sn = 2;   // the slot of layer l+1: that of layer l-2, last read a barrier ago
    for (int l = l0; l < l1; l++) {
        stash(sn, l + 1);
        const z2 f = fn;
        // past the chunk's halo: one address, never used
        fetch(l + 2 <= l1 ? l + 2 : -1);
        fn = F[id0 + (long)min(l + 1, l1 - 1) * Nxy];
        __syncthreads();
        plane(sn, pp);
        if (out) {
            const z2 *cl = coef + 12 * ((long)(b % nop) * Nz + l);   // a..d, ap..dp, am..dm
            z2 acc = layer(pm, cl + 8);
            acc = za(acc, layer(pc, cl));
            acc = za(acc, layer(pp, cl + 4));
            const C2<To> r = cconv<To, double>(zd(acc, f));
            res[id0 + (long)l * Nxy] = r;
            if constexpr (NORM) {
                r2 = fmax(r2, cabs2<double>(cconv<double, To>(r)));
                f2 = fmax(f2, cabs2<double>(f));
            }
        }
        pm = pc;
        pc = pp;
        // slot sn is next rewritten two steps on; every thread has passed
        // the next step's barrier, after its read here, by then
        sn = sn == 2 ? 0 : sn + 1;
    }
    if constexpr (NORM)
        block_norms<NT>(r2, f2, norms, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}

hipError_t launch_residual2d(int Nx, int Ny, int batch, const void *coef, int nop, const void *u, const void *F,
                             void *res, int res_f32, void *norms, hipStream_t st) {
    if (norms && !res_f32) return hipErrorInvalidValue;
    for (int b0 = 0; b0 < batch; b0 += 65535) {   // grid z holds at most 65535 right-hand sides
        const int nb = batch - b0 < 65535 ? batch - b0 : 65535;
        dim3 g((unsigned)((Nx + 255) / 256), (unsigned)((Ny + RES_ROWS - 1) / RES_ROWS), (unsigned)nb);
        auto run = [&](auto kfn, auto *out) {
            hipLaunchKernelGGL(kfn, g, dim3(256), 0, st, Nx, Ny, (const z2 *)coef, nop, (const z2 *)u, (const z2 *)F, out,
                               b0, (unsigned long long *)norms);
        };
        if (norms) run(k_residual2d<float, true>, (float2 *)res);
        else if (res_f32) run(k_residual2d<float, false>, (float2 *)res);
        else run(k_residual2d<double, false>, (z2 *)res);
    }
    return hipGetLastError();
}

hipError_t launch_residual3d(int Nx, int Ny, int Nz, int batch, const void *coef, int nop, const void *u,
                             const void *F, void *res, int res_f32, void *norms, hipStream_t st) {
    const int nchunk = (Nz + RZ - 1) / RZ;
    const int per = 65535 / nchunk;   // right-hand sides per launch (grid z)
    if (per < 1 || (norms && !res_f32)) return hipErrorInvalidValue;
    const int RX = (Nx + 63) / 64 * 64 > (Nx + 31) / 32 * 32 ? 32 : 64;
    for (int b0 = 0; b0 < batch; b0 += per) {
        const int nb = batch - b0 < per ? batch - b0 : per;
        dim3 g((unsigned)((Nx + RX - 1) / RX), (unsigned)((Ny + RY - 1) / RY), (unsigned)(nchunk * nb));
        auto run = [&](auto kfn, auto *out) {
            hipLaunchKernelGGL(kfn, g, dim3(RX, RY), 0, st, Nx, Ny, Nz, nchunk, (const z2 *)coef, nop, (const z2 *)u,
                               (const z2 *)F, out, b0, (unsigned long long *)norms);
        };
        if (norms) run(RX == 64 ? k_residual3d<float, 64, true> : k_residual3d<float, 32, true>, (float2 *)res);
        else if (res_f32) run(RX == 64 ? k_residual3d<float, 64, false> : k_residual3d<float, 32, false>, (float2 *)res);
        else run(RX == 64 ? k_residual3d<double, 64, false> : k_residual3d<double, 32, false>, (z2 *)res);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- norms
// max |x| and max |x - y| (L2 = false), or sqrt(sum |x|^2) and
// sqrt(sum |x - y|^2) (L2 = true), over n complex values, in two passes
// without atomics: each block writes the maxima (sums) of |x|^2 and
// |x - y|^2 over its share to part[blockIdx.x] and part[NORM_BLOCKS +
// blockIdx.x], then one block combines them and roots the result once (sqrt
// is correctly rounded and monotonic, so the maximum equals the maximum of
// the rooted values).  The grid and the reduction tree are fixed, so a sum
// is the same bits from run to run.  Four values per thread and step are
// loaded before any is used.
template <bool L2> HH_DEV double norm_join(double a, double b) { return L2 ? a + b : fmax(a, b); }

template <bool L2>
__global__ __launch_bounds__(256) void k_norms(long n, const z2 *x, const z2 *y, double *part) {
    __shared__ double s0[256], s1[256];
    double m0 = 0, m1 = 0;
    const long stride = (long)gridDim.x * blockDim.x;
    long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
    for (; id + 3 * stride < n; id += 4 * stride) {
        z2 a[4], c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) a[u] = x[id + u * stride];
        if (y) {
#pragma unroll
            for (int u = 0; u < 4; u++) c[u] = y[id + u * stride];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            m0 = norm_join<L2>(m0, cabs2<double>(a[u]));
            if (y) m1 = norm_join<L2>(m1, cabs2<double>(zd(a[u], c[u])));
        }
    }
    for (; id < n; id += stride) {
        const z2 a = x[id];
        m0 = norm_join<L2>(m0, cabs2<double>(a));
        if (y) m1 = norm_join<L2>(m1, cabs2<double>(zd(a, y[id])));
    }
    s0[threadIdx.x] = m0;
    s1[threadIdx.x] = m1;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            s0[threadIdx.x] = norm_join<L2>(s0[threadIdx.x], s0[threadIdx.x + s]);
            s1[threadIdx.x] = norm_join<L2>(s1[threadIdx.x], s1[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = s0[0];
        part[NORM_BLOCKS + blockIdx.x] = s1[0];
    }
}

template <bool L2>
__global__ __launch_bounds__(256) void k_norms_final(int nb, const double *part, double *out) {
    __shared__ double s0[256], s1[256];
    double m0 = 0, m1 = 0;
    for (int b = threadIdx.x; b < nb; b += 256) {
        m0 = norm_join<L2>(m0, part[b]);
        m1 = norm_join<L2>(m1, part[NORM_BLOCKS + b]);
    }
    s0[threadIdx.x] = m0;
    s1[threadIdx.x] = m1;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            s0[threadIdx.x] = norm_join<L2>(s0[threadIdx.x], s0[threadIdx.x + s]);
            s1[threadIdx.x] = norm_join<L2>(s1[threadIdx.x], s1[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = sqrt(s0[0]);
        out[1] = sqrt(s1[0]);
    }
}

// The two maxima that the residuals left in `norms`, rooted, which are zeroed for the next sweep.
static_assert(NORM_SLOTS == 256, "one slot of each maximum per thread");
__global__ __launch_bounds__(256) void k_residual_norms(unsigned long long *norms, double *out) {
    __shared__ double part[8];
    const int t = threadIdx.x;
    double m[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        m[k] = __longlong_as_double((long long)norms[k * NORM_SLOTS + t]);
        norms[k * NORM_SLOTS + t] = 0;
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) m[k] = fmax(m[k], __shfl_xor(m[k], s));
        if (t % 64 == 0) part[4 * k + t / 64] = m[k];
    }
    __syncthreads();
    if (t < 2) out[t] = sqrt(fmax(fmax(part[4 * t], part[4 * t + 1]), fmax(part[4 * t + 2], part[4 * t + 3])));
}

hipError_t launch_residual_norms(void *norms, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_residual_norms, dim3(1), dim3(256), 0, st, (unsigned long long *)norms, out);
    return hipGetLastError();
}

hipError_t launch_norms(long n, const void *x, const void *y, double *part, double *out, hipStream_t st, bool l2) {
    long blocks = (n + 2047) / 2048;   // about eight values per thread
    if (blocks > NORM_BLOCKS) blocks = NORM_BLOCKS;
    if (blocks < 1) blocks = 1;
    auto run = [&](auto L) -> hipError_t {
        constexpr bool B = decltype(L)::value;
        hipLaunchKernelGGL(k_norms<B>, dim3((unsigned)blocks), dim3(256), 0, st, n, (const z2 *)x, (const z2 *)y, part);
        hipLaunchKernelGGL(k_norms_final<B>, dim3(1), dim3(256), 0, st, (int)blocks, (const double *)part, out);
        return hipGetLastError();
    };
    return l2 ? run(std::true_type()) : run(std::false_type());
}

}  // namespace hh
