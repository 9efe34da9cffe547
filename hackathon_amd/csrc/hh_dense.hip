// Dense DST-I kernels for gfx950: line lengths N whose N+1 is not a power of
// two (e.g. N = 100), the sine matrix times the lines.  Counterpart of the
// reference's FFTW / cuFFT transforms at such sizes (2D_Program/
// solver_functions/DST.c:6-44, 3D_Program/solver_functions/DST.c:13-204).
#include "hh_common.h"
#include "hh_internal.h"

namespace hh {

// Dense DST: out[line][k] = sum_n S[k][n] in[line][n].  Block tile: 32 lines x
// 64 outputs, 256 threads, each thread 8 outputs of one line.
template <typename Ti, typename T, typename To>
__global__ __launch_bounds__(256) void k_dst_gemm(const C2<Ti> *__restrict__ in, C2<To> *__restrict__ out,
                                                  Lines ln, long nlines, const T *__restrict__ S) {
    constexpr int TL = 32, TK = 64, TN = 32;
    __shared__ C2<T> xs[TL][TN + 1];
    __shared__ T ss[TN][TK + 1];
    const int N = ln.N, HP = half_dst_rows(N), WP = half_dst_cols(N);
    const long l0 = (long)blockIdx.x * TL;
    const int k0 = blockIdx.y * TK;
    const int tl = threadIdx.x % TL, tk = threadIdx.x / TL;  // tk in [0,8)
    C2<T> acc[8];
#pragma unroll
    for (int u = 0; u < 8; u++) acc[u] = mk<T>(0, 0);
    auto line_base = [&](long l) -> long {
        long p = l / ln.ncols, c = l % ln.ncols;
        return p * ln.plane_stride + c * ln.col_stride;
    };
    for (int n0 = 0; n0 < N; n0 += TN) {
        for (int e = threadIdx.x; e < TL * TN; e += 256) {
            int a, b;  // a: line in tile, b: n in tile
            if (ln.elem_stride == 1) { a = e / TN; b = e % TN; }
            else { a = e % TL; b = e / TL; }
            long l = l0 + a;
            int n = n0 + b;
            C2<T> v = mk<T>(0, 0);
            if (l < nlines && n < N) v = cconv<T, Ti>(in[line_base(l) + (long)n * ln.elem_stride]);
            xs[a][b] = v;
        }
        for (int e = threadIdx.x; e < TN * TK; e += 256) {
            int b = e / TK, kk = e % TK;
            const int n = n0 + b, k = k0 + kk;
            T v = 0;
            if (n < N && k < N) {   // the second half of a line mirrors the first, the middle has its full weight
                const bool mirror = 2 * n >= N, mid = 2 * n + 1 == N;
                v = S[((long)(k & 1) * HP + (mirror ? N - 1 - n : n)) * WP + k / 2];
                v = mid ? 2 * v : mirror && (k & 1) ? -v : v;
            }
            ss[b][kk] = v;
        }
        __syncthreads();
#pragma unroll 4
        for (int b = 0; b < TN; b++) {
            C2<T> xv = xs[tl][b];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                T s = ss[b][tk + 8 * u];
                acc[u].x += xv.x * s;
                acc[u].y += xv.y * s;
            }
        }
        __syncthreads();
    }
    long l = l0 + tl;
    if (l < nlines) {
        long bse = line_base(l);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            int k = k0 + tk + 8 * u;
            if (k < N) put_out<To, T>(out + bse + (long)k * ln.elem_stride, acc[u], ln.acc);
        }
    }
}

// Dense DST on the matrix cores, N+1 not a power of two.  The sine matrix is
// symmetric or antisymmetric about the middle of a line, sin(pi (M-j) k/M) =
// +-sin(pi j k/M) for odd / even k (M = N+1), so the odd outputs are a
// transform of x_j + x_{M-j} and the even ones of x_j - x_{M-j}: two products
// of half the length and half the width, half the operations of the full
// matrix.  The lines' real and imaginary parts form the rows of a real matrix
// (row 2l + c = part c of line l) and each parity is a real GEMM
// (v_mfma_f64_16x16x4f64 in FP64, v_mfma_f32_16x16x4f32 in FP32).
//
// A block computes ROWS rows x 2 BN neighbouring outputs: WR x WC waves per
// parity, each of RT x CT MFMA tiles.  K goes through LDS BK at a time, sums
// and differences formed on the way in, the next chunk loaded into registers
// meanwhile.  LDS row strides are 16 mod 32 elements, which puts the two k
// rows that a half wave reads on distinct banks, and row r of step k sits at
// r ^ 2 (k/2 mod 8), which does the same for the writes (threads along k); the
// plain order had 8-way conflicts there.  The output tile goes back through
// LDS so that stores are coalesced for contiguous and for strided lines.
// Operand layouts (lane l): A[l % 16][l / 16], B[l / 16][l % 16]; result j of
// lane l is row l / 16 + 4 j (FP64) or 4 (l / 16) + j (FP32) of column l % 16.
//
// What bounds it: the matrix cores where K is long.  3000 lines of N = 500,
// FP64: 41 us a pass (82 us for the full matrix), 36 TFLOP/s of the half
// product against 72 measured for a large FP64 matrix product on this card;
// 125^3 with N = 125: 18.5 us (38 us), of which the 62 MB of lines take 8 us.
// Eight waves of 32 x 16 against four of 32 x 32: 108 against 112 us and 101
// against 104 us for the whole solves of those grids (500 x 375 x 8, 125^3);
// chunks of 32, 128-row tiles and three waves per SIMD were slower.
//
// Tables (half_dst_rows, half_dst_cols): per parity [HP][WP], zero past the parity's size,
// the middle point of an odd N (its own mirror) at half weight.
template <typename T> struct Mfma16;
template <> struct Mfma16<double> {
    typedef double V __attribute__((ext_vector_type(4)));
    static HH_DEV V step(double a, double b, V c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static HH_DEV int row(int l, int j) { return l / 16 + 4 * j; }
};
template <> struct Mfma16<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    static HH_DEV V step(float a, float b, V c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static HH_DEV int row(int l, int j) { return 4 * (l / 16) + j; }
};

template <int RT_, int CT_, int WR_, int WC_, int BK_> struct DenseTile {
    static constexpr int RT = RT_, CT = CT_, WR = WR_, WC = WC_, BK = BK_;
    static constexpr int ROWS = 16 * RT * WR, BL = ROWS / 2, BN = 16 * CT * WC, NT = 128 * WR * WC;
    static constexpr int XS = ROWS % 32 == 16 ? ROWS : ROWS + 16;   // LDS row strides: 16 mod 32
    static constexpr int SS = BN % 32 == 16 ? BN : BN + 16;
    static constexpr int OS = 2 * BN + 1;
    static constexpr int STAGE = 2 * BK * (XS + SS), OUTT = ROWS * OS;
    static constexpr int LDS = STAGE > OUTT ? STAGE : OUTT;
    static_assert(HH_DENSE_HP % BK == 0 && HH_DENSE_WP % BN == 0, "tables are padded to whole tiles");
};

template <typename Ti, typename T, typename To, class C>
__global__ __launch_bounds__(C::NT, 4) void k_dst_mfma(const C2<Ti> *__restrict__ in, C2<To> *__restrict__ out, Lines ln,
                                                    long nlines, const T *__restrict__ S) {
    using M = Mfma16<T>;
    constexpr int RT = C::RT, CT = C::CT, BL = C::BL, BN = C::BN, BK = C::BK, NT = C::NT, XS = C::XS, SS = C::SS;
    __shared__ __align__(16) T sh[C::LDS];
    __shared__ long lbase[BL];   // first element of the block's lines: one 64-bit division per line
    T *xs = sh, *ss = sh + 2 * BK * XS;
    const int N = ln.N, H = (N + 1) / 2;
    // Block -> (lines, outputs): the ny output tiles of one tile of lines run
    // next to each other on one XCD (blocks go round-robin to the 8 XCDs), so
    // that the lines are read from HBM once and then from that XCD's L2
    const unsigned ny = ((unsigned)(N + 1) / 2 + BN - 1) / BN;
    const unsigned nl8 = (gridDim.x / ny) & ~7u;
    unsigned lt, nt;
    if (blockIdx.x < nl8 * ny) {
        const unsigned s = blockIdx.x >> 3;
        nt = s % ny;
        lt = (s / ny) * 8 + (blockIdx.x & 7);
    } else {
        const unsigned s = blockIdx.x - nl8 * ny;
        nt = s % ny;
        lt = nl8 + s / ny;
    }
    const long l0 = (long)lt * BL;
    const int n0 = nt * BN;   // first output of each parity
    const int t = threadIdx.x, lane = t % 64, wv = t / 64;
    const int par = wv & 1, wr = (wv >> 1) % C::WR, wc = (wv >> 1) / C::WR;
    const int HP = half_dst_rows(N), WP = half_dst_cols(N);
    const bool rows = ln.elem_stride == 1;
    if (t < BL) {
        const long l = min(l0 + t, nlines - 1);   // lines past the end repeat the last one and are not stored
        const long p = l / ln.ncols, c = l - p * ln.ncols;
        lbase[t] = p * ln.plane_stride + c * ln.col_stride;
    }
    __syncthreads();
    typename M::V acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++) acc[i][j] = typename M::V{0, 0, 0, 0};
    // a thread's slots of the chunk: XI (line, k) pairs with their mirrors
    // (contiguous lines: threads along the line, strided lines: threads across
    // lines) and SI pairs of neighbouring table entries
    constexpr int XI = BL * BK / NT, SI = 2 * BK * BN / 2 / NT;
    static_assert(XI * NT == BL * BK && SI * NT == BK * BN, "whole slots per thread");
    const C2<Ti> *xp[XI];
    int xk[XI], xo[XI];
#pragma unroll
    for (int i = 0; i < XI; i++) {
        const int e = t + NT * i;
        const int a = rows ? e / BK : e % BL, b = rows ? e % BK : e / BL;
        xp[i] = in + lbase[a];
        xk[i] = b;
        xo[i] = b * XS + 2 * (a ^ ((b >> 1) & 7));
    }
    C2<Ti> xa[XI], xb[XI];
    C2<T> sv[SI];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int k = min(k0 + xk[i], N - 1);   // past the end: in bounds, zeroed on the way to LDS
            xa[i] = xp[i][(long)k * ln.elem_stride];
            xb[i] = xp[i][(long)(N - 1 - k) * ln.elem_stride];
        }
#pragma unroll
        for (int i = 0; i < SI; i++) {
            const int e = 2 * (t + NT * i);
            const int b = e / BN, c = e % BN;   // b: parity, then row of the chunk
            const C2<T> v = *reinterpret_cast<const C2<T> *>(S + ((long)(b / BK) * HP + k0 + b % BK) * WP + n0 + c);
            sv[i] = mk<T>(v.x, v.y);
        }
    };
    load(0);
    for (int k0 = 0; k0 < H; k0 += BK) {
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const bool ok = k0 + xk[i] < H;
            const C2<T> s = cconv<T, Ti>(cadd<Ti>(xa[i], xb[i])), d = cconv<T, Ti>(csub<Ti>(xa[i], xb[i]));
            *reinterpret_cast<C2<T> *>(xs + xo[i]) = ok ? s : mk<T>(0, 0);
            *reinterpret_cast<C2<T> *>(xs + BK * XS + xo[i]) = ok ? d : mk<T>(0, 0);
        }
#pragma unroll
        for (int i = 0; i < SI; i++) {
            const int e = 2 * (t + NT * i);
            *reinterpret_cast<C2<T> *>(ss + (e / BN) * SS + e % BN) = mk<T>(sv[i].x, sv[i].y);
        }
        __syncthreads();
        if (k0 + BK < H) load(k0 + BK);
        const T *xw = xs + par * BK * XS + wr * 16 * RT + (lane / 16) * XS;
        const int xr = lane % 16 ^ 2 * (lane >> 5);
        const T *sw = ss + par * BK * SS + wc * 16 * CT + lane % 16 + (lane / 16) * SS;
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            T a[RT], b[CT];
#pragma unroll
            for (int i = 0; i < RT; i++) a[i] = xw[kk * XS + 16 * i + (xr ^ (kk & 12))];
#pragma unroll
            for (int j = 0; j < CT; j++) b[j] = sw[kk * SS + 16 * j];
#pragma unroll
            for (int i = 0; i < RT; i++)
#pragma unroll
                for (int j = 0; j < CT; j++) acc[i][j] = M::step(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
    // output tile through LDS, the parities interleaved
    constexpr int OS = C::OS;
    T *os = sh;
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int j = 0; j < CT; j++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                os[(wr * 16 * RT + 16 * i + M::row(lane, q)) * OS + 2 * (wc * 16 * CT + 16 * j + lane % 16) + par] =
                    acc[i][j][q];
    __syncthreads();
#pragma unroll
    for (int e = t; e < BL * 2 * BN; e += NT) {
        const int a = rows ? e / (2 * BN) : e % BL, c = rows ? e % (2 * BN) : e / BL;
        const int n = 2 * n0 + c;
        if (l0 + a < nlines && n < N)
            put_out<To, T>(out + lbase[a] + (long)n * ln.elem_stride, mk<T>(os[2 * a * OS + c], os[(2 * a + 1) * OS + c]),
                           ln.acc);
    }
}

template <typename Ti, typename T, typename To>
static hipError_t launch_dense_t(const Lines &ln, int algo, const void *in, void *out, const void *S, hipStream_t st) {
    if (in == out || S == nullptr) return hipErrorInvalidValue;
    long nlines = ln.ncols * ln.nplanes;
    if (algo & 8) {   // vector-FMA form (kept for comparison)
        dim3 grid((unsigned)((nlines + 31) / 32), (unsigned)((ln.N + 63) / 64));
        hipLaunchKernelGGL((k_dst_gemm<Ti, T, To>), grid, dim3(256), 0, st, (const C2<Ti> *)in, (C2<To> *)out, ln,
                           nlines, (const T *)S);
        return hipGetLastError();
    }
    auto run = [&](auto tile) -> hipError_t {
        using C = decltype(tile);
        const long blocks = ((nlines + C::BL - 1) / C::BL) * (((ln.N + 1) / 2 + C::BN - 1) / C::BN);
        if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_dst_mfma<Ti, T, To, C>), dim3((unsigned)blocks), dim3(C::NT), 0, st, (const C2<Ti> *)in,
                           (C2<To> *)out, ln, nlines, (const T *)S);
        return hipGetLastError();
    };
    // Whole tiles of 64 rows x 64 outputs when they give every CU a block;
    // fewer lines take tiles of 16 rows (8 lines) x 64 outputs with K in
    // chunks of 32, where the latency of a chunk, not the matrix rate, counts
    // (100 lines of N = 100: 4.3 us a pass, 13.2 us before in 64-row tiles).
    using Big = DenseTile<2, 1, 2, 2, 16>;
    using Small = DenseTile<1, 1, 1, 2, 32>;
    const long big = ((nlines + Big::BL - 1) / Big::BL) * (((ln.N + 1) / 2 + Big::BN - 1) / Big::BN);
    return big >= 256 ? run(Big{}) : run(Small{});
}

hipError_t launch_dense(const Lines &ln, int algo, int ti, int tc, int to, const void *in, void *out, const void *S,
                        hipStream_t st) {
    if (tc == 0) {
        if (ti == 0 && to == 0) return launch_dense_t<double, double, double>(ln, algo, in, out, S, st);
        return hipErrorInvalidValue;
    }
    if (ti == 0 && to == 1) return launch_dense_t<double, float, float>(ln, algo, in, out, S, st);
    if (ti == 1 && to == 1) return launch_dense_t<float, float, float>(ln, algo, in, out, S, st);
    if (ti == 1 && to == 0) return launch_dense_t<float, float, double>(ln, algo, in, out, S, st);
    return hipErrorInvalidValue;
}

}  // namespace hh
