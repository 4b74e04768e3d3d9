#pragma once

#include "sc_internal.h"

// Shared by the transform sources (fft_kernels.hip, fft_x.hip, fft_z.hip):
// the small DFTs, the compile-time plans and the kernels' argument blocks.
//
// The sources are compiled twice: as they are (sc::fp64, FP64 transforms) and with
// SC_FFT_F32 defined (sc::fp32: transforms, products and the intermediate
// arrays W1, W2 and the cached fields in FP32).  The state arrays read at
// the start (U, FP64) and the results written at the end (the Gauss-point
// slots, FP64) are FP64 in both; values are converted on load and store.
#ifdef SC_FFT_F32
#define SC_FFT_NS fp32
#else
#define SC_FFT_NS fp64
#endif

namespace sc {
namespace SC_FFT_NS {

#ifdef SC_FFT_F32
using real = float;
using real2 = float2;
#else
using real = double;
using real2 = double2;
#endif

__host__ __device__ __forceinline__ real2 mk2(real a, real b)
{
    real2 v;
    v.x = a;
    v.y = b;
    return v;
}
__device__ __forceinline__ real2 to_real2(const double2 &v) { return mk2((real) v.x, (real) v.y); }
__device__ __forceinline__ double2 to_cplx(const real2 &v) { return make_double2(v.x, v.y); }
// member stride of an array viewed as real2 values
static inline size_t rstride(const Context &c, const void *p) { return mstride_bytes(c, p) / sizeof(real2); }

constexpr int BLK = FFT_BLOCK;   // threads per block of the runtime-length kernels

// Rounding.  A sum of two products is one product rounded and one multiply-add,
// and which of the two is which is written out below: left to the compiler, the
// choice would follow the code around it, and a transform would round
// differently in kernels of another length, tile or mode.  (The Galerkin solves
// amplify a last-bit difference to 1e-9 of the state and the FP32 build's to
// 1e-5, so kernels that share a result have to agree to the bit.)
__device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// a t for a twiddle t of the table, conjugated for sign < 0
__device__ __forceinline__ real2 twiddle(real2 a, real2 t, real sign)
{
    if (sign > 0) return mk2(fma_(a.x, t.x, -(a.y * t.y)), fma_(a.y, t.x, a.x * t.y));
#ifdef SC_FFT_F32
    return mk2(fma_(a.y, t.y, a.x * t.x), fma_(a.y, t.x, -(a.x * t.y)));
#else
    return mk2(fma_(a.x, t.x, a.y * t.y), fma_(a.y, t.x, -(a.x * t.y)));
#endif
}

// cos and sin of 2 pi j / R, j < R (correctly rounded; exact where the value
// is 0, +-1/2 or +-1)
template <int R> struct RootTab;
template <> struct RootTab<6> {
    static constexpr double c[6] = {1.0, 0.5, -0.5, -1.0, -0.5, 0.5};
    static constexpr double s[6] = {0.0, 0.8660254037844386, 0.8660254037844386, 0.0, -0.8660254037844386, -0.8660254037844386};
};
template <> struct RootTab<8> {
    static constexpr double c[8] = {1.0, 0.7071067811865476, 0.0, -0.7071067811865476, -1.0, -0.7071067811865476, 0.0, 0.7071067811865476};
    static constexpr double s[8] = {0.0, 0.7071067811865476, 1.0, 0.7071067811865476, 0.0, -0.7071067811865476, -1.0, -0.7071067811865476};
};
template <> struct RootTab<12> {
    static constexpr double c[12] = {1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0, -0.8660254037844386, -0.5, 0.0, 0.5, 0.8660254037844386};
    static constexpr double s[12] = {0.0, 0.5, 0.8660254037844386, 1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0, -0.8660254037844386, -0.5};
};
template <> struct RootTab<16> {
    static constexpr double c[16] = {1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0, -0.3826834323650898, -0.7071067811865476, -0.9238795325112867, -1.0, -0.9238795325112867, -0.7071067811865476, -0.3826834323650898, 0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867};
    static constexpr double s[16] = {0.0, 0.3826834323650898, 0.7071067811865476, 0.9238795325112867, 1.0, 0.9238795325112867, 0.7071067811865476, 0.3826834323650898, 0.0, -0.3826834323650898, -0.7071067811865476, -0.9238795325112867, -1.0, -0.9238795325112867, -0.7071067811865476, -0.3826834323650898};
};

// In-place DFTs in registers: v[q] <- sum_m v[m] exp(sign 2 pi i m q / R).
__device__ __forceinline__ void dft2(real2 *v)
{
    real2 a = v[0], b = v[1];
    v[0] = mk2(a.x + b.x, a.y + b.y);
    v[1] = mk2(a.x - b.x, a.y - b.y);
}

__device__ __forceinline__ void dft4(real2 *v, real sign)
{
    real2 a0 = v[0], a1 = v[1], a2 = v[2], a3 = v[3];
    real2 s02 = mk2(a0.x + a2.x, a0.y + a2.y);
    real2 d02 = mk2(a0.x - a2.x, a0.y - a2.y);
    real2 s13 = mk2(a1.x + a3.x, a1.y + a3.y);
    real2 d13 = mk2(a1.x - a3.x, a1.y - a3.y);
    // w d13 with w = sign * i
    real2 wd = mk2(-sign * d13.y, sign * d13.x);
    v[0] = mk2(s02.x + s13.x, s02.y + s13.y);
    v[1] = mk2(d02.x + wd.x, d02.y + wd.y);
    v[2] = mk2(s02.x - s13.x, s02.y - s13.y);
    v[3] = mk2(d02.x - wd.x, d02.y - wd.y);
}

__device__ __forceinline__ void dft3(real2 *v, real sign)
{
    const real h = sign * (real) 0.86602540378443864676;   // sqrt(3)/2
    real2 a0 = v[0], a1 = v[1], a2 = v[2];
    real2 t1 = mk2(a1.x + a2.x, a1.y + a2.y);
    real2 t2 = mk2(fma_((real) -0.5, t1.x, a0.x), fma_((real) -0.5, t1.y, a0.y));
    real2 d = mk2(a1.x - a2.x, a1.y - a2.y);
    v[0] = mk2(a0.x + t1.x, a0.y + t1.y);
    v[1] = mk2(fma_(-h, d.y, t2.x), fma_(h, d.x, t2.y));
    v[2] = mk2(fma_(h, d.y, t2.x), fma_(-h, d.x, t2.y));
}

__device__ __forceinline__ void dft5(real2 *v, real sign)
{
    const real c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    const real s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    real2 a0 = v[0], a1 = v[1], a2 = v[2], a3 = v[3], a4 = v[4];
    real2 b1 = mk2(a1.x + a4.x, a1.y + a4.y);
    real2 b2 = mk2(a2.x + a3.x, a2.y + a3.y);
    real2 d1 = mk2(a1.x - a4.x, a1.y - a4.y);
    real2 d2 = mk2(a2.x - a3.x, a2.y - a3.y);
    real2 t1 = mk2(fma_(c2, b2.x, fma_(c1, b1.x, a0.x)), fma_(c2, b2.y, fma_(c1, b1.y, a0.y)));
    real2 t2 = mk2(fma_(c1, b2.x, fma_(c2, b1.x, a0.x)), fma_(c1, b2.y, fma_(c2, b1.y, a0.y)));
    real2 u1 = mk2(sign * fma_(s2, d2.x, s1 * d1.x), sign * fma_(s2, d2.y, s1 * d1.y));
    real2 u2 = mk2(sign * fma_(s2, d1.x, -(s1 * d2.x)), sign * fma_(s2, d1.y, -(s1 * d2.y)));
    v[0] = mk2(a0.x + b1.x + b2.x, a0.y + b1.y + b2.y);
    v[1] = mk2(t1.x - u1.y, t1.y + u1.x);
    v[4] = mk2(t1.x + u1.y, t1.y - u1.x);
    v[2] = mk2(t2.x - u2.y, t2.y + u2.x);
    v[3] = mk2(t2.x + u2.y, t2.y - u2.x);
}

template <int R> __device__ __forceinline__ void dft_prime(real2 *v, real sign)
{
    if constexpr (R == 2) dft2(v);
    else if constexpr (R == 3) dft3(v, sign);
    else if constexpr (R == 4) dft4(v, sign);
    else dft5(v, sign);
}

// How the first pass of a transform rounds its constant twiddles (see
// rounds_by_y).  Two lengths, 48 and 96, have an order of their own on the grids
// that tile evenly (even_columns, even_rows), the general one on the others.
// Both are as accurate; each grid keeps its order, so that a transform has the same
// bits in whatever kernel of the same fields.  (The merged adjoint kernel packs
// eight sequences, the single one five: on grids whose z rows come in the groups of
// the one only, 4 against 8 at 48 points and 2 against 4 at 96, an adjoint with
// cached fields and one without differ in the last bits.)
enum DftStart : int {
    DS_ANY = 0,        // the general order; every pass but the first
    DS_FORWARD = 1,    // forward transforms
    DS_ZINV_A = 2,     // z inverse transforms of a slot
    DS_ZINV_B = 3,     // ... of a field formed as a curl
};
constexpr bool start_length(int n) { return n == 48 || n == 96; }
// z transforms: the columns come in groups of 16
inline bool even_columns(int Mx) { return Mx % 16 == 0; }
// x transforms: the z rows come in groups of a 2048-value tile, nseq packed
// sequences a row
constexpr int even_group(int px, int nseq)
{
    int rows = 1;
    while (2 * rows <= 64 && 2 * rows * nseq * (px + 1) + px <= 2048) rows *= 2;
    return rows;
}
inline bool even_rows(int Px, int Pz, int nseq) { return Pz % even_group(Px, nseq) == 0; }

// Whether the real (im = 0) or imaginary (im = 1) part of t w, w = (c, s) the
// twiddle of (m2, k1) in a composite DFT, takes its t.y term (t.x otherwise) in
// the multiply-add and rounds the other one.
constexpr bool rounds_by_y(int R, int m2, int k1, bool fwd, int start, int im)
{
    if (!im) return R == 12 && start == DS_FORWARD && m2 == 2 && k1 == 2;
    if (R == 12 && start == DS_ZINV_A) return m2 == 1 && k1 == 1;
    if (R == 12 && start == DS_ZINV_B) return m2 == 1 && k1 == 2;
    if (R == 16) return (m2 * k1) % 2 != 0 && m2 * k1 != 9;
    if (R == 12) return k1 == 1 || (m2 == 1 && k1 == 2 && fwd);
    if (R == 8) return false;
    return k1 == 1 && fwd;             // 6
}

// Composite R = R1 R2 in registers: with m = R2 m1 + m2 and q = k1 + R1 k2,
// DFT_R = (R1 DFTs of length R2) . twiddles exp(sign 2 pi i m2 k1 / R) .
// (R2 DFTs of length R1).  The twiddles are compile-time constants; i, -1 and
// -i take no product.
template <int R1, int R2, int START>
__device__ __forceinline__ void dft_comp(real2 *v, real sign)
{
    constexpr int R = R1 * R2;
    real2 a[R];
#pragma unroll
    for (int m2 = 0; m2 < R2; ++m2) {
        real2 t[R1];
#pragma unroll
        for (int m1 = 0; m1 < R1; ++m1) t[m1] = v[R2 * m1 + m2];
        dft_prime<R1>(t, sign);
#pragma unroll
        for (int k1 = 0; k1 < R1; ++k1) {
            const int e = (m2 * k1) % R;
            const real2 x = t[k1];
            real2 &o = a[m2 * R1 + k1];
            if (e == 0) {
                o = x;
            } else if (2 * e == R) {
                o = mk2(-x.x, -x.y);
            } else if (4 * e == R) {
                o = mk2(-sign * x.y, sign * x.x);
            } else {
                const real c = (real) RootTab<R>::c[e], s = sign * (real) RootTab<R>::s[e];
                o.x = rounds_by_y(R, m2, k1, sign < 0, START, 0) ? fma_(-x.y, s, x.x * c)
                                                                 : fma_(x.x, c, -(x.y * s));
                o.y = rounds_by_y(R, m2, k1, sign < 0, START, 1) ? fma_(x.y, c, x.x * s)
                                                                 : fma_(x.x, s, x.y * c);
            }
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
        real2 t[R2];
#pragma unroll
        for (int m2 = 0; m2 < R2; ++m2) t[m2] = a[m2 * R1 + k1];
        dft_prime<R2>(t, sign);
#pragma unroll
        for (int k2 = 0; k2 < R2; ++k2) v[k1 + R1 * k2] = t[k2];
    }
}

template <int R, int START = DS_ANY> __device__ __forceinline__ void dft(real2 *v, real sign)
{
    if constexpr (R == 16) dft_comp<4, 4, START>(v, sign);
    else if constexpr (R == 12) dft_comp<4, 3, START>(v, sign);
    else if constexpr (R == 8) dft_comp<4, 2, START>(v, sign);
    else if constexpr (R == 6) dft_comp<3, 2, START>(v, sign);
    else dft_prime<R>(v, sign);
}

// ---------------------------------------------------------------- fixed lengths
// Transform lengths with a compile-time plan (k_xrow<MODE, PX>, k_zinv_c<PZ>,
// k_zfwd_c<PZ>, k_zadj_c<PZ>): radices, strides, the tile shape and all index
// divisions fold into constants.  The same rule as the host planner: fewest
// passes over the radices below, then the smallest per-thread tile; the same
// radices in the same order as the runtime plan, so a length gives the same
// bits through either.
struct PBest {
    int passes, worst, first;
};

constexpr int FIX_RADICES[] = {16, 12, 8, 6, 5, 4, 3, 2};

constexpr int fix_tile(int r) { return (FFT_TILE / BLK + r - 1) / r * r; }

constexpr PBest plan_best(int m)
{
    if (m == 1) return PBest{0, 0, 0};
    PBest b{1 << 20, 0, 0};
    for (int r : FIX_RADICES) {
        if (m % r) continue;
        const PBest sub = plan_best(m / r);
        if (sub.passes >= (1 << 20)) continue;
        const int np = sub.passes + 1, nw = sub.worst > fix_tile(r) ? sub.worst : fix_tile(r);
        if (np < b.passes || (np == b.passes && nw < b.worst)) b = PBest{np, nw, r};
    }
    return b;
}

// radix of pass p of the length-n plan
constexpr int plan_radix(int n, int p)
{
    int m = n;
    for (int i = 0; i < p; ++i) m /= plan_best(m).first;
    return plan_best(m).first;
}


// The dealiased lengths 3 Nx / 2 (Nx a multiple of 4) and 3 Nz / 2 (Nz even)
// up to 192 with at least two passes: these have kernels of their own.
#define SC_X_LENGTHS(F) \
    F(18) F(24) F(30) F(36) F(48) F(54) F(60) F(72) F(90) F(96) F(108) F(120) F(144) F(150) F(162) \
    F(180) F(192)
#define SC_Z_LENGTHS(F) \
    F(15) F(18) F(24) F(27) F(30) F(36) F(45) F(48) F(54) F(60) F(72) F(75) F(81) F(90) F(96) F(108) \
    F(120) F(135) F(144) F(150) F(162) F(180) F(192)

// Passes of a fixed-length transform by T threads over NSEQ sequences in LDS,
// element e of sequence s at s*SSTR + e*ESTR; item b of a pass is butterfly
// b / NSEQ of sequence b % NSEQ.
//
// First pass: the R1 inputs of a butterfly (elements j + q N/R1) come from
// ld(i, j, s, q) (i: the thread's item counter), so the load stage and the pass
// are one; nothing is read from LDS.  The caller synchronises afterwards.
template <int START, int N, int NSEQ, int SSTR, int ESTR, int T, class LD>
__device__ __forceinline__ void fft_first(real2 *data, real sign, LD ld)
{
    constexpr int R = plan_radix(N, 0), NBS = N / R, TOTAL = NSEQ * NBS;
    constexpr int NBT = (TOTAL + T - 1) / T;
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        const int b = threadIdx.x + i * T;
        if (TOTAL % T != 0 && b >= TOTAL) break;
        const int j = b / NSEQ, s = b - j * NSEQ;
        real2 v[R];
        ld(j, s, v);
        dft<R, START>(v, sign);
        real2 *dst = data + s * SSTR + j * R * ESTR;
#pragma unroll
        for (int q = 0; q < R; ++q) dst[q * ESTR] = v[q];
    }
}

// The same with the inputs in the memory that the outputs take: they wait in
// registers for the block's barrier.
template <int START, int N, int NSEQ, int SSTR, int ESTR, int T, class LD>
__device__ __forceinline__ void fft_first_in_place(real2 *data, real sign, LD ld)
{
    constexpr int R = plan_radix(N, 0), NBS = N / R, TOTAL = NSEQ * NBS;
    constexpr int NBT = (TOTAL + T - 1) / T;
    real2 v[NBT][R];
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        const int b = threadIdx.x + i * T, j = b / NSEQ, s = b - j * NSEQ;
        if (TOTAL % T == 0 || b < TOTAL) ld(j, s, v[i]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        const int b = threadIdx.x + i * T, j = b / NSEQ, s = b - j * NSEQ;
        if (TOTAL % T == 0 || b < TOTAL) {
            dft<R, START>(v[i], sign);
            real2 *dst = data + s * SSTR + j * R * ESTR;
#pragma unroll
            for (int q = 0; q < R; ++q) dst[q * ESTR] = v[i][q];
        }
    }
}

// inputs of butterfly j of sequence src, twiddled, and their DFT
template <int R, int N, int NS, int ESTR, int START = DS_ANY>
__device__ __forceinline__ void fft_butterfly(const real2 *src, int j, int k, const real2 *tw,
                                              real sign, real2 *v)
{
    constexpr int NBS = N / R, TWS = N / (NS * R);
#pragma unroll
    for (int q = 0; q < R; ++q) {
        real2 a = src[(j + q * NBS) * ESTR];
        if (q > 0 && NS > 1) {
            a = twiddle(a, tw[q * k * TWS], sign);
        }
        v[q] = a;
    }
    dft<R, START>(v, sign);
}

// a pass in place: the inputs wait in registers for the block's barrier
template <int START, int R, int N, int NS, int NSEQ, int SSTR, int ESTR, int T>
__device__ __forceinline__ void fft_pass_c(real2 *data, const real2 *tw, real sign)
{
    constexpr int NBS = N / R, TOTAL = NSEQ * NBS, NBT = (TOTAL + T - 1) / T;
    real2 v[NBT][R];
    int off[NBT];
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        const int b = threadIdx.x + i * T;
        const int j = b / NSEQ, s = b - j * NSEQ;
        off[i] = -1;
        if (TOTAL % T == 0 || b < TOTAL) {
            const int jq = j / NS, k = j - jq * NS;
            off[i] = s * SSTR + (jq * NS * R + k) * ESTR;
            fft_butterfly<R, N, NS, ESTR, START>(data + s * SSTR, j, k, tw, sign, v[i]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        if (off[i] >= 0) {
            real2 *dst = data + off[i];
#pragma unroll
            for (int q = 0; q < R; ++q) dst[q * NS * ESTR] = v[i][q];
        }
    }
    __syncthreads();
}

// passes P .. P1 - 1 in place
template <int N, int NSEQ, int SSTR, int ESTR, int T, int P1, int P = 0, int NS = 1, int START = DS_ANY>
__device__ __forceinline__ void lds_fft_c(real2 *data, const real2 *tw, real sign)
{
    if constexpr (P < P1) {
        constexpr int R = plan_radix(N, P);
        fft_pass_c<START, R, N, NS, NSEQ, SSTR, ESTR, T>(data, tw, sign);
        lds_fft_c<N, NSEQ, SSTR, ESTR, T, P1, P + 1, NS * R>(data, tw, sign);
    }
}

// Last pass: the outputs of a butterfly (elements k + q N/R) go to
// st(k, s, v) from registers; no barrier.
template <int N, int NSEQ, int SSTR, int ESTR, int T, class ST>
__device__ __forceinline__ void fft_last(const real2 *data, const real2 *tw, real sign, ST st)
{
    constexpr int P = plan_best(N).passes - 1, R = plan_radix(N, P), NS = N / R;
    constexpr int TOTAL = NSEQ * NS, NBT = (TOTAL + T - 1) / T;
#pragma unroll
    for (int i = 0; i < NBT; ++i) {
        const int b = threadIdx.x + i * T;
        if (TOTAL % T != 0 && b >= TOTAL) break;
        const int k = b / NSEQ, s = b - k * NSEQ;
        real2 v[R];
        fft_butterfly<R, N, NS, ESTR>(data + s * SSTR, k, k, tw, sign, v);
        st(k, s, v);
    }
}

template <int N, int T>
__device__ __forceinline__ void stage_twiddles_c(const double2 *tw, real2 *twl)
{
#pragma unroll
    for (int m = 0; m < N; m += T)
        if (m + T <= N || (int) threadIdx.x < N - m) twl[m + threadIdx.x] = to_real2(tw[m + threadIdx.x]);
}

// ---------------------------------------------------------------- arguments
struct ZinvArgs {
    FieldSpec fs;
    const double2 *tw;
    int Nz, Mx, qpts, Pz, XB, nm;
    double ax, az;                 // 2 pi / Lx, 2 pi / Lz
    const int *abort_flag;
    size_t ms_w1;                  // member stride of W1
};

struct XmixArgs {
    int mode, nf, nout, Mx, Px, Pz, qpts, ZB, check_cfl;
    int nm;                    // members (k_xrow_shared)
    const double2 *tw;
    int nf1;                   // fields 0..nf1-1 from the first source, the rest from W1b
    const real2 *W1b;
    int nf2;                   // XM_ADJ2: fields nf1..nf2-1 from W1b, nf2..nf-1 from W1c
    const real2 *W1c;
    real2 *W2b;                 // XM_ADJ2: the second product set
    double cfl1, cfl3;
    const double *cfl2;
    double *cflmax;        // [qpts], as ordered bit patterns
    double *flow;          // XM_PHYS output
    const int *abort_flag;
    // member strides of W1, W1b, W1c, W2, W2b (grid z = member)
    size_t ms_in, ms_inb, ms_inc, ms_out, ms_outb;
};

struct ZfwdArgs {
    int nout, Nz, Mx, Pz, qpts, XB, dst_kind, nm;
    const double2 *tw;
    double norm;
    const int *abort_flag;
    // cfl_slot >= 0: the first block runs the CFL check of the products
    // kernel's maxima first (in place of a separate launch)
    int cfl_slot;
    double *cflmax;
    double dt;
    int *abort_rw;
    size_t ms_in, ms_out;      // member strides of W2 and dst
    int p32;                   // ZF_USLOTS stored as FP32 complex (same element index)
};

struct ZadjArgs {
    int Nz, Mx, Pz, qpts, XA;
    const double2 *tw;
    double norm;
    const double *Kx, *Kz;
    const int *abort_flag;
    // a second problem (W2b -> Ub) in the same grid: nprob = 2
    int nprob;
    const real2 *W2b;
    cplx *Ub;
    // members (strides of W2 / W2b and U / Ub)
    int nm;
    size_t ms_in, ms_out;
    int p32;                   // the five slots stored as FP32 complex
};

__device__ __forceinline__ void atomic_max_nonneg(double *addr, double v)
{
    atomicMax((unsigned long long *) addr, (unsigned long long) __double_as_longlong(v));
}

// A Gauss-point slot value at element index i of src: FP64 complex, or
// FP32 complex (S32) where the mixed-precision rebuild stored the slots.
template <bool S32>
__device__ __forceinline__ double2 ld_slot(const cplx *src, size_t i)
{
    if constexpr (S32) {
        const float2 v = ((const float2 *) src)[i];
        return make_double2(v.x, v.y);
    } else {
        return src[i];
    }
}

// a product slot value at element index i of U: FP64 or FP32 complex
template <class V>
__device__ __forceinline__ void st_slot(cplx *U, size_t i, bool p32, V re, V im)
{
    if (p32)
        ((float2 *) U)[i] = make_float2((float) re, (float) im);
    else
        U[i] = make_double2((double) re, (double) im);
}

// The five adjoint slots at one (kz, y, kx) from the transforms before the
// scale `norm`: Hz = -Tz - i kx Sy, Hx = -Tx + i kz Sy, Hy = -Ty - i kz Sx +
// i kx Sz, then S_x, S_z (channel/pass2.c:474-566).  e: element of slot 0, ss
// the slots' stride.
__device__ __forceinline__ void st_adjoint(cplx *U, size_t e, size_t ss, bool p32, real norm, double kx,
                                           double kz, const real2 *S, const real2 *T)
{
    const real2 Sx = mk2(norm * S[0].x, norm * S[0].y), Sy = mk2(norm * S[1].x, norm * S[1].y);
    const real2 Sz = mk2(norm * S[2].x, norm * S[2].y);
    // k s - norm t and -(norm t) - k s
#ifdef SC_FFT_F32
    auto minus = [&](double k, float s, float t) { return __builtin_fma(k, (double) s, -(double) (norm * t)); };
    auto neg = [&](double k, float s, float t) { return __builtin_fma(-k, (double) s, -(double) (norm * t)); };
#else
    auto minus = [&](double k, double s, double t) { return __builtin_fma(k, s, -(norm * t)); };
    auto neg = [&](double k, double s, double t) { return __builtin_fma(-norm, t, -(k * s)); };
#endif
    st_slot(U, e, p32, minus(kx, Sy.y, T[2].x), neg(kx, Sy.x, T[2].y));
    st_slot(U, e + ss, p32, neg(kz, Sy.y, T[0].x), minus(kz, Sy.x, T[0].y));
    st_slot(U, e + 2 * ss, p32, __builtin_fma(-kx, (double) Sz.y, minus(kz, Sx.y, T[1].x)),
            __builtin_fma(kx, (double) Sz.x, neg(kz, Sx.x, T[1].y)));
    st_slot(U, e + 3 * ss, p32, Sx.x, Sx.y);
    st_slot(U, e + 4 * ss, p32, Sz.x, Sz.y);
}

template <int MODE> struct XmixShape;
template <> struct XmixShape<XM_PRIMAL> { static constexpr int NF = 6, NOUT = 3; };
template <> struct XmixShape<XM_TANGENT> { static constexpr int NF = 12, NOUT = 3; };
template <> struct XmixShape<XM_ADJOINT> { static constexpr int NF = 9, NOUT = 6; };
template <> struct XmixShape<XM_PHYS> { static constexpr int NF = 3, NOUT = 0; };
template <> struct XmixShape<XM_ADJ2> { static constexpr int NF = 15, NOUT = 12; };

// a b - c d, the second product rounded
__device__ __forceinline__ real det(real a, real b, real c, real d) { return fma_(a, b, -(c * d)); }

// The products of one point from its fields f[0 .. NF) (packed pairs in
// order), into out[0 .. NOUT).
template <int MODE>
__device__ __forceinline__ void xmix_products(const real *f, real *out)
{
    const real u = f[0], v = f[1], w = f[2], oz = f[3], ox = f[4], oy = f[5];
    if constexpr (MODE == XM_PRIMAL) {
        out[1] = det(v, oz, w, oy);         // Hx
        out[2] = det(w, ox, u, oz);         // Hy
        out[0] = det(u, oy, v, ox);         // Hz
    } else if constexpr (MODE == XM_TANGENT) {
        const real Iu = f[6], Iv = f[7], Iw = f[8], Ioz = f[9], Iox = f[10], Ioy = f[11];
        out[1] = fma_(-w, Ioy, fma_(v, Ioz, det(Iv, oz, Iw, oy)));
        out[2] = fma_(-u, Ioz, fma_(w, Iox, det(Iw, ox, Iu, oz)));
        out[0] = fma_(-v, Iox, fma_(u, Ioy, det(Iu, oy, Iv, ox)));
    } else if constexpr (MODE == XM_ADJOINT) {
        const real lx = f[6], ly = f[7], lz = f[8];
        out[0] = det(v, lz, w, ly);           // Sx
        out[1] = det(w, lx, u, lz);           // Sy
        out[2] = det(u, ly, v, lx);           // Sz
        out[3] = det(ly, oz, lz, oy);         // Tx
        out[4] = det(lz, ox, lx, oz);         // Ty
        out[5] = det(lx, oy, ly, ox);         // Tz
    } else if constexpr (MODE == XM_ADJ2) {
        // the adjoint products of lambda with two states: (u, omega) in
        // f[0..5] and f[6..11], lambda in f[12..14]
        const real lx = f[12], ly = f[13], lz = f[14];
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const real pu = f[6 * p], pv = f[6 * p + 1], pw = f[6 * p + 2];
            const real qz = f[6 * p + 3], qx = f[6 * p + 4], qy = f[6 * p + 5];
            out[6 * p + 0] = det(pv, lz, pw, ly);     // Sx
            out[6 * p + 1] = det(pw, lx, pu, lz);     // Sy
            out[6 * p + 2] = det(pu, ly, pv, lx);     // Sz
            out[6 * p + 3] = det(ly, qz, lz, qy);     // Tx
            out[6 * p + 4] = det(lz, qx, lx, qz);     // Ty
            out[6 * p + 5] = det(lx, qy, ly, qx);     // Tz
        }
    }
}

// ---------------------------------------------------------------- fixed kernels
// A kernel of fft_x.hip / fft_z.hip for a length, with its launch shape; null
// where the length has none.
typedef void (*XrowKernel)(XmixArgs, const real2 *, real2 *);
typedef void (*ZinvKernel)(ZinvArgs, real2 *);
typedef void (*ZfwdKernel)(ZfwdArgs, const real2 *, cplx *);
typedef void (*ZadjKernel)(ZadjArgs, const real2 *, cplx *);
template <class K> struct Fixed {
    K kernel = nullptr;
    int group = 0;             // rows (x) or columns (z) of a block
    int threads = 0;
    size_t lds = 0;            // bytes
};
template <int MODE> Fixed<XrowKernel> xrow_fixed(int Px, int Pz);
// nm tangent members along one trajectory (fft_x.hip, k_xrow_shared)
Fixed<XrowKernel> xrow_shared_fixed(int Px, int Pz, int nm);
Fixed<ZinvKernel> zinv_fixed(int Pz, int Mx, bool s32);
Fixed<ZfwdKernel> zfwd_fixed(int Pz, int Mx);
Fixed<ZadjKernel> zadj_fixed(int Pz, int Mx);

}  // namespace SC_FFT_NS
}  // namespace sc
