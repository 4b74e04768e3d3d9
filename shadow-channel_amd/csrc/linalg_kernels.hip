// Legendre-Galerkin kernels: y-transforms, banded Helmholtz solves with the
// (kx,kz) = (0,0) mode, and small vector kernels.
//
// y-transforms (channel/initAlphaBeta2.c:96-240 rebuild, channel/project.c:
// 95-115,176-191 and channel/adjproject.c:108-134,213-234 projections) are
// real dense products (qpts x dim or dim x qpts) applied to the complex
// columns of every kz row; they run on the FP64 matrix cores, the complex
// columns split into real and imaginary parts.
//
// Band solves (channel/mvOps.c:29-144, used by channel/project.c,
// increproject.c, adjproject.c): the matrices of the implicit stage are
// time-invariant, so their LU factors (no pivoting, same elimination order as
// the reference) are computed once on the host.  Even and odd rows decouple
// (bands sit on every other diagonal), so one thread solves one parity of
// one (kz, kx, field) system.  Explicit band products are formed on the fly
// from the Gram tables.
#include <type_traits>

#include "sc_internal.h"

namespace sc {

// ------------------------------------------------------------ MFMA helpers
// v_mfma_f64_16x16x4f64: D[16][16] += A[16][4] B[4][16].  Lane l supplies
// A[l%16][l/16] and B[l/16][l%16]; item r of its result holds D[4r + l/16][l%16].
typedef double mf4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ mf4 mfma_f64(double a, double b, mf4 c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The FP32 form for the mixed-precision rebuild, v_mfma_f32_16x16x4f32: the
// same operand layout (A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k),
// but result row i sits in lane group i / 4, item i % 4, where the FP64 form
// puts it in lane group i % 4, item i / 4 (both measured on gfx950).  The
// FP32 instance therefore feeds A row i with the data of row
// 4 (i % 4) + i / 4 (mfma_arow), which leaves every result where the FP64
// instance, and the shared store code, have it.
typedef float ff4 __attribute__((ext_vector_type(4)));
template <class T> __device__ __forceinline__ int mfma_arow(int i)
{
    return sizeof(T) == sizeof(double) ? i : ((i & 3) << 2) | (i >> 2);
}

__device__ __forceinline__ mf4 mfma_t(double a, double b, mf4 c) { return mfma_f64(a, b, c); }
__device__ __forceinline__ ff4 mfma_t(float a, float b, ff4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// accumulator type of the y-transform products in arithmetic type T
template <class T> struct YAcc;
template <> struct YAcc<double> { typedef mf4 type; };
template <> struct YAcc<float> { typedef ff4 type; };
template <class T> __device__ __forceinline__ typename YAcc<T>::type yacc_zero()
{
    typename YAcc<T>::type z = {0, 0, 0, 0};
    return z;
}

// The 16 real columns of an n-tile are eight complex columns; real column n
// is complex column 2(n%4) + n/8, part (n/4)%2.  Item r of lane l then holds
// complex column 2(l/16) + r/2, part r%2: both parts of two neighbouring
// columns sit in one lane.
__device__ __forceinline__ int ncol_x(int n) { return 2 * (n & 3) + (n >> 3); }
__device__ __forceinline__ int ncol_part(int n) { return (n >> 2) & 1; }


// most blocks per XCD of the parity rebuild, split over its half-domain y-tiles:
// two a CU for FP64 (61 KB of basis at 24 k-steps), three for FP32 (32 members at
// 64x97x64: 216 us, 230 with two)
constexpr int RB_BLOCKS = 64, RB_BLOCKS_F32 = 96;

// wave index within the block, in a scalar register: the compiler then
// treats everything derived from it as uniform across the wave
__device__ __forceinline__ int wave_id()
{
    return __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
}

__device__ __forceinline__ mf4 mf4_zero()
{
    mf4 z = {0.0, 0.0, 0.0, 0.0};
    return z;
}

// Wavenumbers formed in registers, bit-identical to the host tables
// (kx = x 2pi/Lx; kz = z 2pi/Lz, z - Nz above Nz/2): no global load, and so
// no wait on the in-order memory counter behind prefetched operands.
__device__ __forceinline__ double wave_kx(int x, double ax) { return x * ax; }
__device__ __forceinline__ double wave_kz(int z, int Nz, double az)
{
    return (z <= Nz / 2 ? z : z - Nz) * az;
}

// ------------------------------------------------------------ rebuild
struct RebuildArgs {
    const double *frag, *Kx, *Kz;
    int Nz, Mx, qpts, dimR, dimQ, nks, nyt, nseg;
    double ax, az;                      // 2 pi / Lx, 2 pi / Lz
    const int *abort_flag;
    unsigned *queue;                    // [8][nyt][2] task and exit counters, zero between launches
    int bpq;                            // blocks per (XCD, y-tile) queue
    int nprob;                          // 2: a second rebuild C1 -> U1 in the same launch
    const cplx *C1;
    cplx *U1;
    // members: problem p = m nprob + sub (sub 1: C1 -> U1) reads C (or C1)
    // + m ms_c and writes U (or U1) + m ms_u; k_rebuild: grid y = member
    int nm;
    size_t ms_c, ms_u;
};

// the coefficient and Gauss-point arrays of problem p (member p / nprob)
__device__ __forceinline__ const cplx *rb_src(const RebuildArgs &a, const cplx *C, int p)
{
    const int m = p / a.nprob;
    return (p - m * a.nprob ? a.C1 : C) + m * a.ms_c;
}
__device__ __forceinline__ cplx *rb_dst(const RebuildArgs &a, cplx *U, int p)
{
    const int m = p / a.nprob;
    return (p - m * a.nprob ? a.U1 : U) + m * a.ms_u;
}

// U[z][0..4][y][x] from C[z][0..1][j][x]; 1-D grid over the (kz row, y-tile)
// tiles, y-tile fastest, XCD-aware (xcd_tile); 256 threads.
// D[n][y] = sum_j C[j][n] B_m[y][j] for the bases m = Q, Qp, Qpp (alpha
// columns) and R, Rp (beta columns); wave w takes the n-tiles w, w+4, ... of
// the block's y-tile.  The basis fragments of a chunk of KC_REBUILD k-steps are
// staged in LDS (double-buffered) and shared by the four waves; the
// coefficient fragments are prefetched one chunk ahead in registers.
// Epilogue: u, w, du/dy, dw/dy from v', v'', omega_y, omega_y'
// (channel/initAlphaBeta2.c:96-240).
// The Nyquist row kz = Nz/2 carries no data, so its blocks rebuild the mean
// column (kx, kz) = (0, 0) instead: u = R alpha, du/dy = Rp alpha,
// w = R beta, dw/dy = Rp beta, v = 0 (channel/initAlphaBeta2.c:22-68), with
// the n rows 0..3 of one tile holding Re/Im alpha, Re/Im beta.
__global__ __launch_bounds__(256, SC_YT_WAVES) void k_rebuild(RebuildArgs a, const cplx *C, cplx *U)
{
    constexpr int KC = KC_REBUILD, CH = KC * 5 * 64, PT = CH / 256;
    static_assert(CH % 256 == 0, "chunk must split over the block");
    __shared__ double bs[2][CH];
    if (*a.abort_flag) return;
    const int tile = xcd_tile(a.nyt * a.Nz);
    if (tile < 0) return;
    C += blockIdx.y * a.ms_c;
    U += blockIdx.y * a.ms_u;
    const int zrow = tile / a.nyt, yt = tile - zrow * a.nyt;
    const bool meanb = zrow == a.Nz / 2;
    const int z = meanb ? 0 : zrow;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int Mx = a.Mx, q = a.qpts, nR = a.dimR, nQ = a.dimQ;
    const int nnt = meanb ? 1 : (Mx + 7) / 8, nch = a.nks / KC;
    const int kq = lane >> 4, nl = lane & 15;
    const double *frag = a.frag + (size_t) yt * a.nks * 5 * 64;
    const double *Cd = (const double *) (C + (size_t) z * 2 * nR * Mx);
    const size_t ss = (size_t) q * Mx;
    cplx *Uz = U + (size_t) z * 5 * ss;
    const double kz = a.Kz[z];
    for (int nt0 = 0; nt0 < nnt; nt0 += 4) {
        const int nt = nt0 + wave;
        const bool active = nt < nnt;
        int xcol, part;
        bool okA, okB;
        size_t offA, offB;
        if (meanb) {
            // n = 0, 1: Re, Im alpha(0,0); n = 2, 3: Re, Im beta(0,0)
            xcol = 0;
            part = nl & 1;
            okA = active && nl < 4;
            okB = false;
            offA = (size_t) (nl >> 1) * nR * Mx * 2 + part;
            offB = 0;
        } else {
            xcol = nt * 8 + ncol_x(nl);
            part = ncol_part(nl);
            okA = okB = active && xcol < Mx;
            offA = (size_t) xcol * 2 + part;
            offB = (size_t) nR * Mx * 2 + offA;
        }
        const int limA = meanb ? nR : nQ;
        mf4 acc[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) acc[m] = mf4_zero();
        // two register sets of coefficient fragments, used alternately
        double ca0[KC], cb0[KC], ca1[KC], cb1[KC], st[PT];
        auto load_coef = [&](int ch, double *ca, double *cb) {
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                const int j = (ch * KC + s) * 4 + kq;
                ca[s] = (okA && j < limA) ? Cd[offA + (size_t) j * Mx * 2] : 0.0;
                cb[s] = (okB && j < nR) ? Cd[offB + (size_t) j * Mx * 2] : 0.0;
            }
        };
        auto load_basis = [&](int ch) {
            const double *src = frag + (size_t) ch * CH;
#pragma unroll
            for (int i = 0; i < PT; ++i) st[i] = src[threadIdx.x + 256 * i];
        };
        auto put_basis = [&](int buf) {
#pragma unroll
            for (int i = 0; i < PT; ++i) bs[buf][threadIdx.x + 256 * i] = st[i];
        };
        auto compute = [&](const double *xa, const double *xb, const double *b) {
            if (active && meanb) {
#pragma unroll
                for (int s = 0; s < KC; ++s) {
                    acc[3] = mfma_f64(xa[s], b[(s * 5 + 3) * 64 + lane], acc[3]);
                    acc[4] = mfma_f64(xa[s], b[(s * 5 + 4) * 64 + lane], acc[4]);
                }
            } else if (active) {
#pragma unroll
                for (int s = 0; s < KC; ++s) {
                    const double b0 = b[(s * 5 + 0) * 64 + lane], b1 = b[(s * 5 + 1) * 64 + lane];
                    const double b2 = b[(s * 5 + 2) * 64 + lane], b3 = b[(s * 5 + 3) * 64 + lane];
                    const double b4 = b[(s * 5 + 4) * 64 + lane];
                    acc[0] = mfma_f64(xa[s], b0, acc[0]);
                    acc[1] = mfma_f64(xa[s], b1, acc[1]);
                    acc[2] = mfma_f64(xa[s], b2, acc[2]);
                    acc[3] = mfma_f64(xb[s], b3, acc[3]);
                    acc[4] = mfma_f64(xb[s], b4, acc[4]);
                }
            }
        };
        load_coef(0, ca0, cb0);
        load_basis(0);
        put_basis(0);
        __syncthreads();
        for (int ch = 0; ch < nch; ch += 2) {
            const bool n1 = ch + 1 < nch;
            if (n1) {
                load_coef(ch + 1, ca1, cb1);
                load_basis(ch + 1);
            }
            compute(ca0, cb0, bs[0]);
            if (n1) put_basis(1);
            __syncthreads();
            if (!n1) break;
            const bool n2 = ch + 2 < nch;
            if (n2) {
                load_coef(ch + 2, ca0, cb0);
                load_basis(ch + 2);
            }
            compute(ca1, cb1, bs[1]);
            if (n2) put_basis(0);
            __syncthreads();
        }
        const int y = yt * 16 + nl;
        if (!active || y >= q) continue;
        if (meanb) {
            // item 0 of lane group kq holds n = kq: u (kq < 2) or w (kq >= 2)
            double *Ur = (double *) (Uz + (size_t) y * Mx) + (kq & 1);
            const int su = kq < 2 ? 0 : 2;
            Ur[(size_t) su * ss * 2] = acc[3][0];
            Ur[(size_t) (su == 0 ? 3 : 4) * ss * 2] = acc[4][0];
            Ur[(size_t) 1 * ss * 2] = 0.0;
            continue;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int x = nt * 8 + 2 * kq + h;
            if (x >= Mx || (z == 0 && x == 0)) continue;
            const size_t o = (size_t) y * Mx + x;
            const double kx = a.Kx[x], k2 = kz * kz + kx * kx;
            const double2 v = make_double2(acc[0][2 * h], acc[0][2 * h + 1]);
            const double2 f = make_double2(-acc[1][2 * h], -acc[1][2 * h + 1]);
            const double2 q2 = make_double2(acc[2][2 * h], acc[2][2 * h + 1]);
            const double2 g = make_double2(acc[3][2 * h], acc[3][2 * h + 1]);
            const double2 gp = make_double2(acc[4][2 * h], acc[4][2 * h + 1]);
            Uz[o + 1 * ss] = v;
            Uz[o + 0 * ss] = make_double2((kx * f.y + kz * g.y) / k2, -(kx * f.x + kz * g.x) / k2);
            Uz[o + 2 * ss] = make_double2((-kx * g.y + kz * f.y) / k2, (kx * g.x - kz * f.x) / k2);
            Uz[o + 3 * ss] = make_double2((-kx * q2.y + kz * gp.y) / k2, (kx * q2.x - kz * gp.x) / k2);
            Uz[o + 4 * ss] = make_double2(-(kx * gp.y + kz * q2.y) / k2, (kx * gp.x + kz * q2.x) / k2);
        }
    }
}

// Operands of one (kz row, n-tile) task of the rebuild: lane offsets into C
// of its alpha and beta fragments.  Every lane loads (the loads carry no
// predicate, so nothing waits on them before use): columns past Mx read the
// last column and are never stored, rows past the basis meet zero basis
// fragments, and in the mean row only the n rows 0..3 are stored.
struct RebuildTask {
    size_t offA, offB;
    const double *cd;                   // coefficient array of the task's rebuild
};

__device__ __forceinline__ RebuildTask rebuild_task(const RebuildArgs &a, int zrow, int nt, int nl)
{
    RebuildTask t;
    const int Mx = a.Mx, nR = a.dimR;
    if (zrow == a.Nz / 2) {
        // n = 0, 1: Re, Im alpha(0,0); n = 2, 3: Re, Im beta(0,0)
        t.offA = (size_t) ((nl >> 1) & 1) * nR * Mx * 2 + (nl & 1);
        t.offB = t.offA;
    } else {
        const int xcol = min(nt * 8 + ncol_x(nl), Mx - 1);
        t.offA = (size_t) zrow * 2 * nR * Mx * 2 + (size_t) xcol * 2 + ncol_part(nl);
        t.offB = t.offA + (size_t) nR * Mx * 2;
    }
    return t;
}

// Gauss-point values of one task from its five accumulators (D[n][y] layout)
// VEL: the velocity slots u, v, w only (acc[2], acc[4] unused).  The slots
// are stored as O: double2, or float2 for the FP32 instance (the mixed-
// precision steps, whose z-inverse transform reads FP32 slots at the same
// element index; the member base address stays that of the FP64 layout).
// DIV: divisions by kx^2 + kz^2 as k_rebuild's, not products with its inverse.
template <bool VEL = false, class ACC = mf4, class O = double2, bool DIV = false>
__device__ __forceinline__ void rebuild_store(const RebuildArgs &a, int zrow, int nt, int y, int kq,
                                              const ACC *acc, cplx *U)
{
    typedef decltype(O().x) S;
    const int Mx = a.Mx, q = a.qpts;
    if (y >= q) return;
    const size_t ss = (size_t) q * Mx;
    O *Uo = (O *) U;
    if (zrow == a.Nz / 2) {
        // mean column: item 0 of lane group kq holds n = kq, Re/Im of
        // alpha (kq < 2: u, du/dy) or beta (kq >= 2: w, dw/dy)
        S *Ur = (S *) (Uo + (size_t) y * Mx) + (kq & 1);
        const int su = kq < 2 ? 0 : 2;
        Ur[(size_t) su * ss * 2] = (S) acc[3][0];
        if (!VEL) Ur[(size_t) (su == 0 ? 3 : 4) * ss * 2] = (S) acc[4][0];
        Ur[(size_t) 1 * ss * 2] = (S) 0;
        return;
    }
    O *Uz = Uo + (size_t) zrow * 5 * ss;
    const double kz = wave_kz(zrow, a.Nz, a.az);
    O v[2][5];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        auto put = [&](int s, double re, double im) { v[h][s] = O{(S) re, (S) im}; };
        // one reciprocal per column instead of eight divisions
        const double kx = wave_kx(nt * 8 + 2 * kq + h, a.ax), k2 = kz * kz + kx * kx, r2 = 1.0 / k2;
        auto over = [&](double w) { return DIV ? w / k2 : w * r2; };
        const double2 f = make_double2(-acc[1][2 * h], -acc[1][2 * h + 1]);
        const double2 g = make_double2(acc[3][2 * h], acc[3][2 * h + 1]);
        put(0, over(kx * f.y + kz * g.y), -over(kx * f.x + kz * g.x));
        put(1, acc[0][2 * h], acc[0][2 * h + 1]);
        put(2, over(-kx * g.y + kz * f.y), over(kx * g.x - kz * f.x));
        if (VEL) continue;
        const double2 q2 = make_double2(acc[2][2 * h], acc[2][2 * h + 1]);
        const double2 gp = make_double2(acc[4][2 * h], acc[4][2 * h + 1]);
        put(3, over(-kx * q2.y + kz * gp.y), over(kx * q2.x - kz * gp.x));
        put(4, -over(kx * gp.y + kz * q2.y), over(kx * gp.x + kz * q2.x));
    }
    // the lane's columns x0 and x0 + 1; (0, 0) is the mean task's
    const int x0 = nt * 8 + 2 * kq;
    const bool in0 = x0 < Mx && !(zrow == 0 && x0 == 0), in1 = x0 + 1 < Mx;
    O *Ux = Uz + (size_t) y * Mx + x0;
    // FP32: both columns in one 16-byte store where a row of slots is a whole
    // number of them (Mx even: x0, y Mx and a slot's elements all are)
    typedef S s4 __attribute__((ext_vector_type(4)));
    const bool both = sizeof(S) == sizeof(float) && Mx % 2 == 0 && in0;
#pragma unroll
    for (int s = 0; s < (VEL ? 3 : 5); ++s) {
        if (both) {
            *(s4 *) (Ux + s * ss) = s4{v[0][s].x, v[0][s].y, v[1][s].x, v[1][s].y};
        } else {
            if (in0) Ux[s * ss] = v[0][s];
            if (in1) Ux[s * ss + 1] = v[1][s];
        }
    }
}

// Rebuild for dimR <= 4*NKS with dynamic task queues: a block owns one
// y-tile and stages its whole basis (NKS k-steps) in LDS once; its waves then
// take (kz row, n-tile) tasks (load the 2 NKS coefficient fragments, 5 NKS
// products, store) from the queue of their (XCD, y-tile) until it is empty,
// so the products spread evenly over the SIMDs.  Blocks are dispatched
// round-robin over the 8 XCDs (block b on XCD b % 8), and the queue of XCD x
// holds the kz rows [x Nz/8, (x+1) Nz/8): the coefficient rows of an XCD's
// tasks stay in its L2.  A queue is a task counter and an exit counter; the
// last wave of the queue to exit clears both, so they are zero between
// launches.  Two blocks share a CU.  Grid: 8 * nyt * bpq blocks.
template <int NKS>
__global__ __launch_bounds__(256, 2) void k_rebuild_rows(RebuildArgs a, const cplx *C, cplx *U)
{
    __shared__ double bs[NKS * 5 * 64];
    if (*a.abort_flag) return;
    const int xcd = blockIdx.x & 7, ib = blockIdx.x >> 3;
    const int yt = ib % a.nyt;
    const int z0 = xcd * a.Nz / 8, z1 = (xcd + 1) * a.Nz / 8;
    unsigned *qc = a.queue + ((size_t) xcd * a.nyt + yt) * 2;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int kq = lane >> 4, nl = lane & 15;
    const int nnt = (a.Mx + 7) / 8, nR = a.dimR;
    const double *frag = a.frag + (size_t) yt * NKS * 5 * 64;
    {
        // all loads in flight before the first LDS store
        constexpr int PT = NKS * 5 * 64 / 256;
        static_assert(NKS * 5 * 64 % 256 == 0, "basis must split over the block");
        double st[PT];
#pragma unroll
        for (int i = 0; i < PT; ++i) st[i] = frag[threadIdx.x + 256 * i];
#pragma unroll
        for (int i = 0; i < PT; ++i) bs[threadIdx.x + 256 * i] = st[i];
    }
    // task t of the queue: rows z0..z1-1 in order, nnt n-tiles each (one in
    // the mean row); tasks p ntask1 .. belong to problem p (rb_src)
    const int zm = a.Nz / 2;
    const bool has_mean = zm >= z0 && zm < z1;
    const int ntask1 = (z1 - z0) * nnt - (has_mean ? nnt - 1 : 0);
    const int ntask = ntask1 * a.nprob * a.nm;
    auto task_of = [&](int t, int &zrow, int &nt) {
        t -= (t / ntask1) * ntask1;
        const int tm = has_mean ? (zm - z0) * nnt : ntask1;  // first task of the mean row
        if (t < tm) {
            zrow = z0 + t / nnt;
            nt = t % nnt;
        } else if (t == tm) {
            zrow = zm;
            nt = 0;
        } else {
            const int u = t - tm - 1;
            zrow = zm + 1 + u / nnt;
            nt = u % nnt;
        }
    };
    auto grab = [&]() {
        unsigned t0 = 0;
        if (lane == 0) t0 = atomicAdd(&qc[0], 1u);
        return __builtin_amdgcn_readfirstlane((int) t0);
    };
    // The coefficient fragments of a task move in two halves, one register
    // buffer each: the loads of the second half are issued before the
    // products of the first, those of the next task's first half before the
    // products of the second.
    constexpr int CK = NKS / 2, NCH = 2;
    static_assert(CK % 4 == 0, "a half must be whole groups of four k-steps");
    double ca[NCH][CK], cb[NCH][CK];
    // row j = 4 s + kq of k-step s: a lane base (row kq) plus a uniform step;
    // only the last k-step can pass row dimR - 1 (4 (NKS-1) < dimR), so only
    // it is clamped
    const size_t rstep = (size_t) 4 * a.Mx * 2;
    auto load = [&](const RebuildTask &t, int ch) {
        const double *Cd = t.cd;
        const double *pa = Cd + t.offA + (size_t) kq * a.Mx * 2;
        const double *pb = Cd + t.offB + (size_t) kq * a.Mx * 2;
#pragma unroll
        for (int s = 0; s < CK; ++s) {
            const int ks = ch * CK + s;
            if (ks == NKS - 1) {
                const size_t j = min(ks * 4 + kq, nR - 1);
                ca[ch][s] = Cd[t.offA + j * a.Mx * 2];
                cb[ch][s] = Cd[t.offB + j * a.Mx * 2];
            } else {
                ca[ch][s] = pa[ks * rstep];
                cb[ch][s] = pb[ks * rstep];
            }
        }
    };
    // products of chunk ch (basis fragments LDS -> registers two k-steps at a
    // time, one group ahead; the scheduling barriers keep the compiler from
    // sinking those loads to their uses)
    auto chunk = [&](bool mean, int ch, mf4 *acc) {
        const double *xa = ca[ch], *xb = cb[ch];
        if (mean) {
#pragma unroll
            for (int t = 0; t < CK; ++t) {
                const int s = ch * CK + t;
                acc[3] = mfma_f64(xa[t], bs[(s * 5 + 3) * 64 + lane], acc[3]);
                acc[4] = mfma_f64(xa[t], bs[(s * 5 + 4) * 64 + lane], acc[4]);
            }
            return;
        }
        double p0[10], p1[10];
        auto ldb = [&](int s0, double *p) {
#pragma unroll
            for (int e = 0; e < 10; ++e) p[e] = bs[(s0 * 5 + e) * 64 + lane];
        };
        auto mm = [&](int t0, const double *p) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = t0 + u;
                acc[0] = mfma_f64(xa[t], p[u * 5 + 0], acc[0]);
                acc[1] = mfma_f64(xa[t], p[u * 5 + 1], acc[1]);
                acc[2] = mfma_f64(xa[t], p[u * 5 + 2], acc[2]);
                acc[3] = mfma_f64(xb[t], p[u * 5 + 3], acc[3]);
                acc[4] = mfma_f64(xb[t], p[u * 5 + 4], acc[4]);
            }
        };
        const int sb = ch * CK;
        ldb(sb, p0);
#pragma unroll
        for (int t0 = 0; t0 < CK; t0 += 4) {
            if (t0 + 2 < CK) ldb(sb + t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0, p0);
            __builtin_amdgcn_sched_barrier(0);
            if (t0 + 2 >= CK) break;
            if (t0 + 4 < CK) ldb(sb + t0 + 4, p0);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    __syncthreads();
    (void) wave;
    // operands of task t: offsets and the coefficient array of its rebuild
    auto task_ops = [&](int t, int zr, int nt) {
        RebuildTask r = rebuild_task(a, zr, nt, nl);
        r.cd = (const double *) rb_src(a, C, t / ntask1);
        return r;
    };
    int t = grab();
    if (t >= ntask) {
        t = ntask;
    } else {
        int zr, nt;
        task_of(t, zr, nt);
        load(task_ops(t, zr, nt), 0);
    }
    while (t < ntask) {
        int zr, nt;
        task_of(t, zr, nt);
        const RebuildTask cur = task_ops(t, zr, nt);
        const bool mean = zr == zm;
        mf4 acc[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) acc[m] = mf4_zero();
        int tn = ntask;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            if (ch + 1 < NCH) {
                load(cur, ch + 1);
            } else {
                tn = grab();
                if (tn < ntask) {
                    int zn, ntn;
                    task_of(tn, zn, ntn);
                    load(task_ops(tn, zn, ntn), 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            chunk(mean, ch, acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        rebuild_store(a, zr, nt, yt * 16 + nl, kq, acc, rb_dst(a, U, t / ntask1));
        t = tn;
    }
    // every wave of the queue's blocks exits here once; the last clears it
    if (lane == 0) {
        const unsigned done = atomicAdd(&qc[1], 1u);
        if (done == (unsigned) (a.bpq * 4 - 1)) {
            atomicExch(&qc[0], 0u);
            atomicExch(&qc[1], 0u);
        }
    }
}

// k_rebuild for dimR <= 4 NKS (NKS = 32: dimR 97 to 128), the whole basis of a
// y-tile in LDS: the same products in the same order, so the same bits.  The
// tasks of an XCD's kz rows, eight waves' at a time, are numbered y-tile by
// y-tile and split evenly over its blocks, one a CU; a block stages the basis
// of its first y-tile and, once or twice, of the next.  A wave's coefficients
// move in four quarters through two register buffers, the next quarter's loads
// (or the next task's first) issued before the current quarter's products.
// Bound by the FP64 products (113 us for two members at 128x129x128); the form
// that stages the basis chunk by chunk behind a barrier, for four waves that
// start and end every n-tile together, took 262 us, this one 187: the products take
// 61% of its clocks and the divisions and other vector instructions, which share
// their unit, 12%; the rest is the change of basis and re-reading coefficients.
constexpr int RW_THREADS = 512;
template <int NKS>
__global__ __launch_bounds__(RW_THREADS) void k_rebuild_wide(RebuildArgs a, const cplx *C, cplx *U)
{
    constexpr int CK = NKS / 4, NW = RW_THREADS / 64;
    static_assert(CK % 4 == 0, "a quarter is whole groups of four k-steps");
    __shared__ double bs[NKS * 5 * 64];
    if (*a.abort_flag) return;
    const int xcd = blockIdx.x & 7, ib = blockIdx.x >> 3;
    const int z0 = xcd * a.Nz / 8, z1 = (xcd + 1) * a.Nz / 8;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int kq = lane >> 4, nl = lane & 15;
    const int nnt = (a.Mx + 7) / 8, nR = a.dimR, M2 = a.Mx * 2;
    const int zm = a.Nz / 2;
    const bool has_mean = zm >= z0 && zm < z1;
    const int ntask1 = (z1 - z0) * nnt - (has_mean ? nnt - 1 : 0);
    const int ntask = ntask1 * a.nprob * a.nm;
    // groups of NW tasks: ng a y-tile, this block's g0 .. g1 - 1 of all
    const int ng = (ntask + NW - 1) / NW;
    const int g0 = (int) ((long long) ib * a.nyt * ng / a.bpq), g1 = (int) ((long long) (ib + 1) * a.nyt * ng / a.bpq);
    auto task_of = [&](int t, int &zrow, int &nt) {
        t -= (t / ntask1) * ntask1;
        const int tm = has_mean ? (zm - z0) * nnt : ntask1;
        const int u = t <= tm ? t : t - tm - 1;
        zrow = t == tm ? zm : (t < tm ? z0 : zm + 1) + u / nnt;
        nt = t == tm ? 0 : u % nnt;
    };
    auto task_ops = [&](int t) {
        int zr, nt;
        task_of(t, zr, nt);
        RebuildTask r = rebuild_task(a, zr, nt, nl);
        r.cd = (const double *) rb_src(a, C, t / ntask1);
        return r;
    };
    double ca[2][CK], cb[2][CK];
    // quarter ch of a task's coefficients as buffer loads over the whole array.
    // Rows past the matrix read as zero (an offset past the array), as whatever
    // else lies there may not be finite: the alpha rows dimQ and dimQ + 1, which
    // carry nothing, and the rows after a column's last.  Only the k-steps from
    // RP on can hold one (dimQ >= 95 at 32 k-steps).
    const unsigned cbytes = (unsigned) ((size_t) a.Nz * 2 * nR * M2 * sizeof(double));
    constexpr int RP = NKS - 9, PAST = 0x7ffffff8;
    auto load = [&](const RebuildTask &t, int ch) {
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *) t.cd, 0, cbytes, 0x00020000);
        const int va = (int) (unsigned) ((t.offA + kq * M2) * 8), vb = (int) (unsigned) ((t.offB + kq * M2) * 8);
        // (the mean task's fragments are both R rows)
        const int limA = t.offA == t.offB ? nR : a.dimQ;
#pragma unroll
        for (int s = 0; s < CK; ++s) {
            const int ks = ch * CK + s, so = ks * 4 * M2 * 8, j = ks * 4 + kq;
            const int oa = ks >= RP && j >= limA ? PAST : va, ob = ks >= RP && j >= nR ? PAST : vb;
            ca[ch & 1][s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, oa, so, 0));
            cb[ch & 1][s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, ob, so, 0));
        }
    };
    auto chunk = [&](int ch, mf4 *acc) {
        const double *xa = ca[ch & 1], *xb = cb[ch & 1];
        double p0[10], p1[10];
        auto ldb = [&](int s0, double *p) {
#pragma unroll
            for (int e = 0; e < 10; ++e) p[e] = bs[(s0 * 5 + e) * 64 + lane];
        };
        auto mm = [&](int t0, const double *p) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                acc[0] = mfma_f64(xa[t0 + u], p[u * 5 + 0], acc[0]);
                acc[1] = mfma_f64(xa[t0 + u], p[u * 5 + 1], acc[1]);
                acc[2] = mfma_f64(xa[t0 + u], p[u * 5 + 2], acc[2]);
                acc[3] = mfma_f64(xb[t0 + u], p[u * 5 + 3], acc[3]);
                acc[4] = mfma_f64(xb[t0 + u], p[u * 5 + 4], acc[4]);
            }
        };
        const int sb = ch * CK;
        ldb(sb, p0);
#pragma unroll
        for (int t0 = 0; t0 < CK; t0 += 4) {
            ldb(sb + t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0, p0);
            __builtin_amdgcn_sched_barrier(0);
            if (t0 + 4 < CK) ldb(sb + t0 + 4, p0);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int gs = g0; gs < g1;) {
        const int yt = gs / ng, ge = min(g1, (yt + 1) * ng);
        int t = (gs - yt * ng) * NW + wave;
        const int te = min(ntask, (ge - yt * ng) * NW);
        if (t < te) load(task_ops(t), 0);
        if (gs > g0) __syncthreads();                          // the last y-tile's products
        {
            const double *frag = a.frag + (size_t) yt * NKS * 5 * 64;
            constexpr int PT = NKS * 5 * 64 / RW_THREADS;
            static_assert(NKS * 5 * 64 % RW_THREADS == 0, "basis must split over the block");
            double st[PT];
#pragma unroll
            for (int i = 0; i < PT; ++i) st[i] = frag[threadIdx.x + RW_THREADS * i];
#pragma unroll
            for (int i = 0; i < PT; ++i) bs[threadIdx.x + RW_THREADS * i] = st[i];
        }
        __syncthreads();
        for (; t < te; t += NW) {
            const RebuildTask cur = task_ops(t);
            mf4 acc[5];
#pragma unroll
            for (int m = 0; m < 5; ++m) acc[m] = mf4_zero();
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                if (ch < 3)
                    load(cur, ch + 1);
                else if (t + NW < te)
                    load(task_ops(t + NW), 0);
                __builtin_amdgcn_sched_barrier(0);
                // (the mean task's alpha and beta fragments are one load's, and
                // its first three sums are not used)
                chunk(ch, acc);
                __builtin_amdgcn_sched_barrier(0);
            }
            int zr, nt;
            task_of(t, zr, nt);
            rebuild_store<false, mf4, double2, true>(a, zr, nt, yt * 16 + nl, kq, acc, rb_dst(a, U, t / ntask1));
        }
        gs = ge;
    }
}

// Parity form of the queued rebuild.  The Gauss points are mirror images
// (y[q-1-i] = -y[i], exactly) and every basis column has a parity, exactly:
// Q_j, Qpp_j and R_j that of j, Qp_j and Rp_j the opposite.  With E and O
// the sums over the even and the odd j at a point y_i of the half domain
// i < (q+1)/2,
//     U(y_i) = E + O,    U(y_{q-1-i}) = s (E - O),
// s = +1 for Q, Qpp, R and -1 for Qp, Rp.  A task covers 16 half-domain
// points and their mirrors with the 5 NKS products that the direct form
// spends on 16 points, so the products halve.  For odd q the middle point is
// y = 0, where the columns of the other parity vanish exactly and E + O is
// stored once.  k-step s < NKS/2 holds the even rows j = 8s + 2(l/16), the
// others the odd rows; the coefficients move in four quarters (even rows,
// then odd rows, two halves each) through two register buffers, the next
// quarter's loads issued before the current quarter's products.  Blocks and
// the mean task as in k_rebuild_rows (a.nyt is the number of half-domain
// y-tiles, a.frag the parity-ordered basis), but the tasks are assigned
// statically: wave w of the bpq blocks of an (XCD, y-tile) takes the tasks
// w, w + 4 bpq, ..., and issues its first coefficient loads before it
// stages the basis.
template <int NKS, bool VEL, class T>
__global__ __launch_bounds__(256, sizeof(T) == sizeof(float) ? 3 : 2) void k_rebuild_par(RebuildArgs a, const cplx *C, cplx *U)
{
    using ACC = typename YAcc<T>::type;
    __shared__ T bs[NKS * 5 * 64];
    if (*a.abort_flag) return;
    const int xcd = blockIdx.x & 7, ib = blockIdx.x >> 3;
    const int yt = ib % a.nyt;
    const int z0 = xcd * a.Nz / 8, z1 = (xcd + 1) * a.Nz / 8;
    const int lane = threadIdx.x & 63;
    const int kq = lane >> 4, nl = lane & 15;
    const int nnt = (a.Mx + 7) / 8, nR = a.dimR, M2 = a.Mx * 2;
    const int tstep = 4 * a.bpq;
    const int zm = a.Nz / 2;
    const bool has_mean = zm >= z0 && zm < z1;
    const int ntask1 = (z1 - z0) * nnt - (has_mean ? nnt - 1 : 0);
    const int ntask = ntask1 * a.nprob * a.nm;
    auto task_of = [&](int t, int &zrow, int &nt) {
        t -= (t / ntask1) * ntask1;
        const int tm = has_mean ? (zm - z0) * nnt : ntask1;
        if (t < tm) {
            zrow = z0 + t / nnt;
            nt = t % nnt;
        } else if (t == tm) {
            zrow = zm;
            nt = 0;
        } else {
            const int u = t - tm - 1;
            zrow = zm + 1 + u / nnt;
            nt = u % nnt;
        }
    };
    constexpr int NKH = NKS / 2, CK = NKS / 4;
    static_assert(CK % 2 == 0, "a quarter must be whole pairs of k-steps");
    double ca[2][CK], cb[2][CK];
    // quarter ch: parity ch / 2, k-steps (ch % 2) CK .. + CK - 1 of that
    // parity, as buffer loads over the whole coefficient array: a lane
    // offset plus a uniform k-step offset.  Rows past dimR - 1 (whose basis
    // fragments are zero) read the next rows of the array, or zero past its
    // end, so no row index is clamped.
    const unsigned cbytes = (unsigned) ((size_t) a.Nz * 2 * nR * M2 * sizeof(double));
    auto load = [&](const RebuildTask &t, int ch, int buf) {
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *) t.cd, 0, cbytes, 0x00020000);
        const int par = ch >> 1, s0 = (ch & 1) * CK;
        const int row = (2 * kq + par) * M2;
        const int va = (int) (unsigned) ((t.offA + row) * 8), vb = (int) (unsigned) ((t.offB + row) * 8);
#pragma unroll
        for (int s = 0; s < CK; ++s) {
            const int so = (s0 + s) * 8 * M2 * 8;
            ca[buf][s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, va, so, 0));
            cb[buf][s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, vb, so, 0));
        }
    };
    auto chunk = [&](bool mean, int ch, int buf, ACC *acc) {
        const double *xa = ca[buf], *xb = cb[buf];
        const int sb = (ch >> 1) * NKH + (ch & 1) * CK;
        if (mean) {
#pragma unroll
            for (int t = 0; t < CK; ++t) {
                acc[3] = mfma_t((T) xa[t], bs[((sb + t) * 5 + 3) * 64 + lane], acc[3]);
                if (!VEL) acc[4] = mfma_t((T) xa[t], bs[((sb + t) * 5 + 4) * 64 + lane], acc[4]);
            }
            return;
        }
        T p0[10], p1[10];
        auto ldb = [&](int s0, T *p) {
#pragma unroll
            for (int e = 0; e < 10; ++e)
                if (!VEL || (e % 5 != 2 && e % 5 != 4)) p[e] = bs[(s0 * 5 + e) * 64 + lane];
        };
        auto mm = [&](int t0, const T *p) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = t0 + u;
                acc[0] = mfma_t((T) xa[t], p[u * 5 + 0], acc[0]);
                acc[1] = mfma_t((T) xa[t], p[u * 5 + 1], acc[1]);
                if (!VEL) acc[2] = mfma_t((T) xa[t], p[u * 5 + 2], acc[2]);
                acc[3] = mfma_t((T) xb[t], p[u * 5 + 3], acc[3]);
                if (!VEL) acc[4] = mfma_t((T) xb[t], p[u * 5 + 4], acc[4]);
            }
        };
        ldb(sb, p0);
#pragma unroll
        for (int t0 = 0; t0 < CK; t0 += 4) {
            if (t0 + 2 < CK) ldb(sb + t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0, p0);
            __builtin_amdgcn_sched_barrier(0);
            if (t0 + 2 >= CK) break;
            if (t0 + 4 < CK) ldb(sb + t0 + 4, p0);
            __builtin_amdgcn_sched_barrier(0);
            mm(t0 + 2, p1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto task_ops = [&](int t, int zr, int nt) {
        RebuildTask r = rebuild_task(a, zr, nt, mfma_arow<T>(nl));
        r.cd = (const double *) rb_src(a, C, t / ntask1);
        return r;
    };
    const int hq = (a.qpts + 1) / 2;
    const int y = yt * 16 + nl, ym = a.qpts - 1 - y;
    int t = (ib / a.nyt) * 4 + wave_id();
    if (t < ntask) {
        int zr, nt;
        task_of(t, zr, nt);
        load(task_ops(t, zr, nt), 0, 0);
    }
    {
        const double *frag = a.frag + (size_t) yt * NKS * 5 * 64;
        constexpr int PT = NKS * 5 * 64 / 256;
        static_assert(NKS * 5 * 64 % 256 == 0, "basis must split over the block");
        double st[PT];
#pragma unroll
        for (int i = 0; i < PT; ++i) st[i] = frag[threadIdx.x + 256 * i];   // converted when stored
#pragma unroll
        for (int i = 0; i < PT; ++i) bs[threadIdx.x + 256 * i] = (T) st[i];
    }
    __syncthreads();
    while (t < ntask) {
        int zr, nt;
        task_of(t, zr, nt);
        const RebuildTask cur = task_ops(t, zr, nt);
        const bool mean = zr == zm;
        ACC ae[5], ao[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            ae[m] = yacc_zero<T>();
            ao[m] = yacc_zero<T>();
        }
        int tn = ntask;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
            if (ch < 3) {
                load(cur, ch + 1, (ch + 1) & 1);
            } else {
                tn = t + tstep;
                if (tn < ntask) {
                    int zn, ntn;
                    task_of(tn, zn, ntn);
                    load(task_ops(tn, zn, ntn), 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            chunk(mean, ch, ch & 1, ch < 2 ? ae : ao);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (y < hq) {
            cplx *Ud = rb_dst(a, U, t / ntask1);
            // values at y (E + O), then at the mirror point (s (E - O))
#pragma unroll
            for (int m = 0; m < 5; ++m) {
                const ACC e = ae[m], o = ao[m];
                ae[m] = e + o;
                ao[m] = (m == 1 || m == 4) ? o - e : e - o;
            }
            // FP32 products: FP32 slots
            typedef typename std::conditional<sizeof(T) == sizeof(float), float2, double2>::type O;
            rebuild_store<VEL, ACC, O>(a, zr, nt, y, kq, ae, Ud);
            if (ym != y) rebuild_store<VEL, ACC, O>(a, zr, nt, ym, kq, ao, Ud);
        }
        t = tn;
    }
}

// one or two rebuilds (C1 null: one); the queued kernel runs both in one
// launch (they share the staged basis), the chunked kernel one launch each
void launch_rebuild2(Context &c, const cplx *C0, cplx *U0, const cplx *C1, cplx *U1, bool vel_only)
{
    const Dims &d = c.d;
    // segments of kz rows for the chunked kernel
    const int nseg = std::max(1, std::min(d.Nz, 512 / c.nyt));
    // queued form: blocks per (XCD, y-tile), about two blocks per CU
    const int bpq = std::max(1, 64 / c.nyt);
    int nprob = C1 ? 2 : 1;
    const int nm = c.nrun;
    const size_t ms_c = mstride(c, C0), ms_u = mstride(c, U0);
    if (C1 && (mstride(c, C1) != ms_c || mstride(c, U1) != ms_u)) {
        // the two problems' arrays have other member strides: two launches
        launch_rebuild2(c, C0, U0, nullptr, nullptr, vel_only);
        launch_rebuild2(c, C1, U1, nullptr, nullptr, vel_only);
        return;
    }
    RebuildArgs a{c.dFragR, c.dKx, c.dKz, d.Nz, d.Mx, d.qpts, d.dimR, d.dimQ, c.nksR, c.nyt,
                  nseg, 2. * M_PI / d.Lx, 2. * M_PI / d.Lz, c.abort_flag, c.rb_queue, bpq,
                  nprob, C1, U1, nm, ms_c, ms_u};
    const double slot_bytes = slots32(c) ? 8.0 : 16.0;
    double bytes = nm * nprob * (double) (d.Nz - 1) * d.Mx *
                   (16.0 * 2.0 * d.dimR + slot_bytes * (vel_only ? 3.0 : 5.0) * d.qpts);
    const hipStream_t st = c.stream;
    const int nks = c.nksR;
    const dim3 grows(8 * c.nyt * bpq), gchunk(xcd_grid(c.nyt * d.Nz), nm);
    const int nksp = c.nksP;
    const bool par = c.ypar && (nksp == 8 || nksp == 16 || nksp == 24);
    // mixed precision: the parity rebuild's products on the FP32 matrix cores
    // and FP32 slots, except for outputs such as spec2phys
    const bool f32 = slots32(c);
    RebuildArgs ap = a;
    ap.frag = c.dFragP;
    ap.nyt = c.nht;
    ap.nks = nksp;
    {
        // enough waves for one task each (of one rebuild of all members), at
        // most about two (FP32: three) blocks per CU
        const int ntmax = nm * ((d.Nz + 7) / 8 * ((d.Mx + 7) / 8));
        const int rbb = tuning().rebuild_blocks > 0 ? tuning().rebuild_blocks : f32 ? RB_BLOCKS_F32 : RB_BLOCKS;
        ap.bpq = std::max(1, std::min((ntmax + 3) / 4, rbb / c.nht));
    }
    const dim3 gpar(8 * c.nht * ap.bpq);
    // whole basis of a y-tile in LDS (80 KB at 32 k-steps): a block a CU, never
    // more than there are tasks for its first wave
    RebuildArgs aw = a;
    aw.bpq = std::max(1, std::min(32, c.nyt * (nm * nprob * ((d.Nz + 7) / 8) * ((d.Mx + 7) / 8) + 7) / 8));
    const dim3 gwide(8 * aw.bpq);
    typedef void (*RebuildKernel)(RebuildArgs, const cplx *, cplx *);
#define SC_RB_PAR(N, V) (f32 ? (RebuildKernel) k_rebuild_par<N, V, float> : (RebuildKernel) k_rebuild_par<N, V, double>)
    auto go = [=]() {
        if (par && vel_only) {
            if (nksp == 8)
                hipLaunchKernelGGL(SC_RB_PAR(8, true), gpar, dim3(256), 0, st, ap, C0, U0);
            else if (nksp == 16)
                hipLaunchKernelGGL(SC_RB_PAR(16, true), gpar, dim3(256), 0, st, ap, C0, U0);
            else
                hipLaunchKernelGGL(SC_RB_PAR(24, true), gpar, dim3(256), 0, st, ap, C0, U0);
        } else if (par) {
            if (nksp == 8)
                hipLaunchKernelGGL(SC_RB_PAR(8, false), gpar, dim3(256), 0, st, ap, C0, U0);
            else if (nksp == 16)
                hipLaunchKernelGGL(SC_RB_PAR(16, false), gpar, dim3(256), 0, st, ap, C0, U0);
            else
                hipLaunchKernelGGL(SC_RB_PAR(24, false), gpar, dim3(256), 0, st, ap, C0, U0);
        } else if (nks == 8)
            hipLaunchKernelGGL(k_rebuild_rows<8>, grows, dim3(256), 0, st, a, C0, U0);
        else if (nks == 16)
            hipLaunchKernelGGL(k_rebuild_rows<16>, grows, dim3(256), 0, st, a, C0, U0);
        else if (nks == 24)
            hipLaunchKernelGGL(k_rebuild_rows<24>, grows, dim3(256), 0, st, a, C0, U0);
        else if (nks == 32)
            hipLaunchKernelGGL(k_rebuild_wide<32>, gwide, dim3(RW_THREADS), 0, st, aw, C0, U0);
        else
            for (int p = 0; p < nprob; ++p)
                hipLaunchKernelGGL(k_rebuild, gchunk, dim3(256), 0, st, a, p ? C1 : C0, p ? U1 : U0);
    };
    prof_begin(c, st, 4, bytes);
    go();
    prof_end(c, st, 4, go);
}
#undef SC_RB_PAR

void launch_rebuild(Context &c, const cplx *Csrc, cplx *Udst, bool vel_only)
{
    launch_rebuild2(c, Csrc, Udst, nullptr, nullptr, vel_only);
}

// ------------------------------------------------------------ projection
struct ForceArgs {
    const double *frag, *Kx, *Kz;
    int Nz, Mx, qpts, dimR, dimQ, nks, nit;
    double ax, az;                      // 2 pi / Lx, 2 pi / Lz
    const int *abort_flag;
    // members: problem p = m nprob + sub of the staged-basis kernels reads
    // U (sub 0: U0, 1: U1) + m ms_u and writes Fa, Fb + m ms_fa, m ms_fb;
    // k_force: grid y = member
    int nm;
    size_t ms_u, ms_fa, ms_fb;
};

// Fa[z][i][x] (i < dimQ), Fb[z][i][x] (i < dimR); 1-D grid over the (kz row,
// i-tile) tiles, i-tile fastest, XCD-aware (xcd_tile); 256 threads.
// D[n][i] = sum_y A_m[y][n] W_m[i][y] (channel/project.c:95-115,176-191,
// channel/adjproject.c:108-134,213-234) with the pointwise combinations
//   fa = Qpw P - k2 Qw Hy (+ Qppw Z),     P  = i kx Hx + i kz Hz
//   fb = Rw P2 (+ Rpw Z2),                P2 = i kz Hx - i kx Hz
//   (adjoint) Z = -i kz Sx + i kx Sz,     Z2 = i kz Sz + i kx Sx
// summed into two accumulators.  Each lane forms its A entries from the parts
// of Hx, Hz, Hy, Sx, Sz it needs.  Mean column (channel/project0.c:110-146,
// channel/adjproject0.c:98-140): Fb(0,0) = (Rw Re Hx + Rpw Re Sz,
// Rw Re Hz - Rpw Re Sx).  Wave w takes the n-tiles w, w+4, ... of the
// block's i-tile; the weighted-basis fragments of a chunk of KC_FORCE k-steps are
// staged in LDS (double-buffered), the field values prefetched a chunk ahead.
template <bool ADJ>
__global__ __launch_bounds__(256, SC_YT_WAVES) void k_force(ForceArgs a, const cplx *U, cplx *Fa, cplx *Fb)
{
    constexpr int KC = KC_FORCE, CH = KC * 5 * 64, PT = CH / 256;
    static_assert(CH % 256 == 0, "chunk must split over the block");
    __shared__ double bs[2][CH];
    if (*a.abort_flag) return;
    const int tile = xcd_tile(a.nit * a.Nz);
    if (tile < 0) return;
    U += blockIdx.y * a.ms_u;
    Fa += blockIdx.y * a.ms_fa;
    Fb += blockIdx.y * a.ms_fb;
    const int z = tile / a.nit, it = tile - z * a.nit;
    if (z == a.Nz / 2) return;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int Mx = a.Mx, q = a.qpts, nR = a.dimR, nQ = a.dimQ;
    constexpr bool adj = ADJ;
    const int nnt = (Mx + 7) / 8, nch = a.nks / KC;
    const int kq = lane >> 4, nl = lane & 15;
    const double *frag = a.frag + (size_t) it * a.nks * 5 * 64;
    const size_t ss = (size_t) q * Mx;
    const double *Ud = (const double *) (U + (size_t) z * 5 * ss);
    const double kz = wave_kz(z, a.Nz, a.az);
    for (int nt0 = 0; nt0 < nnt; nt0 += 4) {
        const int nt = nt0 + wave;
        const bool active = nt < nnt;
        // columns past Mx read the last column and are never stored
        const int xcol = min(nt * 8 + ncol_x(nl), Mx - 1), part = ncol_part(nl);
        const bool mean = z == 0 && xcol == 0;
        const double kx = wave_kx(xcol, a.ax), k2 = kz * kz + kx * kx;
        const double sg = part ? 1.0 : -1.0;
        const int other = mean ? 0 : 1 - part;
        mf4 accA = mf4_zero(), accB = mf4_zero();
        // two register sets of field values, used alternately:
        // r[0] Hx, r[1] Hz, r[2] Hy, r[3] Sx, r[4] Sz
        double r0[5][KC], r1[5][KC], st[PT];
        // unpredicated loads: Gauss points past qpts read the last point and
        // meet zero basis fragments
        auto load_fields = [&](int ch, double (*r)[KC]) {
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                const int y = min((ch * KC + s) * 4 + kq, q - 1);
                const size_t e = ((size_t) y * Mx + xcol) * 2;
                r[1][s] = Ud[e + other];
                r[0][s] = Ud[e + 2 * ss + other];
                r[2][s] = Ud[e + 4 * ss + part];
                if (adj) {
                    r[3][s] = Ud[e + 6 * ss + other];
                    r[4][s] = Ud[e + 8 * ss + other];
                }
            }
        };
        auto load_basis = [&](int ch) {
            const double *src = frag + (size_t) ch * CH;
#pragma unroll
            for (int i = 0; i < PT; ++i) st[i] = src[threadIdx.x + 256 * i];
        };
        auto put_basis = [&](int buf) {
#pragma unroll
            for (int i = 0; i < PT; ++i) bs[buf][threadIdx.x + 256 * i] = st[i];
        };
        auto compute = [&](double (*r)[KC], const double *b) {
            if (!active) return;
#pragma unroll
            for (int s = 0; s < KC; ++s) {
                const double hx = r[0][s], hz = r[1][s], hy = r[2][s];
                double vP, vY, vP2, vZ = 0.0, vZ2 = 0.0;
                if (mean) {
                    vP = 0.0;
                    vY = 0.0;
                    vP2 = part ? hz : hx;
                    if (adj) vZ2 = part ? -r[3][s] : r[4][s];
                } else {
                    vP = sg * (kx * hx + kz * hz);
                    vY = -k2 * hy;
                    vP2 = sg * (kz * hx - kx * hz);
                    if (adj) {
                        vZ = -sg * (kz * r[3][s] - kx * r[4][s]);
                        vZ2 = sg * (kz * r[4][s] + kx * r[3][s]);
                    }
                }
                accA = mfma_f64(vP, b[(s * 5 + 0) * 64 + lane], accA);
                accB = mfma_f64(vP2, b[(s * 5 + 3) * 64 + lane], accB);
                accA = mfma_f64(vY, b[(s * 5 + 1) * 64 + lane], accA);
                if (adj) {
                    accA = mfma_f64(vZ, b[(s * 5 + 2) * 64 + lane], accA);
                    accB = mfma_f64(vZ2, b[(s * 5 + 4) * 64 + lane], accB);
                }
            }
        };
        load_fields(0, r0);
        load_basis(0);
        put_basis(0);
        __syncthreads();
        for (int ch = 0; ch < nch; ch += 2) {
            const bool n1 = ch + 1 < nch;
            if (n1) {
                load_fields(ch + 1, r1);
                load_basis(ch + 1);
            }
            compute(r0, bs[0]);
            if (n1) put_basis(1);
            __syncthreads();
            if (!n1) break;
            const bool n2 = ch + 2 < nch;
            if (n2) {
                load_fields(ch + 2, r0);
                load_basis(ch + 2);
            }
            compute(r1, bs[1]);
            if (n2) put_basis(0);
            __syncthreads();
        }
        const int i = it * 16 + nl;
        if (!active || i >= nR) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int x = nt * 8 + 2 * kq + h;
            if (x >= Mx) continue;
            if (i < nQ && !(z == 0 && x == 0))
                Fa[((size_t) z * nQ + i) * Mx + x] = make_double2(accA[2 * h], accA[2 * h + 1]);
            Fb[((size_t) z * nR + i) * Mx + x] = make_double2(accB[2 * h], accB[2 * h + 1]);
        }
    }
}

// Projection with the i-tile's whole weighted basis in LDS (NKS k-steps;
// the three bases Qpw, Qw, Rw of the primal, all five for the adjoint), for
// NKS in {16, 28, 40}.  A block of 8 waves owns one i-tile and a contiguous
// range of its (kz row, n-tile) tasks; wave w takes tasks w, w+8, ... of the
// range.  No barrier after the staging: each wave streams its field values
// through two register buffers of CK k-steps (the loads of chunk c+1, or of
// the next task's chunk 0, issued before the products of chunk c).  The
// products enter the accumulators in the same order as in k_force.
// Grid: nit * bpi blocks, block b -> i-tile b / bpi.  With nprob = 2 the
// task range covers two projections sharing the staged basis (fields U0 ->
// Fa0, Fb0, then U1 -> Fa1, Fb1).
constexpr int FR_THREADS = 512;

template <bool ADJ, int NKS>
struct ForceRowsShape {
    static constexpr int NB = ADJ ? 5 : 3;                   // bases staged per k-step
    static constexpr int NF = ADJ ? 5 : 3;                   // field values per k-step
    // chunk: the largest CK <= CKMAX with an even number of chunks
    static constexpr int CKMAX = ADJ ? 4 : 5;
    static constexpr int pick(int ck) { return (NKS % ck == 0 && (NKS / ck) % 2 == 0) ? ck : pick(ck - 1); }
    static constexpr int CK = pick(CKMAX), NCH = NKS / CK;
};

template <bool ADJ, int NKS>
__global__ __launch_bounds__(FR_THREADS) void k_force_rows(ForceArgs a, int bpi, int nprob,
                                                           const cplx *U0, cplx *Fa0, cplx *Fb0,
                                                           const cplx *U1, cplx *Fa1, cplx *Fb1)
{
    using SH = ForceRowsShape<ADJ, NKS>;
    constexpr int NB = SH::NB, NF = SH::NF, CK = SH::CK, NCH = SH::NCH;
    static_assert(NCH % 2 == 0 && CK >= 1, "chunks alternate between two buffers");
    extern __shared__ double bsf[];
    if (*a.abort_flag) return;
    const int it = blockIdx.x / bpi, lb = blockIdx.x - it * bpi;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int kq = lane >> 4, nl = lane & 15;
    const int Mx = a.Mx, q = a.qpts, nR = a.dimR, nQ = a.dimQ;
    const int nnt = (Mx + 7) / 8;
    const int ntask = (a.Nz - 1) * nnt;                       // every row but the Nyquist row
    const int nall = ntask * nprob * a.nm;
    const int t0 = lb * nall / bpi, t1 = (lb + 1) * nall / bpi;
    {
        // bases of the i-tile: fragF [nit][nksF][5][64] -> [NKS][NB][64]
        const double *frag = a.frag + (size_t) it * a.nks * 5 * 64;
        constexpr int TOT = NKS * NB * 64, PT = (TOT + FR_THREADS - 1) / FR_THREADS;
        double st[PT];
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int e = min((int) threadIdx.x + FR_THREADS * i, TOT - 1);
            const int s = e / (NB * 64), r = e - s * NB * 64, m = r >> 6, l = r & 63;
            const int mm = ADJ ? m : (m == 2 ? 3 : m);       // primal: Qpw, Qw, Rw
            st[i] = frag[((size_t) s * 5 + mm) * 64 + l];
        }
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int e = threadIdx.x + FR_THREADS * i;
            if (e < TOT) bsf[e] = st[i];
        }
    }
    __syncthreads();
    // staged bases per k-step: Qpw, Qw, Qppw, Rw, Rpw (adjoint); Qpw, Qw, Rw (primal)
    struct Task {
        int z, nt, xcol, part, p, m;
        size_t off;
    };
    auto task_of = [&](int t) {
        Task k;
        const int pr = t / ntask;                             // problem: member, projection
        k.m = pr / nprob;
        k.p = pr - k.m * nprob;
        t -= pr * ntask;
        const int zr = t / nnt;
        k.z = zr < a.Nz / 2 ? zr : zr + 1;
        k.nt = t - zr * nnt;
        k.xcol = min(k.nt * 8 + ncol_x(nl), Mx - 1);
        k.part = ncol_part(nl);
        k.off = (size_t) k.z * 5 * q * Mx * 2 + (size_t) k.xcol * 2;
        return k;
    };
    const size_t ss2 = (size_t) q * Mx * 2;                   // slot stride in doubles
    double r[2][NF][CK];
    auto load = [&](const Task &k, int ch, int buf) {
        const double *Ud = (const double *) ((k.p ? U1 : U0) + k.m * a.ms_u);
        const bool mean = k.z == 0 && k.xcol == 0;
        const int other = mean ? 0 : 1 - k.part;
#pragma unroll
        for (int s = 0; s < CK; ++s) {
            const int y = min((ch * CK + s) * 4 + kq, q - 1);
            const size_t e = k.off + (size_t) y * Mx * 2;
            r[buf][1][s] = Ud[e + other];
            r[buf][0][s] = Ud[e + ss2 + other];
            r[buf][2][s] = Ud[e + 2 * ss2 + k.part];
            if (ADJ) {
                r[buf][3 % NF][s] = Ud[e + 3 * ss2 + other];
                r[buf][4 % NF][s] = Ud[e + 4 * ss2 + other];
            }
        }
    };
    int t = t0 + wave;
    if (t < t1) load(task_of(t), 0, 0);
    while (t < t1) {
        const Task k = task_of(t);
        const bool mean = k.z == 0 && k.xcol == 0;
        const double kz = wave_kz(k.z, a.Nz, a.az);
        const double kx = wave_kx(k.xcol, a.ax), k2 = kz * kz + kx * kx;
        const double sg = k.part ? 1.0 : -1.0;
        mf4 accA = mf4_zero(), accB = mf4_zero();
        const int tn = t + 8;
        // products of chunk ch from buffer buf
        auto chunk = [&](int ch, int buf) {
            const double *bc = bsf + (size_t) ch * CK * NB * 64 + lane;
#pragma unroll
            for (int u = 0; u < CK; ++u) {
                const double hx = r[buf][0][u], hz = r[buf][1][u], hy = r[buf][2][u];
                double vP, vY, vP2, vZ = 0.0, vZ2 = 0.0;
                if (mean) {
                    vP = 0.0;
                    vY = 0.0;
                    vP2 = k.part ? hz : hx;
                    if (ADJ) vZ2 = k.part ? -r[buf][3 % NF][u] : r[buf][4 % NF][u];
                } else {
                    vP = sg * (kx * hx + kz * hz);
                    vY = -k2 * hy;
                    vP2 = sg * (kz * hx - kx * hz);
                    if (ADJ) {
                        vZ = -sg * (kz * r[buf][3 % NF][u] - kx * r[buf][4 % NF][u]);
                        vZ2 = sg * (kz * r[buf][4 % NF][u] + kx * r[buf][3 % NF][u]);
                    }
                }
                const double *b = bc + u * NB * 64;
                accA = mfma_f64(vP, b[(ADJ ? 0 : 0) * 64], accA);
                accB = mfma_f64(vP2, b[(ADJ ? 3 : 2) * 64], accB);
                accA = mfma_f64(vY, b[1 * 64], accA);
                if (ADJ) {
                    accA = mfma_f64(vZ, b[2 * 64], accA);
                    accB = mfma_f64(vZ2, b[4 * 64], accB);
                }
            }
        };
        // two chunks per iteration, one per buffer; the loads of the chunk
        // after next (or of the next task's first chunk) go into the buffer
        // just used
#pragma unroll 1
        for (int ch = 0; ch < NCH; ch += 2) {
            load(k, ch + 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            chunk(ch, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (ch + 2 < NCH)
                load(k, ch + 2, 0);
            else if (tn < t1)
                load(task_of(tn), 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            chunk(ch + 1, 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int i = it * 16 + nl;
        if (i < nR) {
            cplx *Fa = (k.p ? Fa1 : Fa0) + k.m * a.ms_fa, *Fb = (k.p ? Fb1 : Fb0) + k.m * a.ms_fb;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = k.nt * 8 + 2 * kq + h;
                if (x >= Mx) continue;
                if (i < nQ && !(k.z == 0 && x == 0))
                    Fa[((size_t) k.z * nQ + i) * Mx + x] = make_double2(accA[2 * h], accA[2 * h + 1]);
                Fb[((size_t) k.z * nR + i) * Mx + x] = make_double2(accB[2 * h], accB[2 * h + 1]);
            }
        }
        t = tn;
    }
}

// Parity form of the staged-basis projection.  The weighted basis functions
// have the parity of the Gauss-point mirror (Qw, Qppw, Rw of row i that of
// i, Qpw and Rpw the opposite), so over a mirrored pair of points
//     W(y) v(y) + W(-y) v(-y) = W(y) (v(y) + v(-y))  or  W(y) (v(y) - v(-y)),
// and a projection onto 16 even and 16 odd rows i takes the half domain's
// points once each: the products of one k-step feed both row tiles.  Each
// lane forms the pointwise combinations (P, Hy, P2, Z, Z2 as in k_force) at
// y and at its mirror, then their sum S and difference D:
//     even rows:  Qpw D_P + Qw S_Y + Qppw S_Z,   Rw S_P2 + Rpw D_Z2
//     odd rows:   Qpw S_P + Qw D_Y + Qppw D_Z,   Rw D_P2 + Rpw S_Z2
// The middle point of an odd qpts (y = 0) is its own mirror: its staged
// weights are halved, so that S = 2 v(0) gives the weight once, and the
// functions that D multiplies vanish there.  A block owns one pair of row
// tiles (even rows 2(16p + n), odd rows 2(16p + n) + 1), stages their
// weighted bases [NKS][2][NB][64] and runs the (kz row, n-tile) tasks of a
// contiguous range.  Field values are read with buffer loads over the whole
// field array: the points past the half domain, whose staged weights are zero,
// read values in or past the array (zero past its end) and need no clamp.
//
// What bounds it: the FP64 unit, which FP64 products and FP64 vector
// instructions share (a product 65 clocks a SIMD, a multiply-add or add 4.5, a
// conversion 6.5, one after the other), and with members the loads' way through
// the L1.  So a k-step is held to the products and as few other FP64
// instructions as the combinations need: their signs and the mean column's case
// sit in per-lane coefficients.  The fields come through a ring of PD k-steps,
// refilled for the k-step PD later, or for the next task's, as soon as a
// k-step's combinations are formed; the first ring is requested before the
// bases, and FP32 slots are converted when used (when loaded, the conversion
// waited for the load).  Measured against chunks requested task by task, 104
// instead of 55 vector instructions a k-step: 32 mixed members at 64x97x64 588
// -> 460 us (adjoint) and 259 -> 206 us, two at 128x129x128 216 -> 193 and 95 ->
// 77 us, nine FP64 members 50 -> 44.5 us, one FP64 solution 25.6 -> 24.7 and 13.4
// -> 13.0 us.
//
// The sums of the two halves of the k-steps are added at the end (NH = 2).
// KS = 2: two waves share a task, one half each, and add through LDS.  KS = 1: a
// wave sums both halves, no barrier.
template <bool ADJ, int NKS, bool P32, int KS>
struct ForceParShape {
    static constexpr int NB = ADJ ? 5 : 3;
    static constexpr int NF = ADJ ? 5 : 3;
    // the bases of 28 adjoint k-steps leave no room for an exchange of halves
    static constexpr int NH = ADJ && NKS == 28 ? 1 : 2;
    static constexpr int KW = NKS / NH;                      // k-steps of a half
    static constexpr int KT = NKS / KS;                      // k-steps of a wave's task
    static constexpr int TPR = FR_THREADS / 64 / KS;         // tasks per round of the block
    static constexpr int XCH1 = 4 * 4 * 64;                  // doubles of one wave's partials
    static constexpr int XCH = KS > 1 ? TPR * XCH1 : 0;
    // ring: 4, 5 or 7 k-steps, a divisor of KW; 2 where those would not leave
    // the registers for two waves a SIMD (FP64 adjoint, FP64 28 k-steps)
    static constexpr int PD = !P32 && (ADJ || NKS == 28) ? 2 : KW % 5 == 0 ? 5 : KW % 4 == 0 ? 4 : 7;
    // k-steps of an unrolled group: whole turns of the ring and of the two
    // buffers of basis fragments
    static constexpr int UN = PD % 2 ? 2 * PD : PD;
    static_assert(KT % UN == 0 && KW % PD == 0 && KS <= NH, "a task is whole groups");
    static constexpr size_t lds_bytes() { return sizeof(double) * ((size_t) NKS * 2 * NB * 64 + XCH); }
};
// P32: the product slots are FP32 complex (mixed precision; same element
// index), converted to FP64 when used
template <bool ADJ, int NKS, bool P32, int KS>
__global__ __launch_bounds__(FR_THREADS) void k_force_par(ForceArgs a, int bpi, int nprob,
                                                          const cplx *U0, cplx *Fa0, cplx *Fb0,
                                                          const cplx *U1, cplx *Fa1, cplx *Fb1)
{
    using SH = ForceParShape<ADJ, NKS, P32, KS>;
    constexpr int NB = SH::NB, NF = SH::NF, PD = SH::PD, UN = SH::UN, KT = SH::KT, NG = KT / UN;
    constexpr unsigned ESZ = P32 ? 8 : 16;                   // bytes of a slot value
    constexpr int TPR = SH::TPR, XCH1 = SH::XCH1;
    typedef typename std::conditional<P32, float, double>::type V;
    extern __shared__ double bsf[];
    if (*a.abort_flag) return;
    // XCD-aware: block b runs task range lb = (b / 8 / npair) 8 + b % 8 of
    // row-tile pair tp = (b / 8) % npair, so the pairs' blocks of one task
    // range (which read the same fields) share an XCD and its L2; bpi is a
    // multiple of 8
    const int npair = a.nit;
    const int rest = blockIdx.x >> 3, tp = rest % npair;
    const int lb = (rest / npair) * 8 + (blockIdx.x & 7);
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int kq = lane >> 4, nl = lane & 15;
    const int Mx = a.Mx, q = a.qpts, nR = a.dimR, nQ = a.dimQ;
    const int nnt = (Mx + 7) / 8;
    const int ntask = (a.Nz - 1) * nnt;
    const int nall = ntask * nprob * a.nm;
    const int t0 = (int) ((long long) lb * nall / bpi), t1 = (int) ((long long) (lb + 1) * nall / bpi);
    const int part = ncol_part(nl), half = KS > 1 ? wave % KS : 0, slot = wave / KS, kb = half * KT;
    const unsigned ubytes = (unsigned) ((size_t) a.Nz * 5 * q * Mx * ESZ);
    const unsigned rowb = (unsigned) Mx * ESZ, slotb = (unsigned) q * rowb;
    struct Task {
        int z, nt, p, m;
        // bytes of the lane's column at its first point (row kb 4 + kq): the
        // part that P, P2, Z, Z2 read and the part that Hy does
        unsigned other, own;
    };
    auto task_of = [&](int t) {
        Task k;
        const int pr = t / ntask;                             // problem: member, projection
        k.m = pr / nprob;
        k.p = pr - k.m * nprob;
        t -= pr * ntask;
        const int zr = t / nnt;
        k.z = zr < a.Nz / 2 ? zr : zr + 1;
        k.nt = t - zr * nnt;
        const int xcol = min(k.nt * 8 + ncol_x(nl), Mx - 1);
        const bool mean = k.z == 0 && xcol == 0;
        const unsigned off = (unsigned) (((size_t) k.z * 5 * q * Mx + xcol) * ESZ) + (unsigned) (kb * 4 + kq) * rowb;
        k.other = off + (mean ? 0 : 1 - part) * (ESZ / 2);
        k.own = off + part * (ESZ / 2);
        return k;
    };
    // r[slot of the ring][0: y, 1: mirror][field]
    V r[PD][2][NF];
    // k-step kb + s of task k (s = g PD + u) into slot u: uniform offsets for the
    // field and the point; the mirror runs down from row q - 1 - (kb 4 + kq)
    const unsigned md = (unsigned) (q - 1 - 2 * (kb * 4 + kq)) * rowb;
    auto load = [&](const Task &k, int s, int u) {
        __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void *) ((k.p ? U1 : U0) + k.m * a.ms_u), 0, ubytes, 0x00020000);
        auto ld = [&](unsigned v, unsigned so) {
            if constexpr (P32)
                return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int) v, (int) so, 0));
            else
                return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, (int) v, (int) so, 0));
        };
        const unsigned step = (unsigned) s * 4 * rowb;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned vo = h ? k.other + md - step : k.other, vw = h ? k.own + md - step : k.own;
            const unsigned so = h ? 0 : step;
            r[u][h][1] = ld(vo, so);
            r[u][h][0] = ld(vo, so + slotb);
            r[u][h][2] = ld(vw, so + 2 * slotb);
            if constexpr (ADJ) {
                r[u][h][3] = ld(vo, so + 3 * slotb);
                r[u][h][4] = ld(vo, so + 4 * slotb);
            }
        }
    };
    int t = t0 + slot;
    Task k = task_of(min(t, nall - 1));
    if (t < t1) {
#pragma unroll
        for (int u = 0; u < PD; ++u) load(k, u, u);
    }
    __builtin_amdgcn_sched_barrier(0);
    {
        // fragQ [npair][NKS][2][5][64] -> [NKS][2][NB][64]
        const double *frag = a.frag + (size_t) tp * NKS * 2 * 5 * 64;
        constexpr int TOT = NKS * 2 * NB * 64, PT = (TOT + FR_THREADS - 1) / FR_THREADS;
        double st[PT];
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int e = min((int) threadIdx.x + FR_THREADS * i, TOT - 1);
            const int sp = e / (NB * 64), rr = e - sp * NB * 64, m = rr >> 6, l = rr & 63;
            const int mm = ADJ ? m : (m == 2 ? 3 : m);       // primal: Qpw, Qw, Rw
            st[i] = frag[((size_t) sp * 5 + mm) * 64 + l];
        }
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int e = threadIdx.x + FR_THREADS * i;
            if (e < TOT) bsf[e] = st[i];
        }
    }
    __syncthreads();
    double *xch = bsf + (size_t) NKS * 2 * NB * 64;
    // the lane's basis fragments of a k-step: even rows' NB, then odd rows'
    double bf[2][2 * NB];
    auto fragments = [&](double *f, int s) {
        const double *b = bsf + (size_t) (kb + s) * 2 * NB * 64 + lane;
#pragma unroll
        for (int e = 0; e < 2 * NB; ++e) f[e] = b[e * 64];
    };
    fragments(bf[0], 0);
    // rounds of TPR tasks, the same count in every wave of a KS = 2 block
    for (int tb = t0; KS > 1 ? tb < t1 : t < t1; tb += TPR, t += TPR) {
        const bool act = t < t1, more = t + TPR < t1;
        const Task kn = task_of(more ? t + TPR : min(t, nall - 1));
        mf4 aAe = mf4_zero(), aBe = mf4_zero(), aAo = mf4_zero(), aBo = mf4_zero();
        mf4 bAe, bBe, bAo, bBo;                              // the first half's sums (KS = 1)
        if (act) {
            // the lane's combinations, signs in the coefficients:
            //   P = px hx + pz hz, Y = ky hy, P2 = qx hx - qz hz,
            //   Z = px sz - pz sx, Z2 = wz sz + wx sx
            // the mean column takes P = Y = Z = 0, P2 = hx (first part) or hz,
            // Z2 = sz or -sx
            const int xcol = min(k.nt * 8 + ncol_x(nl), Mx - 1);
            const bool mean = k.z == 0 && xcol == 0;
            const double kz = wave_kz(k.z, a.Nz, a.az);
            const double kx = wave_kx(xcol, a.ax), k2 = __builtin_fma(kx, kx, kz * kz);
            const double sg = part ? 1.0 : -1.0;
            const double px = mean ? 0.0 : sg * kx, pz = mean ? 0.0 : sg * kz, ky = mean ? 0.0 : -k2;
            const double qx = mean ? 1.0 - part : pz, qz = mean ? -part : px;
            const double wz = mean ? 1.0 - part : pz, wx = mean ? -part : px;
#pragma unroll 1
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int u = 0; u < UN; ++u) {
#pragma clang fp contract(off)   // Y is rounded before its sums
                    const int w = u % PD;                    // ring slot
                    if (KS < SH::NH && u == SH::KW % UN && g == SH::KW / UN) {
                        bAe = aAe; bBe = aBe; bAo = aAo; bBo = aBo;
                        aAe = aBe = aAo = aBo = mf4_zero();
                    }
                    double vP[2], vY[2], vP2[2], vZ[2] = {0.0, 0.0}, vZ2[2] = {0.0, 0.0};
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const double hx = r[w][h][0], hz = r[w][h][1], hy = r[w][h][2];
                        // which product is rounded: either is as accurate, and the
                        // primal's results with eight k-steps (qpts <= 64) have been
                        // those of the second form, which keeps their last bits
                        vP[h] = ADJ || NKS != 8 ? __builtin_fma(px, hx, pz * hz)
                                                : __builtin_fma(pz, hz, px * hx);
                        vY[h] = ky * hy;
                        vP2[h] = __builtin_fma(qx, hx, -(qz * hz));
                        if constexpr (ADJ) {
                            const double sx = r[w][h][3], sz = r[w][h][4];
                            vZ[h] = __builtin_fma(-pz, sx, px * sz);
                            vZ2[h] = __builtin_fma(wx, sx, wz * sz);
                        }
                    }
                    const double sP = vP[0] + vP[1], dP = vP[0] - vP[1];
                    const double sY = vY[0] + vY[1], dY = vY[0] - vY[1];
                    const double sP2 = vP2[0] + vP2[1], dP2 = vP2[0] - vP2[1];
                    const double sZ = vZ[0] + vZ[1], dZ = vZ[0] - vZ[1];
                    const double sZ2 = vZ2[0] + vZ2[1], dZ2 = vZ2[0] - vZ2[1];
                    __builtin_amdgcn_sched_barrier(0);
                    // the k-step PD on, of this task or the next
                    if (u + PD < UN || g + 1 < NG)
                        load(k, g * UN + u + PD, w);
                    else if (more)
                        load(kn, u + PD - UN, w);
                    // the next k-step's basis fragments
                    fragments(bf[(u + 1) & 1], u + 1 < UN || g + 1 < NG ? g * UN + u + 1 : 0);
                    __builtin_amdgcn_sched_barrier(0);
                    const double *be = bf[u & 1], *bo = be + NB;
                    aAe = mfma_f64(dP, be[0], aAe);
                    aAo = mfma_f64(sP, bo[0], aAo);
                    aBe = mfma_f64(sP2, be[ADJ ? 3 : 2], aBe);
                    aBo = mfma_f64(dP2, bo[ADJ ? 3 : 2], aBo);
                    aAe = mfma_f64(sY, be[1], aAe);
                    aAo = mfma_f64(dY, bo[1], aAo);
                    if constexpr (ADJ) {
                        aAe = mfma_f64(sZ, be[2], aAe);
                        aAo = mfma_f64(dZ, bo[2], aAo);
                        aBe = mfma_f64(dZ2, be[4], aBe);
                        aBo = mfma_f64(sZ2, bo[4], aBo);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (KS < SH::NH) {
                aAe = bAe + aAe;
                aBe = bBe + aBe;
                aAo = bAo + aAo;
                aBo = bBo + aBo;
            }
        }
        if constexpr (KS > 1) {
            // the second half's sums go through LDS to the first half's wave
            double *xw = xch + (size_t) slot * XCH1 + lane;
            if (act && half > 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xw[(0 * 4 + e) * 64] = aAe[e];
                    xw[(1 * 4 + e) * 64] = aBe[e];
                    xw[(2 * 4 + e) * 64] = aAo[e];
                    xw[(3 * 4 + e) * 64] = aBo[e];
                }
            }
            __syncthreads();
            if (act && half == 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    aAe[e] += xw[(0 * 4 + e) * 64];
                    aBe[e] += xw[(1 * 4 + e) * 64];
                    aAo[e] += xw[(2 * 4 + e) * 64];
                    aBo[e] += xw[(3 * 4 + e) * 64];
                }
            }
        }
        if (act && half == 0) {
            cplx *Fa = (k.p ? Fa1 : Fa0) + k.m * a.ms_fa, *Fb = (k.p ? Fb1 : Fb0) + k.m * a.ms_fb;
#pragma unroll
            for (int par = 0; par < 2; ++par) {
                const int i = 2 * (tp * 16 + nl) + par;
                if (i >= nR) continue;
                const mf4 &A = par ? aAo : aAe, &B = par ? aBo : aBe;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int x = k.nt * 8 + 2 * kq + h;
                    if (x >= Mx) continue;
                    if (i < nQ && !(k.z == 0 && x == 0))
                        Fa[((size_t) k.z * nQ + i) * Mx + x] = make_double2(A[2 * h], A[2 * h + 1]);
                    Fb[((size_t) k.z * nR + i) * Mx + x] = make_double2(B[2 * h], B[2 * h + 1]);
                }
            }
        }
        // the exchange area is reused by the next round
        if (KS > 1) __syncthreads();
        k = kn;
    }
}

template <bool ADJ, int NKS, bool P32, int KS>
static void launch_force_par_ks(const ForceArgs &a, int npair, int bpi, int nprob, const cplx *U0,
                                cplx *Fa0, cplx *Fb0, const cplx *U1, cplx *Fa1, cplx *Fb1,
                                hipStream_t st)
{
    const size_t lds = ForceParShape<ADJ, NKS, P32, KS>::lds_bytes();
    static bool attr = false;
    if (!attr) {
        (void) hipFuncSetAttribute((const void *) k_force_par<ADJ, NKS, P32, KS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        attr = true;
    }
    hipLaunchKernelGGL((k_force_par<ADJ, NKS, P32, KS>), dim3(npair * bpi), dim3(FR_THREADS), lds, st, a, bpi,
                       nprob, U0, Fa0, Fb0, U1, Fa1, Fb1);
}

template <bool ADJ, int NKS, bool P32>
static void launch_force_par(const ForceArgs &a, int npair, int ntask, int nprob, const cplx *U0,
                             cplx *Fa0, cplx *Fb0, const cplx *U1, cplx *Fa1, cplx *Fb1,
                             hipStream_t st)
{
    // blocks per pair: a multiple of 8 (XCD-aware mapping), one block per CU
    const int cap = tuning().force_blocks > 0 ? tuning().force_blocks : 256 / npair / 8 * 8;
    const int nall = ntask * nprob * a.nm;
    const int bpi = std::max(8, std::min((nall + 7) / 8 * 8, cap));
    // a task per wave where a block has eight tasks or more, for FP32 slots (32
    // members: 460 us, with two waves a task 480; FP64 slots leave no registers
    // for both halves' sums: nine members 73 us, with two waves 44.5); two waves
    // a task otherwise
    constexpr bool pairs = ForceParShape<ADJ, NKS, P32, 1>::NH > 1;
    if constexpr (pairs) {
        if (!P32 || nall < 8 * bpi) {
            launch_force_par_ks<ADJ, NKS, P32, 2>(a, npair, bpi, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
            return;
        }
    }
    if constexpr (P32 || !pairs)
        launch_force_par_ks<ADJ, NKS, P32, 1>(a, npair, bpi, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
}

template <bool ADJ, int NKS>
static void launch_force_rows(const ForceArgs &a, int nit, int ntask, int nprob, const cplx *U0,
                              cplx *Fa0, cplx *Fb0, const cplx *U1, cplx *Fa1, cplx *Fb1,
                              hipStream_t st)
{
    using SH = ForceRowsShape<ADJ, NKS>;
    const size_t lds = sizeof(double) * NKS * SH::NB * 64;
    static bool attr = false;
    if (!attr) {
        (void) hipFuncSetAttribute((const void *) k_force_rows<ADJ, NKS>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        attr = true;
    }
    // blocks per i-tile: one 8-wave block per CU in total (the registers of
    // the wave's two field buffers allow no second block), never more than
    // the tasks
    const int bpi = std::max(1, std::min(ntask * nprob * a.nm, 256 / nit));
    hipLaunchKernelGGL((k_force_rows<ADJ, NKS>), dim3(nit * bpi), dim3(FR_THREADS), lds, st, a, bpi,
                       nprob, U0, Fa0, Fb0, U1, Fa1, Fb1);
}

// one or two projections (U1 null: one); the staged-basis kernel runs both in
// one launch, the chunked kernel one launch each
void launch_force2(Context &c, int adj, const cplx *U0, cplx *Fa0, cplx *Fb0, const cplx *U1,
                   cplx *Fa1, cplx *Fb1)
{
    const Dims &d = c.d;
    const int nm = c.nrun;
    const size_t ms_u = mstride(c, U0), ms_fa = mstride(c, Fa0), ms_fb = mstride(c, Fb0);
    if (U1 && (mstride(c, U1) != ms_u || mstride(c, Fa1) != ms_fa || mstride(c, Fb1) != ms_fb)) {
        // the two problems' arrays have other member strides: two launches
        launch_force2(c, adj, U0, Fa0, Fb0, nullptr, nullptr, nullptr);
        launch_force2(c, adj, U1, Fa1, Fb1, nullptr, nullptr, nullptr);
        return;
    }
    ForceArgs a{c.dFragF, c.dKx, c.dKz, d.Nz, d.Mx, d.qpts, d.dimR, d.dimQ, c.nksF, c.nit,
                2. * M_PI / d.Lx, 2. * M_PI / d.Lz, c.abort_flag, nm, ms_u, ms_fa, ms_fb};
    dim3 grid(xcd_grid(c.nit * d.Nz), nm);
    const int nprob = U1 ? 2 : 1;
    // mixed precision: FP32 product slots (the z-forward transforms wrote them)
    const bool p32 = prods32(c);
    double bytes = nm * nprob * (double) (d.Nz - 1) * d.Mx *
                   ((p32 ? 8.0 : 16.0) * (adj ? 5.0 : 3.0) * d.qpts + 16.0 * (d.dimQ + d.dimR));
    const hipStream_t st = c.stream;
    const int nks = c.nksF, nit = c.nit, ntask = (d.Nz - 1) * ((d.Mx + 7) / 8);
    const int nksq = c.nksQ, npair = c.npair;
    const bool par = c.ypar && (nksq == 8 || nksq == 16 || nksq == 20 || nksq == 28);
    ForceArgs ap = a;
    ap.frag = c.dFragQ;
    ap.nks = nksq;
    ap.nit = npair;
    auto go = [=]() {
        if (par) {
#define SC_FORCE_PAR(A, N)                                                                   \
    (p32 ? launch_force_par<A, N, true>(ap, npair, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st) \
         : launch_force_par<A, N, false>(ap, npair, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st))
            if (adj) {
                if (nksq == 8) SC_FORCE_PAR(true, 8);
                else if (nksq == 16) SC_FORCE_PAR(true, 16);
                else if (nksq == 20) SC_FORCE_PAR(true, 20);
                else SC_FORCE_PAR(true, 28);
            } else {
                if (nksq == 8) SC_FORCE_PAR(false, 8);
                else if (nksq == 16) SC_FORCE_PAR(false, 16);
                else if (nksq == 20) SC_FORCE_PAR(false, 20);
                else SC_FORCE_PAR(false, 28);
            }
#undef SC_FORCE_PAR
            return;
        }
        // staged-basis kernel for the k-step counts it is built for
        if (nks == 40 || nks == 28 || nks == 16) {
            if (adj) {
                if (nks == 40)
                    launch_force_rows<true, 40>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
                else if (nks == 28)
                    launch_force_rows<true, 28>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
                else
                    launch_force_rows<true, 16>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
            } else {
                if (nks == 40)
                    launch_force_rows<false, 40>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
                else if (nks == 28)
                    launch_force_rows<false, 28>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
                else
                    launch_force_rows<false, 16>(a, nit, ntask, nprob, U0, Fa0, Fb0, U1, Fa1, Fb1, st);
            }
            return;
        }
        for (int p = 0; p < nprob; ++p) {
            const cplx *U = p ? U1 : U0;
            cplx *Fa = p ? Fa1 : Fa0, *Fb = p ? Fb1 : Fb0;
            if (adj)
                hipLaunchKernelGGL(k_force<true>, grid, dim3(256), 0, st, a, U, Fa, Fb);
            else
                hipLaunchKernelGGL(k_force<false>, grid, dim3(256), 0, st, a, U, Fa, Fb);
        }
    };
    prof_begin(c, st, 5, bytes);
    go();
    prof_end(c, st, 5, go);
}

void launch_force(Context &c, const cplx *Usrc, int adj, cplx *Fa, cplx *Fb)
{
    launch_force2(c, adj, Usrc, Fa, Fb, nullptr, nullptr, nullptr);
}

void launch_force(Context &c, const cplx *Usrc, int adj) { launch_force(c, Usrc, adj, c.Fa, c.Fb); }

// ------------------------------------------------------------ band solves
// Stage solve of every (kz, kx) column (channel/project.c:22-151,
// channel/increproject.c:13-194, channel/adjproject.c:9-226): the right-hand
// side E C + dt c_k F (E applied only at the first stage, where C still holds
// the state), the LU solve with the stage's implicit operator, then
// C <- E' X + dt d_{k+1} F2, the next stage's carried right-hand side.  The
// even and odd rows of the stride-2 bands decouple, so one chain is one
// (column, field, parity), and the real and imaginary parts are chains of
// their own.
//
// A block solves SBT columns of one (field, parity) for up to MB members, which
// all have the same operator.  One wave runs the chains (2 SBT lanes a member,
// the last DL values in registers); the other three, the workers, own the rows:
// they form the right-hand sides, bring the U factors into LDS and form the next
// stage's operator entries while the chain wave runs its forward sweep, and write
// the results.  The chain is what the kernel waits for, and a lone wave issues
// one instruction every four or five clocks, so its cost is its instructions: the
// factors are laid out (setup.cpp) so that a row's operands are whole 16-byte LDS
// reads at immediate offsets, rows and vectors are padded with zeros to groups
// of eight so that nothing is clamped or predicated.  Two sweeps of 48 rows took
// 7 us with a row-major image and clamped rows, and take 4.2 with four blocks'
// chains on a CU (10000 clocks; 32 rows 2 us).  Measured, stage average: one
// 64x97x64 solution 23.0 -> 16.0 us, 32 members 455 -> 232 us, 32x65x32 12.7 ->
// 8.0 us, 128x129x128 with two members 185 -> 143 us; the members' launch is
// bound by its 0.8 GB of vectors (4.9 TB/s of a large copy: 165 us).
//
// The mean mode (kz = kx = 0; channel/project0.c:22-271,
// channel/increproject0.c:14-312, channel/adjproject0.c:8-310): real-part-only
// forcing fa = Re(Hx)-projection and fb = Re(Hz)-projection, read as the pair
// Fb(0,0) = (fa, fb); the flux correction
// alpha += (target - sum_i rowsum_i Re alpha_i) add / 2.
struct SolveArgs {
    const double *Qs, *Qps, *Qpps, *Rs, *Rps, *Kx, *Kz;
    const double *La, *Lb;             // factor images of this stage (SolveImage)
    const double *Lm, *add, *rowsum;   // mean mode: its image, flux vector, row sums
    const cplx *Fa, *Fb;               // projection for this stage's RHS
    const cplx *Fa2, *Fb2;             // projection for the next-stage RHS
    int Nz, Mx, dimR, dimQ, k, has_next;
    int nblk;                          // column blocks of SBT columns
    int ngrp;                          // groups of MB members
    int nyq_mean;                      // the mean mode runs in the Nyquist blocks' first (1) or in an extra block (0)
    int mirror;                        // factor images of rows z > Nz/2 are those of row Nz - z
    double dtc, dtd;                   // dt c_k, dt d_{k+1}
    double ce0[2], cn[2];              // explicit-operator coefficients per field (stage 0, next)
    double target;                     // mean-mode flux target
    double target_alt;                 // ... of the members m with bit m of alt_mask set
    unsigned alt_mask;
    const int *abort_flag;
    // member strides of C, Cs, Fa, Fb, Fa2, Fb2, Src
    size_t ms_c, ms_cs, ms_fa, ms_fb, ms_fa2, ms_fb2, ms_src;
    // optional right-hand-side source of the stage (C layout), added after
    // the explicit part and the forcing, before the solve (all modes)
    const cplx *Src;
    // adjoint only: the mean column as the exact transpose of the tangent's
    // flux correction: at stages 0 and 1 the right-hand side's real alpha
    // loses w1 (add_mass . rhs) / 2 before the solve, and no correction
    // follows the solve (the host loop applies P at each step's start)
    int exact_mean;
    const double *add_mass;            // Rs^{-1} w1
    int nm;                            // members of the launch
};

// Entries A(i, i + 2m), m = -DL .. DL, of the explicit operator of a row: the v
// operator -(k2 Qs + Qps) + coef (k2^2 Qs + 2 k2 Qps + Qpps) (DL = 4), the omega_y
// operator Rs + coef (Rps + k2 Rs) (DL = 2).  The Gram bands are zero outside the
// matrix; Qs reaches |m| = 4, Qps 3, Qpps 2, Rs 2 and Rps 1.  Which product of
// k2^2 Qs + 2 k2 Qps is rounded is written out, so that every block shape forms
// the same bits.
template <int DL>
__device__ __forceinline__ void op_row(const SolveArgs &a, int i, double k2, double coef, double *e)
{
    if constexpr (DL == 4) {
        const double s = k2 * k2, t = 2. * k2;
        const double *qs = a.Qs + i * 9, *qp = a.Qps + i * 9, *qq = a.Qpps + i * 9;
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            const bool p = j > 0 && j < 8, q = j > 1 && j < 7;
            double v = p ? __builtin_fma(s, qs[j], t * qp[j]) : s * qs[j];
            if (q) v += qq[j];
            e[j] = __builtin_fma(coef, v, -(p ? __builtin_fma(k2, qs[j], qp[j]) : k2 * qs[j]));
        }
    } else {
        const double *rs = a.Rs + i * 5, *rp = a.Rps + i * 5;
#pragma unroll
        for (int j = 0; j < 5; ++j)
            e[j] = __builtin_fma(coef, j > 0 && j < 4 ? __builtin_fma(k2, rs[j], rp[j]) : k2 * rs[j], rs[j]);
    }
}

// Forward and back substitution of one part (real or imaginary) of one column
// held in LDS: fl, bu, bi the image's factors of the column (rows SBT DL, SBT DL
// and SBT apart), v its part of the vector, rows vr apart, nrp rows (a multiple
// of eight) between rows of zeros.  Factors of rows past the chain are zero.
//
// Forward sweep, row s: x_s = v_s - L(s,DL) x_{s-DL} - ... - L(s,1) x_{s-1},
// the terms applied farthest first (the reference's order).  It runs skewed:
// the step that produces x_r applies it to the rows r+1 .. r+DL at once, so its
// DL multiply-adds are independent and only one of them is on the path to the
// next step.  P[k] holds row r+k with its terms DL .. k+2 applied;
// fl[r][k] = L(r+k, k+1).
//
// Backward sweep, row r: x_r = (v_r - U(r,1) x_{r+1} - ... - U(r,DL) x_{r+DL})
// / U(r,r), nearest term first (the reference's order); bu[r][m-1] = U(r, r+m),
// bi[r] = 1 / U(r, r).
//
// Operands stream through two register buffers of four rows each: the loads of
// the next four rows are issued before the arithmetic of the current ones (a
// scheduling barrier keeps them there).
// (one row's operands are named values: arrays of rows would be kept in
// scratch memory)
template <int DL> struct RowFactors;
template <> struct RowFactors<4> {
    double2 p, q;
    __device__ __forceinline__ void load(const double *f)
    {
        p = ((const double2 *) f)[0];
        q = ((const double2 *) f)[1];
    }
    template <int K> __device__ __forceinline__ double get() const
    {
        return K == 0 ? p.x : K == 1 ? p.y : K == 2 ? q.x : q.y;
    }
};
template <> struct RowFactors<2> {
    double2 p;
    __device__ __forceinline__ void load(const double *f) { p = ((const double2 *) f)[0]; }
    template <int K> __device__ __forceinline__ double get() const { return K == 0 ? p.x : p.y; }
};

template <int DL> struct FwdRow {
    RowFactors<DL> c;
    double vn;
};
template <int DL, int FR, int VR> struct FwdRows {
    FwdRow<DL> a, b, c, d;
    __device__ __forceinline__ void load1(FwdRow<DL> &o, const double *fl, const double *v)
    {
        o.c.load(fl);
        o.vn = v[(DL - 1) * VR];
    }
    __device__ __forceinline__ void load(const double *fl, const double *v)
    {
        load1(a, fl, v);
        load1(b, fl + FR * DL, v + VR);
        load1(c, fl + 2 * FR * DL, v + 2 * VR);
        load1(d, fl + 3 * FR * DL, v + 3 * VR);
    }
};

// P0 .. P2 (P0 only for DL = 2): the next rows with their terms applied so far
struct FwdState {
    double P0, P1, P2, x;
};

template <int DL>
__device__ __forceinline__ void fwd_step(const FwdRow<DL> &o, FwdState &s, double *v)
{
    const double x = __builtin_fma(-o.c.template get<0>(), s.x, s.P0);
    if constexpr (DL == 4) {
        s.P0 = __builtin_fma(-o.c.template get<1>(), s.x, s.P1);
        s.P1 = __builtin_fma(-o.c.template get<2>(), s.x, s.P2);
        s.P2 = __builtin_fma(-o.c.template get<3>(), s.x, o.vn);
    } else {
        s.P0 = __builtin_fma(-o.c.template get<1>(), s.x, o.vn);
    }
    v[0] = x;
    s.x = x;
}

template <int DL, int FR, int VR>
__device__ __forceinline__ void chain_forward(const double *fl, double *v, int nrp)
{
    FwdState s{v[0], DL == 4 ? v[VR] : 0.0, DL == 4 ? v[2 * VR] : 0.0, 0.0};
    FwdRows<DL, FR, VR> A, B;
    A.load(fl, v);
    for (int r = 0; r < nrp; r += 8) {
        B.load(fl + 4 * FR * DL, v + 4 * VR);
        __builtin_amdgcn_sched_barrier(0);
        fwd_step<DL>(A.a, s, v);
        fwd_step<DL>(A.b, s, v + VR);
        fwd_step<DL>(A.c, s, v + 2 * VR);
        fwd_step<DL>(A.d, s, v + 3 * VR);
        // past the last row: the rows after the image and the vector's padding,
        // loaded and not used
        A.load(fl + 8 * FR * DL, v + 8 * VR);
        __builtin_amdgcn_sched_barrier(0);
        fwd_step<DL>(B.a, s, v + 4 * VR);
        fwd_step<DL>(B.b, s, v + 5 * VR);
        fwd_step<DL>(B.c, s, v + 6 * VR);
        fwd_step<DL>(B.d, s, v + 7 * VR);
        fl += 8 * FR * DL;
        v += 8 * VR;
    }
}

template <int DL> struct BwdRow {
    RowFactors<DL> u;
    double d, v;
};
template <int DL, int FR, int VR> struct BwdRows {
    BwdRow<DL> a, b, c, d;
    __device__ __forceinline__ void load1(BwdRow<DL> &o, const double *bu, const double *bi, const double *v)
    {
        o.u.load(bu);
        o.d = bi[0];
        o.v = v[0];
    }
    __device__ __forceinline__ void load(const double *bu, const double *bi, const double *v)
    {
        load1(a, bu, bi, v);
        load1(b, bu - FR * DL, bi - FR, v - VR);
        load1(c, bu - 2 * FR * DL, bi - 2 * FR, v - 2 * VR);
        load1(d, bu - 3 * FR * DL, bi - 3 * FR, v - 3 * VR);
    }
};

// w0 .. w3: the solutions of the rows above, nearest first
struct BwdState {
    double w0, w1, w2, w3;
};

template <int DL>
__device__ __forceinline__ void bwd_step(const BwdRow<DL> &o, BwdState &s, double *v)
{
    double x = __builtin_fma(-o.u.template get<0>(), s.w0, o.v);
    x = __builtin_fma(-o.u.template get<1>(), s.w1, x);
    if constexpr (DL == 4) {
        x = __builtin_fma(-o.u.template get<2>(), s.w2, x);
        x = __builtin_fma(-o.u.template get<3>(), s.w3, x);
    }
    x *= o.d;
    s.w3 = s.w2;
    s.w2 = s.w1;
    s.w1 = s.w0;
    s.w0 = x;
    v[0] = x;
}

template <int DL, int FR, int VR>
__device__ __forceinline__ void chain_backward(const double *bu, const double *bi, double *v, int nrp)
{
    BwdState s{0.0, 0.0, 0.0, 0.0};
    bu += (nrp - 1) * FR * DL;
    bi += (nrp - 1) * FR;
    v += (nrp - 1) * VR;
    BwdRows<DL, FR, VR> A, B;
    A.load(bu, bi, v);
    for (int r = nrp; r > 0; r -= 8) {
        B.load(bu - 4 * FR * DL, bi - 4 * FR, v - 4 * VR);
        __builtin_amdgcn_sched_barrier(0);
        bwd_step<DL>(A.a, s, v);
        bwd_step<DL>(A.b, s, v - VR);
        bwd_step<DL>(A.c, s, v - 2 * VR);
        bwd_step<DL>(A.d, s, v - 3 * VR);
        if (r > 8) A.load(bu - 8 * FR * DL, bi - 8 * FR, v - 8 * VR);
        __builtin_amdgcn_sched_barrier(0);
        bwd_step<DL>(B.a, s, v - 4 * VR);
        bwd_step<DL>(B.b, s, v - 5 * VR);
        bwd_step<DL>(B.c, s, v - 6 * VR);
        bwd_step<DL>(B.d, s, v - 7 * VR);
        bu -= 8 * FR * DL;
        bi -= 8 * FR;
        v -= 8 * VR;
    }
}

// 16 bytes of an image (a plain vector: arrays of double2 copied whole stay in
// scratch memory)
typedef double v2d __attribute__((ext_vector_type(2)));

struct ColumnOf {
    int z, x;
    bool valid, chain;
};

__device__ __forceinline__ ColumnOf column_of(const SolveArgs &a, int col)
{
    ColumnOf c;
    c.valid = col < a.Nz * a.Mx;
    c.z = c.valid ? col / a.Mx : 0;
    c.x = c.valid ? col - c.z * a.Mx : 0;
    c.chain = c.valid && c.z != a.Nz / 2 && !(c.z == 0 && c.x == 0);
    return c;
}

constexpr int SOLVE_THREADS = 256, SOLVE_WORKERS = 192;
constexpr int SOLVE_VR_MAX = 4;
// zero rows before a vector (the operator's reach) and after it (that, and the
// forward sweep's read ahead)
constexpr int SOLVE_LEAD = 4, SOLVE_TAIL = 12;

// The wave that runs the chains: the one whose SIMD equals the block's workgroup
// slot on the CU (mod 4), so that the blocks resident on one CU run their chains
// on different SIMDs (wave 0 when no wave matches).
__device__ __forceinline__ int pick_chain_wave()
{
    __shared__ int chain_wave[1];
    if (threadIdx.x == 0) chain_wave[0] = 0;
    __syncthreads();
    // HW_ID: SIMD in bits 5:4, workgroup slot in bits 19:16
    const unsigned hw = __builtin_amdgcn_s_getreg(4 | (0 << 6) | (31 << 11));
    if ((threadIdx.x & 63) == 0 && ((hw >> 4) & 3) == ((hw >> 16) & 3)) chain_wave[0] = threadIdx.x >> 6;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(chain_wave[0]);
}

// One (field, parity) of SBT consecutive columns, for the members m0 ..
// m0 + nmb - 1 (nmb <= MB).  lds: the factor image (L, then U and the inverse
// pivots), then per member SOLVE_LEAD + nrp + SOLVE_TAIL vector rows of SBT
// complex values.  Worker w owns column w % SBT and the rows w / SBT + t RSTEP,
// t < VR.
template <int DL, int SBT, int VR, int MB>
__device__ __forceinline__ void solve_block(const SolveArgs &a, int var, int par, int blk, int m0, int nmb,
                            int stop, cplx *C, cplx *Cs, double *lds)
{
    constexpr int RSTEP = SOLVE_WORKERS / SBT, NE = 2 * DL + 1;
    static_assert(2 * SBT * MB <= 64, "one chain lane per member, part and column");
    const int Mx = a.Mx, nR = a.dimR, nQ = a.dimQ;
    const int N = var == 0 ? nQ : nR;
    const int nr = (N - par + 1) / 2, nrp = solve_rows(N);
    const int tid = threadIdx.x;
    const int vrows = SOLVE_LEAD + nrp + SOLVE_TAIL;
    double *fl = lds, *bu = fl + nrp * DL * SBT, *bi = bu + nrp * DL * SBT;
    double2 *vec = (double2 *) (bi + nrp * SBT) + SOLVE_LEAD * SBT;     // row 0 of member 0
    const int vm = vrows * SBT;                                          // member stride
    // the factor image: mirror rows kz <-> Nz - kz share one
    int fb = blk;
    if (a.mirror) {
        const int z = blk * SBT / Mx;
        if (z > a.Nz / 2) fb = blk - (2 * z - a.Nz) * (Mx / SBT);
    }

    // L factors: every thread, in flight while the chain wave is chosen (LB and
    // UB 16-byte loads a thread cover the rows that VR slots hold, whole eights)
    constexpr int LB = DL == 4 ? (3 * VR + 1) / 2 : VR, UB = DL == 4 ? (5 * VR + 1) / 2 : (3 * VR + 1) / 2;
    static_assert(RSTEP % 8 == 0 && 2 * LB * SOLVE_THREADS >= VR * RSTEP * DL * SBT &&
                      2 * UB * SOLVE_WORKERS >= VR * RSTEP * (DL + 1) * SBT,
                  "the loads cover the image");
    const v2d *src = (const v2d *) (var == 0 ? a.La : a.Lb) + ((size_t) fb * 2 + par) * (nrp * NE * SBT / 2);
    const int nl = nrp * DL * SBT / 2, nu = nrp * (DL + 1) * SBT / 2;
    v2d lt[LB], ut[UB];
#pragma unroll
    for (int i = 0; i < LB; ++i) lt[i] = src[min(tid + i * SOLVE_THREADS, nl - 1)];
    const int cw = pick_chain_wave();
    if (stop) return;                                    // (its load is under the others')
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto store_L = [&]() {
#pragma unroll
        for (int i = 0; i < LB; ++i)
            if (tid + i * SOLVE_THREADS < nl) ((v2d *) fl)[tid + i * SOLVE_THREADS] = lt[i];
    };
    // The chain wave and the workers take separate paths with the same barriers
    // (each is uniform in its waves), so that neither holds the other's values in
    // registers.
    if (wave == cw) {
        store_L();
        // lane cl < 2 SBT nmb: member cl / (2 SBT), part (cl / SBT) % 2 (real,
        // imaginary) of column cl % SBT
        const int cl = tid & 63, mb = cl / (2 * SBT), col = cl % SBT;
        double *vd = (double *) (vec + mb * vm) + 2 * col + ((cl / SBT) & 1);
        if (a.k == 0) {
            __syncthreads();
            __syncthreads();
        }
        __syncthreads();
        if (mb < nmb) chain_forward<DL, SBT, 2 * SBT>(fl + col * DL, vd, nrp);
        __syncthreads();
        if (mb < nmb) chain_backward<DL, SBT, 2 * SBT>(bu + col * DL, bi + col, vd, nrp);
        __syncthreads();
        return;
    }
    const int wt = tid - (wave > cw ? 64 : 0);
    const int cc = wt % SBT, rt = wt / SBT;
    const ColumnOf co = column_of(a, blk * SBT + cc);
    const double kx = a.Kx[co.x], kz = a.Kz[co.z], k2 = __builtin_fma(kz, kz, kx * kx);
    const size_t cbase = (((size_t) co.z * 2 + var) * nR + par) * Mx + co.x;   // C row par
    const size_t fbase = ((size_t) co.z * N + par) * Mx + co.x;                 // F row par
    const size_t rs = (size_t) 2 * Mx;                                          // next chain row
    // the members' arrays (member m0 + mb; the last one again past the group)
    auto of = [&](int mb) { return (size_t) (m0 + min(mb, nmb - 1)); };
    auto Cm = [&](int mb) { return C + of(mb) * a.ms_c; };
    auto Csm = [&](int mb) { return Cs + of(mb) * a.ms_cs; };
    auto Fm = [&](int mb) { return var == 0 ? a.Fa + of(mb) * a.ms_fa : a.Fb + of(mb) * a.ms_fb; };
    auto F2m = [&](int mb) { return var == 0 ? a.Fa2 + of(mb) * a.ms_fa2 : a.Fb2 + of(mb) * a.ms_fb2; };

    double2 cv[MB][VR], fv[MB][VR];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int t = 0; t < VR; ++t) {
            const int r = max(min(rt + t * RSTEP, nr - 1), 0);
            cv[mb][t] = Cm(mb)[cbase + r * rs];
            fv[mb][t] = Fm(mb)[fbase + r * rs];
        }
    // U factors and pivots, stored after the barrier
#pragma unroll
    for (int i = 0; i < UB; ++i) ut[i] = src[nl + min(wt + i * SOLVE_WORKERS, nu - 1)];
    store_L();
    // right-hand sides (at stage 0 the state itself first, for the explicit
    // operator), zero outside the chain and its column set
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb >= nmb) break;
        double2 *vv = vec + mb * vm + cc;
#pragma unroll
        for (int t = 0; t < VR; ++t) {
            const int r = rt + t * RSTEP;
            if (r >= nr) continue;
            double2 v = cv[mb][t];
            if (a.k != 0) {
                v.x = __builtin_fma(a.dtc, fv[mb][t].x, v.x);
                v.y = __builtin_fma(a.dtc, fv[mb][t].y, v.y);
                if (a.Src) {
                    const double2 s = a.Src[of(mb) * a.ms_src + cbase + r * rs];
                    v.x += s.x;
                    v.y += s.y;
                }
            }
            vv[r * SBT] = co.chain ? v : make_double2(0.0, 0.0);
        }
        const int npad = vrows - nr;
        for (int p = rt; p < npad; p += RSTEP)
            vv[(p < SOLVE_LEAD ? p - SOLVE_LEAD : nr + p - SOLVE_LEAD) * SBT] = make_double2(0.0, 0.0);
    }
    if (a.k == 0) {
        // E C + dt c_0 F with the stage-0 explicit operator, its entries formed
        // once for the members
        __syncthreads();
        double2 acc[MB][VR];
#pragma unroll
        for (int t = 0; t < VR; ++t) {
            const int r = max(min(rt + t * RSTEP, nr - 1), 0);
            double e[NE] = {};
            if (nr > 0) op_row<DL>(a, par + 2 * r, k2, a.ce0[var], e);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const double2 *vv = vec + min(mb, nmb - 1) * vm + r * SBT + cc;
                double2 s = make_double2(0.0, 0.0);
#pragma unroll
                for (int m = -DL; m <= DL; ++m) {
                    const double2 y = vv[m * SBT];
                    s.x = __builtin_fma(e[DL + m], y.x, s.x);
                    s.y = __builtin_fma(e[DL + m], y.y, s.y);
                }
                s.x = __builtin_fma(a.dtc, fv[mb][t].x, s.x);
                s.y = __builtin_fma(a.dtc, fv[mb][t].y, s.y);
                if (a.Src) {
                    const double2 q = a.Src[of(mb) * a.ms_src + cbase + r * rs];
                    s.x += q.x;
                    s.y += q.y;
                }
                acc[mb][t] = s;
            }
            __builtin_amdgcn_sched_barrier(0);       // one row's bands at a time
        }
        __syncthreads();
        if (co.chain) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int t = 0; t < VR; ++t)
                    if (mb < nmb && rt + t * RSTEP < nr) vec[mb * vm + (rt + t * RSTEP) * SBT + cc] = acc[mb][t];
        }
    }
    __syncthreads();
    double2 f2[MB][VR];
    double en[VR][NE];
    v2d *dst = (v2d *) bu;
#pragma unroll
    for (int i = 0; i < UB; ++i)
        if (wt + i * SOLVE_WORKERS < nu) dst[wt + i * SOLVE_WORKERS] = ut[i];
    if (a.has_next && nr > 0) {
#pragma unroll
        for (int t = 0; t < VR; ++t) {
            const int r = max(min(rt + t * RSTEP, nr - 1), 0);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) f2[mb][t] = F2m(mb)[fbase + r * rs];
            op_row<DL>(a, par + 2 * r, k2, a.cn[var], en[t]);
            __builtin_amdgcn_sched_barrier(0);       // one row's bands at a time
        }
    }
    __syncthreads();
    __syncthreads();
    // the solutions and the next stage's right-hand sides
    if (co.chain) {
#pragma unroll
        for (int t = 0; t < VR; ++t) {
            const int r = rt + t * RSTEP;
            if (r >= nr) continue;
            const size_t gi = cbase + r * rs;
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                if (mb >= nmb) continue;
                const double2 *vv = vec + mb * vm + r * SBT + cc;
                const double2 sol = vv[0];
                Csm(mb)[gi] = sol;
                double2 s = sol;
                if (a.has_next) {
                    s = make_double2(0.0, 0.0);
#pragma unroll
                    for (int m = -DL; m <= DL; ++m) {
                        const double2 y = vv[m * SBT];
                        s.x = __builtin_fma(en[t][DL + m], y.x, s.x);
                        s.y = __builtin_fma(en[t][DL + m], y.y, s.y);
                    }
                    s.x = __builtin_fma(a.dtd, f2[mb][t].x, s.x);
                    s.y = __builtin_fma(a.dtd, f2[mb][t].y, s.y);
                }
                Cm(mb)[gi] = s;
            }
        }
    }
    // rows of v beyond dimQ are carried unchanged; the Nyquist row is zeroed
    const int nrest = (nR - par + 1) / 2;
    if (!co.valid || (co.z == 0 && co.x == 0)) return;
    for (int mb = 0; mb < nmb; ++mb)
        for (int r = rt; r < nrest; r += RSTEP) {
            const size_t gi = cbase + r * rs;
            if (co.z == a.Nz / 2)
                Cm(mb)[gi] = make_double2(0.0, 0.0);
            else if (var == 0 && par + 2 * r >= nQ)
                Csm(mb)[gi] = Cm(mb)[gi];
        }
}

// Sum of red[0 .. 255] by halving (128, 64, ..., 1), the same order in every
// call; every thread gets it.
__device__ __forceinline__ double halving_sum(double v, double *red)
{
    const int tid = threadIdx.x;
    __syncthreads();
    red[tid] = v;
    __syncthreads();
    if (tid < 64) {
        double s = (red[tid] + red[tid + 128]) + (red[tid + 64] + red[tid + 192]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o);
        if (tid == 0) red[0] = s;
    }
    __syncthreads();
    return red[0];
}

// The mean mode of the members m0 .. m0 + nmb - 1: alpha (streamwise mean) and
// beta (spanwise mean) columns as the two columns of one chain image.  lds: the
// image ([parity]: L, U, inverse pivots), then per member and parity the padded
// rows of (alpha, beta), then 256 partial sums.  Rows per thread:
// i = tid + 256 t, t < MEAN_ROWS (dimR <= 512).
constexpr int MEAN_ROWS = 2;
__device__ __forceinline__ void solve_mean(const SolveArgs &a, int m0, int nmb, cplx *C, cplx *Cs, double *lds)
{
    constexpr int T = SOLVE_THREADS;
    const int nR = a.dimR, Mx = a.Mx, tid = threadIdx.x;
    const int nrp = solve_rows(nR), img = nrp * 5, vrows = SOLVE_LEAD + nrp + SOLVE_TAIL;
    double2 *vec = (double2 *) (lds + 2 * img);
    const int pv = vrows * 2, mv = 2 * pv;                 // parity and member strides
    double *red = (double *) (vec + nmb * mv);
    // row i of member mb: (alpha, beta)
    auto row = [&](int mb, int i) { return vec + mb * mv + (i & 1) * pv + (SOLVE_LEAD + (i >> 1)) * 2; };
    for (int e = tid; e < 2 * img; e += T) lds[e] = a.Lm[e];
    for (int e = tid; e < nmb * mv; e += T) vec[e] = make_double2(0.0, 0.0);
    __syncthreads();
    // Rs + coef Rps of the rows' two columns
    auto mult = [&](int mb, int i, double coef, double2 &al, double2 &be) {
        double e[5];
        const double *rs = a.Rs + i * 5, *rp = a.Rps + i * 5;
#pragma unroll
        for (int j = 0; j < 5; ++j) e[j] = __builtin_fma(coef, rp[j], rs[j]);
        const double2 *v = row(mb, i);
        al = be = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = -2; m <= 2; ++m) {
            const double2 x = v[2 * m], y = v[2 * m + 1];
            al.x = __builtin_fma(e[m + 2], x.x, al.x);
            al.y = __builtin_fma(e[m + 2], x.y, al.y);
            be.x = __builtin_fma(e[m + 2], y.x, be.x);
            be.y = __builtin_fma(e[m + 2], y.y, be.y);
        }
    };
    for (int mb = 0; mb < nmb; ++mb) {
        const size_t m = m0 + mb;
        const cplx *Ca = C + m * a.ms_c, *Cb = Ca + (size_t) nR * Mx;
        const cplx *Fm = a.Fb + m * a.ms_fb, *Sm = a.Src ? a.Src + m * a.ms_src : nullptr;
        double2 fr[MEAN_ROWS], al[MEAN_ROWS], be[MEAN_ROWS];
#pragma unroll
        for (int t = 0; t < MEAN_ROWS; ++t) {
            const int i = tid + T * t;
            if (i >= nR) continue;
            al[t] = Ca[(size_t) i * Mx];
            be[t] = Cb[(size_t) i * Mx];
            fr[t] = Fm[(size_t) i * Mx];
        }
        if (a.k == 0) {
#pragma unroll
            for (int t = 0; t < MEAN_ROWS; ++t) {
                const int i = tid + T * t;
                if (i >= nR) continue;
                row(mb, i)[0] = al[t];
                row(mb, i)[1] = be[t];
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < MEAN_ROWS; ++t) {
                const int i = tid + T * t;
                if (i < nR) mult(mb, i, a.ce0[1], al[t], be[t]);
            }
            __syncthreads();
        }
        double q = 0.0;
#pragma unroll
        for (int t = 0; t < MEAN_ROWS; ++t) {
            const int i = tid + T * t;
            if (i >= nR) continue;
            al[t].x = __builtin_fma(a.dtc, fr[t].x, al[t].x);
            be[t].x = __builtin_fma(a.dtc, fr[t].y, be[t].x);
            if (Sm) {
                const double2 sa = Sm[(size_t) i * Mx], sb = Sm[(size_t) (nR + i) * Mx];
                al[t].x += sa.x;
                al[t].y += sa.y;
                be[t].x += sb.x;
                be[t].y += sb.y;
            }
            if (a.exact_mean) q = __builtin_fma(a.add_mass[i], al[t].x, q);
        }
        double h = 0.0;
        // the transpose of the flux correction on the right-hand side
        if (a.exact_mean && a.k < 2) h = 0.5 * halving_sum(q, red);
#pragma unroll
        for (int t = 0; t < MEAN_ROWS; ++t) {
            const int i = tid + T * t;
            if (i >= nR) continue;
            if (a.exact_mean && a.k < 2) al[t].x = __builtin_fma(-h, a.rowsum[i], al[t].x);
            row(mb, i)[0] = al[t];
            row(mb, i)[1] = be[t];
        }
    }
    __syncthreads();
    // eight chains a member: parity, column, part
    if (tid < 8 * nmb) {
        const int mb = tid >> 3, p = (tid >> 2) & 1;
        double *v = (double *) row(mb, p) + (tid & 3);
        const double *f = lds + p * img;
        chain_forward<2, 1, 4>(f, v, nrp);
        chain_backward<2, 1, 4>(f + nrp * 2, f + nrp * 4, v, nrp);
    }
    __syncthreads();
    for (int mb = 0; mb < nmb; ++mb) {
        const size_t m = m0 + mb;
        cplx *Ca = C + m * a.ms_c, *Cb = Ca + (size_t) nR * Mx, *Sa = Cs + m * a.ms_cs;
        const cplx *Fm2 = a.Fb2 + m * a.ms_fb2;
        double p = 0.0;
        for (int i = tid; i < nR; i += T) p = __builtin_fma(a.rowsum[i], row(mb, i)[0].x, p);
        const double target = (a.alt_mask >> m) & 1u ? a.target_alt : a.target;
        const double flux_t = target - halving_sum(p, red);
#pragma unroll
        for (int t = 0; t < MEAN_ROWS; ++t) {
            const int i = tid + T * t;
            if (i >= nR) continue;
            double2 v = row(mb, i)[0];
            if (!a.exact_mean) {
                v.x = __builtin_fma(flux_t * a.add[i], 0.5, v.x);
                row(mb, i)[0] = v;
            }
            Sa[(size_t) i * Mx] = v;
            Sa[(size_t) (nR + i) * Mx] = row(mb, i)[1];
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MEAN_ROWS; ++t) {
            const int i = tid + T * t;
            if (i >= nR) continue;
            double2 xa = row(mb, i)[0], xb = row(mb, i)[1];
            if (a.has_next) {
                const double2 f = Fm2[(size_t) i * Mx];
                mult(mb, i, a.cn[1], xa, xb);
                xa.x = __builtin_fma(a.dtd, f.x, xa.x);
                xb.x = __builtin_fma(a.dtd, f.y, xb.x);
            }
            Ca[(size_t) i * Mx] = xa;
            Cb[(size_t) i * Mx] = xb;
        }
    }
}

// The Nyquist row kz = Nz/2 carries no data: a block whose columns all lie
// in it only clears its C rows.
template <int SBT>
__device__ void nyquist_clear(const SolveArgs &a, int var, int par, int blk, cplx *C)
{
    const int nR = a.dimR, Mx = a.Mx, nrest = (nR - par + 1) / 2;
    const int x0 = blk * SBT - (a.Nz / 2) * Mx;
    const size_t base = (((size_t) (a.Nz / 2) * 2 + var) * nR + par) * Mx + x0;
    for (int e = threadIdx.x; e < nrest * SBT; e += SOLVE_THREADS)
        C[base + (size_t) (e / SBT) * 2 * Mx + e % SBT] = make_double2(0.0, 0.0);
}

// Tiles (column block, field and parity, group of MB members), groups fastest and
// XCD-aware: the groups of a column block read the same factor image from one L2.
// With Mx % SBT == 0 the blocks of the Nyquist row hold no chains; they come
// first, and the first of them with field 0 and parity 0 runs the mean mode (so
// the grid is exactly the column blocks, and the long mean chains start early);
// otherwise the extra column block nblk does.  The registers are bounded for the
// blocks that a CU's LDS holds: 36 KB a block at 48 rows, one member; 44 KB with
// two, 47 KB at 64 rows; 57 KB and more beyond.
template <int SBT, int VR, int MB>
__global__ __launch_bounds__(SOLVE_THREADS, VR <= 2 && MB == 1 ? 4 : VR * MB <= 4 && VR <= 3 && MB <= 2 ? 3 : 2)
void k_solve(SolveArgs a, cplx *C, cplx *Cs)
{
    extern __shared__ __align__(16) double lds_solve[];
    const int stop = *a.abort_flag;
    const int ncol = a.nblk + (a.nyq_mean ? 0 : 1);
    const int tile = xcd_tile(ncol * 4 * a.ngrp);
    if (tile < 0) return;
    const int cv = tile / a.ngrp, m0 = (tile - cv * a.ngrp) * MB, nmb = min(MB, a.nm - m0);
    const int var = (cv & 3) >> 1, par = cv & 1, nyq = (a.Nz / 2) * a.Mx / SBT;
    int blk = cv >> 2;
    if (a.nyq_mean) {
        const int per = a.Mx / SBT;                        // blocks of a kz row
        blk = blk < per ? nyq + blk : blk < nyq + per ? blk - per : blk;
    }
    const bool clear = a.nyq_mean && blk * SBT / a.Mx == a.Nz / 2;
    if ((clear || blk == a.nblk) && stop) return;
    if (clear)
        for (int mb = 0; mb < nmb; ++mb)
            nyquist_clear<SBT>(a, var, par, blk, C + (m0 + mb) * a.ms_c);
    if (clear || blk == a.nblk) {
        if ((cv & 3) == 0 && (blk == nyq || !clear)) solve_mean(a, m0, nmb, C, Cs, lds_solve);
        return;
    }
    if (var == 0)
        solve_block<4, SBT, VR, MB>(a, 0, par, blk, m0, nmb, stop, C, Cs, lds_solve);
    else
        solve_block<2, SBT, VR, MB>(a, 1, par, blk, m0, nmb, stop, C, Cs, lds_solve);
}

// coefficient tables for the stages
static const double FA_[3] = {1. / 3., -1. / 2, 1. / 3.};
static const double FC_[3] = {1. / 2, 1. / 3., 1.};
static const double FD_[3] = {0., -1. / 6, -2. / 3};
static const double BA_[3] = {1. / 3., -1. / 2, 1. / 3.};
static const double BC_[3] = {1., 1. / 3., 1. / 2.};
static const double BD_[3] = {0., -2. / 3, -1. / 6};

size_t solve_lds_bytes(int dimR, int sbt, int mb)
{
    const size_t nrp = solve_rows(dimR), vrows = SOLVE_LEAD + nrp + SOLVE_TAIL;
    const size_t blk = nrp * sbt * 9 * 8 + mb * vrows * sbt * 16;
    const size_t mean = 2 * nrp * 5 * 8 + mb * 2 * vrows * 2 * 16 + SOLVE_THREADS * 8;
    return blk > mean ? blk : mean;
}

// Row slots of a worker: the chains' rows over the workers' rows of a pass
static int solve_slots(int dimR, int sbt)
{
    const int step = SOLVE_WORKERS / sbt;
    return ((dimR + 1) / 2 + step - 1) / step;
}

// Columns per solve block: 8, 4 or 2 (an even count keeps every block's
// factor image a whole number of 16-byte pairs), within 64 KB of LDS and with
// a row slot for every chain row; 0 when none fits.
int solve_columns_per_block(int dimR)
{
    for (int sbt = 8; sbt >= 2; sbt >>= 1)
        if (solve_lds_bytes(dimR, sbt, 1) <= 64 * 1024 && solve_slots(dimR, sbt) <= SOLVE_VR_MAX)
            return sbt;
    return 0;
}

// Members per solve block (1, 2 or 4) of a run of nrun members: the tuning's choice
// when set, else 2 (32 members at 64x97x64: 232 us a launch, 262 with one: the second
// member's vectors come while the first's chain runs, and a third would take the LDS
// of a block) while a worker holds no more than six rows of them in registers; fewer
// when the run has fewer members, when two blocks would not fit a CU's LDS, or when a
// worker's rows would not fit its registers (four members of more than three rows).
int solve_members(int dimR, int sbt, int nrun, int tuned)
{
    const int slots = solve_slots(dimR, sbt);
    int mb = tuned > 0 ? tuned : 2;
    while (mb > 1 && (mb > nrun || (tuned > 0 ? mb == 4 && slots > 3 : mb * slots > 6) ||
                      2 * solve_lds_bytes(dimR, sbt, mb) > 160 * 1024))
        mb /= 2;
    return mb;
}

typedef void (*SolveKernel)(SolveArgs, cplx *, cplx *);

template <int SBT, int VR>
static SolveKernel solve_kernel_mb(int mb)
{
    if constexpr (VR <= 3)
        if (mb == 4) return k_solve<SBT, VR, 4>;
    return mb == 2 ? k_solve<SBT, VR, 2> : k_solve<SBT, VR, 1>;
}

// the shapes that solve_columns_per_block leads to: one row slot only with 8
// columns, four only with 8 or 4 (256 rows at most)
template <int SBT>
static SolveKernel solve_kernel(int slots, int mb)
{
    if constexpr (SBT == 8)
        if (slots == 1) return solve_kernel_mb<SBT, 1>(mb);
    if constexpr (SBT > 2)
        if (slots == 4) return solve_kernel_mb<SBT, 4>(mb);
    return slots == 3 ? solve_kernel_mb<SBT, 3>(mb) : solve_kernel_mb<SBT, 2>(mb);
}

void launch_solve(Context &c, cplx *Ccarry, cplx *Csol, int k, int adj, const cplx *Fa2,
                  const cplx *Fb2, double target, double target_alt, unsigned alt_mask,
                  const cplx *Src, int exact_mean)
{
    const Dims &d = c.d;
    const double *A = adj ? BA_ : FA_, *Cc = adj ? BC_ : FC_, *D = adj ? BD_ : FD_;
    SolveArgs a;
    a.Qs = c.dQs; a.Qps = c.dQps; a.Qpps = c.dQpps; a.Rs = c.dRs; a.Rps = c.dRps;
    a.Kx = c.dKx; a.Kz = c.dKz;
    a.La = c.dLa[adj][k];
    a.Lb = c.dLb[adj][k];
    a.Lm = c.dLm[adj][k];
    a.add = c.dAdd[adj][k];
    a.rowsum = c.dRowsum;
    a.Fa = c.Fa; a.Fb = c.Fb;
    a.Fa2 = Fa2; a.Fb2 = Fb2;
    a.Nz = d.Nz; a.Mx = d.Mx; a.dimR = d.dimR; a.dimQ = d.dimQ; a.k = k;
    a.has_next = k != 2;
    a.dtc = d.dt * Cc[k];
    a.dtd = k != 2 ? d.dt * D[k + 1] : 0.0;
    // v: -(K2 Qs + Qps) + re a dt (K2^2 Qs + 2 K2 Qps + Qpps);
    // omega_y: Rs - re a dt (Rps + K2 Rs)  (channel/project.c:55-71,140-151)
    a.ce0[0] = d.re * A[0] * d.dt;
    a.ce0[1] = -(d.re * A[0] * d.dt);
    a.cn[0] = k != 2 ? d.re * A[k + 1] * d.dt : 0.0;
    a.cn[1] = k != 2 ? -(d.re * A[k + 1] * d.dt) : 0.0;
    a.target = target;
    a.target_alt = target_alt;
    a.alt_mask = alt_mask;
    a.Src = Src;
    a.ms_src = mstride(c, Src);
    a.exact_mean = adj && exact_mean;
    a.add_mass = c.dAdd[0][k];
    a.abort_flag = c.abort_flag;
    a.ms_c = mstride(c, Ccarry);
    a.ms_cs = mstride(c, Csol);
    a.ms_fa = mstride(c, a.Fa);
    a.ms_fb = mstride(c, a.Fb);
    a.ms_fa2 = mstride(c, Fa2);
    a.ms_fb2 = mstride(c, Fb2);
    // RHS in, projections in (the next stage's only when they are other
    // arrays: the primal's are the same), solution and next right-hand side
    // out, and the factor images in (each stored image once: mirror rows
    // share one)
    const bool f2 = k != 2 && Fa2 != c.Fa;
    const double fcols = (double) (c.factor_mirror ? d.Nz / 2 + 1 : d.Nz) * d.Mx;
    double bytes = c.nrun * (double) (d.Nz - 1) * d.Mx *
                       (16.0 * (2.0 * d.dimR) * 3.0 + 16.0 * (d.dimQ + d.dimR) * (f2 ? 2.0 : 1.0)) +
                   fcols * 8.0 * (9.0 * d.dimQ + 5.0 * d.dimR);
    const int sbt = c.sbt;
    const int ncol = d.Nz * d.Mx;
    const int mb = solve_members(d.dimR, sbt, c.nrun, tuning().solve_mb);
    const size_t lds = solve_lds_bytes(d.dimR, sbt, mb);
    a.nm = c.nrun;
    a.ngrp = (c.nrun + mb - 1) / mb;
    a.nblk = (ncol + sbt - 1) / sbt;
    a.mirror = c.factor_mirror;
    a.nyq_mean = d.Mx % sbt == 0;
    const dim3 grid(xcd_grid((a.nblk + (a.nyq_mean ? 0 : 1)) * 4 * a.ngrp));
    const hipStream_t st = c.stream;
    const int slots = solve_slots(d.dimR, sbt);
    const SolveKernel kern = sbt == 8   ? solve_kernel<8>(slots, mb)
                             : sbt == 4 ? solve_kernel<4>(slots, mb)
                                        : solve_kernel<2>(slots, mb);
    if (lds > 64 * 1024)
        (void) hipFuncSetAttribute((const void *) kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int) lds);
    auto go = [=]() {
        hipLaunchKernelGGL(kern, grid, dim3(SOLVE_THREADS), lds, st, a, Ccarry, Csol);
    };
    prof_begin(c, st, 6, bytes);
    go();
    prof_end(c, st, 6, go);
}

// ------------------------------------------------------------ vectors
// Inner products of ddt_project (channel/channel.c:704-780) straight from the
// coefficients.  The reference forms <f, g> = sum_y W_y sum_{x,z} f g over the
// velocities of f and g rebuilt on the dealiased Px x Pz x qpts grid.  Those
// sums are exact integrals: Parseval in x and z (the fields are band-limited
// below the padded grid's Nyquist bins), and in y the Gauss rule with qpts
// points integrates the products of the rebuilt fields exactly (degree at
// most 2 dimQ + 6 < 2 qpts).  With u = (i kx v' - i kz w_y)/k2 and
// w = (i kz v' + i kx w_y)/k2, u conj(u~) + w conj(w~) = (v' conj(v~') +
// w_y conj(w~_y))/k2, so per column (kz, kx) != (0, 0)
//     <f, g>_col = c Re[ a_f^H (Qs + Qps/k2) a_g + b_f^H (Rs/k2) b_g ]
// with the Gauss-rule Gram bands Qs = sum W Q Q, Qps = sum W Q' Q',
// Rs = sum W R R of the setup, alpha rows a < dimQ, beta rows b < dimR,
// c = 2 for kx > 0 (the conjugate column) and c = 1 at kx = 0, where the
// coefficients are replaced by their Hermitian part (c(kz) + conj c(-kz))/2,
// the only part the complex-to-real x transform sees.  The mean column holds
// the u and w profiles in the R basis: Re a_f^T Rs Re a_g + Re b_f^T Rs Re b_g
// (the Hermitian part of column (0,0) is its real part).  Row Nz/2 is not
// transformed and counts nothing.  The sums differ from the grid sums only
// in rounding.  num = <dudt, V>, den = <dudt, dudt> (times Px Pz, the grid's
// Parseval factor) with dudt = s (P - M) formed on load.
//
// Block: kz row z and ncol columns; dudt and V of the block's columns in
// LDS ([var][row][column]), then one (var, row, column) item per thread and
// pass; one partial pair per block.
// Sums of a and b over the 256 threads of a block, in the same order in every
// block: lane exchanges within each wave (distances 32 .. 1; both partners
// add the same two values, so every lane holds the same bits), then the four
// wave sums in wave order.  Every thread gets both sums.  sh: 8 doubles.
__device__ __forceinline__ double2 block_sum2_256(double a, double b, double *sh)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[threadIdx.x >> 6] = a;
        sh[4 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    return make_double2((sh[0] + sh[1]) + (sh[2] + sh[3]), (sh[4] + sh[5]) + (sh[6] + sh[7]));
}

constexpr int DDT_IT = 4;        // items per thread of k_ddt_gram's load phase
constexpr int DDT_BT = 12;       // Gram band values per thread loaded in one batch

__global__ __launch_bounds__(256) void k_ddt_gram(const cplx *P, const cplx *M, const cplx *V,
                                                  double s, const double *Qs, const double *Qps,
                                                  const double *Rs, const double *Kx,
                                                  const double *Kz, int Nz, int Mx, int dimR,
                                                  int dimQ, int ncol, double scale, double *part,
                                                  const int *abort_flag, size_t ms_p, size_t ms_m,
                                                  size_t ms_v, const cplx *P0, const cplx *M0)
{
    extern __shared__ double2 sh_ddt[];
    __shared__ double rs[8];
    // member blockIdx.y: its partial pairs follow those of the members before;
    // P0, M0 (when given) replace member 0's pair of states
    P += blockIdx.y * ms_p;
    M += blockIdx.y * ms_m;
    if (blockIdx.y == 0 && P0) {
        P = P0;
        M = M0;
    }
    V += blockIdx.y * ms_v;
    part += (size_t) blockIdx.y * 2 * gridDim.x;
    const int nxb = (Mx + ncol - 1) / ncol;
    const int z = blockIdx.x / nxb, x0 = (blockIdx.x - z * nxb) * ncol;
    const bool live = !*abort_flag && z != Nz / 2;
    const int nit = 2 * dimR * ncol;       // at most 256 DDT_IT (host)
    double2 *sd = sh_ddt, *sv = sh_ddt + nit;
    double2 *smd = sv + nit, *smv = smd + 2 * dimR;   // kx = 0 column of row -kz
    // the Gram bands: Qs, Qps [dimQ][9], Rs [dimR][5]
    double *bq = (double *) (smv + 2 * dimR), *bqp = bq + 9 * dimQ, *br = bqp + 9 * dimQ;
    const bool mirror = live && x0 == 0;
    if (live) {
        // every load of the thread in flight before the first store: the
        // block's items, the mirror column, the Gram bands
        double2 rp[DDT_IT], rm[DDT_IT], rv[DDT_IT], qp, qm, qv;
#pragma unroll
        for (int t = 0; t < DDT_IT; ++t) {
            const int e = threadIdx.x + t * 256;
            const int col = e % ncol, j = (e / ncol) % dimR, var = e / (ncol * dimR);
            const int x = min(x0 + col, Mx - 1);
            const size_t o = (((size_t) z * 2 + min(var, 1)) * dimR + j) * Mx + x;
            if (e < nit) {
                rp[t] = P[o];
                rm[t] = M[o];
                rv[t] = V[o];
            }
        }
        const bool mload = mirror && (int) threadIdx.x < 2 * dimR;
        if (mload) {
            const int zm = z == 0 ? 0 : Nz - z;
            const int j = threadIdx.x % dimR, var = threadIdx.x / dimR;
            const size_t om = (((size_t) zm * 2 + var) * dimR + j) * Mx;
            qp = P[om];
            qm = M[om];
            qv = V[om];
        }
        const int nbq = 9 * dimQ, nbt = 18 * dimQ + 5 * dimR;
        auto band = [&](int i) {
            return i < nbq ? Qs[i] : i < 2 * nbq ? Qps[min(i - nbq, nbq - 1)]
                                                 : Rs[min(max(i - 2 * nbq, 0), 5 * dimR - 1)];
        };
        double tb[DDT_BT];
#pragma unroll
        for (int u = 0; u < DDT_BT; ++u) {
            const int i = threadIdx.x + u * 256;
            if (i < nbt) tb[u] = band(i);
        }
#pragma unroll
        for (int u = 0; u < DDT_BT; ++u) {
            const int i = threadIdx.x + u * 256;
            if (i < nbt) bq[i] = tb[u];
        }
        for (int i = threadIdx.x + DDT_BT * 256; i < nbt; i += 256) bq[i] = band(i);
#pragma unroll
        for (int t = 0; t < DDT_IT; ++t) {
            const int e = threadIdx.x + t * 256;
            if (e >= nit) continue;
            const int col = e % ncol;
            const bool in = x0 + col < Mx;
            sd[e] = in ? make_double2(s * (rp[t].x - rm[t].x), s * (rp[t].y - rm[t].y))
                       : make_double2(0.0, 0.0);
            sv[e] = in ? rv[t] : make_double2(0.0, 0.0);
        }
        if (mload) {
            smd[threadIdx.x] = make_double2(s * (qp.x - qm.x), s * (qp.y - qm.y));
            smv[threadIdx.x] = qv;
        }
        if (mirror) {
            // rows beyond the first 256 (var, j) pairs (dimR > 128)
            const int zm = z == 0 ? 0 : Nz - z;
            for (int q = threadIdx.x + 256; q < 2 * dimR; q += 256) {
                const int j = q % dimR, var = q / dimR;
                const size_t om = (((size_t) zm * 2 + var) * dimR + j) * Mx;
                const cplx pm = P[om], mm = M[om];
                smd[q] = make_double2(s * (pm.x - mm.x), s * (pm.y - mm.y));
                smv[q] = V[om];
            }
        }
    }
    __syncthreads();
    if (mirror) {
        // Hermitian part (c(kz) + conj c(-kz)) / 2 of the kx = 0 column
        for (int q = threadIdx.x; q < 2 * dimR; q += 256) {
            const int e = q * ncol;                // (var, j) = q, column 0
            const double2 d = sd[e], v = sv[e], dm = smd[q], vm = smv[q];
            sd[e] = make_double2(0.5 * (d.x + dm.x), 0.5 * (d.y - dm.y));
            sv[e] = make_double2(0.5 * (v.x + vm.x), 0.5 * (v.y - vm.y));
        }
    }
    __syncthreads();
    double num = 0.0, den = 0.0;
    if (live) {
        const double kz = Kz[z];
        for (int e = threadIdx.x; e < nit; e += 256) {
            const int col = e % ncol, j = (e / ncol) % dimR, var = e / (ncol * dimR);
            const int x = x0 + col;
            if (x >= Mx) continue;
            const bool mean = z == 0 && x == 0;
            const bool qrow = var == 0 && !mean;             // v in the Q basis
            if (qrow && j >= dimQ) continue;
            const double kx = Kx[x], k2 = kx * kx + kz * kz;
            const double2 *dc = sd + var * dimR * ncol + col;
            const double2 *vc = sv + var * dimR * ncol + col;
            double gdx = 0.0, gdy = 0.0, gvx = 0.0, gvy = 0.0;   // (G d)_j, (G v)_j
            if (qrow) {
                const double ik2 = 1.0 / k2;
#pragma unroll
                for (int m = -4; m <= 4; ++m) {
                    const int i = j + 2 * m;
                    if (i < 0 || i >= dimQ) continue;
                    const double g = bq[j * 9 + 4 + m] + bqp[j * 9 + 4 + m] * ik2;
                    const double2 di = dc[i * ncol], vi = vc[i * ncol];
                    gdx += g * di.x;
                    gdy += g * di.y;
                    gvx += g * vi.x;
                    gvy += g * vi.y;
                }
            } else {
                const double f = mean ? 1.0 : 1.0 / k2;
#pragma unroll
                for (int m = -2; m <= 2; ++m) {
                    const int i = j + 2 * m;
                    if (i < 0 || i >= dimR) continue;
                    const double g = br[j * 5 + 2 + m] * f;
                    const double2 di = dc[i * ncol], vi = vc[i * ncol];
                    gdx += g * di.x;
                    gdy += g * di.y;
                    gvx += g * vi.x;
                    gvy += g * vi.y;
                }
            }
            const double2 dj = dc[j * ncol];
            const double w = x > 0 ? 2.0 : 1.0;
            num += w * (dj.x * gvx + dj.y * gvy);
            den += w * (dj.x * gdx + dj.y * gdy);
        }
    }
    const double2 t = block_sum2_256(num * scale, den * scale, rs);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = t.x;
        part[2 * blockIdx.x + 1] = t.y;
    }
}

// vout = vin - r dC, dC = s (P - M), with r = num / den from the nparts
// partial pairs of k_ddt_gram, summed by every block in the same order
// (strided over 256 threads, then block_sum2_256); block 0 leaves num, den, r in
// scal.  With acc, also acc -= a vout, twice when `twice` (the adjoint's
// trapezoid forcing at the end of one step and the start of the next,
// applied back to back).
// grid (blocks, members): member blockIdx.y sums its own nparts partial
// pairs and writes its scalars to scal + 8 blockIdx.y
__global__ __launch_bounds__(256) void k_ddt_apply(cplx *vout, const cplx *vin, const cplx *P,
                                                   const cplx *M, double s, const double *part,
                                                   int nparts, double *scal, size_t n, cplx *acc,
                                                   double a, int twice, size_t ms_vo, size_t ms_vi,
                                                   size_t ms_p, size_t ms_m, size_t ms_acc,
                                                   const cplx *P0, const cplx *M0)
{
    __shared__ double rs[8];
    {
        const int m = blockIdx.y;
        vout += m * ms_vo;
        vin += m * ms_vi;
        P += m * ms_p;
        M += m * ms_m;
        if (m == 0 && P0) {
            P = P0;
            M = M0;
        }
        if (acc) acc += m * ms_acc;
        part += (size_t) m * 2 * nparts;
        scal += 8 * m;
    }
    double sa = 0.0, sb = 0.0;
    for (int i = threadIdx.x; i < nparts; i += 256) {
        sa += part[2 * i];
        sb += part[2 * i + 1];
    }
    const double2 t = block_sum2_256(sa, sb, rs);
    const double r = t.x / t.y;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scal[0] = t.x;
        scal[1] = t.y;
        scal[2] = r;
    }
    for (size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x; e < n;
         e += (size_t) gridDim.x * blockDim.x) {
        const cplx p = P[e], m = M[e];
        const double dx = s * (p.x - m.x), dy = s * (p.y - m.y);
        cplx v = vin[e];
        v.x -= r * dx;
        v.y -= r * dy;
        vout[e] = v;
        if (acc) {
            cplx w = acc[e];
            w.x -= a * v.x;
            w.y -= a * v.y;
            if (twice) {
                w.x -= a * v.x;
                w.y -= a * v.y;
            }
            acc[e] = w;
        }
    }
}

// Reynolds-number sensitivity forcing of a stored state S = MC[count]
// (channel/tangent_forcing.c:10-75, channel/tangent_forcing0.c:10-44), band
// products in the order of smMult / smMult0 (channel/mvOps.c:198-237):
//   (kz,kx) != (0,0): fa = -re^2 (K2^2 Qs + 2 K2 Qps + Qpps) alpha   [Nz][dimQ][Mx]
//                     fb =  re^2 (Rps + K2 Rs) beta                   [Nz][dimR][Mx]
//   mean column:      f0 = re^2 Rps alpha(0,0), re^2 Rps beta(0,0)    [2][dimR]
// Column (0,0) of fa and fb is zero.  One thread per output element.
__global__ void k_tangent_forcing(const cplx *S, const double *Qs, const double *Qps,
                                  const double *Qpps, const double *Rs, const double *Rps,
                                  const double *Kx, const double *Kz, double re, int Nz, int Mx,
                                  int nQ, int nR, cplx *fa, cplx *fb, cplx *f0)
{
    const size_t na = (size_t) Nz * nQ * Mx, nb = (size_t) Nz * nR * Mx;
    const size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x;
    if (e >= na + nb + 2 * (size_t) nR) return;
    if (e >= na + nb) {
        const int v = (int) ((e - na - nb) / nR), i = (int) (e - na - nb) - v * nR;
        const cplx *y = S + (size_t) v * nR * Mx;                  // column (0,0) of alpha or beta
        double sr = 0.0, si = 0.0;
        for (int m = -min(2, i / 2); m <= min(2, (nR - i + 1) / 2 - 1); ++m) {
            const double a = re * re * Rps[i * 5 + 2 + m];
            sr += a * y[(size_t) (i + 2 * m) * Mx].x;
            si += a * y[(size_t) (i + 2 * m) * Mx].y;
        }
        f0[e - na - nb] = make_double2(sr, si);
        return;
    }
    const bool alpha = e < na;
    const size_t r = alpha ? e : e - na;
    const int N = alpha ? nQ : nR;
    const int x = (int) (r % Mx), i = (int) ((r / Mx) % N), z = (int) (r / ((size_t) Mx * N));
    cplx *out = alpha ? fa + r : fb + r;
    if (z == 0 && x == 0) {
        *out = make_double2(0.0, 0.0);
        return;
    }
    const double k2 = Kz[z] * Kz[z] + Kx[x] * Kx[x], s = k2 * k2;
    const cplx *y = S + ((size_t) (z * 2 + (alpha ? 0 : 1)) * nR) * Mx + x;
    double sr = 0.0, si = 0.0;
    if (alpha) {
        for (int m = -min(4, i / 2); m <= min(4, (nQ - i + 1) / 2 - 1); ++m) {
            const int b = i * 9 + 4 + m;
            const double a = -re * re * (s * Qs[b] + 2. * k2 * Qps[b] + Qpps[b]);
            sr += a * y[(size_t) (i + 2 * m) * Mx].x;
            si += a * y[(size_t) (i + 2 * m) * Mx].y;
        }
    } else {
        for (int m = -min(2, i / 2); m <= min(2, (nR - i + 1) / 2 - 1); ++m) {
            const int b = i * 5 + 2 + m;
            const double a = re * re * (Rps[b] + k2 * Rs[b]);
            sr += a * y[(size_t) (i + 2 * m) * Mx].x;
            si += a * y[(size_t) (i + 2 * m) * Mx].y;
        }
    }
    *out = make_double2(sr, si);
}

void launch_tangent_forcing(Context &c, const cplx *S, cplx *fa, cplx *fb, cplx *f0)
{
    const Dims &d = c.d;
    const size_t n = (size_t) d.Nz * (d.dimQ + d.dimR) * d.Mx + 2 * (size_t) d.dimR;
    hipLaunchKernelGGL(k_tangent_forcing, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, c.stream,
                       S, c.dQs, c.dQps, c.dQpps, c.dRs, c.dRps, c.dKx, c.dKz, d.re, d.Nz, d.Mx,
                       d.dimQ, d.dimR, fa, fb, f0);
}

// LDS bytes of a k_ddt_gram block of nc columns
static size_t ddt_gram_lds(const Dims &d, int nc)
{
    return sizeof(double2) * 4 * (size_t) d.dimR * (nc + 1) +
           sizeof(double) * (18 * (size_t) d.dimQ + 5 * (size_t) d.dimR);
}

// columns per k_ddt_gram block: 4, fewer while the block's items exceed
// 256 DDT_IT or its LDS 64 KB (grids beyond dimR = 128 with one column ask
// for more)
static int ddt_gram_cols(const Dims &d)
{
    int ncol = 4;
    while (ncol > 1 && (2 * d.dimR * ncol > 256 * DDT_IT || ddt_gram_lds(d, ncol) > 65536))
        ncol /= 2;
    return ncol;
}

int ddt_gram_blocks(const Dims &d)
{
    const int ncol = ddt_gram_cols(d);
    return d.Nz * ((d.Mx + ncol - 1) / ncol);
}

int launch_ddt_gram(Context &c, const cplx *P, const cplx *M, double s, const cplx *V)
{
    return launch_ddt_gram(c, P, M, s, V, c.dotpart, c.ndotpart, c.abort_flag);
}

int launch_ddt_gram(Context &c, const cplx *P, const cplx *M, double s, const cplx *V,
                    double *part, size_t part_cap, const int *stop, const cplx *P0,
                    const cplx *M0)
{
    const Dims &d = c.d;
    const int ncol = ddt_gram_cols(d), nb = ddt_gram_blocks(d);
    if (2 * (size_t) nb * c.nrun > part_cap) {
        last_error() = "ddt_project: partial-sum buffer too small";
        return 0;
    }
    const size_t lds = ddt_gram_lds(d, ncol);
    if (lds > 65536)
        (void) hipFuncSetAttribute((const void *) k_ddt_gram,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
    hipLaunchKernelGGL(k_ddt_gram, dim3(nb, c.nrun), dim3(256), lds, c.stream, P, M, V, s, c.dQs,
                       c.dQps, c.dRs, c.dKx, c.dKz, d.Nz, d.Mx, d.dimR, d.dimQ, ncol,
                       (double) d.Px * (double) d.Pz, part, stop, mstride(c, P), mstride(c, M),
                       mstride(c, V), P0, M0);
    return nb;
}

void launch_ddt_apply(Context &c, cplx *vout, const cplx *vin, const cplx *P, const cplx *M,
                      double s, size_t n, cplx *acc, double a, int nparts, int twice)
{
    launch_ddt_apply(c, vout, vin, P, M, s, n, acc, a, nparts, twice, c.dotpart, c.scal);
}

void launch_ddt_apply(Context &c, cplx *vout, const cplx *vin, const cplx *P, const cplx *M,
                      double s, size_t n, cplx *acc, double a, int nparts, int twice,
                      const double *part, double *scal, const cplx *P0, const cplx *M0)
{
    const int nm = c.nrun;
    hipLaunchKernelGGL(k_ddt_apply, dim3(std::max(128, 1024 / nm), nm), dim3(256), 0, c.stream,
                       vout, vin, P, M, s, part, nparts, scal, n, acc, a, twice, mstride(c, vout),
                       mstride(c, vin), mstride(c, P), mstride(c, M), acc ? mstride(c, acc) : 0,
                       P0, M0);
}

__global__ __launch_bounds__(256) void k_zero(cplx *p, size_t n)
{
    for (size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x; e < n;
         e += (size_t) gridDim.x * blockDim.x)
        p[e] = make_double2(0.0, 0.0);
}

void launch_zero(Context &c, cplx *p, size_t n)
{
    const size_t nb = std::min<size_t>(1024, (n + 255) / 256);
    if (nb) hipLaunchKernelGGL(k_zero, dim3((unsigned) nb), dim3(256), 0, c.stream, p, n);
}

}  // namespace sc
