// The x transforms and pointwise products for the lengths with a compile-time
// plan (channel/pass1.c:107-371, channel/pass2.c:128-472,
// channel/spec2phys.c:67-76): per row (Gauss point y, z row) the c2r transforms
// of the fields, two real fields packed per complex transform, the products,
// and the r2c transforms of the packed products, kept to kx < Nx/2.
// Compiled once per mode (SC_XMODE) and precision (SC_FFT_F32).
#include "fft_common.h"

namespace sc {
namespace SC_FFT_NS {

// Block shape.  The kernel is bound by instruction issue (index work and the
// transforms' arithmetic) and, in FP64, by LDS traffic, so what a shape costs
// is the number of waves its passes issue: a pass of n items takes
// ceil(n / 64) of them whatever the lanes in the last one do.  rows: the count
// that issues the least per row within the LDS tile; threads: the largest
// pass in one go.
struct XrowShape {
    int rows, threads;
};

// LDS tile (complex values).  Lengths up to 128: the smallest tile that fills the
// waves, so that eight (FP64) or more blocks share a CU and cover each other's
// loads and barriers; measured at 96 in FP64 (us, tiles of 1000 / 1300 / 2048 /
// 3400 values): primal 26.4 / 24.9 / 24.8 / 25.4, tangent 48 / 39 / 42 / 38,
// adjoint 36.6 / 33.0 / 34.2 / 33.7.  Longer ones need more for two rows: at 192
// in FP32 the primal takes 221 / 129 us with 1000 / 3400.
constexpr int xrow_tile(int px)
{
    if (px <= 128) return 1300;
    return sizeof(real) == 4 ? 3400 : 2500;
}
constexpr int XROW_THREADS = 256;

constexpr int waves_of(int items) { return (items + 63) / 64; }

constexpr XrowShape xrow_shape(int px, int nseq, int nso)
{
    XrowShape best{1, 64};
    double cost = 1e30;
    for (int rows = 1; rows <= 32; ++rows) {
        if (rows > 1 && rows * nseq * (px + 1) + px > xrow_tile(px)) break;
        double c = 0.0;
        int top = rows * px;
        int m = px;
        while (m > 1) {
            const int r = plan_best(m).first;
            const int ni = rows * nseq * (px / r), no = rows * nso * (px / r);
            c += (waves_of(ni) + waves_of(no)) * (9.0 * r + 30.0);
            if (ni > top) top = ni;
            m /= r;
        }
        c += waves_of(rows * px) * (30.0 + 4.0 * nseq + 8.0 * nso);
        c += waves_of(rows * nso * (px / 3)) * 25.0;
        c = (c + 60.0) / rows;
        if (c < 0.98 * cost) {
            cost = c;
            best.rows = rows;
            best.threads = 64 * waves_of(top < XROW_THREADS ? top : XROW_THREADS);
        }
    }
    return best;
}

// Whether the fields' bins come into LDS first, row by row as they lie in memory
// (the first pass wants each bin twice, directly and mirrored, and a lane its own
// sequence): lengths whose rows of Mx bins lie a multiple of 128 bytes apart (64 at
// 24 points in FP32), which crowd the L1 when lanes read them side by side, as far
// as the two barriers and the LDS traffic cost less.  FP32, direct / staged in us
// (64x97x64, 32 members): primal 404 / 371, tangent 697 / 602, adjoint 628 / 562,
// merged adjoint 950 / 978; 128x129x128, two members: merged adjoint 397 / 308,
// adjoint 235 / 207, primal 132 / 137; three members at Ny = 41: primal 9.0 / 8.1 at
// 24, 14.9 / 12.0 at 48, 19.7 / 17.4 at 144, 22.7 / 22.4 at 192.  The other lengths
// there are 8% slower (30, 90, 180) to 5% faster (72 and 120, whose rows lie 64 bytes
// off a multiple of 128), the merged adjoint at 60 12%, and read directly.  FP64 at
// 48: primal 9.8 / 8.7, tangent 12.5 / 10.8, merged adjoint 34.9 / 36.4; at 96 23.9 /
// 25.0 and 51.5 / 58.2.
constexpr bool xrow_staged(int mode, int px)
{
    if (sizeof(real) == 4) return px == 24 || (px % 48 == 0 && (mode != XM_ADJ2 || px != 96));
    return (px == 24 || px == 48) && (mode == XM_PRIMAL || mode == XM_TANGENT);
}

template <int MODE, int PX> struct XrowPlan {
    static constexpr int NF = XmixShape<MODE>::NF, NOUT = XmixShape<MODE>::NOUT;
    static constexpr int NSEQ = (NF + 1) / 2, NSO = (NOUT + 1) / 2;
    static constexpr XrowShape S = xrow_shape(PX, NSEQ, NSO);
    static constexpr int ROWS = S.rows, T = S.threads, SP = PX + 1;
    static constexpr size_t LDS = sizeof(real2) * ((size_t) ROWS * NSEQ * SP + PX);
};

// First inverse pass, the inputs of butterfly j: bin n < Mx takes X[n] + i Y[n],
// bin n > Px - Mx the conjugates at Px - n, the bins between are zero (c2r uses Re
// only at kx = 0).  Groups of bins in the zero band are not read.
template <int PX>
__device__ __forceinline__ void row_bins(int j, bool hasy, const real2 *X, const real2 *Y, real2 *v)
{
    constexpr int MX = PX / 3, R1 = plan_radix(PX, 0), NB1 = PX / R1;
    const real2 *Xd = X + j, *Yd = Y + j;            // direct bins
    const real2 *Xm = X - j, *Ym = Y - j;            // mirrored ones: Px - n = Px - q NB1 - j
#pragma unroll
    for (int q = 0; q < R1; ++q) {
        const int lo = q * NB1, hi = lo + NB1 - 1, n = j + lo;
        v[q] = mk2(0.0, 0.0);
        if (lo >= MX && hi <= PX - MX) continue;     // zero band for every j
        real2 xv, yl;
        if (hi < MX) {
            xv = Xd[lo];
            yl = Yd[lo];
        } else if (lo > PX - MX) {
            xv = Xm[PX - lo];
            yl = Ym[PX - lo];
        } else {
            const int k = min(n < MX ? n : PX - n, MX - 1);
            xv = X[k];
            yl = Y[k];
        }
        const real2 yv = hasy ? yl : mk2(0.0, 0.0);
        if (hi < MX && lo > 0)
            v[q] = mk2(xv.x - yv.y, xv.y + yv.x);
        else if (lo > PX - MX)
            v[q] = mk2(xv.x + yv.y, -xv.y + yv.x);
        else if (n == 0)
            v[q] = mk2(xv.x, yv.x);
        else if (n < MX)
            v[q] = mk2(xv.x - yv.y, xv.y + yv.x);
        else if (n > PX - MX)
            v[q] = mk2(xv.x + yv.y, -xv.y + yv.x);
    }
}

// One block: ROWS consecutive rows of the flattened (y, z) index, so no block
// has idle rows but the last (ROWS <= Pz: a block meets at most two planes).
// grid (row blocks, members).  LDS: ROWS NSEQ packed sequences at a stride of
// PX + 1 (odd: lanes on neighbouring sequences use different banks), then the
// twiddles.
template <int MODE, int PX, bool EVEN>
__global__ __launch_bounds__((XrowPlan<MODE, PX>::T)) void k_xrow(XmixArgs a, const real2 *W1, real2 *W2)
{
    using P = XrowPlan<MODE, PX>;
    constexpr int NF = P::NF, NOUT = P::NOUT, NSEQ = P::NSEQ, NSO = P::NSO;
    constexpr int ROWS = P::ROWS, T = P::T, SP = P::SP, MX = PX / 3;
    constexpr int R1 = plan_radix(PX, 0), NP = plan_best(PX).passes;
    extern __shared__ __align__(16) char lds_raw[];
    if (*a.abort_flag) return;
    real2 *lds = (real2 *) lds_raw, *twl = lds + ROWS * NSEQ * SP;
    if (const int m = blockIdx.y) {
        W1 += m * a.ms_in;
        W2 += m * a.ms_out;
        a.W1b += m * a.ms_inb;
        a.W1c += m * a.ms_inc;
        a.W2b += m * a.ms_outb;
    }
    const int Pz = a.Pz, nrow = a.qpts * Pz;
    const int row0 = blockIdx.x * ROWS, y0 = row0 / Pz, z0 = row0 - y0 * Pz;
    const int PM = Pz * MX;
    const int nr = min(ROWS, nrow - row0);               // rows of this block
    // plane and z row of row r (ROWS <= Pz: the next plane at most)
    auto plane = [&](int r) { return z0 + r >= Pz ? y0 + 1 : y0; };
    auto zrow = [&](int r) { return z0 + r >= Pz ? z0 + r - Pz : z0 + r; };
    stage_twiddles_c<PX, T>(a.tw, twl);
    const int nf1 = a.nf1, nf2 = MODE == XM_ADJ2 ? a.nf2 : NF;
    // field f of row r in its input array
    auto field = [&](int f, int r) {
        const int src = f < nf1 ? 0 : f < nf2 ? 1 : 2;
        const int f0 = src == 0 ? 0 : src == 1 ? nf1 : nf2;
        const int fn = src == 0 ? nf1 : src == 1 ? nf2 - nf1 : NF - nf2;
        const real2 *B = src == 0 ? W1 : src == 1 ? a.W1b : a.W1c;
        return B + ((size_t) plane(r) * fn + (f - f0)) * PM + zrow(r) * MX;
    };
    if constexpr (xrow_staged(MODE, PX)) {
        // field f of row r at (r NF + f) SB (odd: as SP), inside the sequences' tile
        constexpr int SB = MX | 1, NIN = NF * ROWS * MX, NLD = (NIN + T - 1) / T;
        static_assert(NF * SB <= NSEQ * SP, "the bins fit the tile");
        real bx[NLD], by[NLD];                           // (an array of real2 would go to scratch)
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int e = min((int) threadIdx.x + i * T, NIN - 1);
            const int f = e / (ROWS * MX), rk = e - f * (ROWS * MX), r = rk / MX, k = rk - r * MX;
            const real2 *B = field(f, min(r, nr - 1)) + k;
            bx[i] = B->x;
            by[i] = B->y;
        }
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int e = threadIdx.x + i * T;
            if (NIN % T != 0 && e >= NIN) break;
            const int f = e / (ROWS * MX), rk = e - f * (ROWS * MX), r = rk / MX, k = rk - r * MX;
            lds[(r * NF + f) * SB + k] = mk2(bx[i], by[i]);
        }
        __syncthreads();
        fft_first_in_place<DS_ANY, PX, ROWS * NSEQ, SP, 1, T>(lds, +1.0, [&](int j, int t, real2 *v) {
            const int r = t / NSEQ, s2 = 2 * (t - r * NSEQ);
            const bool hasy = NF % 2 == 0 || s2 + 1 < NF;
            const real2 *X = lds + (r * NF + s2) * SB;
            row_bins<PX>(j, hasy, X, X + (hasy ? SB : 0), v);
        });
    } else {
        fft_first<DS_ANY, PX, ROWS * NSEQ, SP, 1, T>(lds, +1.0, [&](int j, int t, real2 *v) {
            const int r = t / NSEQ, s2 = 2 * (t - r * NSEQ);
            const bool hasy = NF % 2 == 0 || s2 + 1 < NF;
            const real2 *X = field(s2, min(r, nr - 1));
            row_bins<PX>(j, hasy, X, X + (hasy ? PM : 0), v);
        });
    }
    __syncthreads();
    lds_fft_c<PX, ROWS * NSEQ, SP, 1, T, NP, 1, R1>(lds, twl, +1.0);
    // products: every field of a point read, then (after a barrier) the packed
    // outputs written compactly, pair t of row r at sequence r NSO + t
    constexpr int NPT = ROWS * PX, MAXP = (NPT + T - 1) / T;
    real outv[MAXP][NOUT > 0 ? NOUT : 1];
    double cmax[2] = {0.0, 0.0};                         // CFL maxima of planes y0, y0 + 1
#pragma unroll
    for (int i = 0; i < MAXP; ++i) {
        const int e = threadIdx.x + i * T;
        if (NPT % T != 0 && e >= NPT) break;
        // physical output: rows fastest (flow is z-fastest)
        const int r = MODE == XM_PHYS ? e % ROWS : e / PX;
        const int n = MODE == XM_PHYS ? e / ROWS : e - r * PX;
        const real2 *row = lds + r * NSEQ * SP + n;
        real f[2 * NSEQ < 6 ? 6 : 2 * NSEQ] = {};
#pragma unroll
        for (int s = 0; s < NSEQ; ++s) {
            const real2 v = row[s * SP];
            f[2 * s] = v.x;
            f[2 * s + 1] = v.y;
        }
        if constexpr (MODE == XM_PRIMAL || MODE == XM_TANGENT) {
            if (a.check_cfl && r < nr) {
                const int y = plane(r);
                const double t = fabs(f[0]) * a.cfl1 + fabs(f[1]) * a.cfl2[y] + fabs(f[2]) * a.cfl3;
                cmax[0] = fmax(cmax[0], y == y0 ? t : 0.0);
                cmax[1] = fmax(cmax[1], y == y0 ? 0.0 : t);
            }
        }
        if constexpr (MODE == XM_PHYS) {
            if (r < nr) {
                const size_t np = (size_t) PX * a.qpts * Pz;
                const size_t o = ((size_t) n * a.qpts + plane(r)) * Pz + zrow(r);
                a.flow[o] = f[0];
                a.flow[np + o] = f[1];
                a.flow[2 * np + o] = f[2];
            }
        } else {
            xmix_products<MODE>(f, outv[i]);
        }
    }
    if constexpr (MODE == XM_PHYS) return;
    if constexpr (MODE == XM_PRIMAL || MODE == XM_TANGENT) {
        if (a.check_cfl) {
            // block maxima: within each wave by lane exchanges, then the
            // waves' maxima through LDS (a maximum is exact in any order); the
            // second plane only where the block meets it
            __shared__ double cw[2][T / 64];
            const int np = z0 + nr > Pz ? 2 : 1;
            for (int p = 0; p < np; ++p) {
                double m = cmax[p];
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
                if ((threadIdx.x & 63) == 0) cw[p][threadIdx.x >> 6] = m;
            }
            __syncthreads();
            if ((int) threadIdx.x < np) {
                double b = cw[threadIdx.x][0];
#pragma unroll
                for (int w = 1; w < T / 64; ++w) b = fmax(b, cw[threadIdx.x][w]);
                atomic_max_nonneg(&a.cflmax[(y0 + threadIdx.x) * CFL_STRIDE], b);
            }
        }
    }
    if constexpr (NOUT > 0) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MAXP; ++i) {
            const int e = threadIdx.x + i * T;
            if (NPT % T != 0 && e >= NPT) break;
            const int r = e / PX, n = e - r * PX;
#pragma unroll
            for (int t = 0; t < NSO; ++t)
                lds[(r * NSO + t) * SP + n] =
                    mk2(outv[i][2 * t], 2 * t + 1 < NOUT ? outv[i][2 * t + 1 < NOUT ? 2 * t + 1 : 0] : (real) 0);
        }
        __syncthreads();
        lds_fft_c<PX, ROWS * NSO, SP, 1, T, NP, 0, 1, EVEN ? DS_FORWARD : DS_ANY>(lds, twl, -1.0);
        // unpack two real transforms from each packed pair, bins kx < Mx
        constexpr int NU = ROWS * NSO * MX;
#pragma unroll
        for (int i = 0; i < (NU + T - 1) / T; ++i) {
            const int e = threadIdx.x + i * T;
            if (NU % T != 0 && e >= NU) break;
            const int q = e / MX, k = e - q * MX, r = q / NSO, t = q - r * NSO;
            if (r >= nr) break;
            const real2 *Z = lds + q * SP;
            const real2 zk = Z[k], zm = Z[k == 0 ? 0 : PX - k];
            const real2 X = mk2((real) 0.5 * (zk.x + zm.x), (real) 0.5 * (zk.y - zm.y));
            const real2 Yv = mk2((real) 0.5 * (zk.y + zm.y), (real) -0.5 * (zk.x - zm.x));
            constexpr int NO1 = MODE == XM_ADJ2 ? 6 : NOUT;   // fields of an output array
            real2 *D = MODE == XM_ADJ2 && t >= 3 ? a.W2b : W2;
            const int g0 = MODE == XM_ADJ2 && t >= 3 ? 2 * t - 6 : 2 * t;
            D += ((size_t) plane(r) * NO1 + g0) * PM + zrow(r) * MX + k;
            D[0] = X;
            if (NOUT % 2 == 0 || 2 * t + 1 < NOUT) D[PM] = Yv;
        }
    }
}

// The tangent's transforms and products for members along one trajectory: the
// state's six fields, the same for every member, are transformed once for a group
// of members and their point values kept in registers; each member then takes
// three packed inverse transforms instead of six.  The same transforms and
// products as k_xrow<XM_TANGENT>, so the same bits.
// grid (row blocks, groups); group y takes the members y nm / ny ... .  Bound as
// k_xrow is; the next member's bins are fetched while a member is transformed (207
// us for nine FP64 members at 64x97x64, 255 without; k_xrow 279).
template <int PX, bool EVEN>
__global__ __launch_bounds__((XrowPlan<XM_PRIMAL, PX>::T)) void k_xrow_shared(XmixArgs a, const real2 *W1, real2 *W2)
{
    using P = XrowPlan<XM_PRIMAL, PX>;                   // six fields in, three out
    constexpr int NF = 6, NSEQ = 3, NSO = 2;
    constexpr int ROWS = P::ROWS, T = P::T, SP = P::SP, MX = PX / 3;
    constexpr int R1 = plan_radix(PX, 0), NP = plan_best(PX).passes;
    extern __shared__ __align__(16) char lds_raw[];
    if (*a.abort_flag) return;
    real2 *lds = (real2 *) lds_raw, *twl = lds + ROWS * NSEQ * SP;
    const int Pz = a.Pz, nrow = a.qpts * Pz;
    const int row0 = blockIdx.x * ROWS, y0 = row0 / Pz, z0 = row0 - y0 * Pz;
    const int PM = Pz * MX;
    const int nr = min(ROWS, nrow - row0);
    auto plane = [&](int r) { return z0 + r >= Pz ? y0 + 1 : y0; };
    auto zrow = [&](int r) { return z0 + r >= Pz ? z0 + r - Pz : z0 + r; };
    stage_twiddles_c<PX, T>(a.tw, twl);
    // the bins of six fields wait in registers, a member ahead, and come through
    // the tile, field f of row r at (r NF + f) SB
    constexpr int SB = MX | 1, NIN = NF * ROWS * MX, NLD = (NIN + T - 1) / T;
    real bx[NLD], by[NLD];
    auto fetch = [&](const real2 *B) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int e = min((int) threadIdx.x + i * T, NIN - 1);
            const int f = e / (ROWS * MX), rk = e - f * (ROWS * MX), r = min(rk / MX, nr - 1), k = rk % MX;
            const real2 *p = B + ((size_t) plane(r) * NF + f) * PM + zrow(r) * MX + k;
            bx[i] = p->x;
            by[i] = p->y;
        }
    };
    // the fetched fields at the block's points, in the tile; next: fetched meanwhile
    auto inverse = [&](const real2 *next) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int e = threadIdx.x + i * T;
            if (NIN % T != 0 && e >= NIN) break;
            const int f = e / (ROWS * MX), rk = e - f * (ROWS * MX), r = rk / MX, k = rk - r * MX;
            lds[(r * NF + f) * SB + k] = mk2(bx[i], by[i]);
        }
        if (next) fetch(next);
        __syncthreads();
        fft_first_in_place<DS_ANY, PX, ROWS * NSEQ, SP, 1, T>(lds, +1.0, [&](int j, int t, real2 *v) {
            const int r = t / NSEQ;
            const real2 *X = lds + (r * NF + 2 * (t - r * NSEQ)) * SB;
            row_bins<PX>(j, true, X, X + SB, v);
        });
        __syncthreads();
        lds_fft_c<PX, ROWS * NSEQ, SP, 1, T, NP, 1, R1>(lds, twl, +1.0);
    };
    const int m0 = blockIdx.y * a.nm / gridDim.y, m1 = (blockIdx.y + 1) * a.nm / gridDim.y;
    const real2 *Wb = a.W1b + (size_t) m0 * a.ms_inb;
    constexpr int NPT = ROWS * PX, MAXP = (NPT + T - 1) / T;
    auto point = [&](int i, real *f) {
        const int e = min((int) threadIdx.x + i * T, NPT - 1), r = e / PX, n = e - r * PX;
        const real2 *row = lds + r * NSEQ * SP + n;
#pragma unroll
        for (int s = 0; s < NSEQ; ++s) {
            f[2 * s] = row[s * SP].x;
            f[2 * s + 1] = row[s * SP].y;
        }
    };
    fetch(W1);
    inverse(Wb);
    real fb[MAXP][NF];
    double cmax[2] = {0.0, 0.0};                         // CFL maxima of planes y0, y0 + 1
#pragma unroll
    for (int i = 0; i < MAXP; ++i) {
        point(i, fb[i]);
        const int e = threadIdx.x + i * T, r = e / PX;
        if (a.check_cfl && e < NPT && r < nr) {
            const int y = plane(r);
            const double t = fabs(fb[i][0]) * a.cfl1 + fabs(fb[i][1]) * a.cfl2[y] + fabs(fb[i][2]) * a.cfl3;
            cmax[0] = fmax(cmax[0], y == y0 ? t : 0.0);
            cmax[1] = fmax(cmax[1], y == y0 ? 0.0 : t);
        }
    }
    if (a.check_cfl && blockIdx.y == 0) {
        // as k_xrow; the state, and so the maximum, is the same for every group
        __shared__ double cw[2][T / 64];
        const int np = z0 + nr > Pz ? 2 : 1;
        for (int p = 0; p < np; ++p) {
            double m = cmax[p];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
            if ((threadIdx.x & 63) == 0) cw[p][threadIdx.x >> 6] = m;
        }
        __syncthreads();
        if ((int) threadIdx.x < np) {
            double b = cw[threadIdx.x][0];
#pragma unroll
            for (int w = 1; w < T / 64; ++w) b = fmax(b, cw[threadIdx.x][w]);
            atomic_max_nonneg(&a.cflmax[(y0 + threadIdx.x) * CFL_STRIDE], b);
        }
    }
    for (int m = m0; m < m1; ++m) {
        __syncthreads();                                 // the tile's last reads
        Wb += a.ms_inb;
        inverse(m + 1 < m1 ? Wb : nullptr);
        real outv[MAXP][3];
#pragma unroll
        for (int i = 0; i < MAXP; ++i) {
            real f[12];
#pragma unroll
            for (int s = 0; s < NF; ++s) f[s] = fb[i][s];
            point(i, f + NF);
            xmix_products<XM_TANGENT>(f, outv[i]);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < MAXP; ++i) {
            const int e = threadIdx.x + i * T;
            if (NPT % T != 0 && e >= NPT) break;
            const int r = e / PX, n = e - r * PX;
            lds[(r * NSO) * SP + n] = mk2(outv[i][0], outv[i][1]);
            lds[(r * NSO + 1) * SP + n] = mk2(outv[i][2], (real) 0);
        }
        __syncthreads();
        lds_fft_c<PX, ROWS * NSO, SP, 1, T, NP, 0, 1, EVEN ? DS_FORWARD : DS_ANY>(lds, twl, -1.0);
        constexpr int NU = ROWS * NSO * MX;
        real2 *Wm = W2 + (size_t) m * a.ms_out;
#pragma unroll
        for (int i = 0; i < (NU + T - 1) / T; ++i) {
            const int e = threadIdx.x + i * T;
            if (NU % T != 0 && e >= NU) break;
            const int q = e / MX, k = e - q * MX, r = q / NSO, t = q - r * NSO;
            if (r >= nr) break;
            const real2 *Z = lds + q * SP;
            const real2 zk = Z[k], zm = Z[k == 0 ? 0 : PX - k];
            const real2 X = mk2((real) 0.5 * (zk.x + zm.x), (real) 0.5 * (zk.y - zm.y));
            const real2 Yv = mk2((real) 0.5 * (zk.y + zm.y), (real) -0.5 * (zk.x - zm.x));
            real2 *D = Wm + ((size_t) plane(r) * 3 + 2 * t) * PM + zrow(r) * MX + k;
            D[0] = X;
            if (t == 0) D[PM] = Yv;
        }
    }
}

template <int MODE, int PX>
static Fixed<XrowKernel> one(int Pz)
{
    using P = XrowPlan<MODE, PX>;
    Fixed<XrowKernel> f;
    if (P::ROWS > Pz) return f;                          // a block would meet a third plane
    // (the runtime-length kernel, which then runs, has the general order only)
    static_assert(!start_length(PX) || P::ROWS <= even_group(PX, P::NSEQ), "a grid with an order of its own runs this kernel");
    if constexpr (start_length(PX) && P::NOUT > 0)
        f.kernel = even_rows(PX, Pz, P::NSEQ) ? k_xrow<MODE, PX, true> : k_xrow<MODE, PX, false>;
    else
        f.kernel = k_xrow<MODE, PX, false>;
    f.group = P::ROWS;
    f.threads = P::T;
    f.lds = P::LDS;
    return f;
}

template <>
Fixed<XrowKernel> xrow_fixed<SC_XMODE>(int Px, int Pz)
{
    switch (Px) {
#define SC_ONE(N) \
    case N: return one<SC_XMODE, N>(Pz);
        SC_X_LENGTHS(SC_ONE)
#undef SC_ONE
    default: return Fixed<XrowKernel>();
    }
}

// Where the shared form is taken: lengths 48 to 128 that are multiples of 12, from
// four members on below 72.  Per member / shared in us, six members along one
// trajectory, Ny = 41, Nz = 32: FP64 48 25.5 / 20.5, 72 35.1 / 32.6, 96 41.6 / 36.5,
// 120 66.7 / 55.0, but 24 14.6 / 15.5, 54 28.9 / 30.7, 150 75.9 / 81.2; FP32 48 16.4 /
// 14.4, 96 30.1 / 24.6, 120 50.1 / 32.4, but 24 10.5 / 12.3, 162 59.4 / 86.4, 192 52.7 /
// 60.0 (longer rows leave few registers for the waves).  Three members: FP32 48
// 11.3 / 11.8, FP64 60 18.3 / 19.1; two: FP64 72 17.5 / 16.3.  Two lengths outside the
// rule would gain, 90 (FP64 44.0 / 39.7, FP32 33.0 / 27.3) and, in FP32 alone, 54
// (22.3 / 19.3).
constexpr bool xrow_shared_length(int px) { return px >= 48 && px <= 128 && px % 12 == 0; }

// compiled with the tangent's kernels
template <int PX>
static Fixed<XrowKernel> one_shared(int Pz)
{
    using P = XrowPlan<XM_PRIMAL, PX>;
    Fixed<XrowKernel> f;
    if (P::ROWS > Pz) return f;
    // the order of the forward transforms is that of the tangent's six sequences
    if constexpr (start_length(PX))
        f.kernel = even_rows(PX, Pz, 6) ? k_xrow_shared<PX, true> : k_xrow_shared<PX, false>;
    else
        f.kernel = k_xrow_shared<PX, false>;
    f.group = P::ROWS;
    f.threads = P::T;
    f.lds = P::LDS;
    return f;
}

template <int MODE>
static Fixed<XrowKernel> shared_of(int Px, int Pz, int nm)
{
    if (nm < (Px < 72 ? 4 : 2)) return Fixed<XrowKernel>();
    if constexpr (MODE == XM_TANGENT) {
        switch (Px) {
#define SC_ONE(N) \
        case N: \
            if constexpr (xrow_shared_length(N)) return one_shared<N>(Pz); \
            break;
            SC_X_LENGTHS(SC_ONE)
#undef SC_ONE
        }
    }
    return Fixed<XrowKernel>();
}

#define SC_IS_TANGENT_XM_TANGENT 1
#define SC_IS(m) SC_IS_(m)
#define SC_IS_(m) SC_IS_TANGENT_##m
#if SC_IS(SC_XMODE)
Fixed<XrowKernel> xrow_shared_fixed(int Px, int Pz, int nm) { return shared_of<SC_XMODE>(Px, Pz, nm); }
#endif

}  // namespace SC_FFT_NS
}  // namespace sc
