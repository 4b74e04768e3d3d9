// Dealiased x/z transforms of the nonlinear terms, one launch per direction.
//
// The reference does, per Gauss plane y and field, an unnormalised backward
// c2c along z over the Nx/2 stored columns of a 3/2-padded array, then a c2r
// along x, the pointwise products, and the reverse with a 1/(Px Pz) scale and
// truncation (channel/pass1.c:107-114, 312-371; channel/pass2.c:128-221,
// 417-472; channel/spec2phys.c:67-76).  Here the three phases are separate
// batched kernels over all planes at once:
//   zinv : (y, field, kx block) -> length-Pz inverse transforms in LDS, with
//          the spectral curl fused into the load and the zero padding implied
//   xmix : (y, block of z rows) -> pairs of real rows packed into one complex
//          length-Px inverse transform, products, CFL maximum, forward
//          transforms of packed product pairs, unpacking of the kx < Nx/2 bins
//   zfwd : (y, field, kx block) -> forward length-Pz transforms, scale,
//          truncation to the stored kz rows
// The FFTs are Stockham passes run in place in LDS with radices up to 16 (the
// composite ones done as small FFTs in registers, so a length of 96 takes two
// passes): every thread holds its butterflies' inputs in registers across a
// barrier.

// Here: the kernels for any length (runtime plans; the lengths without a
// compile-time plan) and the launchers, which take the fixed-length kernels of
// fft_x.hip and fft_z.hip wherever a grid's lengths have them.
#include "fft_common.h"

namespace sc {
namespace SC_FFT_NS {

// complex values staged in LDS by one x-kernel block, data and twiddles
constexpr int XMIX_TILE = FFT_TILE;

struct PlanDev {
    int n, nf;
    int f[MAX_FACTORS];
    // per pass: ceil(2^32 / Ns), Ns = product of the earlier radices, so that
    // x / Ns = (x * nsm) >> 32 exactly for x <= 8192, Ns <= 4096
    unsigned long long nsm[MAX_FACTORS];
    const double2 *tw;         // the plan's FP64 twiddles (converted when staged)
};

static PlanDev to_dev(const FftPlan &p)
{
    PlanDev d;
    d.n = p.n;
    d.nf = p.nf;
    unsigned long long ns = 1;
    for (int i = 0; i < MAX_FACTORS; ++i) {
        d.f[i] = i < p.nf ? p.f[i] : 0;
        d.nsm[i] = ((1ull << 32) + ns - 1) / ns;
        if (i < p.nf) ns *= (unsigned long long) p.f[i];
    }
    d.tw = p.tw;
    return d;
}

__device__ __forceinline__ int magic_div(int x, unsigned long long m)
{
    return (int) (((unsigned long long) (unsigned) x * m) >> 32);
}

// (index / L, index % L) of the elements threadIdx.x, threadIdx.x + BLK, ...
// of a row-major walk with rows of length L, without divisions in the walk
struct Walk {
    int q, r, dq, dr, L;
    __device__ __forceinline__ Walk(int L_) : L(L_)
    {
        // one division per walk
        q = (int) threadIdx.x / L;
        r = (int) threadIdx.x - q * L;
        dq = BLK / L;
        dr = BLK - dq * L;
    }
    __device__ __forceinline__ void next()
    {
        q += dq;
        r += dr;
        if (r >= L) {
            r -= L;
            ++q;
        }
    }
};

// One Stockham pass of radix R over nseq sequences of length n, in place in
// LDS: element e of sequence s at data[s*sstride + e*estride].  Lanes run
// over the sequences fastest, so with estride = nseq (sequences interleaved)
// every access of a pass is a contiguous run, and with sstride odd and
// estride = 1 neighbouring lanes fall in different banks.  Each thread keeps
// its butterflies' inputs in registers across the barrier; a block of BLK
// threads transforms at most FFT_TILE complex values, so a thread owns at most
// ceil(FFT_TILE / (BLK R)) butterflies.
template <int R>
__device__ __forceinline__ void fft_pass(real2 *data, int nseq, int sstride, int estride, int n,
                                         int Ns, unsigned long long nsm, const real2 *tw,
                                         real sign)
{
    constexpr int NB = (FFT_TILE / BLK + R - 1) / R;
    const int nb = n / R;
    const int twstep = magic_div(nb, nsm);      // n / (Ns R)
    real2 v[NB][R];
    int off[NB];                                // output position of the butterfly
    Walk w(nseq);                               // w.q = butterfly index j, w.r = sequence s
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int j = w.q, s = w.r;
        off[i] = -1;
        if (j < nb) {
            const real2 *src = data + s * sstride;
            const int jq = magic_div(j, nsm), k = j - jq * Ns;
            off[i] = s * sstride + (jq * Ns * R + k) * estride;
#pragma unroll
            for (int q = 0; q < R; ++q) {
                real2 a = src[(j + q * nb) * estride];
                if (q > 0) a = twiddle(a, tw[q * k * twstep], sign);
                v[i][q] = a;
            }
            dft<R>(v[i], sign);
        }
        w.next();
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        if (off[i] >= 0) {
            real2 *dst = data + off[i];
#pragma unroll
            for (int q = 0; q < R; ++q) dst[q * Ns * estride] = v[i][q];
        }
    }
    __syncthreads();
}

// tw: the plan's twiddles exp(2 pi i m / n), m < n, staged in LDS
__device__ __forceinline__ void lds_fft(real2 *data, int nseq, int sstride, int estride,
                                        const PlanDev &p, const real2 *tw, real sign)
{
    int Ns = 1;
    for (int pass = 0; pass < p.nf; ++pass) {
        const int r = p.f[pass];
        const unsigned long long m = p.nsm[pass];
        switch (r) {
        case 16: fft_pass<16>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 12: fft_pass<12>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 8: fft_pass<8>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 6: fft_pass<6>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 5: fft_pass<5>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 4: fft_pass<4>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        case 3: fft_pass<3>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign); break;
        default: fft_pass<2>(data, nseq, sstride, estride, p.n, Ns, m, tw, sign);
        }
        Ns *= r;
    }
}

// copy the plan's twiddle table into LDS (visible after the caller's barrier)
__device__ __forceinline__ void stage_twiddles(const PlanDev &p, real2 *twl)
{
    for (int m = threadIdx.x; m < p.n; m += BLK) twl[m] = to_real2(p.tw[m]);
}

constexpr int MAXE = FFT_TILE / BLK;   // LDS elements per thread of a full tile
constexpr int SBAT = 8;                // stage-in loads in flight per thread and batch
static_assert(MAXE % SBAT == 0, "stage-in batches must tile the per-thread elements");

// Stage a (Pz x XB) tile of one field into LDS in its memory layout
// [zp][x], zero rows for the padding, the spectral curl formed on the fly.
// A batch's loads are all issued before its first LDS store: indices are
// clamped into the array and the padding masked arithmetically, so no load
// sits behind a branch.
template <int KIND, bool S32>
__device__ __forceinline__ void zinv_stage(const ZinvArgs &a, const cplx *src, int slot, int y,
                                           int x0, int XB, real2 *lds)
{
    constexpr int NE = MAXE, SB = SBAT;
    const int Pz = a.Pz, Nz = a.Nz, Mx = a.Mx;
    const int total = XB * Pz;
    const size_t zs = (size_t) 5 * a.qpts * Mx;        // stride of kz in U
    const size_t ss = (size_t) a.qpts * Mx;            // stride of slot in U
    Walk wk(XB);                                       // (zp, xl)
#pragma unroll 1
    for (int i0 = 0; i0 < NE; i0 += SB) {
        if ((int) threadIdx.x + i0 * BLK >= total) break;
        double2 p[SB], q[SB];
        bool ok[SB];
        int kzi[SB], xi[SB];
#pragma unroll
        for (int i = 0; i < SB; ++i) {
            const int e = threadIdx.x + (i0 + i) * BLK;
            const int zp = min(wk.q, Pz - 1), xl = wk.r;
            wk.next();
            const int kz = zp < Nz / 2 ? zp : (zp > Nz ? zp - Nz / 2 : -1);
            ok[i] = e < total && kz >= 0;
            kzi[i] = max(kz, 0);
            xi[i] = x0 + xl;
            const size_t b = kzi[i] * zs + (size_t) y * Mx + xi[i];
            if (KIND == FK_SLOT) {
                p[i] = ld_slot<S32>(src, b + slot * ss);
            } else if (KIND == FK_OMEGA_Z) {
                p[i] = ld_slot<S32>(src, b + 3 * ss);
                q[i] = ld_slot<S32>(src, b + 1 * ss);
            } else if (KIND == FK_OMEGA_X) {
                p[i] = ld_slot<S32>(src, b + 4 * ss);
                q[i] = ld_slot<S32>(src, b + 1 * ss);
            } else {
                p[i] = ld_slot<S32>(src, b);
                q[i] = ld_slot<S32>(src, b + 2 * ss);
            }
        }
#pragma unroll
        for (int i = 0; i < SB; ++i) {
            const int e = threadIdx.x + (i0 + i) * BLK;
            if (e >= total) break;
            const double kx = xi[i] * a.ax;
            const int kz = kzi[i];
            const double kzv = (kz <= Nz / 2 ? kz : kz - Nz) * a.az;
            // formed in FP64 from the FP64 state, then stored as real
            double2 val;
            if (KIND == FK_SLOT) {
                val = p[i];
            } else if (KIND == FK_OMEGA_Z) {            // -du/dy + i kx v
                const double2 du = p[i], v = q[i];
                val = make_double2(-(du.x + kx * v.y), -du.y + kx * v.x);
            } else if (KIND == FK_OMEGA_X) {            // dw/dy - i kz v
                const double2 dw = p[i], v = q[i];
                val = make_double2(dw.x + kzv * v.y, dw.y - kzv * v.x);
            } else {                                    // i kz u - i kx w
                const double2 u = p[i], w = q[i];
                val = make_double2(fma_(kx, w.y, -(kzv * u.y)), fma_(kzv, u.x, -(kx * w.x)));
            }
            lds[e] = ok[i] ? to_real2(val) : mk2(0.0, 0.0);
        }
    }
}

// grid (ceil(Mx/XB), nf * members, qpts): blockIdx.y = member nf + field
template <bool S32>
__global__ __launch_bounds__(BLK) void k_zinv(ZinvArgs a, PlanDev pz, real2 *W1)
{
    extern __shared__ real2 lds[];
    if (*a.abort_flag) return;
    const int nf = a.fs.nf, m = blockIdx.y / nf, f = blockIdx.y - m * nf;
    const int x0 = blockIdx.x * a.XB, y = blockIdx.z;
    const int XB = min(a.XB, a.Mx - x0);
    const int Pz = a.Pz, Mx = a.Mx;
    const cplx *src = a.fs.src[f] + m * a.fs.ms[f];
    const int kind = a.fs.kind[f], slot = a.fs.slot[f];
    real2 *twl = lds + a.XB * Pz;
    stage_twiddles(pz, twl);
    // columns interleaved in LDS exactly as in memory: no transpose
    if (kind == FK_SLOT) zinv_stage<FK_SLOT, S32>(a, src, slot, y, x0, XB, lds);
    else if (kind == FK_OMEGA_Z) zinv_stage<FK_OMEGA_Z, S32>(a, src, slot, y, x0, XB, lds);
    else if (kind == FK_OMEGA_X) zinv_stage<FK_OMEGA_X, S32>(a, src, slot, y, x0, XB, lds);
    else zinv_stage<FK_OMEGA_Y, S32>(a, src, slot, y, x0, XB, lds);
    __syncthreads();
    lds_fft(lds, XB, 1, XB, pz, twl, +1.0);
    real2 *dst = W1 + m * a.ms_w1 + (((size_t) y * nf + f) * Pz) * Mx;
    Walk wk(XB);
    for (int e = threadIdx.x; e < XB * Pz; e += BLK, wk.next())
        dst[(size_t) wk.q * Mx + x0 + wk.r] = lds[e];
}

// grid (Pz/ZB, qpts, members); LDS: ZB * nseq sequences of Px complex at a stride of
// Px + 1 (odd, so lanes on neighbouring sequences use different banks),
// nseq = ceil(nf/2).
template <int MODE>
__global__ __launch_bounds__(BLK) void k_xmix(XmixArgs a, PlanDev px, const real2 *W1, real2 *W2)
{
    extern __shared__ real2 lds[];
    if (*a.abort_flag) return;
    constexpr int nf = XmixShape<MODE>::NF;
    constexpr int NOUT = XmixShape<MODE>::NOUT;
    constexpr int nseq = (nf + 1) / 2;
    constexpr int nso = (NOUT + 1) / 2;
    const int zb = blockIdx.x, y = blockIdx.y;
    if (const int m = blockIdx.z) {
        W1 += m * a.ms_in;
        W2 += m * a.ms_out;
        a.W1b += m * a.ms_inb;
    }
    const int Px = a.Px, Mx = a.Mx, Pz = a.Pz, ZB = a.ZB;
    const int SP = Px + 1;
    const int z0 = zb * ZB;
    real2 *twl = lds + ZB * nseq * SP;
    stage_twiddles(px, twl);
    // load packed pairs with Hermitian extension (c2r uses Re only at kx=0):
    // bin n < Mx takes X[n] + i Y[n], bin n > Px - Mx the conjugates at
    // Px - n, the bins between are zero.  Loads unpredicated (index clamped
    // into the row), all issued before the LDS stores.
    {
        const int tot = ZB * nseq * Px;
        constexpr int MAXL = (XMIX_TILE + BLK - 1) / BLK;
        constexpr int LB = 4;                              // loads in flight per batch
        Walk wl(Px);                                       // (packed row t, bin n)
#pragma unroll 1
        for (int i0 = 0; i0 < MAXL; i0 += LB) {
            if ((int) threadIdx.x + i0 * BLK >= tot) break;
            real2 lx[LB], ly[LB];
            int tn[LB];
#pragma unroll
            for (int i = 0; i < LB; ++i) {
                const int t = min(wl.q, ZB * nseq - 1), n = wl.r;
                tn[i] = wl.q * Px + n;
                wl.next();
                const int s = t % nseq, r = t / nseq;
                const int k = min(n < Mx ? n : Px - n, Mx - 1);
                const int f0 = 2 * s, nf1 = a.nf1;
                const real2 *X = f0 < nf1 ? W1 + (((size_t) y * nf1 + f0) * Pz + z0 + r) * Mx
                                         : a.W1b + (((size_t) y * (nf - nf1) + f0 - nf1) * Pz + z0 + r) * Mx;
                const int sy = min(2 * s + 1, nf - 1) - 2 * s;     // 1, or 0 for a lone field
                lx[i] = X[k];
                ly[i] = X[(size_t) sy * Pz * Mx + k];
            }
#pragma unroll
            for (int i = 0; i < LB; ++i) {
                const int e = threadIdx.x + (i0 + i) * BLK;
                if (e >= tot) break;
                const int t = tn[i] / Px, n = tn[i] - t * Px;
                const int s = t % nseq, r = t / nseq;
                const bool hasy = 2 * s + 1 < nf;
                real2 xv = lx[i], yv = hasy ? ly[i] : mk2(0.0, 0.0);
                real2 val;
                if (n == 0)
                    val = mk2(xv.x, yv.x);
                else if (n < Mx)
                    val = mk2(xv.x - yv.y, xv.y + yv.x);
                else if (n > Px - Mx)
                    val = mk2(xv.x + yv.y, -xv.y + yv.x);
                else
                    val = mk2(0.0, 0.0);
                lds[(r * nseq + s) * SP + n] = val;
            }
        }
    }
    __syncthreads();
    lds_fft(lds, ZB * nseq, SP, 1, px, twl, +1.0);
    // pointwise stage: read all fields of a point, compute, then (after a
    // barrier) write the packed outputs compactly: row r, pair t at sequence
    // r*nso + t
    constexpr int MAXP = (XMIX_TILE / nseq + BLK - 1) / BLK;          // points per thread
    constexpr int NO = NOUT > 0 ? NOUT : 1;
    real outv[MAXP][NO];
    double cmax = 0.0;
    const int npt = ZB * Px;
    Walk wp(Px);                                       // (z row r, point n)
#pragma unroll
    for (int i = 0; i < MAXP; ++i) {
        int e = threadIdx.x + i * BLK;
        if (e >= npt) break;
        const int n = wp.r, r = wp.q;
        wp.next();
        const real2 *row = lds + (size_t) r * nseq * SP + n;
        real f[16];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            if (s < nseq) {
                real2 v = row[s * SP];
                f[2 * s] = v.x;
                f[2 * s + 1] = v.y;
            } else {
                f[2 * s] = 0.0;
                f[2 * s + 1] = 0.0;
            }
        }
        const real u = f[0], v = f[1], w = f[2];
        if (a.check_cfl) {
            double t = fabs(u) * a.cfl1 + fabs(v) * a.cfl2[y] + fabs(w) * a.cfl3;
            cmax = fmax(cmax, t);
        }
        xmix_products<MODE>(f, outv[i]);
        if constexpr (MODE == XM_PHYS) {
            int zp = z0 + r;
            size_t plane = (size_t) Px * a.qpts * Pz;
            size_t o = ((size_t) n * a.qpts + y) * Pz + zp;
            a.flow[o] = u;
            a.flow[plane + o] = v;
            a.flow[2 * plane + o] = w;
        }
    }
    if (a.check_cfl) {
        // block maximum: within each wave by lane exchanges, then the waves'
        // maxima through LDS (the maximum is exact in any order)
        __shared__ double cw[BLK / 64];
        double m = cmax;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
        if ((threadIdx.x & 63) == 0) cw[threadIdx.x >> 6] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            double b = cw[0];
#pragma unroll
            for (int w = 1; w < BLK / 64; ++w) b = fmax(b, cw[w]);
            atomic_max_nonneg(&a.cflmax[y * CFL_STRIDE], b);
        }
    }
    if constexpr (MODE == XM_PHYS) return;
    if constexpr (NOUT > 0) {
    __syncthreads();
    wp = Walk(Px);
#pragma unroll
    for (int i = 0; i < MAXP; ++i) {
        int e = threadIdx.x + i * BLK;
        if (e >= npt) break;
        const int n = wp.r, r = wp.q;
        wp.next();
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            if (t < nso) {
                real re = outv[i][2 * t < NO ? 2 * t : 0];
                real im = (2 * t + 1 < NOUT) ? outv[i][2 * t + 1 < NO ? 2 * t + 1 : 0] : (real) 0;
                lds[(size_t) (r * nso + t) * SP + n] = mk2(re, im);
            }
        }
    }
    __syncthreads();
    lds_fft(lds, ZB * nso, SP, 1, px, twl, -1.0);
    // unpack two real transforms from each packed pair, bins kx < Mx
    const int tot2 = ZB * nso * Mx;
    Walk wu(Mx);                                       // (packed row, bin k)
    for (int e = threadIdx.x; e < tot2; e += BLK, wu.next()) {
        const int k = wu.r, t = wu.q % nso, r = wu.q / nso;
        const real2 *Z = lds + (size_t) (r * nso + t) * SP;
        real2 zk = Z[k], zm = Z[k == 0 ? 0 : Px - k];
        real2 X = mk2((real) 0.5 * (zk.x + zm.x), (real) 0.5 * (zk.y - zm.y));
        real2 Yv = mk2((real) 0.5 * (zk.y + zm.y), (real) -0.5 * (zk.x - zm.x));
        int zp = z0 + r;
        int g0 = 2 * t, g1 = 2 * t + 1;
        W2[(((size_t) y * NOUT + g0) * Pz + zp) * Mx + k] = X;
        if (g1 < NOUT) W2[(((size_t) y * NOUT + g1) * Pz + zp) * Mx + k] = Yv;
    }
    }
}

// grid (ceil(Mx/XB), nout * members, qpts): blockIdx.y = member nout + field
__global__ __launch_bounds__(BLK) void k_zfwd(ZfwdArgs a, PlanDev pz, const real2 *W2, cplx *dst)
{
    extern __shared__ real2 lds[];
    if (a.cfl_slot >= 0 && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)
        cfl_check_block(a.cflmax, a.qpts, a.dt, a.abort_rw, a.cfl_slot);
    if (*a.abort_flag) return;
    const int XB0 = a.XB;
    const int m = blockIdx.y / a.nout, g = blockIdx.y - m * a.nout;
    const int x0 = blockIdx.x * XB0, y = blockIdx.z;
    const int XB = min(a.XB, a.Mx - x0);
    const int Nz = a.Nz, Pz = a.Pz, Mx = a.Mx;
    const real2 *src = W2 + m * a.ms_in + (((size_t) y * a.nout + g) * Pz) * Mx;
    dst += m * a.ms_out;
    real2 *twl = lds + XB0 * Pz;
    stage_twiddles(pz, twl);
    {
        // a batch's loads all issued before its LDS stores
        constexpr int NE = MAXE, SB = SBAT;
        const int total = XB * Pz;
        Walk wk(XB);
#pragma unroll 1
        for (int i0 = 0; i0 < NE; i0 += SB) {
            if ((int) threadIdx.x + i0 * BLK >= total) break;
            real2 v[SB];
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                const int zp = min(wk.q, Pz - 1), xl = wk.r;
                wk.next();
                v[i] = src[(size_t) zp * Mx + x0 + xl];
            }
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                const int e = threadIdx.x + (i0 + i) * BLK;
                if (e < total) lds[e] = v[i];
            }
        }
    }
    __syncthreads();
    lds_fft(lds, XB, 1, XB, pz, twl, -1.0);
    Walk wt(XB);
    for (int e = threadIdx.x; e < XB * (Nz - 1); e += BLK, wt.next()) {
        const int r = wt.q, xl = wt.r;
        int kz = r < Nz / 2 ? r : r + 1;             // skip the Nyquist row
        int zp = kz < Nz / 2 ? kz : kz + Nz / 2;
        real2 v = lds[zp * XB + xl];
        v.x *= (real) a.norm;
        v.y *= (real) a.norm;
        if (a.dst_kind == ZF_USLOTS)
            st_slot(dst, (((size_t) kz * 5 + g) * a.qpts + y) * Mx + x0 + xl, a.p32, v.x, v.y);
        else
            dst[(((size_t) g * Nz + kz) * a.qpts + y) * Mx + x0 + xl] = to_cplx(v);
    }
}

// Forward z transforms of the six adjoint products with the assembly fused
// (channel/pass2.c:417-566): a block transforms all six fields of XA
// columns, interleaved in LDS as 6 XA sequences ([zp][field][x], no
// transpose), and forms the five state slots at the stored kz rows:
// Hz = -Tz - i kx Sy, Hx = -Tx + i kz Sy, Hy = -Ty - i kz Sx + i kx Sz, then
// S_x, S_z (each field scaled first, as the separate transform does).
// grid (ceil(Mx / XA), qpts, members)
__global__ __launch_bounds__(BLK) void k_zfwd_adj(ZadjArgs a, PlanDev pz, const real2 *W2, cplx *U)
{
    extern __shared__ real2 lds[];
    if (*a.abort_flag) return;
    const int XA = a.XA;
    const int x0 = blockIdx.x * XA, y = blockIdx.y;
    W2 += blockIdx.z * a.ms_in;
    U += blockIdx.z * a.ms_out;
    const int XB = min(a.XA, a.Mx - x0);                 // columns of this block
    const int Nz = a.Nz, Pz = a.Pz, Mx = a.Mx;
    const int NS = 6 * XA;                               // interleaved sequences
    real2 *twl = lds + NS * Pz;
    stage_twiddles(pz, twl);
    {
        // element (zp, field f, column xl) at (zp * 6 + f) * XA + xl
        const int total = 6 * Pz * XA;
        const real2 *src = W2 + (size_t) y * 6 * Pz * Mx;
        Walk wk(XA);                                     // (zp * 6 + f, xl)
        constexpr int NE = MAXE, SB = SBAT;
#pragma unroll 1
        for (int i0 = 0; i0 < NE; i0 += SB) {
            if ((int) threadIdx.x + i0 * BLK >= total) break;
            real2 v[SB];
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                const int q = min(wk.q, 6 * Pz - 1), xl = min(wk.r, XB - 1);
                wk.next();
                const int zp = q / 6, f = q - zp * 6;
                v[i] = src[((size_t) f * Pz + zp) * Mx + x0 + xl];
            }
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                const int e = threadIdx.x + (i0 + i) * BLK;
                if (e < total) lds[e] = v[i];
            }
        }
    }
    __syncthreads();
    lds_fft(lds, NS, 1, NS, pz, twl, -1.0);
    const size_t ss = (size_t) a.qpts * Mx;
    Walk wt(XA);                                         // (stored kz row r, xl)
    for (int e = threadIdx.x; e < XA * (Nz - 1); e += BLK, wt.next()) {
        const int r = wt.q, xl = wt.r;
        if (xl >= XB) continue;
        const int kz = r < Nz / 2 ? r : r + 1;           // skip the Nyquist row
        const int zp = kz < Nz / 2 ? kz : kz + Nz / 2;
        real2 S[3], T[3];
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            S[f] = lds[(zp * 6 + f) * XA + xl];
            T[f] = lds[(zp * 6 + 3 + f) * XA + xl];
        }
        const int x = x0 + xl;
        st_adjoint(U, ((size_t) kz * 5 * a.qpts + y) * Mx + x, ss, a.p32, (real) a.norm, a.Kx[x], a.Kz[kz], S, T);
    }
}

// adjoint assembly (channel/pass2.c:474-566):
// Hz = -Tz - i kx Sy, Hx = -Tx + i kz Sy, Hy = -Ty - i kz Sx + i kx Sz
// grid (blocks, members): SP and U of member blockIdx.y at the given strides
__global__ void k_assemble_adj(const cplx *SP, cplx *U, const double *Kx, const double *Kz,
                               int Nz, int qpts, int Mx, const int *abort_flag, size_t ms_sp,
                               size_t ms_u, int p32)
{
    if (*abort_flag) return;
    SP += blockIdx.y * ms_sp;
    U += blockIdx.y * ms_u;
    size_t n = (size_t) Nz * qpts * Mx;
    for (size_t e = blockIdx.x * (size_t) blockDim.x + threadIdx.x; e < n;
         e += (size_t) gridDim.x * blockDim.x) {
        int x = e % Mx;
        int y = (e / Mx) % qpts;
        int z = e / ((size_t) Mx * qpts);
        if (z == Nz / 2) continue;
        double kx = Kx[x], kz = Kz[z];
        double2 Sx = SP[e], Sy = SP[n + e], Sz = SP[2 * n + e];
        double2 Tx = SP[3 * n + e], Ty = SP[4 * n + e], Tz = SP[5 * n + e];
        size_t b = ((size_t) z * 5 * qpts + y) * Mx + x, ss = (size_t) qpts * Mx;
        st_slot(U, b + 0 * ss, p32, -Tz.x + kx * Sy.y, -Tz.y - kx * Sy.x);
        st_slot(U, b + 1 * ss, p32, -Tx.x - kz * Sy.y, -Tx.y + kz * Sy.x);
        st_slot(U, b + 2 * ss, p32, -Ty.x + kz * Sx.y - kx * Sz.y, -Ty.y - kz * Sx.x + kx * Sz.x);
        st_slot(U, b + 3 * ss, p32, Sx.x, Sx.y);
        st_slot(U, b + 4 * ss, p32, Sz.x, Sz.y);
    }
}

// ---------------------------------------------------------------- launches
int xmix_zblock(Context &c, int nf);

static int pick_block(int Mx, int P, int nper)
{
    // columns per block so that the LDS tile plus the P twiddles stay within
    // FFT_TILE complex
    int xb = Mx;
    while (xb > 1 && (size_t) xb * P * nper + P > FFT_TILE) xb = (xb + 1) / 2;
    return xb;
}

void launch_zinv(Context &c, const FieldSpec &fs, cplx *W1)
{
    const Dims &d = c.d;
    ZinvArgs a;
    a.fs = fs;
    a.tw = c.pz.tw;
    a.nm = c.nrun;
    a.Nz = d.Nz;
    a.Mx = d.Mx;
    a.qpts = d.qpts;
    a.Pz = d.Pz;
    a.XB = pick_block(d.Mx, d.Pz, 1);
    a.ax = 2. * M_PI / d.Lx;
    a.az = 2. * M_PI / d.Lz;
    a.abort_flag = c.abort_flag;
    for (int f = 0; f < fs.nf; ++f) a.fs.ms[f] = mstride(c, fs.src[f]);
    a.ms_w1 = rstride(c, W1);
    const int nm = c.nrun;
    // the FP32 build reads FP32 slots where the rebuild wrote them
#ifdef SC_FFT_F32
    const bool s32 = slots32(c);
#else
    const bool s32 = false;
#endif
    const double plane = (double) d.qpts * d.Mx;
    int slots = 0;
    for (int f = 0; f < fs.nf; ++f) {
        bool seen = false;
        for (int g = 0; g < f; ++g) seen |= fs.src[g] == fs.src[f];
        if (!seen) slots += fs.nf >= 6 ? 5 : 3;
    }
    if (fs.nf == 9) slots = 8;            // adjoint: 5 state slots + 3 adjoint
    if (fs.nf == 6 && fs.kind[3] == FK_SLOT) slots = 6;   // two velocity triples
    double bytes = nm * plane * ((s32 ? 8.0 : 16.0) * slots * (d.Nz - 1) +
                                 (double) sizeof(real2) * fs.nf * d.Pz);
    const hipStream_t st = c.stream;
    real2 *W1r = (real2 *) W1;
    std::function<void()> go;
    if (const auto fx = zinv_fixed(d.Pz, d.Mx, s32); fx.kernel) {
        const int ncb = (d.qpts * d.Mx + fx.group - 1) / fx.group;
        const dim3 grid(xcd_grid(nm * ncb * fs.nf));
        go = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, a, W1r); };
    } else {
        const dim3 grid((d.Mx + a.XB - 1) / a.XB, fs.nf * nm, d.qpts);
        const size_t lds = sizeof(real2) * (a.XB * d.Pz + d.Pz);
        const PlanDev pd = to_dev(c.pz);
        const auto kern = s32 ? k_zinv<true> : k_zinv<false>;
        go = [=]() { hipLaunchKernelGGL(kern, grid, dim3(BLK), lds, st, a, pd, W1r); };
    }
    prof_begin(c, st, 1, bytes);
    go();
    prof_end(c, st, 1, go);
}

typedef void (*XmixKernel)(XmixArgs, PlanDev, const real2 *, real2 *);

static XmixKernel xmix_kernel(int mode)
{
    switch (mode) {
    case XM_PRIMAL: return k_xmix<XM_PRIMAL>;
    case XM_TANGENT: return k_xmix<XM_TANGENT>;
    case XM_ADJOINT: return k_xmix<XM_ADJOINT>;
    default: return k_xmix<XM_PHYS>;
    }
}

// the fixed-length kernel of a mode for this grid, where there is one
static Fixed<XrowKernel> xrow_kernel(int mode, const Dims &d)
{
    switch (mode) {
    case XM_PRIMAL: return xrow_fixed<XM_PRIMAL>(d.Px, d.Pz);
    case XM_TANGENT: return xrow_fixed<XM_TANGENT>(d.Px, d.Pz);
    case XM_ADJOINT: return xrow_fixed<XM_ADJOINT>(d.Px, d.Pz);
    case XM_ADJ2: return xrow_fixed<XM_ADJ2>(d.Px, d.Pz);
#ifndef SC_FFT_F32
    case XM_PHYS: return xrow_fixed<XM_PHYS>(d.Px, d.Pz);   // FP64 in both precisions
#endif
    default: return Fixed<XrowKernel>();
    }
}

void launch_xmix(Context &c, int mode, const cplx *W1, cplx *W2, int check_cfl,
                 double *flow, const cplx *W1b, int nf1)
{
    const Dims &d = c.d;
    XmixArgs a;
    a.mode = mode;
    a.nf = mode == XM_PRIMAL ? 6 : mode == XM_TANGENT ? 12 : mode == XM_ADJOINT ? 9 : 3;
    a.nout = mode == XM_ADJOINT ? 6 : (mode == XM_PRIMAL || mode == XM_TANGENT) ? 3 : 0;
    a.nf1 = W1b ? nf1 : a.nf;
    a.W1b = (const real2 *) (W1b ? W1b : W1);
    a.nf2 = a.nf;
    a.W1c = nullptr;
    a.W2b = nullptr;
    a.tw = c.px.tw;
    a.Mx = d.Mx;
    a.Px = d.Px;
    a.Pz = d.Pz;
    a.qpts = d.qpts;
    int nseq = (a.nf + 1) / 2;
    int zb = SC_FFT_NS::xmix_zblock(c, a.nf);
    a.ZB = zb;
    a.check_cfl = check_cfl;
    a.cfl1 = d.cfl1;
    a.cfl3 = d.cfl3;
    a.cfl2 = c.dcfl2;
    a.cflmax = c.cflmax;
    a.flow = flow;
    a.abort_flag = c.abort_flag;
    a.ms_in = rstride(c, W1);
    a.ms_inb = rstride(c, a.W1b);
    a.ms_inc = 0;
    a.ms_out = rstride(c, W2);
    a.ms_outb = 0;
    // the physical output exists for one member
    const int nm = mode == XM_PHYS ? 1 : c.nrun;
    const double rows = (double) sizeof(real2) * d.qpts * d.Pz * d.Mx;
    double bytes = nm * rows * (a.nf + a.nout);
    if (mode == XM_PHYS) bytes += 8.0 * 3 * d.Px * d.qpts * d.Pz;
    const hipStream_t st = c.stream;
    const real2 *W1r = (const real2 *) W1;
    real2 *W2r = (real2 *) W2;
    // the CFL maximum accumulates across launches, so a replay skips it
    XmixArgs ar = a;
    ar.check_cfl = 0;
    std::function<void()> go, again;
    a.nm = ar.nm = nm;
    Fixed<XrowKernel> shared;
    if (mode == XM_TANGENT && W1b && nf1 == 6 && a.ms_in == 0) shared = xrow_shared_fixed(d.Px, d.Pz, nm);
    if (shared.kernel) {
        // members along one trajectory: all of them in a block, unless that leaves
        // fewer than four blocks a CU
        const int blocks = (d.qpts * d.Pz + shared.group - 1) / shared.group;
        const dim3 grid(blocks, std::max(1, std::min(nm, 1024 / blocks)));
        go = [=]() { hipLaunchKernelGGL(shared.kernel, grid, dim3(shared.threads), shared.lds, st, a, W1r, W2r); };
        again = [=]() { hipLaunchKernelGGL(shared.kernel, grid, dim3(shared.threads), shared.lds, st, ar, W1r, W2r); };
    } else if (const auto fx = xrow_kernel(mode, d); fx.kernel) {
        const dim3 grid((d.qpts * d.Pz + fx.group - 1) / fx.group, nm);
        go = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, a, W1r, W2r); };
        again = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, ar, W1r, W2r); };
    } else {
        const dim3 grid(d.Pz / zb, d.qpts, nm);
        const size_t lds = sizeof(real2) * (zb * nseq * (d.Px + 1) + d.Px);
        const PlanDev pd = to_dev(c.px);
        const XmixKernel kern = xmix_kernel(mode);
        go = [=]() { hipLaunchKernelGGL(kern, grid, dim3(BLK), lds, st, a, pd, W1r, W2r); };
        again = [=]() { hipLaunchKernelGGL(kern, grid, dim3(BLK), lds, st, ar, pd, W1r, W2r); };
    }
    prof_begin(c, st, 2, bytes);
    go();
    // replays only the modes whose launches are side-effect free
    if (mode == XM_ADJOINT || mode == XM_PRIMAL || mode == XM_TANGENT)
        prof_end(c, st, 2, again);
    else
        prof_end(c, st, 2);
}

bool xmix_adj2_available(Context &c) { return xrow_kernel(XM_ADJ2, c.d).kernel != nullptr; }

void launch_xmix_adj2(Context &c, const cplx *Wa, const cplx *Wb, const cplx *Wl, cplx *W2,
                      cplx *W2b)
{
    const Dims &d = c.d;
    XmixArgs a;
    a.mode = XM_ADJ2;
    a.nf = 15;
    a.nout = 12;
    a.nf1 = 6;
    a.W1b = (const real2 *) Wb;
    a.nf2 = 12;
    a.W1c = (const real2 *) Wl;
    a.W2b = (real2 *) W2b;
    a.tw = c.px.tw;
    a.Mx = d.Mx;
    a.Px = d.Px;
    a.Pz = d.Pz;
    a.qpts = d.qpts;
    const auto fx = xrow_kernel(XM_ADJ2, d);
    a.ZB = fx.group;
    a.check_cfl = 0;
    a.cfl1 = d.cfl1;
    a.cfl3 = d.cfl3;
    a.cfl2 = c.dcfl2;
    a.cflmax = c.cflmax;
    a.flow = nullptr;
    a.abort_flag = c.abort_flag;
    a.ms_in = rstride(c, Wa);
    a.ms_inb = rstride(c, Wb);
    a.ms_inc = rstride(c, Wl);
    a.ms_out = rstride(c, W2);
    a.ms_outb = rstride(c, W2b);
    const dim3 grid((d.qpts * d.Pz + fx.group - 1) / fx.group, c.nrun);
    const double bytes = c.nrun * (double) sizeof(real2) * d.qpts * d.Pz * d.Mx * (a.nf + a.nout);
    const hipStream_t st = c.stream;
    const real2 *War = (const real2 *) Wa;
    real2 *W2r = (real2 *) W2;
    auto go = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, a, War, W2r); };
    prof_begin(c, st, 7, bytes);
    go();
    prof_end(c, st, 7, go);
}

int xmix_zblock(Context &c, int nf)
{
    int nseq = (nf + 1) / 2, zb = 1;
    while (zb * 2 <= c.d.Pz && zb * 2 <= 64 && c.d.Pz % (zb * 2) == 0 &&
           (size_t) zb * 2 * nseq * (c.d.Px + 1) + c.d.Px <= (size_t) XMIX_TILE)
        zb *= 2;
    return zb;
}

void launch_zfwd(Context &c, const cplx *W2, int nout, cplx *dst, int dst_kind, int cfl_slot)
{
    const Dims &d = c.d;
    ZfwdArgs a;
    a.cfl_slot = cfl_slot;
    a.cflmax = c.cflmax;
    a.dt = d.dt;
    a.abort_rw = c.abort_flag;
    a.nout = nout;
    a.Nz = d.Nz;
    a.Mx = d.Mx;
    a.Pz = d.Pz;
    a.qpts = d.qpts;
    a.tw = c.pz.tw;
    a.nm = c.nrun;
    a.XB = pick_block(d.Mx, d.Pz, 1);
    a.dst_kind = dst_kind;
    a.norm = 1.0 / ((3. * d.Nx / 2.) * (3. * d.Nz / 2.));
    a.abort_flag = c.abort_flag;
    a.ms_in = rstride(c, W2);
    a.ms_out = mstride(c, dst);
    a.p32 = dst_kind == ZF_USLOTS && prods32(c);
    double bytes = c.nrun * (double) d.qpts * d.Mx * nout *
                   (sizeof(real2) * d.Pz + (a.p32 ? 8.0 : 16.0) * (d.Nz - 1));
    const hipStream_t st = c.stream;
    const real2 *W2r = (const real2 *) W2;
    std::function<void()> go;
    if (const auto fx = zfwd_fixed(d.Pz, d.Mx); fx.kernel) {
        const int ncb = (d.qpts * d.Mx + fx.group - 1) / fx.group;
        const dim3 grid(xcd_grid(c.nrun * ncb * nout));
        go = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, a, W2r, dst); };
    } else {
        const dim3 grid((d.Mx + a.XB - 1) / a.XB, nout * c.nrun, d.qpts);
        const size_t lds = sizeof(real2) * (a.XB * d.Pz + d.Pz);
        const PlanDev pd = to_dev(c.pz);
        go = [=]() { hipLaunchKernelGGL(k_zfwd, grid, dim3(BLK), lds, st, a, pd, W2r, dst); };
    }
    prof_begin(c, st, 3, bytes);
    go();
    prof_end(c, st, 3, go);
}

// the fused transform + assembly; false when its tile does not fit (the
// caller then transforms into scratch and assembles separately)
bool launch_zfwd_adj(Context &c, const cplx *W2, cplx *Udst)
{
    return SC_FFT_NS::launch_zfwd_adj2(c, W2, Udst, nullptr, nullptr);
}

bool launch_zfwd_adj2(Context &c, const cplx *W2, cplx *Udst, const cplx *W2b, cplx *Udstb)
{
    const Dims &d = c.d;
    const auto fx = zadj_fixed(d.Pz, d.Mx);
    // the pair in one grid only with a fixed-length kernel
    if (W2b && !fx.kernel) {
        if (!SC_FFT_NS::launch_zfwd_adj2(c, W2, Udst, nullptr, nullptr)) return false;
        return SC_FFT_NS::launch_zfwd_adj2(c, W2b, Udstb, nullptr, nullptr);
    }
    ZadjArgs a;
    a.nprob = W2b ? 2 : 1;
    a.W2b = (const real2 *) W2b;
    a.Ub = Udstb;
    a.Nz = d.Nz;
    a.Mx = d.Mx;
    a.Pz = d.Pz;
    a.qpts = d.qpts;
    a.tw = c.pz.tw;
    // generic tile: 6 XA Pz values and the twiddles within FFT_TILE
    a.XA = fx.kernel ? fx.group : std::min(d.Mx, (FFT_TILE - d.Pz) / (6 * d.Pz));
    if (a.XA < 1) return false;
    a.norm = 1.0 / ((3. * d.Nx / 2.) * (3. * d.Nz / 2.));
    a.Kx = c.dKx;
    a.Kz = c.dKz;
    a.abort_flag = c.abort_flag;
    a.nm = c.nrun;
    a.ms_in = rstride(c, W2);
    a.ms_out = mstride(c, Udst);
    a.p32 = prods32(c);
    if (W2b && (rstride(c, W2b) != a.ms_in || mstride(c, Udstb) != a.ms_out)) return false;
    double bytes = a.nm * a.nprob * (double) d.qpts * d.Mx *
                   (sizeof(real2) * 6.0 * d.Pz + (a.p32 ? 8.0 : 16.0) * 5.0 * (d.Nz - 1));
    const hipStream_t st = c.stream;
    const real2 *W2r = (const real2 *) W2;
    std::function<void()> go;
    if (fx.kernel) {
        const int ncb = (d.qpts * d.Mx + fx.group - 1) / fx.group;
        const dim3 grid(xcd_grid(a.nm * a.nprob * ncb));
        go = [=]() { hipLaunchKernelGGL(fx.kernel, grid, dim3(fx.threads), fx.lds, st, a, W2r, Udst); };
    } else {
        const dim3 grid((d.Mx + a.XA - 1) / a.XA, d.qpts, a.nm);
        const size_t lds = sizeof(real2) * (6 * (size_t) a.XA * d.Pz + d.Pz);
        const PlanDev pd = to_dev(c.pz);
        go = [=]() { hipLaunchKernelGGL(k_zfwd_adj, grid, dim3(BLK), lds, st, a, pd, W2r, Udst); };
    }
    prof_begin(c, st, 3, bytes);
    go();
    prof_end(c, st, 3, go);
    return true;
}

void launch_assemble_adj(Context &c, const cplx *SP, cplx *Udst)
{
    const Dims &d = c.d;
    size_t n = (size_t) d.Nz * d.qpts * d.Mx;
    int blocks = (int) std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_assemble_adj, dim3(blocks, c.nrun), dim3(256), 0, c.stream, SP, Udst,
                       c.dKx, c.dKz, d.Nz, d.qpts, d.Mx, c.abort_flag, mstride(c, SP),
                       mstride(c, Udst), (int) prods32(c));
}

}  // namespace SC_FFT_NS
}  // namespace sc
