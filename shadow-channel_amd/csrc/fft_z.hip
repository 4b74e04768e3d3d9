// The z transforms for the lengths with a compile-time plan: the inverse
// transforms of the velocity and vorticity slots, the forward transforms of
// the products, and the adjoint's forward transforms with the assembly of its
// five slots (channel/pass1.c:52-114, 312-371; channel/pass2.c:128-221,
// 417-566).  Compiled once per precision.
//
// These kernels stream: their reads and writes are the bound.  Blocks take
// whole groups of the flattened column index c = y Nx/2 + x, which is
// contiguous in a slot of U for every kz row, so that no lane is idle whatever
// Nx, and the first pass reads from and the last pass writes to memory (LDS is
// crossed once per pass boundary).  The tiles of one column group (its fields)
// follow each other in the XCD-aware order, so the slots that several fields
// read come from one L2.
#include "fft_common.h"

#include <type_traits>

namespace sc {
namespace SC_FFT_NS {

constexpr int ZT = 256;                                   // threads

// columns of a block: 16 where the tile stays within 30 KB in FP64, else 8
constexpr int zcols(int pz) { return 16 * pz <= 1900 ? 16 : 8; }

template <int PZ> struct ZPlan {
    static constexpr int XB = zcols(PZ), NZ = 2 * PZ / 3;
    static constexpr size_t LDS = sizeof(real2) * (XB * PZ + PZ);
};

// the inputs of a first-pass butterfly: rows zp = j + q NB1 of column c of one
// field, from the state slots, the vorticity formed on the fly in FP64; rows in
// the zero band (the Nyquist row and the padding) are zero
template <int KIND, int PZ, bool S32>
__device__ __forceinline__ void zinv_rows(const ZinvArgs &a, const cplx *src, int slot, size_t ss,
                                          size_t zs, double kx, int j, real2 *v)
{
    constexpr int Nz = 2 * PZ / 3, R1 = plan_radix(PZ, 0), NB1 = PZ / R1;
#pragma unroll
    for (int q = 0; q < R1; ++q) {
        if (q * NB1 >= Nz / 2 && q * NB1 + NB1 - 1 <= Nz) {
            v[q] = mk2(0.0, 0.0);
            continue;
        }
        const int zp = j + q * NB1;
        const int kz = zp < Nz / 2 ? zp : (zp > Nz ? zp - Nz / 2 : -1);
        const int kzi = max(kz, 0);
        const size_t bp = kzi * zs;
        const double kzv = (kzi <= Nz / 2 ? kzi : kzi - Nz) * a.az;
        double2 val;
        if (KIND == FK_SLOT) {
            val = ld_slot<S32>(src, bp + slot * ss);
        } else if (KIND == FK_OMEGA_Z) {                // -du/dy + i kx v
            const double2 du = ld_slot<S32>(src, bp + 3 * ss), vv = ld_slot<S32>(src, bp + 1 * ss);
            val = make_double2(-fma_(kx, vv.y, du.x), fma_(kx, vv.x, -du.y));
        } else if (KIND == FK_OMEGA_X) {                // dw/dy - i kz v
            const double2 dw = ld_slot<S32>(src, bp + 4 * ss), vv = ld_slot<S32>(src, bp + 1 * ss);
            val = make_double2(fma_(kzv, vv.y, dw.x), fma_(-kzv, vv.x, dw.y));
        } else {                                        // i kz u - i kx w
            const double2 u = ld_slot<S32>(src, bp), w = ld_slot<S32>(src, bp + 2 * ss);
            val = make_double2(fma_(kx, w.y, -(kzv * u.y)), fma_(kzv, u.x, -(kx * w.x)));
        }
        v[q] = kz >= 0 ? to_real2(val) : mk2(0.0, 0.0);
    }
}

// tile (member, column group, field), fields fastest
template <int PZ, bool S32, bool EVEN>
__global__ __launch_bounds__(ZT) void k_zinv_c(ZinvArgs a, real2 *W1)
{
    constexpr int XB = ZPlan<PZ>::XB, R1 = plan_radix(PZ, 0), NP = plan_best(PZ).passes;
    constexpr int RL = plan_radix(PZ, NP - 1), NSL = PZ / RL;
    extern __shared__ __align__(16) char lds_raw[];
    if (*a.abort_flag) return;
    const int Mx = a.Mx, nc = a.qpts * Mx, ncb = (nc + XB - 1) / XB, nf = a.fs.nf;
    const int tile = xcd_tile(a.nm * ncb * nf);
    if (tile < 0) return;
    const int cbm = tile / nf, f = tile - cbm * nf, m = cbm / ncb, cb = cbm - m * ncb;
    real2 *lds = (real2 *) lds_raw, *twl = lds + XB * PZ;
    // this thread's column in every pass (ZT is a multiple of XB)
    const int c0 = cb * XB + (int) threadIdx.x % XB, c = min(c0, nc - 1);
    const int y = c / Mx, x = c - y * Mx;
    const size_t ss = (size_t) nc, zs = 5 * ss;
    const int slot = a.fs.slot[f], kind = a.fs.kind[f];
    const cplx *src = a.fs.src[f] + m * a.fs.ms[f];
    if constexpr (S32) src = (const cplx *) ((const float2 *) src + c);
    else src += c;
    stage_twiddles_c<PZ, ZT>(a.tw, twl);
    const double kx = x * a.ax;
    auto first = [&](auto K) {
        constexpr int START = !EVEN ? DS_ANY : decltype(K)::value == FK_SLOT ? DS_ZINV_A : DS_ZINV_B;
        fft_first<START, PZ, XB, 1, XB, ZT>(lds, +1.0, [&](int j, int, real2 *v) {
            zinv_rows<decltype(K)::value, PZ, S32>(a, src, slot, ss, zs, kx, j, v);
        });
    };
    if (kind == FK_SLOT) first(std::integral_constant<int, FK_SLOT>());
    else if (kind == FK_OMEGA_Z) first(std::integral_constant<int, FK_OMEGA_Z>());
    else if (kind == FK_OMEGA_X) first(std::integral_constant<int, FK_OMEGA_X>());
    else first(std::integral_constant<int, FK_OMEGA_Y>());
    __syncthreads();
    lds_fft_c<PZ, XB, 1, XB, ZT, NP - 1, 1, R1>(lds, twl, +1.0);
    real2 *dst = W1 + m * a.ms_w1 + ((size_t) y * nf + f) * (PZ * Mx) + x;
    fft_last<PZ, XB, 1, XB, ZT>(lds, twl, +1.0, [&](int k, int, const real2 *v) {
        if (c0 >= nc) return;
#pragma unroll
        for (int q = 0; q < RL; ++q) dst[(k + q * NSL) * Mx] = v[q];
    });
}

// tile (member, column group, product), products fastest
template <int PZ, bool EVEN>
__global__ __launch_bounds__(ZT) void k_zfwd_c(ZfwdArgs a, const real2 *W2, cplx *dst)
{
    constexpr int XB = ZPlan<PZ>::XB, Nz = ZPlan<PZ>::NZ;
    constexpr int R1 = plan_radix(PZ, 0), NB1 = PZ / R1, NP = plan_best(PZ).passes;
    constexpr int RL = plan_radix(PZ, NP - 1), NSL = PZ / RL;
    extern __shared__ __align__(16) char lds_raw[];
    if (a.cfl_slot >= 0 && blockIdx.x == 0)
        cfl_check_block(a.cflmax, a.qpts, a.dt, a.abort_rw, a.cfl_slot);
    if (*a.abort_flag) return;
    const int Mx = a.Mx, nc = a.qpts * Mx, ncb = (nc + XB - 1) / XB, no = a.nout;
    const int tile = xcd_tile(a.nm * ncb * no);
    if (tile < 0) return;
    const int cbm = tile / no, g = tile - cbm * no, m = cbm / ncb, cb = cbm - m * ncb;
    real2 *lds = (real2 *) lds_raw, *twl = lds + XB * PZ;
    const int c0 = cb * XB + (int) threadIdx.x % XB, c = min(c0, nc - 1);
    const int y = c / Mx, x = c - y * Mx;
    const real2 *src = W2 + m * a.ms_in + ((size_t) y * no + g) * (PZ * Mx) + x;
    dst += m * a.ms_out;
    stage_twiddles_c<PZ, ZT>(a.tw, twl);
    fft_first<EVEN ? DS_FORWARD : DS_ANY, PZ, XB, 1, XB, ZT>(lds, -1.0, [&](int j, int, real2 *v) {
#pragma unroll
        for (int q = 0; q < R1; ++q) v[q] = src[(j + q * NB1) * Mx];
    });
    __syncthreads();
    lds_fft_c<PZ, XB, 1, XB, ZT, NP - 1, 1, R1>(lds, twl, -1.0);
    fft_last<PZ, XB, 1, XB, ZT>(lds, twl, -1.0, [&](int k, int, const real2 *v) {
        if (c0 >= nc) return;
#pragma unroll
        for (int q = 0; q < RL; ++q) {
            const int zp = k + q * NSL;                  // stored rows: kz < Nz/2, kz > Nz/2
            if (q * NSL >= Nz / 2 && q * NSL + NSL - 1 <= Nz) continue;
            const int kz = zp < Nz / 2 ? zp : zp - Nz / 2;
            if (zp >= Nz / 2 && zp <= Nz) continue;
            real2 s = v[q];
            s.x *= (real) a.norm;
            s.y *= (real) a.norm;
            if (a.dst_kind == ZF_USLOTS)
                st_slot(dst, ((size_t) kz * 5 + g) * nc + c, a.p32, s.x, s.y);
            else
                dst[((size_t) g * Nz + kz) * nc + c] = to_cplx(s);
        }
    });
}

// Forward z transforms of the six adjoint products with the assembly fused
// (channel/pass2.c:417-566), in two phases over one 3-field tile: S =
// (Sx, Sy, Sz) of the ZA columns is transformed first and each thread keeps the
// values of its (stored kz row, column) pairs; then T = (Tx, Ty, Tz) in the
// same LDS, and the thread forms its slots: Hz = -Tz - i kx Sy,
// Hx = -Tx + i kz Sy, Hy = -Ty - i kz Sx + i kx Sz, then S_x, S_z.  A tile of
// half the fields lets more blocks share a CU, which cover each other's loads.
#ifdef SC_FFT_F32
constexpr int ZA = 8;                                     // 64-byte column runs
#else
constexpr int ZA = 4;
#endif
template <int PZ, bool EVEN>
__global__ __launch_bounds__(ZT) void k_zadj_c(ZadjArgs a, const real2 *W2, cplx *U)
{
    constexpr int Nz = 2 * PZ / 3, NS = 3 * ZA, OWN = (ZA * (Nz - 1) + ZT - 1) / ZT;
    constexpr int R1 = plan_radix(PZ, 0), NB1 = PZ / R1, NP = plan_best(PZ).passes;
    extern __shared__ __align__(16) char lds_raw[];
    if (*a.abort_flag) return;
    const int Mx = a.Mx, nc = a.qpts * Mx, ncb = (nc + ZA - 1) / ZA;
    const int tile = xcd_tile(a.nm * a.nprob * ncb);
    if (tile < 0) return;
    const int prob = tile / ncb, m = prob / a.nprob, cb = tile - prob * ncb;
    if (prob - m * a.nprob) {
        W2 = a.W2b;                                       // the second problem's tiles
        U = a.Ub;
    }
    W2 += m * a.ms_in;
    U += m * a.ms_out;
    real2 *lds = (real2 *) lds_raw, *twl = lds + NS * PZ;
    stage_twiddles_c<PZ, ZT>(a.tw, twl);
    const int xl = threadIdx.x % ZA;                      // this thread's column (ZT % ZA == 0)
    const int c0 = cb * ZA + xl, c = min(c0, nc - 1), y = c / Mx, x = c - y * Mx;
    // phase h: element (zp, f, xl) of field 3h + f at (zp 3 + f) ZA + xl
    auto phase = [&](int h, real2 (*P)[3]) {
        fft_first<EVEN ? DS_FORWARD : DS_ANY, PZ, NS, 1, NS, ZT>(lds, -1.0, [&](int j, int s, real2 *v) {
            // a sequence's column is not the thread's own where ZT % NS != 0
            const int f = s / ZA, cc = min(cb * ZA + s - f * ZA, nc - 1), yy = cc / Mx;
            const real2 *src = W2 + ((size_t) yy * 6 + 3 * h + f) * (PZ * Mx) + (cc - yy * Mx);
#pragma unroll
            for (int q = 0; q < R1; ++q) v[q] = src[(j + q * NB1) * Mx];
        });
        __syncthreads();
        lds_fft_c<PZ, NS, 1, NS, ZT, NP, 1, R1>(lds, twl, -1.0);
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int r = threadIdx.x / ZA + o * (ZT / ZA), kz = r < Nz / 2 ? r : r + 1;
            const int zp = min(kz < Nz / 2 ? kz : kz + Nz / 2, PZ - 1);
#pragma unroll
            for (int f = 0; f < 3; ++f) P[o][f] = lds[(zp * 3 + f) * ZA + xl];
        }
    };
    real2 S[OWN][3], Tt[OWN][3];
    phase(0, S);
    __syncthreads();                                      // S read before T is stored
    phase(1, Tt);
    if (c0 >= nc) return;
    const double kx = a.Kx[x];
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
        const int r = threadIdx.x / ZA + o * (ZT / ZA);
        if (r >= Nz - 1) continue;
        const int kz = r < Nz / 2 ? r : r + 1;            // skip the Nyquist row
        st_adjoint(U, ((size_t) kz * 5) * nc + c, (size_t) nc, a.p32, (real) a.norm, kx, a.Kz[kz], S[o], Tt[o]);
    }
}

template <class K>
static Fixed<K> fixed(K kernel, int group, size_t lds)
{
    Fixed<K> f;
    f.kernel = kernel;
    f.group = group;
    f.threads = ZT;
    f.lds = lds;
    return f;
}

// the instance for a length: both first-pass orders exist for the lengths with
// an order of their own
#define SC_PICK(N, NAME, ...) \
    (start_length(N) && even_columns(Mx) ? NAME<N, __VA_ARGS__ start_length(N)> : NAME<N, __VA_ARGS__ false>)
#define SC_ARG(A) A,

Fixed<ZinvKernel> zinv_fixed(int Pz, int Mx, bool s32)
{
    switch (Pz) {
#ifdef SC_FFT_F32
#define SC_ONE(N)                                                                              \
    case N:                                                                                    \
        return fixed<ZinvKernel>(s32 ? SC_PICK(N, k_zinv_c, SC_ARG(true)) : SC_PICK(N, k_zinv_c, SC_ARG(false)), \
                                 ZPlan<N>::XB, ZPlan<N>::LDS);
#else
#define SC_ONE(N) \
    case N: return fixed<ZinvKernel>(SC_PICK(N, k_zinv_c, SC_ARG(false)), ZPlan<N>::XB, ZPlan<N>::LDS);
#endif
        SC_Z_LENGTHS(SC_ONE)
#undef SC_ONE
    default: return Fixed<ZinvKernel>();
    }
}

Fixed<ZfwdKernel> zfwd_fixed(int Pz, int Mx)
{
    switch (Pz) {
#define SC_ONE(N) \
    case N: return fixed<ZfwdKernel>(SC_PICK(N, k_zfwd_c, ), ZPlan<N>::XB, ZPlan<N>::LDS);
        SC_Z_LENGTHS(SC_ONE)
#undef SC_ONE
    default: return Fixed<ZfwdKernel>();
    }
}

Fixed<ZadjKernel> zadj_fixed(int Pz, int Mx)
{
    switch (Pz) {
#define SC_ONE(N) \
    case N: return fixed<ZadjKernel>(SC_PICK(N, k_zadj_c, ), ZA, sizeof(real2) * (3 * ZA * N + N));
        SC_Z_LENGTHS(SC_ONE)
#undef SC_ONE
    default: return Fixed<ZadjKernel>();
    }
}

}  // namespace SC_FFT_NS
}  // namespace sc
