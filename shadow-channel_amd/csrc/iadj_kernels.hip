// Incremental adjoint stage: one Runge-Kutta stage k of the second-order
// (incremental) adjoint over every mode, increadjproject0
// (channel/increadjproject0.c:14-357) for (kx, kz) = (0, 0) and
// increadjproject (channel/increadjproject.c:10-645) for the others, as the
// driver loop calls them (shan/increadjoint_test7.c:673-685):
//   - right-hand side: at k = 0 the explicit operator on IAC plus the tangent
//     coupling re dt (a0 + b0) V MIC[count] (V the viscous part); the
//     Galerkin projection of the stage's products (IU: H slots, S_x, S_z as
//     the adjoint's); the forcing; the wall-lift terms of Uxb, Uzb, their
//     values Uxbt, Uzbt at the previous stage and the adjoint walls AUxb,
//     AUzb;
//   - the implicit solve (stride-2 band LU without pivoting, per parity);
//   - the Gauss-point values IAU with the wall lifts and the wall values
//     IAUxb, IAUzb;
//   - for k < 2 the next stage's explicit part from the products LIU and
//     MIC[count - 1].
// Layouts as the reference's arrays (complex {re, im}, kx fastest):
//   IAC [Nz][2][dimR][Mx], IU, LIU, IAU [Nz][5][qpts][Mx],
//   walls [6][Nz][Mx] (Uxb, Uzb, Uxbt, Uzbt, AUxb, AUzb), IAUb [2][Nz][Mx],
//   forcing [2 stages][2 sides: alpha, beta][Nz][Mx][dimR].
//
// The Galerkin projections of IU and LIU are the adjoint's (the same
// operator on other products) and run on the adjoint path's FP64 matrix-core
// kernels in one launch; so does the y-transform to the Gauss points, on the
// solved coefficients with the omega_y coefficients beyond dimQ cleared (the
// reference's sums stop there), the wall lifts added after it by a streaming
// pass.  What is particular to this stage (right-hand sides, lifts, tangent
// coupling, band solves, wall values, next stage's explicit part) is one
// kernel over the modes: IA_XG neighbouring kx columns of one kz row per
// block, one band row per thread; the implicit operators are the adjoint's,
// whose LU factors the setup stores, so each parity chain (one per thread)
// only substitutes.
#include "sc_internal.h"

#include <algorithm>

namespace sc {

namespace {

constexpr int IA_XG = 4;          // kx columns per block
typedef double v2d __attribute__((ext_vector_type(2)));   // stays in registers in arrays
constexpr int IA_THREADS = 256;   // rows: alpha on threads 0..127, beta on 128..255

// adjoint RK3/CN coefficients (channel/increadjproject.c:34-37)
__constant__ double kA[3] = {1. / 3., -1. / 2, 1. / 3.};
__constant__ double kB[3] = {2. / 3, 1. / 6, 0.};
__constant__ double kC[3] = {1., 1. / 3., 1. / 2.};
__constant__ double kD[3] = {0., -2. / 3, -1. / 6};
// Galerkin projections of the wall lifts (channel/increadjproject.c:40-46):
// LG[i] = 2 (R_i, (1-y)/2), LX[i] = (Q_i, lv), LR[i] = 2 (Q_i, lv''),
// lv = (1-y)^2 (1+y)/4; zero beyond these entries
__constant__ double kLG[4] = {4. / 3., -4. / 15., -4. / 15., 4. / 35.};
__constant__ double kLR[8] = {-16. / 15., 16. / 35., 32. / 105., -32. / 105.,
                              -16. / 315., 16. / 231., 0., 0.};
__constant__ double kLX[8] = {8. / 35., -8. / 315., -8. / 105., 8. / 385.,
                              8. / 385., -8. / 1001., -8. / 3003., 8. / 6435.};

struct IadjArgs {
    const cplx *IU, *LIU, *W, *F, *mic0, *mic1;
    // projections of IU (Fa, Fb) and LIU (FLa, FLb): [Nz][dimQ|dimR][Mx]
    const cplx *Fa, *Fb, *FLa, *FLb;
    cplx *IAC, *IAU, *IAUb;
    cplx *Ctr;             // solved coefficients for the y-transform
    const double *Kx, *Kz, *Qs, *Qps, *Qpps, *Rs, *Rps, *Rp0;
    const double *tRw, *tRpw;   // [q][dimR]: Rw, Rpw transposed
    // LU factors of the stage's implicit operators (the adjoint's): the solve
    // images of the setup (alpha La, beta Lb: blocks of sbt columns over columns
    // z Mx + x, rows z <= Nz/2 only when mirror) and the mean's
    const double *La, *Lb, *Lm;
    int sbt, mirror;
    const double *lift;    // [4][q]: lv, lv', lv'', lg
    const double *mlift;   // [dimR]: sum_j Rw[i][j] (1 - y_j)/2
    int Nz, Mx, q, dQ, dR, k;
    double re, dt;
};

__device__ __forceinline__ cplx cadd(cplx a, cplx b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ cplx cscale(cplx a, double s) { return make_double2(a.x * s, a.y * s); }

// Forward and back substitution of one part (real or imaginary) of the nr rows
// of one parity of a stride-2 band system (no pivoting), in LDS: row r at v[4 r],
// its factors at L[r XG DL + m - 1] = L(r + m - 1, m), U[r XG DL + m - 1] =
// U(r, r + m) and D[r XG] = 1 / U(r, r), for rows up to the next multiple of
// eight (zero past the chain).  Nearest terms first in both sweeps; the last DL
// values stay in registers, and the operands of eight rows are read while the
// eight before them are computed.
template <int DL, int XG>
__device__ __forceinline__ void chain_subst(double *v, const double *L, const double *U, const double *D, int nr)
{
    constexpr int B = 8, FR = XG * DL;
    const int nrp = (nr + B - 1) / B * B;
    double y[DL], f[B][DL], b[B], d[B];
#pragma unroll
    for (int m = 0; m < DL; ++m) y[m] = 0.0;
    auto fwd = [&](int r0) {
#pragma unroll
        for (int i = 0; i < B; ++i) {
            // rows before the first multiply zeros
#pragma unroll
            for (int m = 0; m < DL; ++m) f[i][m] = L[max(r0 + i - m, 0) * FR + m];
            b[i] = v[4 * min(r0 + i, nr - 1)];
        }
    };
    if (nr > 0) fwd(0);
    for (int r0 = 0; r0 < nrp; r0 += B) {
        double fc[B][DL], bc[B];
#pragma unroll
        for (int i = 0; i < B; ++i) {
#pragma unroll
            for (int m = 0; m < DL; ++m) fc[i][m] = f[i][m];
            bc[i] = b[i];
        }
        if (r0 + B < nrp) fwd(r0 + B);
#pragma unroll
        for (int i = 0; i < B; ++i) {
            double x = bc[i];
#pragma unroll
            for (int m = 0; m < DL; ++m) x = __builtin_fma(-fc[i][m], y[m], x);
#pragma unroll
            for (int m = DL - 1; m > 0; --m) y[m] = y[m - 1];
            y[0] = x;
            if (r0 + i < nr) v[4 * (r0 + i)] = x;
        }
    }
#pragma unroll
    for (int m = 0; m < DL; ++m) y[m] = 0.0;
    auto bwd = [&](int r0) {
#pragma unroll
        for (int i = 0; i < B; ++i) {
#pragma unroll
            for (int m = 0; m < DL; ++m) f[i][m] = U[(r0 + i) * FR + m];
            b[i] = r0 + i < nr ? v[4 * (r0 + i)] : 0.0;
            d[i] = D[(r0 + i) * XG];
        }
    };
    if (nr > 0) bwd(nrp - B);
    for (int r0 = nrp - B; r0 >= 0; r0 -= B) {
        double fc[B][DL], bc[B], dc[B];
#pragma unroll
        for (int i = 0; i < B; ++i) {
#pragma unroll
            for (int m = 0; m < DL; ++m) fc[i][m] = f[i][m];
            bc[i] = b[i];
            dc[i] = d[i];
        }
        if (r0 >= B) bwd(r0 - B);
#pragma unroll
        for (int i = B - 1; i >= 0; --i) {
            double x = bc[i];
#pragma unroll
            for (int m = 0; m < DL; ++m) x = __builtin_fma(-fc[i][m], y[m], x);
            x *= dc[i];
#pragma unroll
            for (int m = DL - 1; m > 0; --m) y[m] = y[m - 1];
            y[0] = x;
            if (r0 + i < nr) v[4 * (r0 + i)] = x;
        }
    }
}

// Row i of the operator (alpha: -(k2 Qs + Qps) + cv V, V = k2^2 Qs + 2 k2 Qps +
// Qpps; beta: Rs - cv V, V = -(Rps + k2 Rs)) on v and of the viscous part V on m
// (rows in LDS): e, mm.  No column is skipped: the Gram bands are zero outside the
// matrix, and what they meet there is a zero of its own (a clamped column would
// be one of the other parity's, and that need not be finite).  Qps reaches three
// off-diagonals of the four, Qpps two, Rps one of two.
template <bool B>
struct BandRow {
    static constexpr int DL = B ? 2 : 4, W = 2 * DL + 1;
    double s[W], p[W], pp[W];
    __device__ __forceinline__ void load(const IadjArgs &a, int i)
    {
#pragma unroll
        for (int o = 0; o < W; ++o) {
            s[o] = (B ? a.Rs : a.Qs)[i * W + o];
            p[o] = o > 0 && o < W - 1 ? (B ? a.Rps : a.Qps)[i * W + o] : 0.0;
            pp[o] = !B && o > 1 && o < W - 2 ? a.Qpps[i * W + o] : 0.0;
        }
    }
    __device__ __forceinline__ void apply(int i, int N, double k2, double cv, const cplx *v, const cplx *m,
                                          const cplx *zero, cplx &e, cplx &mm) const
    {
        e = mm = make_double2(0.0, 0.0);
        const double k4 = k2 * k2, t2 = 2. * k2;
#pragma unroll
        for (int o = 0; o < W; ++o) {
            const int col = i + 2 * (o - DL);
            const bool in = o == DL || (o < DL ? col >= 0 : col < N);
            const bool hp = o > 0 && o < W - 1;
            const double ks = hp ? __builtin_fma(k2, s[o], p[o]) : k2 * s[o];     // k2 Qs + Qps
            double vs, ex;
            if (B) {
                vs = -ks;
                ex = __builtin_fma(cv, ks, s[o]);
            } else {
                vs = hp ? __builtin_fma(k4, s[o], t2 * p[o]) : k4 * s[o];
                if (o > 1 && o < W - 2) vs += pp[o];
                ex = __builtin_fma(cv, vs, -ks);
            }
            const cplx cv2 = *(in ? v + col : zero), mv = *(in ? m + col : zero);
            e.x = __builtin_fma(ex, cv2.x, e.x);
            e.y = __builtin_fma(ex, cv2.y, e.y);
            mm.x = __builtin_fma(vs, mv.x, mm.x);
            mm.y = __builtin_fma(vs, mv.y, mm.y);
        }
    }
};

// Right-hand sides of row i of the alpha (B = false) or beta coefficients of the
// block's columns
template <bool B, class Valid>
__device__ __forceinline__ void mode_rhs(const IadjArgs &a, int i, int z, int x0, double kz, const cplx *vec,
                                         const cplx *smic, const cplx *zero, const Valid &valid, cplx *acc)
{
    const int dQ = a.dQ, dR = a.dR, Mx = a.Mx, Nz = a.Nz, k = a.k, N = B ? dR : dQ;
    const double dt = a.dt, re = a.re;
    const size_t wp = (size_t) Nz * Mx;
    BandRow<B> g;
    if (k == 0) g.load(a, i);
#pragma unroll
    for (int t = 0; t < IA_XG; ++t) {
        acc[t] = make_double2(0.0, 0.0);
        if (!valid(t)) continue;
        const int x = x0 + t;
        const double kx = a.Kx[x], k2 = kx * kx + kz * kz;
        cplx c = vec[t * dR + i];
        if (k == 0) {
            cplx e, m;
            g.apply(i, N, k2, B ? -re * kA[0] * dt : re * kA[0] * dt, vec + t * dR,
                    smic + t * 2 * dR + (B ? dR : 0), zero, e, m);
            c = cadd(e, cscale(m, re * dt * (kA[0] + kB[0])));
        }
        cplx gf = B ? a.Fb[((size_t) z * dR + i) * Mx + x] : a.Fa[((size_t) z * dQ + i) * Mx + x];
        if (a.F) gf = cadd(gf, a.F[((((size_t) 0 * 2 + (B ? 1 : 0)) * Nz + z) * Mx + x) * dR + i]);
        c = cadd(c, cscale(gf, dt * kC[k]));
        const size_t wo = (size_t) z * Mx + x;
        if (!B && i < 8) {
            const cplx wb = a.W[wp + wo], wbt = a.W[3 * wp + wo], awb = a.W[5 * wp + wo];
            const double mm = kLR[i] / 2. - k2 * kLX[i], vv = -k2 * kLR[i] + k2 * k2 * kLX[i];
            c.x += mm * (wbt.x - wb.x) + dt * re * (kA[k] * wbt.x + kB[k] * wb.x) * vv +
                   dt * re * (kA[k] + kB[k]) * awb.x * vv;
            c.y += mm * (wbt.y - wb.y) + dt * re * (kA[k] * wbt.y + kB[k] * wb.y) * vv +
                   dt * re * (kA[k] + kB[k]) * awb.y * vv;
        }
        if (B && i < 4) {
            const cplx ub = a.W[wo], ubt = a.W[2 * wp + wo], aub = a.W[4 * wp + wo];
            const double h = kLG[i] / 2.;
            c.x += h * (ubt.x - ub.x) + dt * re * (kA[k] * ubt.x + kB[k] * ub.x) * (-k2 * h) +
                   dt * re * (kA[k] + kB[k]) * aub.x * (-k2 * h);
            c.y += h * (ubt.y - ub.y) + dt * re * (kA[k] * ubt.y + kB[k] * ub.y) * (-k2 * h) +
                   dt * re * (kA[k] + kB[k]) * aub.y * (-k2 * h);
        }
        acc[t] = c;
    }
}

// Row i of the next stage's explicit part: projections of LIU, forcing k + 1,
// MIC[count - 1]
template <bool B, class Valid>
__device__ __forceinline__ void mode_next(const IadjArgs &a, int i, int z, int x0, double kz, const cplx *vec,
                                          const cplx *smic, const cplx *zero, const Valid &valid)
{
    const int dQ = a.dQ, dR = a.dR, Mx = a.Mx, Nz = a.Nz, k = a.k, N = B ? dR : dQ;
    const double dt = a.dt, re = a.re;
    BandRow<B> g;
    g.load(a, i);
#pragma unroll
    for (int t = 0; t < IA_XG; ++t) {
        if (!valid(t)) continue;
        const int x = x0 + t;
        const double kx = a.Kx[x], k2 = kx * kx + kz * kz;
        cplx e, m;
        g.apply(i, N, k2, B ? -re * kA[k + 1] * dt : re * kA[k + 1] * dt, vec + t * dR,
                smic + t * 2 * dR + (B ? dR : 0), zero, e, m);
        cplx gf = B ? a.FLb[((size_t) z * dR + i) * Mx + x] : a.FLa[((size_t) z * dQ + i) * Mx + x];
        if (a.F) gf = cadd(gf, a.F[((((size_t) 1 * 2 + (B ? 1 : 0)) * Nz + z) * Mx + x) * dR + i]);
        const cplx c = cadd(cadd(e, cscale(gf, dt * kD[k + 1])), cscale(m, re * dt * (kA[k + 1] + kB[k + 1])));
        a.IAC[((size_t) (z * 2 + (B ? 1 : 0)) * dR + i) * Mx + x] = c;
    }
}

// the (0, 0) mode (channel/increadjproject0.c:14-357), one block.  It is the
// longest of the launch, a chain of latencies, so whatever does not depend on the
// solve is requested at once: both stages' products are projected in one pass over
// the weights (32 Gauss points' in flight), the solve's factors wait in LDS.
__device__ void iadj_mean(const IadjArgs &a, cplx *sh)
{
    const int q = a.q, dR = a.dR, Mx = a.Mx, Nz = a.Nz, k = a.k, tid = threadIdx.x;
    const int lane = tid & 63;
    const size_t plane = (size_t) q * Mx, wp = (size_t) Nz * Mx;
    const double dt = a.dt, re = a.re;
    const int nrp = solve_rows(dR);
    cplx *sal = sh, *sbe = sh + dR, *smic = sh + 2 * dR;          // smic [2][2][dR]: MIC[count], MIC[count - 1]
    double *sp = (double *) (sh + 6 * dR);                        // [2][4][q]: Hx, Sz, Hz, Sx (real) of IU, LIU
    double *sfac = sp + 8 * q;                                    // [2][nrp][5]
    const cplx ub = a.W[0], wb = a.W[wp], ubt = a.W[2 * wp], wbt = a.W[3 * wp];
    // alpha row r on threads < 128, beta row r on the others
    const bool isb = tid >= 128;
    const int r = isb ? tid - 128 : tid, rc = min(r, dR - 1);
    constexpr int PB = 32;
    double w0[PB], w1[PB];                                        // weights of PB Gauss points
    auto weights = [&](int j0) {
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const size_t j = min(j0 + u, q - 1);
            w0[u] = a.tRw[j * dR + rc];
            w1[u] = a.tRpw[j * dR + rc];
        }
    };
    BandRow<true> g;
    cplx fk = make_double2(0.0, 0.0), fn = fk;
    double ml;
    {
        // (q <= 195 and dR <= 128: one Gauss point and one row a thread)
        const size_t o = (size_t) min(tid, q - 1) * Mx, o0 = (size_t) rc * Mx, os = (size_t) (isb ? dR : 0) * Mx;
        const double u0 = a.IU[plane + o].x, u1 = a.IU[4 * plane + o].x, u2 = a.IU[o].x, u3 = a.IU[3 * plane + o].x;
        double l0 = 0.0, l1 = 0.0, l2 = 0.0, l3 = 0.0;
        cplx m0 = make_double2(0.0, 0.0), m1 = m0;
        const cplx c0 = a.IAC[os + o0];
        if (k == 0) m0 = a.mic0[os + o0];
        if (k < 2) {
            l0 = a.LIU[plane + o].x;
            l1 = a.LIU[4 * plane + o].x;
            l2 = a.LIU[o].x;
            l3 = a.LIU[3 * plane + o].x;
            m1 = a.mic1[os + o0];
        }
        double lf[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) lf[i] = a.Lm[min(tid + i * IA_THREADS, 10 * nrp - 1)];
        g.load(a, rc);
        ml = a.mlift[rc];
        if (a.F) {
            fk = a.F[((size_t) (isb ? 1 : 0) * Nz * Mx) * dR + rc];
            if (k < 2) fn = a.F[((size_t) (2 + (isb ? 1 : 0)) * Nz * Mx) * dR + rc];
        }
        weights(0);
        if (tid < q) {
            sp[tid] = u0; sp[q + tid] = u1; sp[2 * q + tid] = u2; sp[3 * q + tid] = u3;
            sp[4 * q + tid] = l0; sp[5 * q + tid] = l1; sp[6 * q + tid] = l2; sp[7 * q + tid] = l3;
        }
        if (r < dR) {
            (isb ? sbe : sal)[r] = c0;
            smic[(isb ? dR : 0) + r] = m0;
            smic[(isb ? 3 : 2) * dR + r] = m1;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (tid + i * IA_THREADS < 10 * nrp) sfac[tid + i * IA_THREADS] = lf[i];
    }
    __syncthreads();
    // f[r] = sum_j Rw Hx + Rpw Sz (alpha), Rw Hz - Rpw Sx (beta): real parts;
    // Rw, Rpw transposed ([q][dimR]); fl the same of LIU
    double f = 0.0, fl = 0.0;
    {
        const double *p0 = sp + (isb ? 2 * q : 0), *p1 = sp + (isb ? 3 * q : q);
        const double sg = isb ? -1.0 : 1.0;
        for (int j0 = 0; j0 < q; j0 += PB) {
            if (j0 > 0) weights(j0);
#pragma unroll
            for (int u = 0; u < PB; ++u)
                if (j0 + u < q) {
                    f += w0[u] * p0[j0 + u] + sg * w1[u] * p1[j0 + u];
                    fl += w0[u] * p0[4 * q + j0 + u] + sg * w1[u] * p1[4 * q + j0 + u];
                }
        }
    }
    cplx c = make_double2(0.0, 0.0);
    if (r < dR) {
        const cplx *v = isb ? sbe : sal;
        c = v[r];
        if (k == 0) {
            // Rs - re a0 dt Rps on the coefficients, - re dt (a0 + b0) Rps MIC[count]
            cplx e = make_double2(0.0, 0.0), m = make_double2(0.0, 0.0);
        #pragma unroll
            for (int o = 0; o < 5; ++o) {
                const int col = r + 2 * (o - 2);
                if (col < 0 || col >= dR) continue;
                const double ex = g.s[o] - re * kA[0] * dt * g.p[o];
                const cplx vv = v[col], mv = smic[(isb ? dR : 0) + col];
                e.x += ex * vv.x; e.y += ex * vv.y;
                m.x += g.p[o] * mv.x; m.y += g.p[o] * mv.y;
            }
            c = cadd(e, cscale(m, -(dt * re * (kA[0] + kB[0]))));
        }
        // only the real part of the stage's forcing reaches the right-hand side
        // (channel/increadjproject0.c:130-141)
        if (a.F) f += fk.x;
        c.x += dt * kC[k] * f;
        const cplx dw = isb ? make_double2(wbt.x - wb.x, wbt.y - wb.y)
                            : make_double2(ubt.x - ub.x, ubt.y - ub.y);
        c.x += ml * dw.x;
        c.y += ml * dw.y;
    }
    __syncthreads();
    if (r < dR) (isb ? sbe : sal)[r] = c;
    __syncthreads();
    // chains: alpha, beta (waves 0, 1), parity, part
    if ((tid & 63) < 4 && tid < 128) {
        const int pr = (tid >> 1) & 1, part = tid & 1;
        const double *L = sfac + pr * nrp * 5, *U = L + nrp * 2, *D = U + nrp * 2;
        chain_subst<2, 1>((double *) (tid < 64 ? sal : sbe) + 2 * pr + part, L, U, D, (dR - pr + 1) / 2);
    }
    __syncthreads();
    // the mean's Gauss-point values sum all dimR coefficients
    for (int i = tid; i < dR; i += IA_THREADS) {
        a.Ctr[(size_t) i * Mx] = sal[i];
        a.Ctr[((size_t) dR + i) * Mx] = sbe[i];
    }
    if (tid < 128) {
        // IAUxb, IAUzb: Rp0 . alpha - Uxb/2, Rp0 . beta - Uzb/2 (wave 0, wave 1)
        const cplx *v = tid < 64 ? sal : sbe;
        double xr = 0.0, xi = 0.0;
        for (int i = lane; i < dR; i += 64) {
            xr += a.Rp0[i] * v[i].x;
            xi += a.Rp0[i] * v[i].y;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            xr += __shfl_xor(xr, off);
            xi += __shfl_xor(xi, off);
        }
        const cplx wv = tid < 64 ? ub : wb;
        if (lane == 0) a.IAUb[tid < 64 ? 0 : wp] = make_double2(xr - wv.x / 2., xi - wv.y / 2.);
    }
    if (k == 2) {
        for (int i = tid; i < dR; i += IA_THREADS) {
            a.IAC[(size_t) i * Mx] = sal[i];
            a.IAC[((size_t) dR + i) * Mx] = sbe[i];
        }
        return;
    }
    if (r < dR) {
        const cplx *v = isb ? sbe : sal;
        cplx e = make_double2(0.0, 0.0), m = make_double2(0.0, 0.0);
        for (int o = 0; o < 5; ++o) {
            const int col = r + 2 * (o - 2);
            if (col < 0 || col >= dR) continue;
            const double ex = g.s[o] - re * kA[k + 1] * dt * g.p[o];
            const cplx vv = v[col], mv = smic[(isb ? 3 : 2) * dR + col];
            e.x += ex * vv.x; e.y += ex * vv.y;
            m.x += g.p[o] * mv.x; m.y += g.p[o] * mv.y;
        }
        cplx gf = make_double2(fl, 0.0);
        if (a.F) gf = cadd(gf, fn);
        const cplx c2 = cadd(cadd(e, cscale(gf, dt * kD[k + 1])),
                             cscale(m, -(dt * re * (kA[k + 1] + kB[k + 1]))));
        a.IAC[((size_t) (isb ? dR : 0) + r) * Mx] = c2;
    }
}

// Right-hand side, solve, wall values and next explicit part of the modes
// (kx, kz) != (0, 0), kz row != Nz/2: IA_XG kx columns of one kz row per
// block; the first block of the grid serves the mean mode (it runs longest).
// Bound by latency and the FP64 band rows.  At 64x97x64 92 -> 51 us (modes alone
// 72 -> 32, the mean alone 34 -> 32) with the factors requested at the start and the
// chains fed from LDS, real and imaginary parts on lanes of their own, and the
// band rows of alpha and beta in code of their own without a test per entry.
__global__ __launch_bounds__(IA_THREADS) void k_iadj_modes(IadjArgs a)
{
    extern __shared__ double2 sh[];
    const int dQ = a.dQ, dR = a.dR, Mx = a.Mx, Nz = a.Nz, k = a.k;
    const int nxg = (Mx + IA_XG - 1) / IA_XG;
    if (blockIdx.x == 0) {
        iadj_mean(a, sh);
        return;
    }
    const int z = (blockIdx.x - 1) / nxg, x0 = ((blockIdx.x - 1) % nxg) * IA_XG;
    const int nx = min(IA_XG, Mx - x0);
    const int tid = threadIdx.x;
    const size_t wp = (size_t) Nz * Mx;
    if (z == Nz / 2) {
        // cleared coefficients (zero Gauss-point values) and wall values
        for (int e = tid; e < 2 * dR * nx; e += IA_THREADS) {
            const int t = e % nx, r = e / nx;
            a.Ctr[((size_t) z * 2 * dR + r) * Mx + x0 + t] = make_double2(0.0, 0.0);
        }
        if (tid < 2 * nx) a.IAUb[(tid / nx) * wp + (size_t) z * Mx + x0 + tid % nx] = make_double2(0.0, 0.0);
        return;
    }
    cplx *zero = sh;                         // a zero (BandRow)
    cplx *sal = zero + 1;                    // [t][dR]
    cplx *sbe = sal + IA_XG * dR;            // [t][dR]
    // MIC[count] for the right-hand sides, the factors for the solves, then
    // MIC[count - 1]: [t][2][dR]
    cplx *smic = sbe + IA_XG * dR;
    const double kz = a.Kz[z];
    auto valid = [&](int t) { return t < nx && !(z == 0 && x0 + t == 0); };
    // MIC rows in registers, four values a thread (2 dR IA_XG <= 4 IA_THREADS)
    v2d mv[4];
    auto load_mic = [&](const cplx *mic) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = min(tid + i * IA_THREADS, 2 * dR * IA_XG - 1), r = e / IA_XG;     // r over [2][dR]
            mv[i] = *(const v2d *) &mic[((size_t) z * 2 * dR + r) * Mx + x0 + min(e % IA_XG, nx - 1)];
        }
    };
    auto put_mic = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = tid + i * IA_THREADS;
            if (e < 2 * dR * IA_XG) smic[(e % IA_XG) * 2 * dR + e / IA_XG] = make_double2(mv[i].x, mv[i].y);
        }
    };
    // The factors of the block's columns, eight rows of a parity at a time: a
    // thread's role in a row is two L or two U values of one column or one
    // inverse pivot (alpha: threads 0 .. 19 of 32, beta: the others).  They are
    // requested here and put into LDS, [parity][L, U, D][row][t], once the
    // right-hand sides no longer need it.
    const int nrq = solve_rows(dQ), nrr = solve_rows(dR);
    const int role = tid & 31, frow = tid >> 5;
    const bool fb = role >= 20, fd = fb ? role >= 28 : role >= 16;         // beta, inverse pivot
    const int fe = fb ? role - (fd ? 28 : role >= 24 ? 24 : 20) : role - (fd ? 16 : role >= 8 ? 8 : 0);
    const int fdl = fb ? 2 : 4, frows = fb ? nrr : nrq, fsec = fd ? 2 : fb ? (role >= 24) : (role >= 8);
    const int ft = fd || fb ? fe : fe >> 1, fm = fd || fb ? 0 : 2 * (fe & 1);
    v2d fv[2][8];
    {
        const int zi = (a.mirror && z > Nz / 2) ? Nz - z : z;
        const size_t col = (size_t) zi * Mx + x0 + min(ft, nx - 1), blk = col / a.sbt;
        const int cc = (int) (col % a.sbt);
        const size_t psize = (size_t) frows * a.sbt * (2 * fdl + 1);
        const double *src = (fb ? a.Lb : a.La) + blk * 2 * psize + (size_t) fsec * frows * a.sbt * fdl +
                            (fd ? cc : cc * fdl + fm);
        const size_t rs = (size_t) a.sbt * (fd ? 1 : fdl);
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r = i * 8 + frow;
                fv[p][i] = v2d{0.0, 0.0};
                if (i * 8 < nrr && r < frows) {
                    if (fd) fv[p][i].x = src[p * psize + r * rs];
                    else fv[p][i] = *(const v2d *) (src + p * psize + r * rs);
                }
            }
    }
    double *fac = (double *) smic, *facb = fac + 2 * nrq * IA_XG * 9;
    auto put_factors = [&]() {
        double *dst = (fb ? facb : fac) + (size_t) fsec * frows * IA_XG * fdl + (fd ? ft : ft * fdl + fm);
        const int psize = frows * IA_XG * (2 * fdl + 1), rs = IA_XG * (fd ? 1 : fdl);
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int r = i * 8 + frow;
                if (i * 8 < nrr && r < frows) {
                    if (fd) dst[p * psize + r * rs] = fv[p][i].x;
                    else *(v2d *) (dst + p * psize + r * rs) = fv[p][i];
                }
            }
    };
    if (k == 0) load_mic(a.mic0);
    for (int e = tid; e < dR * IA_XG; e += IA_THREADS) {
        const int i = e / IA_XG, t = e % IA_XG;
        if (t < nx) {
            const size_t o = ((size_t) (z * 2) * dR + i) * Mx + x0 + t;
            sal[t * dR + i] = a.IAC[o];
            sbe[t * dR + i] = a.IAC[o + (size_t) dR * Mx];
        }
    }
    if (k == 0) put_mic();
    if (tid == 0) *zero = make_double2(0.0, 0.0);
    __syncthreads();
    // right-hand sides: thread rows i (alpha: tid < 128, beta: tid >= 128)
    const bool isb = tid >= 128;
    const int i = isb ? tid - 128 : tid;
    const int N = isb ? dR : dQ;
    cplx acc[IA_XG];
    if (isb) {
        if (i < dR) mode_rhs<true>(a, i, z, x0, kz, sbe, smic, zero, valid, acc);
    } else {
        if (i < dQ) mode_rhs<false>(a, i, z, x0, kz, sal, smic, zero, valid, acc);
    }
    __syncthreads();
    if (i < N) {
#pragma unroll
        for (int t = 0; t < IA_XG; ++t)
            if (valid(t)) (isb ? sbe : sal)[t * dR + i] = acc[t];
    }
    put_factors();                    // the rows of MIC[count] are no longer read
    if (k < 2) load_mic(a.mic1);
    __syncthreads();
    // implicit solves: alpha chains on wave 0, beta chains on wave 1, one lane a
    // parity, column and part
    if ((tid & 63) < 4 * IA_XG && tid < 128) {
        const int pr = (tid >> 3) & 1, t = (tid >> 1) & 3, part = tid & 1;
        if (valid(t)) {
            if (tid < 64) {
                const double *L = fac + pr * nrq * IA_XG * 9, *U = L + nrq * IA_XG * 4, *D = U + nrq * IA_XG * 4;
                chain_subst<4, IA_XG>((double *) (sal + t * dR) + 2 * pr + part, L + 4 * t, U + 4 * t, D + t,
                                      (dQ - pr + 1) / 2);
            } else {
                const double *L = facb + pr * nrr * IA_XG * 5, *U = L + nrr * IA_XG * 2, *D = U + nrr * IA_XG * 2;
                chain_subst<2, IA_XG>((double *) (sbe + t * dR) + 2 * pr + part, L + 2 * t, U + 2 * t, D + t,
                                      (dR - pr + 1) / 2);
            }
        }
    }
    __syncthreads();
    if (k < 2) put_mic();             // the factors are no longer read
    // solved coefficients for the y-transform: alpha rows beyond dimQ and
    // omega_y rows beyond dimQ cleared (channel/increadjproject.c:371-395 sum
    // the omega_y coefficients below dimQ)
    for (int e = tid; e < dR * IA_XG; e += IA_THREADS) {
        const int r = e / IA_XG, t = e % IA_XG;
        if (!valid(t)) continue;
        const size_t o = ((size_t) (z * 2) * dR + r) * Mx + x0 + t;
        a.Ctr[o] = r < dQ ? sal[t * dR + r] : make_double2(0.0, 0.0);
        a.Ctr[o + (size_t) dR * Mx] = r < dQ ? sbe[t * dR + r] : make_double2(0.0, 0.0);
    }
    // wall values IAUxb, IAUzb (channel/increadjproject.c:446-485): wave t
    // of the block sums mode t's coefficients
    for (int t = tid >> 6; t < IA_XG; t += IA_THREADS / 64) {
        if (!valid(t)) continue;
        const int lane = tid & 63, x = x0 + t;
        double br = 0.0, bi = 0.0, ar = 0.0, ai = 0.0;
        for (int r = lane; r < dR; r += 64) {
            const cplx be = sbe[t * dR + r];
            br += a.Rp0[r] * be.x;
            bi += a.Rp0[r] * be.y;
            if (r < dQ) {
                const double sg = (r & 1) ? -8.0 : 8.0;
                const cplx al = sal[t * dR + r];
                ar += sg * al.x;
                ai += sg * al.y;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            br += __shfl_xor(br, off);
            bi += __shfl_xor(bi, off);
            ar += __shfl_xor(ar, off);
            ai += __shfl_xor(ai, off);
        }
        if (lane == 0) {
            const double kx = a.Kx[x], k2 = kx * kx + kz * kz;
            const cplx ub = a.W[(size_t) z * Mx + x], wb = a.W[wp + (size_t) z * Mx + x];
            cplx xb, zb;
            xb.x = bi * kz / k2 - ub.y / 2. * kz / k2 - ai * kx / k2 + wb.y * 2. * kx / k2;
            xb.y = -br * kz / k2 + ub.x / 2. * kz / k2 + 2. * ar * kx / k2 - wb.x * 2. * kx / k2;
            zb.x = -bi * kx / k2 + ub.y / 2. * kx / k2 - ai * kz / k2 + wb.y * 2. * kz / k2;
            zb.y = br * kx / k2 - ub.x / 2. * kx / k2 + 2. * ar * kz / k2 - wb.x * 2. * kz / k2;
            a.IAUb[(size_t) z * Mx + x] = xb;
            a.IAUb[wp + (size_t) z * Mx + x] = zb;
        }
    }
    if (k == 2) {
        for (int e = tid; e < dR * IA_XG; e += IA_THREADS) {
            const int r = e / IA_XG, t = e % IA_XG;
            if (!valid(t)) continue;
            const size_t o = ((size_t) (z * 2) * dR + r) * Mx + x0 + t;
            if (r < dQ) a.IAC[o] = sal[t * dR + r];
            a.IAC[o + (size_t) dR * Mx] = sbe[t * dR + r];
        }
        return;
    }
    __syncthreads();
    if (isb) {
        if (i < dR) mode_next<true>(a, i, z, x0, kz, sbe, smic, zero, valid);
    } else {
        if (i < dQ) mode_next<false>(a, i, z, x0, kz, sal, smic, zero, valid);
    }
}

// The wall lifts added to the Gauss-point values of the y-transform
// (channel/increadjproject.c:315-420, channel/increadjproject0.c:220-290):
// modes: v += Uzb lv, -dv/dy -= Uzb lv', d2v/dy2 += Uzb lv'', omega_y += Uxb lg,
// d omega_y/dy -= Uxb/2, carried through u = -i(kx f + kz g)/k2,
// w = i(kx g - kz f)/k2, du/dy = i(kx q - kz p)/k2, dw/dy = i(kz q + kx p)/k2;
// the mean: u += Uxb lg, w += Uzb lg, du/dy -= Uxb/2, dw/dy -= Uzb/2.
// Row Nz/2 is zero.  One thread per (z, j, x).
__global__ __launch_bounds__(256) void k_iadj_lift(IadjArgs a)
{
    const int q = a.q, Mx = a.Mx, Nz = a.Nz;
    const size_t n = (size_t) Nz * q * Mx;
    const size_t e = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    const int x = (int) (e % Mx), j = (int) ((e / Mx) % q), z = (int) (e / ((size_t) q * Mx));
    const size_t plane = (size_t) q * Mx, wp = (size_t) Nz * Mx;
    cplx *o = a.IAU + (size_t) z * 5 * plane + (size_t) j * Mx + x;
    if (z == Nz / 2) {
        for (int s = 0; s < 5; ++s) o[s * plane] = make_double2(0.0, 0.0);
        return;
    }
    const cplx ub = a.W[(size_t) z * Mx + x], wb = a.W[wp + (size_t) z * Mx + x];
    const double lv = a.lift[j], lv1 = a.lift[q + j], lv2 = a.lift[2 * q + j];
    const double lg = a.lift[3 * q + j];
    if (z == 0 && x == 0) {
        o[0] = cadd(o[0], cscale(ub, lg));
        o[2 * plane] = cadd(o[2 * plane], cscale(wb, lg));
        o[3 * plane] = cadd(o[3 * plane], cscale(ub, -0.5));
        o[4 * plane] = cadd(o[4 * plane], cscale(wb, -0.5));
        return;
    }
    const double kx = a.Kx[x], kz = a.Kz[z], k2 = kx * kx + kz * kz;
    const cplx f = cscale(wb, -lv1), g = cscale(ub, lg), qq = cscale(wb, lv2), p = cscale(ub, -0.5);
    const cplx u = make_double2((kx * f.y + kz * g.y) / k2, -(kx * f.x + kz * g.x) / k2);
    const cplx w = make_double2((-kx * g.y + kz * f.y) / k2, (kx * g.x - kz * f.x) / k2);
    const cplx du = make_double2((-kx * qq.y + kz * p.y) / k2, (kx * qq.x - kz * p.x) / k2);
    const cplx dw = make_double2(-(kx * p.y + kz * qq.y) / k2, (kx * p.x + kz * qq.x) / k2);
    o[0] = cadd(o[0], u);
    o[plane] = cadd(o[plane], cscale(wb, lv));
    o[2 * plane] = cadd(o[2 * plane], w);
    o[3 * plane] = cadd(o[3 * plane], du);
    o[4 * plane] = cadd(o[4 * plane], dw);
}

// a += b, row Nz/2 of a cleared (one thread per complex value)
__global__ __launch_bounds__(256) void k_gauss_sum(cplx *a, const cplx *b, size_t n, size_t per_z,
                                                   int zhalf)
{
    const size_t e = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    a[e] = (e / per_z == (size_t) zhalf) ? make_double2(0.0, 0.0) : cadd(a[e], b[e]);
}

}  // namespace

void launch_gauss_sum(Context &c, cplx *a, const cplx *b)
{
    const size_t n = c.usize, per_z = (size_t) 5 * c.d.qpts * c.d.Mx;
    hipLaunchKernelGGL(k_gauss_sum, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, c.stream, a, b,
                       n, per_z, c.d.Nz / 2);
}

// Constants of the incremental adjoint on the device (the lift values at the
// Gauss points, the mean mode's lift projection, Rw and Rpw transposed) and
// its staging buffer, built at the first call of a context.
int iadj_prepare(Context &c)
{
    if (c.dIadj) return 0;
    const Dims &d = c.d;
    const int q = d.qpts, nQ = d.dimQ, nR = d.dimR;
    std::vector<double> h;
    for (int j = 0; j < q; ++j) {
        const double y = c.y[j];
        h.push_back((1 - y) * (1 - y) * (1 + y) * 0.25);
    }
    for (int j = 0; j < q; ++j) h.push_back((3 * c.y[j] * c.y[j] - 2 * c.y[j] - 1) * 0.25);
    for (int j = 0; j < q; ++j) h.push_back((3 * c.y[j] - 1) * 0.5);
    for (int j = 0; j < q; ++j) h.push_back((1 - c.y[j]) * 0.5);
    for (int i = 0; i < nR; ++i) {
        double s = 0.0;
        for (int j = 0; j < q; ++j) s += c.Rw[(size_t) i * q + j] * (1 - c.y[j]) * 0.5;
        h.push_back(s);
    }
    for (int j = 0; j < q; ++j)
        for (int i = 0; i < nR; ++i) h.push_back(c.Rw[(size_t) i * q + j]);
    for (int j = 0; j < q; ++j)
        for (int i = 0; i < nR; ++i) h.push_back(c.Rpw[(size_t) i * q + j]);
    const size_t np = (size_t) d.Nz * d.Mx;
    const size_t buf = sizeof(cplx) * (3 * c.csize + 3 * c.usize + 6 * np + 4 * np * nR + 2 * np +
                                       2 * np * (nQ + nR));
    if (hipMalloc(&c.dIadj, sizeof(double) * h.size()) != hipSuccess ||
        hipMemcpy(c.dIadj, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMalloc(&c.iadjbuf, buf) != hipSuccess) {
        last_error() = "incremental adjoint: device allocation failed";
        if (c.dIadj) (void) hipFree(c.dIadj);
        c.dIadj = nullptr;
        if (c.iadjbuf) (void) hipFree(c.iadjbuf);
        c.iadjbuf = nullptr;
        return -1;
    }
    return 0;
}

int launch_iadj(Context &c, int k, int count, cplx *IAC, const cplx *IU, const cplx *LIU,
                const cplx *W, const cplx *F, cplx *IAU, cplx *IAUb)
{
    const Dims &d = c.d;
    if (iadj_prepare(c)) return -1;
    const int q = d.qpts, nQ = d.dimQ, nR = d.dimR;
    const size_t np = (size_t) d.Nz * d.Mx;
    // work arrays after the staging of iadjbuf (sc_increadjproject's layout)
    cplx *work = c.iadjbuf + c.csize + 3 * c.usize + 6 * np + 4 * np * nR + 2 * np;
    cplx *Ctr = work, *Fa = Ctr + c.csize, *Fb = Fa + np * nQ, *FLa = Fb + np * nR, *FLb = FLa + np * nQ;
    IadjArgs a;
    a.IU = IU; a.LIU = LIU; a.W = W; a.F = F;
    a.mic0 = c.MIC + c.csize * (size_t) count;
    a.mic1 = count > 0 ? c.MIC + c.csize * (size_t) (count - 1) : nullptr;
    a.Fa = Fa; a.Fb = Fb; a.FLa = FLa; a.FLb = FLb;
    a.IAC = IAC; a.IAU = IAU; a.IAUb = IAUb; a.Ctr = Ctr;
    a.Kx = c.dKx; a.Kz = c.dKz;
    a.Qs = c.dQs; a.Qps = c.dQps; a.Qpps = c.dQpps; a.Rs = c.dRs; a.Rps = c.dRps;
    a.Rp0 = c.dRwall;                     // R_j'(-1) (first row of the wall table)
    a.lift = c.dIadj;
    a.mlift = a.lift + 4 * (size_t) q;
    a.tRw = a.mlift + nR;
    a.tRpw = a.tRw + (size_t) q * nR;
    a.Nz = d.Nz; a.Mx = d.Mx; a.q = q; a.dQ = nQ; a.dR = nR; a.k = k;
    a.re = d.re; a.dt = d.dt;
    a.La = c.dLa[1][k]; a.Lb = c.dLb[1][k]; a.Lm = c.dLm[1][k];
    a.sbt = c.sbt; a.mirror = c.factor_mirror ? 1 : 0;
    const size_t nrq = solve_rows(nQ), nrr = solve_rows(nR);
    const size_t fac = sizeof(double) * 2 * IA_XG * (9 * nrq + 5 * nrr);
    const size_t lds_modes = sizeof(cplx) * (2 * IA_XG * (size_t) nR + 1) +
                             std::max(fac, sizeof(cplx) * 2 * IA_XG * (size_t) nR);
    const size_t lds_mean = sizeof(cplx) * 6 * (size_t) nR +
                            sizeof(double) * (8 * (size_t) q + 10 * nrr);
    const size_t lds = std::max(lds_modes, lds_mean);
    (void) hipFuncSetAttribute((const void *) k_iadj_modes, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int) lds);
    const int nxg = (d.Mx + IA_XG - 1) / IA_XG;
    const size_t nu = (size_t) d.Nz * q * d.Mx;
    // algorithmic bytes of the stage: per mode IAC read and written, the
    // products of this stage (and the next) read, MIC[count] (k = 0) and
    // MIC[count - 1] (k < 2), the forcing, IAU written, the wall planes
    const double modes = (double) (d.Nz - 1) * d.Mx;
    double per = 16.0 * (2.0 * nR + nQ + nR) + 16.0 * 5.0 * q * (k < 2 ? 2 : 1) + 16.0 * 5.0 * q + 16.0 * 8.0;
    if (k == 0) per += 16.0 * 2.0 * nR;
    if (k < 2) per += 16.0 * 2.0 * nR;
    if (F) per += 16.0 * (k < 2 ? 4.0 : 2.0) * nR;
    const double bytes = modes * per;
    // the adjoint path's projections and y-transform in FP64 whatever the
    // context's precision
    const bool mixed = c.mixed;
    c.mixed = false;
    auto go = [=, &c]() {
        if (k < 2) launch_force2(c, 1, IU, Fa, Fb, LIU, FLa, FLb);
        else launch_force(c, IU, 1, Fa, Fb);
        hipLaunchKernelGGL(k_iadj_modes, dim3((unsigned) (d.Nz * nxg + 1)), dim3(IA_THREADS), lds,
                           c.stream, a);
        launch_rebuild(c, Ctr, IAU);
        hipLaunchKernelGGL(k_iadj_lift, dim3((unsigned) ((nu + 255) / 256)), dim3(256), 0, c.stream, a);
    };
    prof_begin(c, c.stream, 8, bytes);
    go();
    prof_end(c, c.stream, 8);
    c.mixed = mixed;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace sc
