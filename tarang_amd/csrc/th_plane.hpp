// th_plane.hpp -- passes 2 to 4 of the fused RK stage in one launch, for boxes whose (y, z) planes fit in LDS.
//
// A workgroup owns one x-plane of one box and one group of real-space products.  For each operand it reads the
// plane's kept modes A[x][cy][cz], transforms them along y (columns) and z (rows, c2r) and keeps the real line in
// registers; each product goes back through z (r2c, kept kz) and y, and its kept ky are written to D[x][cy][cz].
// The plane lives in one LDS array of L2 rows of a padded z line: a column transform exchanges through its own
// column, a row transform through its own row, so nothing else is staged.
//
// What bounds it: the separate passes write and read two buffers of all N2 rows (B and C) between them, 2 x (inputs
// + products) planes per stage, and on small boxes take three launches of a few workgroups each.  Here neither
// buffer exists, and what is left is the arithmetic of the line FFTs at the occupancy that a plane in LDS leaves.
// The product list is cut into ngrp contiguous groups, a workgroup each: an operand is inverse-transformed once per
// group that uses it, so few groups do less work and many groups fill the chip (plane_groups).
#pragma once
#include "th_fused_kern.hpp"

namespace th {

constexpr int plane_EZ(int LZ) { return LZ % 3 == 0 ? (LZ >= 24 ? 12 : 6) : (LZ <= 16 ? 4 : 8); }
constexpr int plane_E2(int L2) { return L2 % 3 == 0 ? 12 : 8; }
template <typename R> constexpr size_t plane_lds(int L2, int LZ, int line) { return sizeof(cplx<R>) * ((size_t)L2 * line + L2 + 2 * LZ); }

template <typename R, int L2, int LZ>
__global__ __launch_bounds__(L2 * (LZ / plane_EZ(LZ))) void k_plane(FG g, PlaneTab tab, int ngrp, const cplx<R>* __restrict__ A,
                                                                     cplx<R>* __restrict__ D, long bD, const cplx<R>* __restrict__ tw2,
                                                                     const cplx<R>* __restrict__ twL,
                                                                     const cplx<R>* __restrict__ twN)
{
    constexpr int EZ = plane_EZ(LZ), PZ = LZ / EZ, E2 = plane_E2(L2), P2 = L2 / E2, NT = L2 * PZ;
    constexpr int NKZ = (2 * LZ) / 3;          // kept kz (a dealiased state)
    using ZI = LineFFT<R, LZ, PZ, +1>;
    using ZF = LineFFT<R, LZ, PZ, -1>;
    using YI = LineFFT<R, L2, P2, +1>;
    using YF = LineFFT<R, L2, P2, -1>;
    using Lay = ZPad<LZ>;
    constexpr int LS = Lay::line;
    static_assert(64 % PZ == 0 && NT <= 1024 && NKZ * P2 <= NT && LS >= LZ + 1, "plane shape");
    extern __shared__ __attribute__((aligned(16))) char plane_raw[];
    cplx<R>* const PL = (cplx<R>*)plane_raw;
    cplx<R>* const t2 = PL + L2 * LS;
    cplx<R>* const tz = t2 + L2;               // W_LZ^k, then W_N3^k
    for (int i = threadIdx.x; i < L2; i += NT) t2[i] = tw2[i];
    for (int i = threadIdx.x; i < 2 * LZ; i += NT) tz[i] = i < LZ ? twL[i] : twN[i - LZ];
    // workgroups of one plane are neighbours (they read the same operands), and neighbours share an XCD's L2
    const int lin = xcd_tile(blockIdx.x, gridDim.x);
    const int q = lin % ngrp, xb = lin / ngrp, x = xb % g.N1, box = xb / g.N1;
    A += (long)x * g.sx;
    D += box * bD + (long)x * g.sx;
    const int np = 3 * tab.npr, s0 = q * np / ngrp, s1 = (q + 1) * np / ngrp;
    // column threads: lanes along kz (memory order), row threads: the PZ lanes of one row in one wavefront
    const int c = threadIdx.x % NKZ, tc = threadIdx.x / NKZ;
    const bool col = tc < P2;
    const int tr = threadIdx.x % PZ;
    cplx<R>* const Z = PL + (threadIdx.x / PZ) * LS;
    __syncthreads();

    // operand a: A -> real line of this thread's row (register order of ZI's output).  Enters with PL free to write
    // once every thread is at the column transform's first barrier.
    auto operand = [&](int a, cplx<R> (&u)[EZ]) {
        cplx<R> v[E2];
        const cplx<R>* src = A + a * g.cA + (a < tab.shared ? 0 : box * g.bA) + c;
#pragma unroll
        for (int i = 0; i < E2; i++) {
            const int l = YI::in_pos(tc, i);
            v[i] = (col && lkept(g.my, l)) ? src[(long)lq(g.my, l) * g.KZP] : czero<R>();
        }
        YI::template run<LS, false, NoPad, false, 1, true>(v, PL + c, tc, t2, col);
        __syncthreads();                       // the last exchange's reads
        if (col) {
#pragma unroll
            for (int i = 0; i < E2; i++) PL[YI::out_pos(tc, i) * LS + c] = v[i];
        }
        __syncthreads();
        // c2r packing: s + i conj(W^k) d with s, d = x_k +- conj(x_{LZ-k}); modes kz >= NKZ are zero
#pragma unroll
        for (int m = 0; m < EZ; m++) {
            const int k = tr + PZ * m, km = LZ - k;
            if (sizeof(R) == 8 && m == EZ / 2) __builtin_amdgcn_sched_barrier(0);   // FP64: half the points in flight
            cplx<R> xv = k < NKZ ? Z[k] : czero<R>();
            const cplx<R> xc = km < NKZ ? conjg(Z[km]) : czero<R>();
            if (k == 0) xv.y = R(0);           // FFTW's c2r ignores Im of kz = 0
            // register of point t + PZ m in ZI's input order
            u[(m % (EZ / ZI::R0)) * ZI::R0 + m / (EZ / ZI::R0)] = add_iwd(xv + xc, conjg(tz[LZ + k]), xv - xc);
        }
        wave_sync();                           // the row's reads above come before the exchange's writes
        ZI::template run<1, true, Lay>(u, Z, tr, tz);
    };
    auto product = [&](cplx<R> (&w)[EZ], int p) {
        if constexpr (ZI::RL != ZF::R0) {
            wave_sync();
#pragma unroll
            for (int i = 0; i < EZ; i++) Z[ZI::out_pos(tr, i)] = w[i];
            wave_sync();
#pragma unroll
            for (int i = 0; i < EZ; i++) w[i] = Z[ZF::in_pos(tr, i)];
        }
        ZF::template run<1, true, Lay>(w, Z, tr, tz);
        constexpr int B = EZ / ZF::RL;
        wave_sync();
#pragma unroll
        for (int m = 0; m < EZ; m++) Z[tr + PZ * m] = w[(m % B) * ZF::RL + m / B];
        if (tr == 0) Z[LZ] = w[0];
        wave_sync();
        // 2 X_k = (z_k + conj z_{LZ-k}) - i W^k (z_k - conj z_{LZ-k}) (FG::norm carries the 1/2)
        cplx<R> o[EZ];
#pragma unroll
        for (int m = 0; m < EZ; m++) {
            const int k = tr + PZ * m;
            const cplx<R> zk = w[(m % B) * ZF::RL + m / B], zc = conjg(Z[LZ - k]), wn = tz[LZ + k];
            o[m] = add_iwd(zk + zc, mk<R>(-wn.x, -wn.y), zk - zc);
        }
        wave_sync();
#pragma unroll
        for (int m = 0; m < EZ; m++) {
            const int k = tr + PZ * m;
            if (k < NKZ) Z[k] = o[m];
        }
        __syncthreads();
        cplx<R> v[E2];
#pragma unroll
        for (int i = 0; i < E2; i++) v[i] = col ? PL[YF::in_pos(tc, i) * LS + c] : czero<R>();
        YF::template run<LS, false, NoPad, false, 1, true>(v, PL + c, tc, t2, col);
        if (col) {
            cplx<R>* dst = D + p * g.cA + c;
#pragma unroll
            for (int i = 0; i < E2; i++) {
                const int l = YF::out_pos(tc, i);
                if (lkept(g.my, l)) dst[(long)lq(g.my, l) * g.KZP] = v[i];
            }
        }
        // the next operand's first barrier covers these reads of PL
    };

    // Products s0..s1-1 in the table's order; an operand that the next product needs again stays in registers.
    cplx<R> ux[EZ], uy[EZ];
    int xh = -1, yh = -1;                      // the inputs that ux and uy hold
#pragma unroll 1
    for (int s = s0; s < s1; s++) {
        const int r = s / tab.npr, j = s - r * tab.npr, xi = tab.x[r], yi = tab.y[r][j];
        if (xh != xi) {
            if (yh == xi) {
#pragma unroll
                for (int i = 0; i < EZ; i++) ux[i] = uy[i];
            } else {
                operand(xi, ux);
            }
            xh = xi;
        }
        cplx<R> w[EZ];
        if (yi == xi) {
#pragma unroll
            for (int i = 0; i < EZ; i++) w[i] = mk<R>(ux[i].x * ux[i].x, ux[i].y * ux[i].y);
            __syncthreads();                   // the previous product's column reads come before this one's row writes
        } else {
            if (yh != yi) operand(yi, uy);
            else __syncthreads();
            yh = yi;
#pragma unroll
            for (int i = 0; i < EZ; i++) w[i] = mk<R>(ux[i].x * uy[i].x, ux[i].y * uy[i].y);
        }
        product(w, tab.o[r][j]);
    }
}

// ------------------------------------------------------------------------------------------
// x-forward for short lines: the same contraction, projection and IF-RK4 update as k_fx_fwd, with the products side
// by side instead of one after another.  A workgroup of NP groups of T x P threads transforms all NP product lines
// of T columns at once, leaves them in LDS, and then takes the kept modes of the tile point by point (all threads);
// CHAIN: the stage outputs go back to LDS and groups 0..NA-1 transform them along x into the next stage's A lines
// (any radix schedule: the line changes order in LDS).
//
// What bounds it: at 64^3 a tile loop of six dependent load-transform rounds ran in 123 one-wave workgroups for 256
// CUs (FP64), 17 us of latency for 5 MB of data.  Here the rounds run at the same time in six times the waves, the state
// and accumulator loads are issued before the first transform, and nothing is written non-temporally (the next
// pass finds its lines in the L2).
// ------------------------------------------------------------------------------------------
template <typename R, int L, int T, int MODE> struct XSplit {
    static constexpr int E = L % 3 == 0 ? 12 : (L == 16 ? 4 : 8), P = L / E;
    static constexpr int NP = MODE == 0 ? 6 : 9, NA = MODE == 0 ? 3 : 6, NX = MODE == 0 ? 2 : 4;
    static constexpr int NT = T * P * NP;
    static constexpr size_t lds = sizeof(cplx<R>) * ((size_t)NP * L * T + L) + sizeof(double) * NX * (L + T);
};

template <typename R, int L, int T, int MODE, bool CHAIN>
__global__ __launch_bounds__((XSplit<R, L, T, MODE>::NT)) void k_fx_split(FG g, const cplx<R>* D, cplx<R>* Aout,
                                                                     cplx<R>* S, cplx<R>* Vs, cplx<R>* acc,
                                                                     const cplx<R>* __restrict__ tw,
                                                                     const StageCoef* __restrict__ coefs)
{
    using X = XSplit<R, L, T, MODE>;
    constexpr int E = X::E, P = X::P, NP = X::NP, NA = X::NA, NX = X::NX, NT = X::NT;
    constexpr int NC = MODE == 1 ? 6 : 3;
    constexpr int RS = P * NP, NR = (2 * (L / 3) - 1 + RS - 1) / RS;   // kept rows per thread
    using F = LineFFT<R, L, P, -1>;
    using FI = LineFFT<R, L, P, +1>;
    extern __shared__ __attribute__((aligned(16))) char split_raw[];
    cplx<R>* const lds = (cplx<R>*)split_raw;
    cplx<R>* const twl = lds + NP * L * T;
    double* const exl = (double*)(twl + L);     // exp(c Kx^2) per row, exp(c (Ky^2 + Kz^2)) per column (k_fx_fwd)
    double* const eyz = exl + NX * L;
    const int c = threadIdx.x % T, row = threadIdx.x / T, t = row % P, gi = row / P;
    const int ntz = (g.nkz + T - 1) / T;
    const int lin = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int tile = lin % gridDim.x, box = lin / gridDim.x;
    const int cy = tile / ntz;
    const int cz = (tile % ntz) * T + c;
    const bool ok = cz < g.nkz;
    const long m = (long)cy * g.KZP + cz;
    D += box * g.bA + m;
    Aout += box * g.bA + m;
    S += box * g.bS + m;
    Vs += box * g.bS + m;
    acc += box * g.bS + m;
    const StageCoef sc = coefs[box];
    const int stage = sc.stage;
    cplx<R> v[E];
#pragma unroll
    for (int i = 0; i < E; i++) v[i] = ok ? D[gi * g.cA + (long)F::in_pos(t, i) * g.sx] : czero<R>();
    const cplx<R>* accr = stage > 1 ? acc : S;   // stage 1 has no accumulator yet (value unused)
    cplx<R> s0[NR][NC], a0[NR][NC];
#pragma unroll
    for (int q = 0; q < NR; q++) {
        const int cx = row + RS * q;
        const bool on = ok && cx < g.mx.nk;
#pragma unroll
        for (int a = 0; a < NC; a++) {
            s0[q][a] = on ? S[a * g.cS + (long)cx * g.sx] : czero<R>();
            a0[q][a] = on ? accr[a * g.cS + (long)cx * g.sx] : czero<R>();
        }
    }
    for (int i = threadIdx.x; i < L; i += NT) {
        twl[i] = tw[i];
        const double kx = kx_four(i, g.N1) * g.f1, kx2 = kx * kx;
        exl[i] = exp(sc.fh[0] * kx2);
        exl[L + i] = exp(sc.f1[0] * kx2);
        if constexpr (MODE == 1) {
            exl[2 * L + i] = exp(sc.fh[1] * kx2);
            exl[3 * L + i] = exp(sc.f1[1] * kx2);
        }
    }
    const double dKy = ky_of(ll(g.my, cy), g.N2) * g.f2, dKz = cz * g.f3;
    if (row < NX) {
        const double kyz2 = dKy * dKy + dKz * dKz;
        const double cf = row == 0 ? sc.fh[0] : row == 1 ? sc.f1[0] : row == 2 ? sc.fh[1] : sc.f1[1];
        eyz[row * T + c] = exp(cf * kyz2);
    }
    __syncthreads();
    cplx<R>* const buf = lds + gi * (L * T);
    F::template run<T, false, NoPad, false, 0>(v, buf + c, t, twl);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; i++) buf[F::out_pos(t, i) * T + c] = v[i];
    __syncthreads();
    const R Ky = (R)dKy, Kz = (R)dKz;
    const bool wvs = !CHAIN || (g.keep3 && stage == 3);
#pragma unroll
    for (int q = 0; q < NR; q++) {
        const int cx = row + RS * q;
        if (!(ok && cx < g.mx.nk)) continue;
        const int l = ll(g.mx, cx);
        const double dKx = kx_four(l, g.N1) * g.f1;
        const R Kx = (R)dKx;
        cplx<R>* const pt = lds + l * T + c;    // product p of this point: pt[p * L * T]
        cplx<R> n[NA];
#pragma unroll
        for (int a = 0; a < NA; a++) n[a] = czero<R>();
#pragma unroll
        for (int p = 0; p < NP; p++) {          // the terms and their order are k_fx_fwd's
            const cplx<R> w = pt[p * L * T];
            const int pi = MODE == 1 ? p / 3 : p < 3 ? p : p - 3;
            const int pj = MODE == 1 ? p % 3 : p < 3 ? p : (p == 5 ? 0 : p - 2);
            acc_iK(n[pi], pj == 0 ? Kx : pj == 1 ? Ky : Kz, w);
            if (MODE == 1) acc_iK(n[MODE == 1 ? 3 + pj : 0], pi == 0 ? Kx : pi == 1 ? Ky : Kz, w);
            else if (pi != pj) acc_iK(n[pj], pi == 0 ? Kx : pi == 1 ? Ky : Kz, w);
        }
        const double K2 = ksq_f(dKx, dKy, dKz);
        Dc Nu[3], rhs[3];
#pragma unroll
        for (int a = 0; a < 3; a++)
            Nu[a] = MODE == 0 ? dsc(dl(n[a]), g.norm) : dsc(dadd(dl(n[a]), dl(n[MODE == 1 ? 3 + a : 0])), 0.5 * g.norm);
        if (K2 > 0) {
            const double iK2 = 1.0 / K2;
            const Dc kn = dmk((dKx * Nu[0].x + dKy * Nu[1].x + dKz * Nu[2].x) * iK2,
                              (dKx * Nu[0].y + dKy * Nu[1].y + dKz * Nu[2].y) * iK2);
            const double Kc[3] = {dKx, dKy, dKz};
#pragma unroll
            for (int a = 0; a < 3; a++) rhs[a] = dmk(-(Nu[a].x - Kc[a] * kn.x), -(Nu[a].y - Kc[a] * kn.y));
        } else {
#pragma unroll
            for (int a = 0; a < 3; a++) rhs[a] = dmk(-Nu[a].x, -Nu[a].y);
        }
        const double eh = exl[l] * eyz[c], e1 = exl[L + l] * eyz[T + c];
        const long o = (long)cx * g.sx;
        cplx<R> keep[NC];
#pragma unroll
        for (int a = 0; a < 3; a++)
            keep[a] = rk_store<R, false>(stage, sc.dt, eh, e1, rhs[a], s0[q][a], a0[q][a], S + a * g.cS + o,
                                         Vs + a * g.cS + o, acc + a * g.cS + o, wvs);
        if constexpr (MODE == 1) {
            const double ehb = exl[2 * L + l] * eyz[2 * T + c], e1b = exl[3 * L + l] * eyz[3 * T + c];
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const Dc np = dl(n[a]), nm = dl(n[3 + a]);
                const Dc nb = dsc(dmk(np.x - nm.x, np.y - nm.y), 0.5 * g.norm);
                keep[3 + a] = rk_store<R, false>(stage, sc.dt, ehb, e1b, dmk(-nb.x, -nb.y), s0[q][3 + a], a0[q][3 + a],
                                                 S + (3 + a) * g.cS + o, Vs + (3 + a) * g.cS + o,
                                                 acc + (3 + a) * g.cS + o, wvs);
            }
        }
        if constexpr (CHAIN) {                  // over this point's own products
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if (MODE == 0) {
                    pt[a * L * T] = keep[a];
                } else {
                    pt[a * L * T] = keep[a] + keep[NC - 3 + a];
                    pt[(3 + a) * L * T] = keep[a] - keep[NC - 3 + a];
                }
            }
        }
    }
    if constexpr (CHAIN) {
        // rows outside the kept modes: 0
        for (int l = g.mx.h + row; l < g.mx.h + g.mx.N - g.mx.nk; l += RS)
#pragma unroll
            for (int a = 0; a < NA; a++) lds[(a * L + l) * T + c] = czero<R>();
        __syncthreads();
#pragma unroll
        for (int i = 0; i < E; i++) v[i] = buf[FI::in_pos(t, i) * T + c];
        FI::template run<T, false, NoPad, false, 1>(v, buf + c, t, twl);   // groups past NA run on their own lines
        if (ok && gi < NA) {
#pragma unroll
            for (int i = 0; i < E; i++) Aout[gi * g.cA + (long)FI::out_pos(t, i) * g.sx] = v[i];
        }
    }
}

// The same for the sine / cosine lines of RB (k_sx_fwd_rb, k_sx_inv): the nine product lines side by side; the mirror
// value V_{N-k} of a point's DCT / DST comes from LDS, where the whole line is.  CHAIN: the stage outputs become the
// next stage's A lines, groups 0-3 transforming V1 (sine), V2, V3 (cosine), T (sine); the stage field is written all
// the same (the next stage's force reads V1 and T of it).
template <typename R, int L, int T, bool CHAIN>
__global__ __launch_bounds__((XSplit<R, L, T, 1>::NT)) void k_sx_split(FG g, const cplx<R>* D, cplx<R>* Aout, cplx<R>* S,
                                                                  cplx<R>* Vs, cplx<R>* acc,
                                                                  const cplx<R>* __restrict__ tw,
                                                                  const cplx<R>* __restrict__ tw4,
                                                                  const StageCoef* __restrict__ coefs)
{
    using X = XSplit<R, L, T, 1>;
    constexpr int E = X::E, P = X::P, NP = X::NP, NT = X::NT, NX = 4;
    constexpr int RS = P * NP;
    static_assert(2 * L / 3 <= RS, "one kept row per thread");
    using F = LineFFT<R, L, P, -1>;
    using FI = LineFFT<R, L, P, +1>;
    extern __shared__ __attribute__((aligned(16))) char split_raw[];
    cplx<R>* const lds = (cplx<R>*)split_raw;
    cplx<R>* const twl = lds + NP * L * T;
    double* const exl = (double*)(twl + L);     // as in k_fx_split
    double* const eyz = exl + NX * L;
    cplx<R>* const w4 = (cplx<R>*)(eyz + NX * T);
    const int c = threadIdx.x % T, row = threadIdx.x / T, t = row % P, gi = row / P;
    const int ntz = (g.nkz + T - 1) / T;
    const int lin = xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    const int tile = lin % gridDim.x, box = lin / gridDim.x;
    const int cy = tile / ntz;
    const int cz = (tile % ntz) * T + c;
    const bool ok = cz < g.nkz;
    const long m = (long)cy * g.KZP + cz;
    D += box * g.bA + m;
    Aout += box * g.bA + m;
    S += box * g.bS + m;
    Vs += box * g.bS + m;
    acc += box * g.bS + m;
    const StageCoef sc = coefs[box];
    const int stage = sc.stage;
    const bool psin = ((0x1A8u >> gi) & 1u) != 0;     // sine products, see k_sx_fwd_rb
    cplx<R> v[E];
#pragma unroll
    for (int i = 0; i < E; i++) {
        const int j = F::in_pos(t, i);
        const cplx<R> d = ok ? D[gi * g.cA + (long)j * g.sx] : czero<R>();
        v[i] = cscale(d, (psin && j >= L / 2) ? R(-1) : R(1));
    }
    const cplx<R>* accr = stage > 1 ? acc : S;        // stage 1 has no accumulator yet (value unused)
    const cplx<R>* F0 = stage == 1 ? S : Vs;          // field the stage's rhs is evaluated on
    const int l = row;                                // this thread's kept mode
    const bool on = ok && l < g.mx.nk;
    cplx<R> s0[4], a0[4], f0[2];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        s0[a] = on ? S[a * g.cS + (long)l * g.sx] : czero<R>();
        a0[a] = on ? accr[a * g.cS + (long)l * g.sx] : czero<R>();
    }
    f0[0] = on ? F0[(long)l * g.sx] : czero<R>();
    f0[1] = on ? F0[3 * g.cS + (long)l * g.sx] : czero<R>();
    for (int i = threadIdx.x; i < L; i += NT) {
        twl[i] = tw[i];
        w4[i] = tw4[i];
        const double kx = i * g.f1, kx2 = kx * kx;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            exl[2 * q * L + i] = exp(sc.fh[q] * kx2);
            exl[(2 * q + 1) * L + i] = exp(sc.f1[q] * kx2);
        }
    }
    const double dKy = ky_of(ll(g.my, cy), g.N2) * g.f2, dKz = cz * g.f3;
    if (row < NX) {
        const double kyz2 = dKy * dKy + dKz * dKz;
        const double cf = row == 0 ? sc.fh[0] : row == 1 ? sc.f1[0] : row == 2 ? sc.fh[1] : sc.f1[1];
        eyz[row * T + c] = exp(cf * kyz2);
    }
    __syncthreads();
    cplx<R>* const buf = lds + gi * (L * T);
    F::template run<T, false, NoPad, false, 0>(v, buf + c, t, twl);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < E; i++) buf[F::out_pos(t, i) * T + c] = v[i];
    __syncthreads();
    cplx<R> keep[4];
    if (on) {
        const double dKx = l * g.f1;
        const R Kx = (R)dKx, Ky = (R)dKy, Kz = (R)dKz;
        const cplx<R> w = w4[l];
        cplx<R> n[4];
#pragma unroll
        for (int a = 0; a < 4; a++) n[a] = czero<R>();
#pragma unroll
        for (int p = 0; p < NP; p++) {                // the terms and their order are k_sx_fwd_rb's
            const bool sn = ((0x1A8u >> p) & 1u) != 0;
            const cplx<R> Pv = cmul(w, lds[(p * L + l) * T + c]);
            const cplx<R> Qv = cmul(conjg(w), lds[(p * L + (l ? L - l : 0)) * T + c]);
            const cplx<R> dv = Pv - Qv, sv = Pv + Qv;
            cplx<R> Av = sn ? mk<R>(-dv.y, dv.x) : sv;
            if (sn && l == 0) Av = czero<R>();
            const int a1 = (p == 0 || p == 3 || p == 5) ? 0 : (p == 1 || p == 4) ? 1 : (p == 2) ? 2 : 3;
            if (p == 0 || p == 6) n[a1] = mk<R>(n[a1].x - Kx * Av.x, n[a1].y - Kx * Av.y);
            else acc_iK(n[a1], (p == 1 || p == 3 || p == 7) ? Ky : Kz, Av);
            const int a2 = p == 3 ? 1 : 2;
            if (p == 3 || p == 5) n[a2] = mk<R>(n[a2].x + Kx * Av.x, n[a2].y + Kx * Av.y);
            else if (p == 4) acc_iK(n[a2], Ky, Av);
        }
        const double K2 = ksq_f(dKx, dKy, dKz);
        Dc Nn[4];
#pragma unroll
        for (int a = 0; a < 4; a++) Nn[a] = dsc(dl(n[a]), g.norm);
        const Dc V1 = dl(f0[0]), Tf = dl(f0[1]);
        Nn[0] = dmk(Nn[0].x - Tf.x, Nn[0].y - Tf.y);
        Nn[3] = dmk(Nn[3].x - V1.x, Nn[3].y - V1.y);
        Dc pr = dmk(0.0, 0.0);
        if (K2 > 0) {
            const double iK2 = 1.0 / K2;
            const double dr = dKx * Nn[0].x - dKy * Nn[1].y - dKz * Nn[2].y;
            const double di = dKx * Nn[0].y + dKy * Nn[1].x + dKz * Nn[2].x;
            pr = dmk(dr * iK2, di * iK2);
        }
        Dc rhs[4];
        rhs[0] = dmk(-(Nn[0].x - dKx * pr.x), -(Nn[0].y - dKx * pr.y));
        rhs[1] = dmk(-(Nn[1].x - dKy * pr.y), -(Nn[1].y + dKy * pr.x));
        rhs[2] = dmk(-(Nn[2].x - dKz * pr.y), -(Nn[2].y + dKz * pr.x));
        rhs[3] = dmk(-Nn[3].x, -Nn[3].y);
        const double eh = exl[l] * eyz[c], e1 = exl[L + l] * eyz[T + c];
        const double ehT = exl[2 * L + l] * eyz[2 * T + c], e1T = exl[3 * L + l] * eyz[3 * T + c];
        const long o = (long)l * g.sx;
#pragma unroll
        for (int a = 0; a < 4; a++)
            keep[a] = rk_store<R, false>(stage, sc.dt, a < 3 ? eh : ehT, a < 3 ? e1 : e1T, rhs[a], s0[a], a0[a],
                                         S + a * g.cS + o, Vs + a * g.cS + o, acc + a * g.cS + o);
    }
    if constexpr (CHAIN) {
        __syncthreads();                              // every point has read its mirror values
        if (on) {
#pragma unroll
            for (int a = 0; a < 4; a++) lds[(a * L + l) * T + c] = keep[a];
        }
        __syncthreads();
        const bool sn = gi == 0 || gi == 3;
        const int nk = g.mx.nk;
#pragma unroll
        for (int i = 0; i < E; i++) {                 // conj(w_k) (X_k - i X_{N-k}), see k_sx_inv
            const int k = FI::in_pos(t, i);
            const cplx<R> ck = (ok && k < nk && !(sn && k == 0)) ? buf[k * T + c] : czero<R>();
            const cplx<R> cm = (ok && k > 0 && L - k < nk) ? buf[(L - k) * T + c] : czero<R>();
            const cplx<R> a = sn ? cm : ck, b = sn ? ck : cm;
            v[i] = cmul(conjg(w4[k]), mk<R>(a.x + b.y, a.y - b.x));
        }
        FI::template run<T, false, NoPad, false, 1>(v, buf + c, t, twl);   // groups past 3 run on their own lines
        if (ok && gi < 4) {
#pragma unroll
            for (int i = 0; i < E; i++) {
                const int j = FI::out_pos(t, i);
                Aout[gi * g.cA + (long)j * g.sx] = cscale(v[i], (sn && j >= L / 2) ? R(-1) : R(1));
            }
        }
    }
}

template <typename R, int L, int T>
static int launch_sxsplit(const FG& g, const cplx<R>* D, cplx<R>* Aout, cplx<R>* S, cplx<R>* Vs, cplx<R>* acc,
                          const cplx<R>* tw, const cplx<R>* tw4, const StageCoef* sc, hipStream_t st, bool chain)
{
    using X = XSplit<R, L, T, 1>;
    constexpr size_t lds = X::lds + L * sizeof(cplx<R>);
    static_assert(X::NT <= 1024 && lds <= 160 * 1024, "split x-forward shape");
    const dim3 grid(g.my.nk * ((g.nkz + T - 1) / T), g.nbox);
    auto go = [&](auto k) -> int {
        if (lds > 64 * 1024)
            TH_CHECK_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k, grid, dim3(X::NT), lds, st, g, D, Aout, S, Vs, acc, tw, tw4, sc);
        TH_CHECK_HIP(hipGetLastError());
        return OK;
    };
    return chain ? go(k_sx_split<R, L, T, true>) : go(k_sx_split<R, L, T, false>);
}

template <typename R, int L, int T, int MODE>
static int launch_xsplit(const FG& g, const cplx<R>* D, cplx<R>* Aout, cplx<R>* S, cplx<R>* Vs, cplx<R>* acc,
                         const cplx<R>* tw, const StageCoef* sc, hipStream_t st, bool chain)
{
    using X = XSplit<R, L, T, MODE>;
    static_assert(X::NT <= 1024 && X::lds <= 160 * 1024, "split x-forward shape");
    const dim3 grid(g.my.nk * ((g.nkz + T - 1) / T), g.nbox);
    auto go = [&](auto k) -> int {
        if (X::lds > 64 * 1024)
            TH_CHECK_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)X::lds));
        hipLaunchKernelGGL(k, grid, dim3(X::NT), X::lds, st, g, D, Aout, S, Vs, acc, tw, sc);
        TH_CHECK_HIP(hipGetLastError());
        return OK;
    };
    return chain ? go(k_fx_split<R, L, T, MODE, true>) : go(k_fx_split<R, L, T, MODE, false>);
}

template <typename R, int L2, int LZ>
static int launch_plane(const FG& g, const PlaneTab& tab, int ngrp, const cplx<R>* A, cplx<R>* D, long bD, const cplx<R>* tw2,
                        const cplx<R>* twL, const cplx<R>* twN, hipStream_t st)
{
    constexpr size_t lds = plane_lds<R>(L2, LZ, ZPad<LZ>::line);
    static_assert(lds <= 160 * 1024, "the plane must fit in one CU's LDS");
    auto k = k_plane<R, L2, LZ>;
    if (lds > 64 * 1024)
        TH_CHECK_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3((unsigned)(g.N1 * g.nbox * ngrp)), dim3(L2 * (LZ / plane_EZ(LZ))), lds, st, g, tab, ngrp, A, D,
                       bD, tw2, twL, twN);
    TH_CHECK_HIP(hipGetLastError());
    return OK;
}

// ---- dispatch: the planes that plane_ok can name ----
template <typename R, int L2>
static int plane_z(const FG& g, const PlaneTab& tab, int ngrp, const cplx<R>* A, cplx<R>* D, long bD, const cplx<R>* tw2,
                   const cplx<R>* twL, const cplx<R>* twN, hipStream_t st)
{
#define C_(n)                                                                                                                   \
    case n:                                                                                                                     \
        if constexpr (2 * n * L2 <= PLANE_MAX) return launch_plane<R, L2, n>(g, tab, ngrp, A, D, bD, tw2, twL, twN, st);        \
        break;
    switch (g.LZ) { C_(8) C_(12) C_(16) C_(24) C_(32) C_(48) C_(64) }
#undef C_
    set_error("plane pass: %d x %d planes unsupported", g.N2, g.N3);
    return E_UNSUPPORTED;
}

}  // namespace th
