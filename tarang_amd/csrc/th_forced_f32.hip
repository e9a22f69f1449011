// th_forced_f32.hip -- the passes of forced FP32 states: the kernels of th_fused_kern.hpp with the FORCED arithmetic of
// LineFFT, and a z pass that holds all three real lines.
//
// A forced FP32 result follows every rounding of the passes (LineFFT), also which of two products the compiler fuses
// with their sum, so these states have kernels of their own, apart from those that are tuned for the other states:
// the same five passes, without the radix 6 and 12 lines, the short-box kernels of th_plane.hpp and loads ahead of the
// x-forward's transforms.  What that costs: 192^3, four steps 2.68 -> 2.86 ms.
#include "th_fused_kern.hpp"

namespace th {

// pass 3 of NS (k_fz MODE 0): all three inputs are transformed first, then the six products are formed one after
// another.  Up to 8 points per thread in a rolled loop over the rotation steps u_r u_r, u_r u_{r+1} (rotating the
// registers by one puts every operand in a fixed one), more points unrolled, each product fenced off for the scheduler.
// 192^3: 62 us (k_fz 52).
template <int LZ, int P, int TZ>
__global__ __launch_bounds__(TZ * P) void k_fz_forced(FG g, const c32* __restrict__ B, c32* __restrict__ Cout,
                                                      const c32* __restrict__ twL, const c32* __restrict__ twN)
{
    using R = float;
    constexpr bool R16 = (LZ / P) % 16 == 0;   // 16 points per thread: radix-16 stages
    using FI = LineFFT<R, LZ, P, +1, R16, true>;
    using FF = LineFFT<R, LZ, P, -1, R16, true>;
    using Lay = std::conditional_t<R16, ZPad16<LZ>, ZPad<LZ, true>>;
    constexpr int E = FI::E;
    static_assert(64 % P == 0, "a z line's threads must share one wavefront");
    constexpr int LZS = Lay::line;
    static_assert(LZS >= LZ + 1, "the mirror exchange uses positions 0..LZ of the line's LDS region");
    __shared__ cplx<R> lds[TZ * LZS];
    __shared__ cplx<R> tws[2 * LZ];            // W_LZ^j, then W_N3^k
    for (int i = threadIdx.x; i < 2 * LZ; i += TZ * P) tws[i] = i < LZ ? twL[i] : twN[i - LZ];
    __syncthreads();
    const int t = threadIdx.x % P, c = threadIdx.x / P;
    const long q = (long)blockIdx.x * TZ + c;
    const bool ok = q < (long)g.N1 * g.N2;
    const long off = q * g.KZP;
    cplx<R>* Z = lds + c * LZS;
    cplx<R> twk[E];                            // W_N3^(t + P m)
#pragma unroll
    for (int m = 0; m < E; m++) twk[m] = tws[LZ + t + P * m];
    // packing, registers that hold no kept kz and mirrors: as in k_fz
    constexpr int NKZ = (2 * LZ) / 3;
    auto zin = [](int m) constexpr { return P * m >= NKZ; };
    auto zmir = [](int m) constexpr { return LZ - (P - 1) - P * m >= NKZ; };
    static_assert(LZ - (P - 1) >= NKZ, "register 0's mirrors (position LZ included) must be dealiased zeros");
    cplx<R> u[3][E];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const cplx<R>* X = B + a * g.cB + off;
        cplx<R> xa[E];
#pragma unroll
        for (int m = 0; m < E; m++) {
            const int k = t + P * m;
            xa[m] = (!zin(m) && ok && k < NKZ) ? ld_nt(X + k) : czero<R>();
        }
        wave_sync();
#pragma unroll
        for (int m = 0; m < E; m++) Z[t + P * m] = xa[m];
        wave_sync();
#pragma unroll
        for (int m = 0; m < E; m++) {
            cplx<R> w = conjg(twk[m]);
            if (zmir(m)) {
                cplx<R> xv = xa[m];
                if (t == 0 && m == 0) xv.y = R(0);
                u[a][zreg<E, FI::R0>(m)] = add_iwd(xv, w, xv);
            } else if (zin(m)) {
                cplx<R> xb = conjg(Z[LZ - t - P * m]);
                u[a][zreg<E, FI::R0>(m)] = add_iwd(xb, mk<R>(-w.x, -w.y), xb);
            } else {
                cplx<R> xb = Z[LZ - t - P * m];
                cplx<R> xv = xa[m];
                xb.y = -xb.y;
                cplx<R> s = xv + xb, d = xv - xb;
                u[a][zreg<E, FI::R0>(m)] = add_iwd(s, w, d);
            }
        }
        FI::template run<1, true, Lay>(u[a], Z, t, tws);
    }
    auto product_out = [&](cplx<R> (&w)[E], int p) {
        if constexpr (FI::R0 != FI::RL) {
            wave_sync();
#pragma unroll
            for (int i = 0; i < E; i++) Z[FI::out_pos(t, i)] = w[i];
            wave_sync();
#pragma unroll
            for (int i = 0; i < E; i++) w[i] = Z[FF::in_pos(t, i)];
        }
        const cplx<R>* tw = tws + opaque_zero();
        FF::template run<1, true, Lay>(w, Z, t, tw);
        const cplx<R>* twp = tw + LZ;
        cplx<R>* X = Cout + p * g.cB + off;
        wave_sync();
#pragma unroll
        for (int m = 0; m < E; m++)
            if (P * m + (P - 1) > LZ - NKZ) Z[t + P * m] = w[zreg<E, FF::RL>(m)];
        if (t == 0) Z[LZ] = w[zreg<E, FF::RL>(0)];
        wave_sync();
        auto unpack = [&](int m) {
            cplx<R> zk = w[zreg<E, FF::RL>(m)];
            cplx<R> zc = conjg(Z[LZ - t - P * m]);
            const cplx<R> tw = twp[t + P * m];
            return add_iwd(zk + zc, mk<R>(-tw.x, -tw.y), zk - zc);
        };
        cplx<R> o[E];
#pragma unroll
        for (int m = 0; m < E; m++)
            if (!zin(m)) o[m] = unpack(m);
#pragma unroll
        for (int m = 0; m < E; m++) {
            const int k = t + P * m;
            if (!zin(m) && ok && k < NKZ) st_nt(X + k, o[m]);
        }
    };
    cplx<R> w[E];
    if constexpr (E <= 8) {
#pragma unroll 1
        for (int r = 0; r < 3; r++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
#pragma unroll
                for (int i = 0; i < E; i++) w[i] = mk<R>(u[0][i].x * u[j][i].x, u[0][i].y * u[j][i].y);
                product_out(w, 3 * j + r);
            }
#pragma unroll
            for (int i = 0; i < E; i++) {
                const cplx<R> t0 = u[0][i];
                u[0][i] = u[1][i];
                u[1][i] = u[2][i];
                u[2][i] = t0;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < 3; r++) {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int y = (r + j) % 3;
#pragma unroll
                for (int i = 0; i < E; i++) w[i] = mk<R>(u[r][i].x * u[y][i].x, u[r][i].y * u[y][i].y);
                product_out(w, 3 * j + r);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

template <int LZ, int V>
static int launch_zf(const FG& g, const c32* B, c32* Cc, const c32* twL, const c32* twN, hipStream_t st)
{
    constexpr int E = (V == 3) ? 16 : pts_per_thread(LZ), P = LZ / E;      // launch shapes: launch_z
    constexpr int NT = (V == 1) ? 128 : (V == 2) ? 512 : 256;
    constexpr int TZ = (NT / P) < 1 ? 1 : NT / P;
    if (g.nkz != (2 * LZ) / 3) {
        set_error("fused z pass: %d kept kz for N3 = %d (a dealiased state keeps %d)", g.nkz, 2 * LZ, (2 * LZ) / 3);
        return E_UNSUPPORTED;
    }
    const long lines = (long)g.N1 * g.N2;
    hipLaunchKernelGGL((k_fz_forced<LZ, P, TZ>), dim3((unsigned)((lines + TZ - 1) / TZ)), dim3(TZ * P), 0, st, g, B, Cc, twL, twN);
    TH_CHECK_HIP(hipGetLastError());
    return OK;
}
template <int LZ>
static int zf_v(const FG& g, const c32* B, c32* Cc, const c32* twL, const c32* twN, int var, hipStream_t st)
{
    if constexpr (LZ >= 64) {
        if (var == 1) return launch_zf<LZ, 1>(g, B, Cc, twL, twN, st);
        if constexpr (LZ % 3 != 0) {
            if (var == 2) return launch_zf<LZ, 2>(g, B, Cc, twL, twN, st);
            if (var == 3) return launch_zf<LZ, 3>(g, B, Cc, twL, twN, st);
        }
    }
    return launch_zf<LZ, 0>(g, B, Cc, twL, twN, st);
}
int d_z_forced(const FG& g, const c32* B, c32* Cc, const c32* twL, const c32* twN, int var, hipStream_t st)
{
#define C_(n) case n: return zf_v<n>(g, B, Cc, twL, twN, var, st);
    switch (g.LZ) { TH_ZLENS(C_) default: set_error("fused: N3 %d unsupported", g.N3); return E_UNSUPPORTED; }
#undef C_
}

template int d_xinv<float, 0, true>(const FG&, const c32*, c32*, int, const c32*, ShellSel, int, hipStream_t);
template int d_yinv<float, true>(const FG&, const c32*, c32*, int, const c32*, int, hipStream_t);
template int d_yfwd<float, true>(const FG&, const c32*, c32*, int, const c32*, int, hipStream_t);
template int d_xfwd<float, 0, true>(const FG&, const c32*, c32*, c32*, c32*, c32*, const c32*, const StageCoef*, int, hipStream_t, bool);
template bool d_xfwd_chainable<float, true>(const FG&);

}  // namespace th
