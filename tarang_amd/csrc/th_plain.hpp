// th_plain.hpp -- the plain steppers' right-hand side on reference-layout fields through the fused passes.
//
// th_step_plain takes arbitrary fields (not only 2/3-dealiased ones), so the inverse half of the pipeline keeps every
// mode: x-inverse from the user's arrays (with the Elsasser sums, or the sin / cos kinds), y-inverse over all ky, z
// pass over all kz.  The reference dealiases the nonlinear term, the pressure and the step's result, so the forward
// half is the pruned one of the fused step, down to the projected right-hand side on the kept modes (compact
// layout); one element-wise launch then applies the stage of single_time_step.cc / time_advance.cc to every mode, and
// the step's input stays in the caller's arrays until the last stage (no copies).
//
// What bounds it: the operation-by-operation sequence moved each field about 150 times per NS evaluation (transforms
// of three passes each, separate products, derivatives, sums, scalings, copies); this moves the inverse lines four
// times, the pruned products four, and each field twice more.  128^3 FP64 forced MHD RK4: 6.05 ms before.
#pragma once
#include "th_force.hpp"
#include "th_fused_kern.hpp"

namespace th {

// components of a step's fields in the reference layout
struct FieldPtrs {
    const void* v[6];
};

// x-inverse of reference-layout fields: column m = (ky, kz) of every mode -> A[x][ky][kz].
//   KIND 0: components as they are; 1: Z+ = U + B (0-2), Z- = U - B (3-5); 2: SCFT V1 (sine), V2, V3 (cosine), T (sine),
//   rows in the order of k_sx_inv.
template <typename R, int L, int P, int T, int KIND>
__global__ __launch_bounds__(T * P) void k_px_inv(FG g, FieldPtrs f, cplx<R>* __restrict__ A, const cplx<R>* __restrict__ tw,
                                                  const cplx<R>* __restrict__ tw4)
{
    using F = LineFFT<R, L, P, +1>;
    __shared__ cplx<R> lds[L * T];
    __shared__ cplx<R> twl[L];
    stage_tw<R, L>(twl, tw);
    const int c = threadIdx.x % T, t = threadIdx.x / T;
    const int m = blockIdx.x * T + c;            // over the N2 x H modes of one kx
    const int M = g.N2 * g.nkz;
    const bool ok = m < M;
    const int oc = blockIdx.y;
    const int y = ok ? m / g.nkz : 0, cz = m - y * g.nkz;
    cplx<R>* out = A + (long)y * g.KZP + cz;
    cplx<R> v[F::E];
    __syncthreads();
    if constexpr (KIND == 1) {
        const cplx<R>* u = (const cplx<R>*)f.v[oc] + m;
        const cplx<R>* b = (const cplx<R>*)f.v[3 + oc] + m;
        cplx<R> d[F::E];
#pragma unroll
        for (int i = 0; i < F::E; i++) {
            const long o = (long)F::in_pos(t, i) * M;
            const cplx<R> p = ok ? u[o] : czero<R>(), q = ok ? b[o] : czero<R>();
            v[i] = p + q;
            d[i] = p - q;
        }
        F::template run<T, false, NoPad, false, 0>(v, lds + c, t, twl);
        if (ok) {
#pragma unroll
            for (int i = 0; i < F::E; i++) out[oc * g.cA + (long)F::out_pos(t, i) * g.sx] = v[i];
        }
        F::template run<T, false, NoPad, false, 1>(d, lds + c, t, twl);
        if (ok) {
#pragma unroll
            for (int i = 0; i < F::E; i++) out[(3 + oc) * g.cA + (long)F::out_pos(t, i) * g.sx] = d[i];
        }
        return;
    }
    const cplx<R>* u = (const cplx<R>*)f.v[oc] + m;
    const bool sn = KIND == 2 && (oc == 0 || oc == 3);
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int k = F::in_pos(t, i);
        if constexpr (KIND == 0) {
            v[i] = ok ? u[(long)k * M] : czero<R>();
        } else {                                 // conj(w_k) (X_k - i X_{N-k}), see k_sx_inv
            const cplx<R> ck = (ok && !(sn && k == 0)) ? u[(long)k * M] : czero<R>();
            const cplx<R> cm = (ok && k > 0) ? u[(long)(L - k) * M] : czero<R>();
            const cplx<R> a = sn ? cm : ck, b = sn ? ck : cm;
            v[i] = cmul(conjg(tw4[k]), mk<R>(a.x + b.y, a.y - b.x));
        }
    }
    F::template run<T, false, NoPad, false, 0>(v, lds + c, t, twl);
    if (ok) {
#pragma unroll
        for (int i = 0; i < F::E; i++) {
            const int j = F::out_pos(t, i);
            const R sg = (sn && j >= L / 2) ? R(-1) : R(1);
            out[oc * g.cA + (long)j * g.sx] = KIND == 2 ? cscale(v[i], sg) : v[i];
        }
    }
}

// One stage of the plain steppers on every mode (single_time_step.cc:54-86 with the a, b, c of time_advance.cc).  r is
// the right-hand side (0 outside the kept modes), acc the RK4 sum on the kept modes; V0 the step's input.
//   0 EULER  V = (V0 + dt r) e1                          1 RK4 1 / RK2 1  V = (V0 + dt/2 r) eh, acc = dt/6 r e1
//   2 RK4 2  V = V0 eh + dt/2 r, acc += dt/3 r eh        3 RK4 3  V = (V0 eh + dt r) eh, acc += dt/3 r eh
//   4 RK4 4  V = V0 e1 + acc + dt/6 r                    5 RK2 2  V = (V0 eh + dt r) eh
// 0, 4 and 5 end the step: modes outside the kept ones become 0 (Dealias).  RB: the buoyancy force of the stage's
// input (Force1 = T, T.Force = V1; compute_force_RB.cc:51-105) enters r here, projected as k_sx_fwd_rb projects it.
template <typename R, int NC, bool RB>
__global__ __launch_bounds__(256) void k_plain_stage(FG g, FastDiv dH, FastDiv dN2, int kind, double dt, double d0, double d1,
                                                     FieldPtrs v0, FieldPtrs in, FieldPtrs out, const cplx<R>* __restrict__ rhs,
                                                     cplx<R>* __restrict__ acc)
{
    // every product and sum rounded by itself, as the separate operations of the general path round them
#pragma clang fp contract(off)
    auto sc = [](Dc a, double b) {
#pragma clang fp contract(off)
        return dmk(a.x * b, a.y * b);
    };
    auto add = [](Dc a, Dc b) {
#pragma clang fp contract(off)
        return dmk(a.x + b.x, a.y + b.y);
    };
    const unsigned n = (unsigned)g.N1 * g.N2 * dH.d;
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const unsigned rw = fdiv(i, dH), x = fdiv(rw, dN2);
        const int l3 = (int)(i - rw * dH.d), l2 = (int)(rw - x * dN2.d), l1 = (int)x;
        const bool kept = l3 < g.nkz && lkept(g.mx, l1) && lkept(g.my, l2);
        const bool last = kind == 0 || kind >= 4;
        if (last && !kept) {
#pragma unroll
            for (int c = 0; c < NC; c++) ((cplx<R>*)out.v[c])[i] = czero<R>();
            continue;
        }
        cplx<R> s[NC], r[NC], a[NC];
        const long j = kept ? (long)lq(g.mx, l1) * g.sx + (long)lq(g.my, l2) * g.KZP + l3 : 0;
        const bool need = kept && (kind == 2 || kind == 3 || kind == 4);
#pragma unroll
        for (int c = 0; c < NC; c++) {
            s[c] = ((const cplx<R>*)v0.v[c])[i];
            r[c] = kept ? rhs[c * g.cS + j] : czero<R>();
            a[c] = need ? acc[c * g.cS + j] : czero<R>();
        }
        const double kx = (g.scft ? l1 : kx_four(l1, g.N1)) * g.f1, ky = ky_of(l2, g.N2) * g.f2, kz = l3 * g.f3;
        const double k2 = ksq_f(kx, ky, kz);
        const double h0 = exp(-d0 * 0.5 * dt * k2), h1 = NC > 3 ? exp(-d1 * 0.5 * dt * k2) : 0.0;
        // the whole step's factors by themselves (not as squares: one rounding, as k_exp_ksqr's)
        const bool whole = kind == 0 || kind == 1 || kind == 4;
        const double w0 = whole ? exp(-d0 * dt * k2) : 0.0, w1 = NC > 3 && whole ? exp(-d1 * dt * k2) : 0.0;
        Dc q[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) q[c] = dl(r[c]);
        if (RB && kept) {
            const Dc T = dl(((const cplx<R>*)in.v[NC - 1])[i]), V1 = dl(((const cplx<R>*)in.v[0])[i]);
            const double w = k2 > 0 ? kx / k2 : 0.0;         // p = -Kx T / K^2 of the force alone
            q[0] = dadd(q[0], dsc(T, 1.0 - kx * w));
            q[1] = dadd(q[1], dmk(-ky * w * T.y, ky * w * T.x));
            q[2] = dadd(q[2], dmk(-kz * w * T.y, kz * w * T.x));
            q[NC - 1] = dadd(q[NC - 1], V1);
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const double eh = c < 3 ? h0 : h1, e1 = c < 3 ? w0 : w1;
            const Dc V = dl(s[c]);
            Dc o;
            if (kind == 0) o = sc(add(V, sc(q[c], dt)), e1);
            else if (kind == 1) o = sc(add(V, sc(q[c], 0.5 * dt)), eh);
            else if (kind == 2) o = add(sc(V, eh), sc(q[c], 0.5 * dt));
            else if (kind == 4) o = add(sc(V, e1), add(dl(a[c]), sc(q[c], dt / 6)));
            else o = sc(add(sc(V, eh), sc(q[c], dt)), eh);
            ((cplx<R>*)out.v[c])[i] = ds<R>(o);
            if (kept && acc) {
                if (kind == 1) acc[c * g.cS + j] = ds<R>(sc(q[c], dt / 6 * e1));
                else if (kind == 2 || kind == 3) acc[c * g.cS + j] = ds<R>(add(dl(a[c]), sc(q[c], dt / 3 * eh)));
            }
        }
    }
}

// The forces of a stage (force_write / force_subtract of th_force.hip) added to the right-hand side on the band's
// modes, all of them kept (plain_fast_force): P(F) for U, F for W (PROJ false), as rhs = -P(N - F).
template <typename R, bool PROJ>
__global__ __launch_bounds__(256) void k_plain_force(FG g, ForceBand b, const cplx<R>* __restrict__ V0,
                                                     const cplx<R>* __restrict__ V1, const cplx<R>* __restrict__ V2,
                                                     cplx<R>* __restrict__ rhs)
{
    const long n = (long)b.nx * b.ny * b.nz, t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    int lx, ly, lz, sx, sy;
    band_mode(b, t, lx, ly, lz);
    if (!(lz < g.nkz && lkept(g.mx, lx) && lkept(g.my, ly))) return;     // carries no force
    const bool mirror = reality_source(b, lx, ly, lz, sx, sy);
    const long si = ((long)sx * b.N2 + sy) * b.H + lz;
    const cplx<R> v[3] = {V0[si], V1[si], V2[si]};
    double fr[3], fi[3];
    mode_force<R>(b, v, sx, sy, lz, fr, fi);
    if (mirror)
        for (int c = 0; c < 3; c++) fi[c] = -fi[c];
    const double K[3] = {kx_four(lx, g.N1) * g.f1, ky_of(ly, g.N2) * g.f2, lz * g.f3};
    const double k2 = ksq_f(K[0], K[1], K[2]);
    if (PROJ && k2 > 0) {
        const double dr = (K[0] * fr[0] + K[1] * fr[1] + K[2] * fr[2]) / k2;
        const double di = (K[0] * fi[0] + K[1] * fi[1] + K[2] * fi[2]) / k2;
        for (int c = 0; c < 3; c++) {
            fr[c] -= K[c] * dr;
            fi[c] -= K[c] * di;
        }
    }
    const long j = (long)lq(g.mx, lx) * g.sx + (long)lq(g.my, ly) * g.KZP + lz;
    for (int c = 0; c < 3; c++) {
        const cplx<R> a = rhs[c * g.cS + j];
        rhs[c * g.cS + j] = mk<R>((R)((double)a.x + fr[c]), (R)((double)a.y + fi[c]));
    }
}

template <typename R, int L, int KIND>
static int launch_px(const FG& g, const FieldPtrs& f, cplx<R>* A, int ncomp, const cplx<R>* tw, const cplx<R>* tw4, hipStream_t st)
{
    constexpr int E = pts_per_thread(L), P = L / E, T = tileT<R>();
    hipLaunchKernelGGL((k_px_inv<R, L, P, T, KIND>), dim3((g.N2 * g.nkz + T - 1) / T, KIND == 1 ? ncomp / 2 : ncomp), dim3(T * P), 0,
                       st, g, f, A, tw, tw4);
    TH_CHECK_HIP(hipGetLastError());
    return OK;
}
template <typename R, int KIND>
static int px_inv(const FG& g, const FieldPtrs& f, cplx<R>* A, int ncomp, const cplx<R>* tw, const cplx<R>* tw4, hipStream_t st)
{
#define C_(n) case n: return launch_px<R, n, KIND>(g, f, A, ncomp, tw, tw4, st);
    switch (g.N1) { TH_FLENS(C_) default: set_error("plain step: N1 %d unsupported", g.N1); return E_UNSUPPORTED; }
#undef C_
}
// z pass with all kz on input (g.KZPi, g.cBi), kept kz on output
template <typename R, int MODE>
static int pz(const FG& g, const cplx<R>* B, cplx<R>* C, const cplx<R>* twL, const cplx<R>* twN, hipStream_t st)
{
#define C_(n) case n: return launch_z<R, n, MODE, 0, true>(g, B, C, twL, twN, st);
    switch (g.LZ) { TH_ZLENS(C_) default: set_error("plain step: N3 %d unsupported", g.N3); return E_UNSUPPORTED; }
#undef C_
}

// The step.  F: the caller's fields (NS 3, MHD 6, RB 4); keep (or null): receives the last stage's input.
template <typename R> int plain_step(th_plan* p, int physics, int scheme, cplx<R>* const* F, double dt, double d0, double d1,
                                     const ForceBand* fu, const ForceBand* fw, cplx<R>* const* keep)
{
    hipStream_t st = p->ctx->stream;
    const int nc = physics == TH_NS ? 3 : physics == TH_MHD ? 6 : 4, nout = physics == TH_NS ? 6 : 9;
    Geo full = p->g;
    full.dealias = 0;
    const int prec = sizeof(R) == 4 ? 1 : 0;
    const FG gf = make_fg(full, prec);
    FG g = make_fg(p->g, prec);
    g.KZPi = gf.KZP;
    g.cBi = gf.cB;
    // X: A, then the product lines C; Y: B, then D; compact: rhs, the RK4 sum, a zero state, the unused accumulator
    const size_t sX = (size_t)std::max(nc * gf.cA, nout * g.cB), sY = (size_t)std::max(nc * gf.cB, nout * g.cA);
    const size_t sC = (size_t)nc * g.cS, nfull = p->g.ncplx();
    PlainBufs& w = p->plain;
    TRY(plain_ensure(w, sizeof(cplx<R>), sX, sY, sC, nfull * nc, st));
    cplx<R>*X = (cplx<R>*)w.X, *Y = (cplx<R>*)w.Y, *rhs = (cplx<R>*)w.rhs(), *acc = (cplx<R>*)w.acc();
    cplx<R>*zero = (cplx<R>*)w.zero(), *junk = (cplx<R>*)w.junk();
    for (int L : {g.N1, g.N2, g.LZ, g.N3, g.scft ? 4 * g.N1 : g.N1})
        if (!p->tw.get(L, prec, st)) { set_error("twiddle table allocation failed"); return E_NOMEM; }
    const cplx<R>*twx = p->twd<R>(g.N1), *twy = p->twd<R>(g.N2), *twz = p->twd<R>(g.LZ), *twn = p->twd<R>(g.N3);
    const cplx<R>* tw4 = g.scft ? p->twd<R>(4 * g.N1) : twx;
    FieldPtrs v0{}, fs{};
    for (int c = 0; c < nc; c++) {
        v0.v[c] = F[c];
        fs.v[c] = (cplx<R>*)w.Fs + (size_t)c * nfull;
    }
    const int nst = scheme == 0 ? 1 : scheme == 1 ? 2 : 4;
    for (int s = 0; s < nst; s++) {
        const bool last = s == nst - 1;
        const FieldPtrs& in = s == 0 ? v0 : fs;
        if (last && keep && keep[0])
            for (int c = 0; c < nc; c++)
                if (keep[c] != F[c])        // the field's own array ends as the step's result
                    TH_CHECK_HIP(hipMemcpyAsync(keep[c], in.v[c], nfull * sizeof(cplx<R>), hipMemcpyDeviceToDevice, st));
        if (physics == TH_NS) TRY((px_inv<R, 0>(gf, in, X, 3, twx, tw4, st)));
        else if (physics == TH_MHD) TRY((px_inv<R, 1>(gf, in, X, 6, twx, tw4, st)));
        else TRY((px_inv<R, 2>(gf, in, X, 4, twx, tw4, st)));
        TRY(d_yinv<R>(gf, X, Y, nc, twy, 0, st));
        if (physics == TH_NS) TRY((pz<R, 0>(g, Y, X, twz, twn, st)));
        else if (physics == TH_MHD) TRY((pz<R, 1>(g, Y, X, twz, twn, st)));
        else TRY((pz<R, 3>(g, Y, X, twz, twn, st)));
        TRY(d_yfwd<R>(g, X, Y, nout, twy, 0, st));
        // the fused x-forward's first stage on a zero state with dt = 2 and no dissipation stores 0 + r
        if (physics == TH_NS) TRY((d_xfwd<R, 0>(g, Y, Y, zero, rhs, junk, twx, (const StageCoef*)w.coef, 0, st, false)));
        else if (physics == TH_MHD) TRY((d_xfwd<R, 1>(g, Y, Y, zero, rhs, junk, twx, (const StageCoef*)w.coef, 0, st, false)));
        else TRY(d_sx_fwd_rb<R>(g, Y, zero, rhs, junk, twx, tw4, (const StageCoef*)w.coef, 0, st));
        auto add_force = [&](const ForceBand* b, int c0, bool proj) -> int {
            const unsigned nb = (unsigned)(((long)b->nx * b->ny * b->nz + 255) / 256);
            auto k = proj ? k_plain_force<R, true> : k_plain_force<R, false>;
            hipLaunchKernelGGL(k, dim3(nb), dim3(256), 0, st, g, *b, (const cplx<R>*)in.v[c0], (const cplx<R>*)in.v[c0 + 1],
                               (const cplx<R>*)in.v[c0 + 2], rhs + c0 * g.cS);
            TH_CHECK_HIP(hipGetLastError());
            return OK;
        };
        if (fu) TRY(add_force(fu, 0, true));
        if (fw) TRY(add_force(fw, 3, false));
        const int kind = scheme == 0 ? 0 : scheme == 1 ? (last ? 5 : 1) : s + 1;
        const FieldPtrs& out = last ? v0 : fs;
        const dim3 grid((unsigned)std::min<size_t>((nfull + 255) / 256, 65536));
        auto go = [&](auto k) {
            hipLaunchKernelGGL(k, grid, dim3(256), 0, st, g, fast_div(p->g.H), fast_div(g.N2), kind, dt, d0, d1, v0, in, out,
                               (const cplx<R>*)rhs, acc);
        };
        if (physics == TH_NS) go(k_plain_stage<R, 3, false>);
        else if (physics == TH_MHD) go(k_plain_stage<R, 6, false>);
        else go(k_plain_stage<R, 4, true>);
        TH_CHECK_HIP(hipGetLastError());
    }
    return OK;
}

}  // namespace th
