// th_xsplit_f64.hip -- the short-line x-forward of th_plane.hpp in FP64.
#include "th_plane.hpp"

namespace th {

// columns per workgroup: rows of 64 bytes, halved where nine products of 128 points would pass 1024 threads
template <int MODE> static int xsplit(const FG& g, const cplx<double>* D, cplx<double>* Aout, cplx<double>* S, cplx<double>* Vs, cplx<double>* acc,
                                      const cplx<double>* tw, const StageCoef* sc, hipStream_t st, bool chain)
{
    constexpr int T = 64 / sizeof(cplx<double>);
#define C_(n) case n: return launch_xsplit<double, n, (MODE == 1 && n == 128 && T > 4) ? T / 2 : T, MODE>(g, D, Aout, S, Vs, acc, tw, sc, st, chain);
    switch (g.N1) {
        C_(16) C_(24) C_(32) C_(48) C_(64) C_(96) C_(128)
        default: set_error("split x-forward: N1 %d unsupported", g.N1); return E_UNSUPPORTED;
    }
#undef C_
}

template <>
int d_xsplit<double, 0>(const FG& g, const cplx<double>* D, cplx<double>* Aout, cplx<double>* S, cplx<double>* Vs, cplx<double>* acc, const cplx<double>* tw,
                    const StageCoef* sc, hipStream_t st, bool chain)
{
    return xsplit<0>(g, D, Aout, S, Vs, acc, tw, sc, st, chain);
}
template <>
int d_xsplit<double, 1>(const FG& g, const cplx<double>* D, cplx<double>* Aout, cplx<double>* S, cplx<double>* Vs, cplx<double>* acc, const cplx<double>* tw,
                    const StageCoef* sc, hipStream_t st, bool chain)
{
    return xsplit<1>(g, D, Aout, S, Vs, acc, tw, sc, st, chain);
}

template <>
int d_sxsplit<double>(const FG& g, const cplx<double>* D, cplx<double>* Aout, cplx<double>* S, cplx<double>* Vs, cplx<double>* acc,
                     const cplx<double>* tw, const cplx<double>* tw4, const StageCoef* sc, hipStream_t st, bool chain)
{
    constexpr int T = 64 / sizeof(cplx<double>);
#define C_(n) case n: return launch_sxsplit<double, n, (n == 128 && T > 4) ? T / 2 : T>(g, D, Aout, S, Vs, acc, tw, tw4, sc, st, chain);
    switch (g.N1) {
        C_(16) C_(24) C_(32) C_(48) C_(64) C_(96) C_(128)
        default: set_error("split x-forward: N1 %d unsupported", g.N1); return E_UNSUPPORTED;
    }
#undef C_
}

}  // namespace th
