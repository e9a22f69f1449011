// th_plane_f64.hip -- the short-box kernels of th_plane.hpp in FP64.
#include "th_plane.hpp"

namespace th {

template <>
int d_plane<double>(const FG& g, const PlaneTab& tab, int ngrp, const cplx<double>* A, cplx<double>* D, long bD, const cplx<double>* tw2,
                const cplx<double>* twL, const cplx<double>* twN, hipStream_t st)
{
#define C_(n) case n: return plane_z<double, n>(g, tab, ngrp, A, D, bD, tw2, twL, twN, st);
    switch (g.N2) {
        C_(16) C_(24) C_(32) C_(48) C_(64) C_(96) C_(128)
        default: set_error("plane pass: N2 %d unsupported", g.N2); return E_UNSUPPORTED;
    }
#undef C_
}

}  // namespace th
