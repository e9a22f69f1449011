// th_grow.hpp -- buffers that grow and are kept: the growth rule and the plain steppers' workspace, independent of the
// allocator (host code only).
#pragma once
#include <stddef.h>

namespace th {

// p holds cap elements; afterwards at least need, or none and cap 0 where the allocation failed, so that no later, smaller
// request takes a lost buffer for a present one.  The old buffer goes first (no need to hold both).  alloc(&p, elements)
// returns 0 or the error to pass on, release(p) gives back.
template <typename T, typename Alloc, typename Release>
int regrow(T*& p, size_t& cap, size_t need, Alloc alloc, Release release)
{
    if (need <= cap) return 0;
    if (p) release(p);
    p = nullptr;
    cap = 0;
    const int r = alloc(&p, need);
    if (r) {
        p = nullptr;
        return r;
    }
    cap = need;
    return 0;
}

// Workspace of the plain steppers (th_plain.hpp), kept in the plan and grown to the largest physics it has stepped: X and
// Y pipeline lines; rhs, acc, zero, junk compact fields; Fs stage fields in the reference layout; coef one StageCoef.
// Mem: alloc(&p, bytes, cleared) -> 0 or an error, release(p).
struct PlainBufs {
    void *X = nullptr, *Y = nullptr, *C[4] = {}, *Fs = nullptr, *coef = nullptr;
    size_t bX = 0, bY = 0, bC[4] = {}, bF = 0, bK = 0;
    void* rhs() const { return C[0]; }
    void* acc() const { return C[1]; }
    void* zero() const { return C[2]; }
    void* junk() const { return C[3]; }

    // sizes in bytes; *fresh: whether coef is new and has to be filled
    template <class Mem> int ensure(Mem& m, size_t nX, size_t nY, size_t nC, size_t nF, size_t nK, bool* fresh)
    {
        auto grow = [&](void*& q, size_t& cap, size_t n, bool clear) {
            return regrow(q, cap, n, [&](void** p, size_t b) { return m.alloc(p, b, clear); }, [&](void* p) { m.release(p); });
        };
        int r = grow(X, bX, nX, true);
        if (!r) r = grow(Y, bY, nY, true);
        for (int i = 0; i < 4 && !r; i++) r = grow(C[i], bC[i], nC, true);
        if (!r) r = grow(Fs, bF, nF, false);
        *fresh = !r && nK > bK;
        if (!r) r = grow(coef, bK, nK, false);
        return r;
    }
    template <class Mem> void release(Mem& m)
    {
        for (void** q : {&X, &Y, &C[0], &C[1], &C[2], &C[3], &Fs, &coef}) {
            if (*q) m.release(*q);
            *q = nullptr;
        }
        bX = bY = bF = bK = 0;
        for (size_t& b : bC) b = 0;
    }
};

}  // namespace th
