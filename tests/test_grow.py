"""The growth of kept buffers (csrc/th_grow.hpp) with an allocator that fails at a chosen call, built with g++."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tarang_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <set>
#include "th_grow.hpp"

static std::set<void*> live;
static int calls = 0, fail_at = -1;
static int get(void** p, size_t bytes)
{
    if (calls++ == fail_at) { *p = (void*)1; return 7; }      // what a failed allocator leaves there is not looked at
    *p = malloc(bytes);
    live.insert(*p);
    return 0;
}
static void put(void* p)
{
    if (!live.erase(p)) { printf("released what is not held\n"); exit(1); }
    free(p);
}
#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

struct Mem {
    int cleared = 0;
    int alloc(void** p, size_t b, bool clear) { cleared += clear; return get(p, b); }
    void release(void* p) { put(p); }
};

int main()
{
    auto alloc = [](double** p, size_t n) { return get((void**)p, n * sizeof(double)); };
    auto rel = [](double* p) { put(p); };
    double* p = nullptr;
    size_t cap = 0;
    CHECK(th::regrow(p, cap, 100, alloc, rel) == 0 && p && cap == 100);
    double* const first = p;
    CHECK(th::regrow(p, cap, 40, alloc, rel) == 0 && p == first && cap == 100);
    fail_at = calls;
    CHECK(th::regrow(p, cap, 200, alloc, rel) == 7 && !p && cap == 0 && live.empty());
    fail_at = calls;                                   // a smaller request after the failure allocates again
    CHECK(th::regrow(p, cap, 40, alloc, rel) == 7 && !p && cap == 0);
    CHECK(th::regrow(p, cap, 40, alloc, rel) == 0 && p && cap == 40 && live.size() == 1);
    put(p);

    // the workspace, failing at each of its eight allocations in turn: everything can be given back, or the call repeated
    for (int k = 0; k < 8; k++)
        for (int repeat = 0; repeat < 2; repeat++) {
            th::PlainBufs w;
            Mem m;
            bool fresh = true;
            fail_at = calls + k;
            CHECK(w.ensure(m, 64, 32, 16, 8, 4, &fresh) == 7 && fresh == (k == 7));
            CHECK((int)live.size() == k);
            if (repeat) {
                CHECK(w.ensure(m, 64, 32, 16, 8, 4, &fresh) == 0 && fresh && live.size() == 8);
                CHECK(w.ensure(m, 64, 32, 16, 8, 4, &fresh) == 0 && !fresh && live.size() == 8);
                fail_at = calls + 1;                   // growing to a larger physics: X goes, Y fails
                CHECK(w.ensure(m, 128, 64, 32, 16, 4, &fresh) == 7 && !w.Y && w.bY == 0 && w.bX == 128 && live.size() == 7);
                CHECK(w.ensure(m, 64, 32, 16, 8, 4, &fresh) == 0 && !fresh && w.Y && w.bY == 32 && live.size() == 8);
            }
            w.release(m);
            CHECK(live.empty() && !w.X && !w.coef && !w.rhs() && w.bX + w.bY + w.bC[0] + w.bC[3] + w.bF + w.bK == 0);
        }
    printf("ok\n");
    return 0;
}
"""


def test_failed_growth_leaves_nothing_behind(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "grow.cpp", str(tmp_path / "grow")
    src.write_text(PROGRAM)
    subprocess.check_call([gxx, "-std=c++17", "-O1", "-Wall", "-I" + CSRC, "-o", exe, str(src)])
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
