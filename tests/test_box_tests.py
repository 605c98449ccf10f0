"""The traversals' two box tests (device_math.hpp, compiled here for the CPU):
slab with the reference's NaN filters and slab_lean without them admit the
same boxes, and slab_lean's entry distance gives slab's answer at every
smaller max_t.  Rays that start on a box's plane with a direction component
whose inverse is infinite, zero or NaN are the forms where they can part."""

import os
import subprocess

import pytest

from sprout_amd import build

HIP_STUB = """
#pragma once
#include <cmath>
#include <cstdint>
#define __device__
#define __host__
#define __forceinline__ inline
struct float4 { float x, y, z, w; };
"""

DRIVER = r"""
#include "device_math.hpp"
#include <cstdio>
#include <vector>
using namespace mi::dev;
struct Axis { float lo, hi, o, inv; };
int main() {
    float const inf = __builtin_inff(), nan = __builtin_nanf("");
    float const dirs[] = {0.f, -0.f, 1e-20f, -1e-20f, 1e-30f, -1e-30f, 3.7e-33f, 5.4e-20f, -5.5e-20f,
                          1e-42f, -1e-42f, 0.01f, 1.f, -2.f, 3e38f, inf, -inf, nan};
    float const at[]   = {-inf, -3e38f, -2.f, -1.f, 0.f, 0.25f, 2.f, 3e38f, inf, nan};
    uint64_t state = 1;
    auto rnd = [&](uint32_t n) {
        state = state * 6364136223846793005ull + 1442695040888963407ull;
        return uint32_t((state >> 33) % n);
    };
    std::vector<Axis> finite, all;  // boxes of an axis in order, and any bounds
    for (float d : dirs)
        for (float lo : at)
            for (float hi : at)
                for (float o : at) {
                    Axis const a = {lo, hi, o, reciprocal_lane(d)};
                    all.push_back(a);
                    if (lo <= hi && std::isfinite(lo) && std::isfinite(hi) && std::isfinite(o))
                        finite.push_back(a);
                }
    float const ts[] = {0.f, 1e-4f, 1.f, 5.f, 3.40282347e+38f, inf, -1.f};
    long tests = 0, admitted = 0, differ = 0, later = 0;
    auto check = [&](Axis const& x, Axis const& y, Axis const& z) {
        float4 const lo = {x.lo, y.lo, z.lo, 0.f}, hi = {x.hi, y.hi, z.hi, 0.f};
        F3 const     o = {x.o, y.o, z.o}, inv = {x.inv, y.inv, z.inv};
        float const  min_t = ts[rnd(7)], max_t = ts[rnd(7)];
        float        entry;
        bool const   a = slab(lo, hi, o, inv, min_t, max_t);
        bool const   b = slab_lean(lo, hi, o, inv, min_t, max_t, entry);
        ++tests;
        admitted += a;
        if (a != b && differ++ < 5)
            std::printf("lo %g %g %g hi %g %g %g o %g %g %g inv %g %g %g t %g %g: %d %d\n", x.lo, y.lo,
                        z.lo, x.hi, y.hi, z.hi, x.o, y.o, z.o, x.inv, y.inv, z.inv, min_t, max_t, a, b);
        for (float t : ts)
            if (a && b && t <= max_t) later += slab(lo, hi, o, inv, min_t, t) == (t < entry);
    };
    Axis const unit = {-1.f, 1.f, 0.f, 1.f};
    for (Axis const& a : all) check(a, unit, unit), check(unit, a, unit), check(unit, unit, a);
    for (int i = 0; i < 2000000; ++i) {
        auto const& set = i & 1 ? finite : all;
        check(set[rnd(set.size())], set[rnd(set.size())], set[rnd(set.size())]);
    }
    std::printf("%ld tests, %ld admitted, %ld differ, %ld entry distances\n", tests, admitted, differ, later);
    return differ || later || admitted < tests / 20;
}
"""


def test_the_lean_box_test_is_the_filtered_one(tmp_path):
    clang = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")
    if not os.path.exists(clang):
        pytest.skip("no clang++")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP_STUB)
    (tmp_path / "driver.cpp").write_text(DRIVER)
    subprocess.run([clang, "-std=c++17", "-O1", "-ffp-contract=off", "-fno-fast-math", "-I", str(tmp_path),
                    "-I", build.CSRC, str(tmp_path / "driver.cpp"), "-o", str(tmp_path / "driver")], check=True)
    r = subprocess.run([str(tmp_path / "driver")], capture_output=True, text=True, timeout=120)
    assert 0 == r.returncode, r.stdout
