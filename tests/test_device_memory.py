"""Device allocations (device_memory.hpp, compiled here for the CPU over a
stub of the runtime): when memory is used up the workspace kept between tree
builds is given back and the allocation tried once more."""

import os
import subprocess

import pytest

from sprout_amd import build

DRIVER = r"""
#include "device_memory.hpp"
#include <cstdio>
static int       tries, released, kept;
static size_t    free_bytes;
static hipError_t pending;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    ++tries;
    if (n > free_bytes) return pending = hipErrorOutOfMemory;
    *p = &tries;
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { hipError_t e = pending; pending = hipSuccess; return e; }
namespace mi {
bool release_build_workspace() {
    if (!kept) return false;
    ++released;
    free_bytes += kept;
    kept = 0;
    return true;
}
}
static int check(size_t room, int held, size_t n, hipError_t want, int want_tries, int want_released) {
    tries = released = 0, kept = held, free_bytes = room, pending = hipSuccess;
    float* p = nullptr;
    hipError_t const e = mi::device_malloc(&p, n);
    bool const ok = e == want && tries == want_tries && released == want_released && (e || (p && !pending));
    if (!ok) std::printf("%zu of %zu + %d: error %d, %d tries, %d released, pending %d\n", n, room, held, e, tries, released, pending);
    return !ok;
}
int main() {
    return check(10, 5, 8, hipSuccess, 1, 0) + check(10, 5, 14, hipSuccess, 2, 1) +
           check(10, 5, 16, hipErrorOutOfMemory, 2, 1) + check(10, 0, 11, hipErrorOutOfMemory, 1, 0);
}
"""


def test_a_kept_workspace_is_given_back(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    clang = os.path.join(rocm, "llvm", "bin", "clang++")
    if not os.path.exists(clang):
        pytest.skip("no clang++")
    (tmp_path / "driver.cpp").write_text(DRIVER)
    subprocess.run([clang, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", build.CSRC, str(tmp_path / "driver.cpp"), "-o", str(tmp_path / "driver")], check=True)
    r = subprocess.run([str(tmp_path / "driver")], capture_output=True, text=True, timeout=120)
    assert 0 == r.returncode, r.stdout
