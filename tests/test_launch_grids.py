"""The traversals' launch grids (trace.hpp, compiled here for the CPU): the
stack area reserved for a launch holds that of every smaller one."""

import os
import subprocess

import pytest

from sprout_amd import build

DRIVER = r"""
#include "trace.hpp"
#include <cstdio>
using mi::TraceResources;
int main() {
    for (uint32_t cus : {1u, 64u, 256u, 304u}) {
        for (uint32_t block : {64u, 256u, 1024u}) {
            for (uint32_t per_cu : {1u, 8u, 32u}) {
                TraceResources r;
                r.num_cus       = cus;
                r.block_size    = block;
                r.blocks_per_cu = per_cu;
                uint32_t most   = 0;
                for (uint32_t n = 1; n < 80 * r.spread_waves(); n += 1 + n / 512) {
                    uint32_t const b = r.grid_blocks(n);
                    most             = b > most ? b : most;
                    if (r.max_blocks(n) < most || r.max_blocks(n) > cus * per_cu) {
                        std::printf("%u CUs, block %u x %u: %u rays reserve %u of %u\n", cus, block, per_cu, n,
                                    r.max_blocks(n), most);
                        return 1;
                    }
                }
                // the largest is reached by a launch of at most spread_waves() or n rays
                if (r.max_blocks(0xFFFFFFFFu) != cus * per_cu) return 2;
            }
        }
    }
    return 0;
}
"""


def test_a_smaller_launch_needs_no_more_stack(tmp_path):
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    clang = os.path.join(rocm, "llvm", "bin", "clang++")
    if not os.path.exists(clang):
        pytest.skip("no clang++")
    (tmp_path / "driver.cpp").write_text(DRIVER)
    subprocess.run([clang, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(rocm, "include"),
                    "-I", os.path.join(build.ROOT, "include"), "-I", build.CSRC, str(tmp_path / "driver.cpp"),
                    "-o", str(tmp_path / "driver")], check=True)
    r = subprocess.run([str(tmp_path / "driver")], capture_output=True, text=True, timeout=120)
    assert 0 == r.returncode, r.stdout
