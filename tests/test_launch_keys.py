"""Keys of captured waves (put_trace_key, put_instances_key, put_guide_key,
compiled here for the CPU): a graph is replayed for an equal key, so whatever
its launches hold has to change the key, also where the addresses come back
with another tree, instance set or network."""

import os
import subprocess

import pytest

from sprout_amd import build

DRIVER = r"""
#include "guide.hpp"
#include "instances.hpp"
#include "trace.hpp"
#include <cstdio>
using namespace mi;
static int failures = 0;
template <class F, class S, class V>
void differs(char const* name, S s, F key_of, V change) {
    Launch_key const a = key_of(s);
    if (a != key_of(s)) std::printf("%s: not repeatable\n", name), ++failures;
    change(s);
    if (a == key_of(s)) std::printf("%s: not in the key\n", name), ++failures;
}
#define TREE(field, value) differs("tree " #field, tree, tree_key, [&](DeviceBvh& t) { t.field = value; })
#define RES(field, value) differs("launch " #field, res, res_key, [&](TraceResources& r) { r.field = value; })
#define TLAS(field, value) differs("instances " #field, tlas, tlas_key, [&](Tlas& t) { t.field = value; })
#define NET(field, value) differs("network " #field, net, net_key, [&](GuideNet& n) { n.field = value; })
int main() {
    DeviceBvh      tree;
    TraceResources res;
    Tlas           tlas;
    GuideNet       net;
    float4* const   f = reinterpret_cast<float4*>(64);
    uint32_t* const u = reinterpret_cast<uint32_t*>(64);
    float* const    x = reinterpret_cast<float*>(64);
    auto tree_key = [&](DeviceBvh const& t) { Launch_key k; put_trace_key(k, t, res); return k; };
    auto res_key  = [&](TraceResources const& r) { Launch_key k; put_trace_key(k, tree, r); return k; };
    auto tlas_key = [](Tlas const& t) { Launch_key k; put_instances_key(k, t); return k; };
    auto net_key  = [](GuideNet const& n) { Launch_key k; put_guide_key(k, n); return k; };
    TREE(nodes, f); TREE(tris, f); TREE(num_nodes, 3); TREE(num_slots, 3); TREE(max_depth, 9);
    TREE(qpairs, reinterpret_cast<uint4*>(64));
    TREE(qorigin[1], 2.f); TREE(qscale[2], 2.f);
    RES(block_size, 64); RES(blocks_per_cu, 1); RES(num_cus, 1); RES(kernel, 2); RES(refill_lanes, 1);
    RES(claim_batch, 1); RES(lds_entries, 1); RES(counter, u); RES(spill, u);
    TLAS(tree.nodes, f); TLAS(tree.tris, f); TLAS(tree.num_nodes, 3); TLAS(spill, u); TLAS(spill_total, 64);
    TLAS(claims, u);
    TLAS(instances, reinterpret_cast<Instance_record*>(64)); TLAS(meshes, reinterpret_cast<Mesh_view*>(64));
    NET(params, x); NET(adam_m, x); NET(adam_v, x); NET(grad, x); NET(partial, x); NET(wsum, x); NET(freq, x);
    NET(wt, reinterpret_cast<uint16_t*>(64)); NET(window, u); NET(step_dev, u); NET(scratch_step, u);
    NET(partial_blocks, 3);
    return failures;
}
"""


def test_everything_a_captured_launch_holds_is_in_its_key(tmp_path):
    if not os.path.exists(build.hipcc()):
        pytest.skip("no hipcc")
    (tmp_path / "driver.hip").write_text(DRIVER)
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "--cuda-host-only", "-c", str(tmp_path / "driver.hip"),
                    "-o", str(tmp_path / "driver.o")], check=True, capture_output=True)
    subprocess.run([build.hipcc(), str(tmp_path / "driver.o"), "-o", str(tmp_path / "driver")], check=True)
    r = subprocess.run([str(tmp_path / "driver")], capture_output=True, text=True, timeout=120)
    assert 0 == r.returncode, r.stdout
