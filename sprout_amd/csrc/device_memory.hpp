// Device allocations of the library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace mi {

// Frees the workspace that the tree builder keeps between builds
// (bvh_build.hip); false when none is kept.
bool release_build_workspace();

// hipMalloc; when the device's memory is used up, once more without the kept
// workspace.
template <class T>
hipError_t device_malloc(T** p, size_t bytes) {
    hipError_t e = hipMalloc(reinterpret_cast<void**>(p), bytes);
    if (hipErrorOutOfMemory == e && release_build_workspace()) {
        (void)hipGetLastError();  // the first try's
        e = hipMalloc(reinterpret_cast<void**>(p), bytes);
    }
    return e;
}

}  // namespace mi
