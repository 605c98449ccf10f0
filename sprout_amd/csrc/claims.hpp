// Ray claims of the persistent refill traversals (device code).
#pragma once

#include "trace.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mi {

// The ray claims of the refill kernels.  Every wave starts on a slice of its
// own, which costs no memory access: `chunk` rays, 64 where the launch has
// that many for every wave it spreads over, fewer for a small launch, whose
// rays then sit in more waves with fewer rays each.  A wave's loop runs as
// long as the union of its rays' walks, so a launch that cannot fill the
// chip ends sooner that way (1 531 camera rays over 5 620 triangles: 64 us
// with 64 rays a wave, 34 us with one; a preview frame of 97x61 546 and 490
// us).  The rays past the slices go out in
// claims of `batch` rays from Claim_parts counter words, each on its own
// 256-byte line (Claim_stride words apart): atomics on one address serialize
// (about 12 ns each).  Wave w claims from part w mod parts only, and the
// parts own runs of Claim_run claims in turn, so all parts hold the same mix
// of rays and end together: a wave whose part is used up is done, after one
// atomic (looking for open parts cost up to one round trip for each of the
// 32, about 25 us also for an empty queue).  Workgroups go round the eight
// XCDs, and with four waves each parts 4x .. 4x + 3 belong to XCD x: its L2
// sees runs of 4 Claim_run claims.
inline constexpr uint32_t Claim_run = 8;

// Rays of a wave's slice.
__host__ __device__ inline uint32_t claim_chunk(uint32_t num_rays, uint32_t waves, uint32_t spread) {
    uint32_t const over = waves < spread ? waves : spread;
    uint32_t const want = num_rays / over + (num_rays % over ? 1u : 0u);
    return want < 64u ? want : 64u;
}

// Whether rays are left over past the slices: only then does a launch touch
// its counters.
inline bool claims_rays(uint32_t num_rays, uint32_t waves, uint32_t spread) {
    return uint64_t(waves) * claim_chunk(num_rays, waves, spread) < num_rays;
}

struct Claims {
    uint32_t part;   // wave-uniform: the part claimed from
    uint32_t parts;  // all parts (at most the launch's waves, so each has a wave)
    uint32_t fixed;  // rays handed out by slices; the parts split the rest

    // The wave's slice [begin, end) of num_rays rays (wave-uniform); waves is
    // the launch's, spread the number of waves a small launch fills first.
    __device__ void init(uint32_t wave, uint32_t waves, uint32_t spread, uint32_t num_rays,
                         uint32_t& begin, uint32_t& end) {
        uint32_t const chunk = claim_chunk(num_rays, waves, spread);
        uint64_t const all   = uint64_t(waves) * chunk;
        fixed                = all < num_rays ? uint32_t(all) : num_rays;
        uint64_t const lo    = uint64_t(wave) * chunk;
        begin                = lo < fixed ? uint32_t(lo) : fixed;
        end                  = fixed - begin < chunk ? fixed : begin + chunk;
        parts                = waves < Claim_parts ? waves : Claim_parts;
        part                 = wave % parts;
    }

    // Claims up to batch rays [begin, end) for the wave; all 64 lanes call
    // it.  False once the wave's part is used up.
    __device__ bool next(uint32_t* counters, uint32_t num_rays, uint32_t batch, uint32_t lane,
                         uint32_t& begin, uint32_t& end) {
        if (fixed == num_rays) {
            return false;
        }
        uint32_t k = 0;
        if (0 == lane) {
            k = atomicAdd(counters + part * Claim_stride, 1u);
        }
        k = __builtin_amdgcn_readfirstlane(k);
        uint64_t const rest  = num_rays - fixed;
        uint64_t const claim = (uint64_t(k / Claim_run) * parts + part) * Claim_run + k % Claim_run;
        uint64_t const lo    = claim * batch;
        if (lo >= rest) {
            return false;
        }
        begin = fixed + uint32_t(lo);
        end   = rest - lo < batch ? num_rays : begin + batch;
        return true;
    }
};

}  // namespace mi
