// GPU construction of sprout's triangle SBVH.
//
// Produces the tree scene::shape::triangle::bvh::Builder_SAH produces
// (triangle_bvh_builder_sah.cpp:21-67 over scene_bvh_builder_base.cpp:26-290
// and scene_bvh_split_candidate.inl:49-151): the same split decisions, the
// same leaves in the same order, serialized depth-first with sibling pairs
// as serialize() does (triangle_bvh_builder_sah.cpp:129-164).
//
// The reference recurses depth-first on a thread pool; the tree it builds
// depends only on each node's reference list, so here all nodes of one
// depth are processed together, level by level.  A level's nodes wait in
// three lists by size, whose lengths stay on the device (the kernels loop
// over them, the host reads them once every few levels):
//
//   wave_nodes   up to 64 references and within the sweep threshold: one
//                wave a node, candidates at every reference's max bound.
//   block_nodes  up to Chunk references: one workgroup a node, references
//                in LDS; sweep candidates, or the grid's (3 centre planes +
//                num_slices planes per axis, object and, above the spatial
//                depth, spatial) from bins.
//   big nodes    more: big_bins bins every Chunk references of the node by
//                one workgroup and merges with integer atomics, big_select
//                decides, big_count and big_move partition chunk by chunk.
//
// Bins: the reference classifies every reference against every candidate;
// here each reference adds its box and count to one bin per axis for its max
// bound and one for its min bound among the axis's sorted planes, and a
// candidate's sides are the merged bins on either side of its plane.  Counts
// and boxes are the same (integer sums; min / max of order-preserving float
// encodings, so the result does not depend on order).  A node's SAH costs
// have the reference's rounding; first minimum, exhausted test and
// leaf/split decision follow it, and the references move in stable order
// (straddling ones clipped to the plane).  Node and list positions come from
// atomic counters (one set per workgroup): the order within a level is free,
// since the tree is laid out depth-first from its parents afterwards.
//
// Finally every leaf adds its slots up the tree (count_subtrees), every node
// finds its depth-first position on the way to the root, and nodes and slots
// are scattered into place (place_nodes).
//
// Departures, all in inputs the reference cannot handle either: a node of
// more than 255 references that cannot be split fails with
// MI_ERR_UNSPLITTABLE (the reference logs and leaves the node
// uninitialized); a grid node whose box has zero extent gets no slice
// candidates (the reference converts NaN to an integer step count).  Bounds
// equal up to the sign of zero may differ in that sign.  A triangle with a
// vertex that is not finite is in the tree with the box of its finite
// coordinates (make_refs): no ray hits it, and NaN or infinite bounds give
// NaN costs, on which nodes split until memory or the levels run out, or drop
// the bounds of the triangles beside it.

#include "bvh_build.hpp"
#include "device_math.hpp"
#include "device_memory.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <utility>

namespace mi {

namespace {

constexpr uint32_t Chunk      = 1024;  // references a workgroup holds at a time
constexpr uint32_t Wave_refs  = 64;    // references of a wave's node
constexpr uint32_t Kind_leaf  = 1;
constexpr uint32_t Kind_split = 4;
constexpr uint32_t Kind_error = 5;

constexpr float Flt_max = 3.40282347e+38f;

// bits of the error word
constexpr uint32_t Err_unsplittable = 1;
constexpr uint32_t Err_index        = 2;
constexpr uint32_t Err_layout       = 8;
constexpr uint32_t Not_finite       = 16;  // no error: an instance's box is not finite
constexpr uint32_t Err_capacity     = 32;  // a list or buffer is full: the host starts over with more
constexpr uint32_t Err_level        = 8;   // from this bit on: the level of an unsplittable node
constexpr uint32_t Err_stop         = Err_unsplittable | Err_index | Err_capacity;

// scene::bvh::Reference: {min.xyz, primitive}{max.xyz, pad}
struct alignas(16) Ref {
    float    lo[3];
    uint32_t prim;
    float    hi[3];
    uint32_t pad;
};
static_assert(sizeof(Ref) == 32);

struct Task {
    uint32_t begin;
    uint32_t count;
    uint32_t node;
    uint32_t depth;
    float    lo[3];
    float    hi[3];
};

struct Decision {
    uint32_t kind;
    uint32_t axis;
    uint32_t spatial;
    uint32_t n0;
    uint32_t n1;
    float    d;
    float    lo0[3];
    float    hi0[3];
    float    lo1[3];
    float    hi1[3];
};

struct Chunk_rec {
    uint32_t task;
    uint32_t begin;
    uint32_t end;
};

// sprout's Node layout (scene_bvh_node.hpp:44-59)
struct Node {
    float    lo[3];
    uint32_t data;
    float    hi[3];
    uint32_t meta;  // axis | num_indices << 8
};
static_assert(sizeof(Node) == 32);

struct Settings {
    uint32_t num_slices;
    uint32_t sweep_threshold;
    uint32_t max_primitives;
    uint32_t spatial_split_threshold;
};

// ---- float helpers with the reference's semantics --------------------------

// SSE minps/maxps: min(a, b) = a < b ? a : b
__device__ __forceinline__ float smin(float a, float b) {
    return a < b ? a : b;
}

__device__ __forceinline__ float smax(float a, float b) {
    return a > b ? a : b;
}

// std::min / std::max
__device__ __forceinline__ float stdmin(float a, float b) {
    return b < a ? b : a;
}

__device__ __forceinline__ float stdmax(float a, float b) {
    return a < b ? b : a;
}

__device__ __forceinline__ uint32_t key(float f) {
    uint32_t const b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ float unkey(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k);
}

// base/math/aabb.inl:39-42 as the reference build contracts it
__device__ __forceinline__ float surface_area(float const lo[3], float const hi[3]) {
    float const d0 = hi[0] - lo[0];
    float const d1 = hi[1] - lo[1];
    float const d2 = hi[2] - lo[2];
    float const s  = __builtin_fmaf(d1, d2, __builtin_fmaf(d0, d1, d0 * d2));
    return s + s;
}

// Split_candidate::evaluate cost (scene_bvh_split_candidate.inl:109-118)
__device__ __forceinline__ float sah_cost(uint32_t n0, uint32_t n1, uint32_t n, float const lo0[3],
                                          float const hi0[3], float const lo1[3],
                                          float const hi1[3], float aabb_surface_area) {
    if (0 == n0 || 0 == n1) {
        return 2.f + float(n);
    }
    float const sa0      = surface_area(lo0, hi0);
    float const sa1      = surface_area(lo1, hi1);
    float const weight_1 = float(n1) * sa1;
    float const weights  = __builtin_fmaf(float(n0), sa0, weight_1);
    float const k        = float(n0 + n1 - n);
    return __builtin_fmaf(k, 0.125f, weights / aabb_surface_area + 2.f);
}

// Component a of a vector, a differing from lane to lane: the three are read
// and one is selected (an array indexed by lane goes to scratch memory, and a
// branch around each read makes three paths of what follows).
__device__ __forceinline__ float pick(float const v[3], uint32_t a) {
    float const x = v[0], y = v[1], z = v[2];
    return 0 == a ? x : 1 == a ? y : z;
}

__device__ __forceinline__ uint32_t index_max_component(float const v[3]) {
    if (v[0] > v[1]) {
        return v[0] > v[2] ? 0 : 2;
    }
    return v[1] > v[2] ? 1 : 2;
}

// Number of grid slices on axis a (scene_bvh_builder_base.cpp:119-129).
__device__ __forceinline__ uint32_t grid_steps(float extent_a, float step, uint32_t num_slices) {
    float const q = extent_a / step;
    // a zero-extent box gives NaN; a count beyond num_slices + 1 cannot come
    // from a finite box (extent_a <= extent of the longest axis)
    if (!(q >= 0.f) || q > float(num_slices + 1)) {
        return 0;
    }
    return uint32_t(ceilf(q));
}

__device__ __forceinline__ bool covers(float const alo[3], float const ahi[3], float const blo[3],
                                       float const bhi[3]) {
    return alo[0] <= blo[0] && alo[1] <= blo[1] && alo[2] <= blo[2] && ahi[0] >= bhi[0] &&
           ahi[1] >= bhi[1] && ahi[2] >= bhi[2];
}

struct Partial {
    uint32_t n0, n1, used;
    float    lo0[3], hi0[3], lo1[3], hi1[3];
};

__device__ __forceinline__ void partial_init(Partial& p) {
    p.n0 = p.n1 = p.used = 0;
    for (int a = 0; a < 3; ++a) {
        p.lo0[a] = Flt_max;
        p.hi0[a] = -Flt_max;
        p.lo1[a] = Flt_max;
        p.hi1[a] = -Flt_max;
    }
}

__device__ __forceinline__ void merge0(Partial& p, Ref const& r) {
    for (int a = 0; a < 3; ++a) {
        p.lo0[a] = smin(p.lo0[a], r.lo[a]);
        p.hi0[a] = smax(p.hi0[a], r.hi[a]);
    }
}

__device__ __forceinline__ void merge1(Partial& p, Ref const& r) {
    for (int a = 0; a < 3; ++a) {
        p.lo1[a] = smin(p.lo1[a], r.lo[a]);
        p.hi1[a] = smax(p.hi1[a], r.hi[a]);
    }
}

// Classification of one reference against a candidate
// (scene_bvh_split_candidate.inl:57-107).
__device__ __forceinline__ void classify(Partial& p, Ref const& r, uint32_t axis, float d,
                                         bool spatial) {
    if (pick(r.hi, axis) < d) {
        ++p.n0;
        merge0(p, r);
    } else if (!spatial || !(pick(r.lo, axis) < d)) {
        ++p.n1;
        merge1(p, r);
    } else {
        ++p.n0;
        ++p.n1;
        merge0(p, r);
        merge1(p, r);
        p.used = 1;
    }
}

// Fills a decision from the winning candidate's counts and boxes
// (scene_bvh_builder_base.cpp:40-88 and the clipping of
// scene_bvh_split_candidate.inl:95-100).
__device__ __forceinline__ void decide(Task const& t, uint32_t axis, float d, bool spatial_cand, Partial const& p,
                       float cost, Decision& out) {
    uint32_t const n = t.count;

    float lo0[3], hi0[3], lo1[3], hi1[3];
    for (int a = 0; a < 3; ++a) {
        lo0[a] = p.lo0[a];
        hi0[a] = p.hi0[a];
        lo1[a] = p.lo1[a];
        hi1[a] = p.hi1[a];
    }
    bool const spatial = spatial_cand && p.used;
    for (int a = 0; a < 3; ++a) {
        if (spatial && int(axis) == a) {
            hi0[a] = stdmin(d, hi0[a]);
            lo1[a] = stdmax(d, lo1[a]);
        }
    }

    bool const exhausted = (covers(lo0, hi0, t.lo, t.hi) && n == p.n0) ||
                           (covers(lo1, hi1, t.lo, t.hi) && n == p.n1);

    uint32_t kind;
    if (n <= 0xFF && (float(n) <= cost || exhausted)) {
        kind = Kind_leaf;
    } else if (exhausted) {
        kind = Kind_error;
    } else if (0 == p.n0 || 0 == p.n1) {
        // a child without references
        kind = n <= 0xFF ? Kind_leaf : Kind_error;
    } else {
        kind = Kind_split;
    }

    out.kind    = kind;
    out.axis    = axis;
    out.spatial = spatial ? 1 : 0;
    out.n0      = p.n0;
    out.n1      = p.n1;
    out.d       = d;
    for (int a = 0; a < 3; ++a) {
        out.lo0[a] = lo0[a];
        out.hi0[a] = hi0[a];
        out.lo1[a] = lo1[a];
        out.hi1[a] = hi1[a];
    }
}

// First minimum of (cost, index) with the reference's scan semantics: a NaN
// cost never wins, except at index 0 where nothing can replace it.
struct Best {
    float    cost;
    uint32_t index;
};

__device__ __forceinline__ bool better(Best a, Best b) {
    // a strictly before b in the reference's sequential scan order
    if (0 == a.index || 0 == b.index) {
        bool const a_nan0 = (0 == a.index) && (a.cost != a.cost);
        bool const b_nan0 = (0 == b.index) && (b.cost != b.cost);
        if (a_nan0) {
            return true;
        }
        if (b_nan0) {
            return false;
        }
    }
    if (a.cost != a.cost) {
        return false;
    }
    if (b.cost != b.cost) {
        return true;
    }
    return a.cost < b.cost || (a.cost == b.cost && a.index < b.index);
}

__device__ Best block_best(Best mine, Best* lds) {
    for (int off = 32; off > 0; off >>= 1) {
        Best o;
        o.cost  = __shfl_xor(mine.cost, off);
        o.index = __shfl_xor(mine.index, off);
        if (better(o, mine)) {
            mine = o;
        }
    }
    uint32_t const wave  = threadIdx.x >> 6;
    uint32_t const waves = blockDim.x >> 6;
    if (0 == (threadIdx.x & 63)) {
        lds[wave] = mine;
    }
    __syncthreads();
    Best b = lds[0];
    for (uint32_t w = 1; w < waves; ++w) {
        if (better(lds[w], b)) {
            b = lds[w];
        }
    }
    __syncthreads();
    return b;
}

__device__ __forceinline__ Best wave_best(Best mine) {
    for (int off = 32; off > 0; off >>= 1) {
        Best o;
        o.cost  = __shfl_xor(mine.cost, off);
        o.index = __shfl_xor(mine.index, off);
        if (better(o, mine)) {
            mine = o;
        }
    }
    return mine;
}

// Counts and boxes of all lanes' partials, in every lane.
__device__ __forceinline__ void wave_merge(Partial& p) {
    for (int off = 32; off > 0; off >>= 1) {
        p.n0 += __shfl_xor(p.n0, off);
        p.n1 += __shfl_xor(p.n1, off);
        p.used |= __shfl_xor(p.used, off);
        for (int a = 0; a < 3; ++a) {
            p.lo0[a] = fminf(p.lo0[a], __shfl_xor(p.lo0[a], off));
            p.hi0[a] = fmaxf(p.hi0[a], __shfl_xor(p.hi0[a], off));
            p.lo1[a] = fminf(p.lo1[a], __shfl_xor(p.lo1[a], off));
            p.hi1[a] = fmaxf(p.hi1[a], __shfl_xor(p.hi1[a], off));
        }
    }
}

// Orders this wave's LDS accesses (writes by some lanes, reads by others).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void side_flags(Ref const& r, Decision const& d, bool& go0, bool& go1) {
    bool const behind_hi = pick(r.hi, d.axis) < d.d;
    go0                  = behind_hi || (d.spatial && pick(r.lo, d.axis) < d.d);
    go1                  = !behind_hi;
}

// Exclusive prefix over the block of per-thread values (blockDim 256).
__device__ uint32_t block_exclusive(uint32_t v, uint32_t* lds) {
    uint32_t const lane = threadIdx.x & 63;
    uint32_t const wave = threadIdx.x >> 6;
    uint32_t       inc  = v;
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t const o = __shfl_up(inc, off);
        if (lane >= uint32_t(off)) {
            inc += o;
        }
    }
    if (63 == lane) {
        lds[wave] = inc;
    }
    __syncthreads();
    uint32_t base = 0;
    for (uint32_t w = 0; w < wave; ++w) {
        base += lds[w];
    }
    __syncthreads();
    return base + inc - v;
}

// ---- build state ------------------------------------------------------------

// Counters: every kind has 256-byte lines of its own (same-line atomics
// serialize), on them one word per level, of which only the next one is hot.
constexpr uint32_t Line       = 64;
constexpr uint32_t Max_levels = Reference_stack_size + 1;  // levels 0 .. 127
constexpr uint32_t Kind_words = 192;
static_assert(Max_levels + 1 <= Kind_words && 0 == Kind_words % Line);

enum Level_counter { Lc_refs, Lc_wave, Lc_block, Lc_big, Lc_chunks, Lc_split, Num_lc };

struct Build {
    Settings   s;
    uint32_t   bins_per_axis;  // planes + 1, at most num_slices + 3
    Ref*       refs[2];        // by the parity of the level
    Task*      wave_tasks[2];
    Task*      block_tasks[2];
    Task*      big_tasks[2];
    uint32_t*  big_chunk[2];   // first chunk of each big task
    Chunk_rec* chunks[2];      // chunks of the big tasks
    uint32_t*  big_bins[2];    // bins of the big tasks
    Decision*  big_decision;
    uint4*     big_place;      // {child 0's destination, child 1's, leaf flags, first chunk}
    uint32_t*  side0;          // per chunk
    uint32_t*  side1;
    Node*      nodes;
    uint32_t*  parent;
    unsigned long long* sums;  // per inner node: {arrived children, inner nodes, slots} below it
    uint32_t*  leaf_refs;
    uint32_t*  counters;       // Num_lc kinds per level 0 .. Max_levels, then nodes, leaf slots, error
    uint32_t   cap_refs, cap_wave, cap_block, cap_big, cap_chunks, cap_nodes;
};

constexpr uint32_t Counter_nodes = Num_lc * Kind_words;  // word offsets
constexpr uint32_t Counter_leafs = Counter_nodes + Line;
constexpr uint32_t Counter_error = Counter_nodes + 2 * Line;
constexpr uint32_t Build_words = Counter_nodes + 3 * Line;

__device__ __forceinline__ uint32_t* counter(Build const& b, uint32_t level, uint32_t which) {
    return b.counters + which * Kind_words + level;
}

__device__ __forceinline__ uint32_t* counter(Build const& b, uint32_t word) {
    return b.counters + word;
}

// Whether an error ends the build here; the workgroup's one answer (another
// workgroup may raise the error meanwhile).  Every thread calls it.
__device__ __forceinline__ bool stopped(Build const& b) {
    __shared__ uint32_t error;
    if (0 == threadIdx.x) {
        error = *counter(b, Counter_error);
    }
    __syncthreads();
    return 0 != (error & Err_stop);
}

// The levels after one with such a node are not built: the level is one.
__device__ __forceinline__ void unsplittable(Build const& b, uint32_t level) {
    atomicOr(counter(b, Counter_error), Err_unsplittable | level << Err_level);
}

__device__ __forceinline__ uint32_t bin_words(Build const& b) {
    return 6 * 7 * b.bins_per_axis;
}

// ---- planes and bins --------------------------------------------------------

constexpr uint32_t Max_planes = 66;  // num_slices + 1 slices (64 slices) and the centre

// The candidate planes of a grid node (scene_bvh_builder_base.cpp:101-140),
// per axis in ascending order: slice k (from 1) is at k - 1, or at k from the
// centre plane on; a NaN centre (of an infinite box) comes first, so that
// "v < plane" is false up to some index and true from it on for every v.
struct Planes {
    float    d[3][Max_planes];
    uint32_t count[3];
    uint32_t centre[3];
    uint32_t steps[3];
};

// Threads 0..2 of the workgroup fill one axis each.
__device__ __forceinline__ void make_planes(Task const& t, Settings const& s, Planes& p) {
    if (threadIdx.x < 3) {
        uint32_t const a = threadIdx.x;
        float          extent[3];
        for (int k = 0; k < 3; ++k) {
            extent[k] = t.hi[k] - t.lo[k];
        }
        uint32_t const la     = index_max_component(extent);
        float const    step   = pick(extent, la) / float(s.num_slices);
        float const    ext    = pick(extent, a);
        float const    lo     = pick(t.lo, a);
        uint32_t const steps  = grid_steps(ext, step, s.num_slices);
        float const    step_a = ext / float(steps);
        float const    mid    = (lo + pick(t.hi, a)) * 0.5f;
        uint32_t       n      = 0;
        uint32_t       centre = 0;
        bool           placed = false;
        for (uint32_t k = 1; k < steps; ++k) {
            float const d = __builtin_fmaf(float(k), step_a, lo);
            if (!placed && !(d < mid)) {
                centre    = n;
                placed    = true;
                p.d[a][n++] = mid;
            }
            p.d[a][n++] = d;
        }
        if (!placed) {
            centre    = n;
            p.d[a][n++] = mid;
        }
        p.count[a]  = n;
        p.centre[a] = centre;
        p.steps[a]  = steps;
    }
}

// Candidates of a grid node in the reference's order: the three centre
// planes (spatial), then per axis and slice the object and, above the
// spatial depth, the spatial split.
__device__ __forceinline__ uint32_t grid_candidates(Planes const& p, uint32_t per_slice) {
    uint32_t n = 3;
    for (int a = 0; a < 3; ++a) {
        n += p.steps[a] > 1 ? (p.steps[a] - 1) * per_slice : 0;
    }
    return n;
}

__device__ __forceinline__ void grid_candidate(Planes const& p, uint32_t per_slice, uint32_t c,
                                               uint32_t& axis, uint32_t& plane, bool& spatial) {
    if (c < 3) {
        axis    = c;
        plane   = p.centre[c];
        spatial = true;
        return;
    }
    c -= 3;
    axis = 0;
    for (int a = 0; a < 2; ++a) {
        uint32_t const n = p.steps[a] > 1 ? (p.steps[a] - 1) * per_slice : 0;
        if (int(axis) == a && c >= n) {
            c -= n;
            ++axis;
        }
    }
    uint32_t const k = c / per_slice;
    plane            = k + (k >= p.centre[axis] ? 1 : 0);
    spatial          = 1 == c % per_slice;
}

// Bins of a node: per axis for the max bound (type 0) and the lesser of the
// min and max bound's bins (type 1): count, box min, box max; a component's
// bins are adjacent, so lanes at different bins use different LDS banks.
__device__ __forceinline__ uint32_t bin_index(uint32_t axis, uint32_t type, uint32_t comp,
                                              uint32_t bin, uint32_t per_axis) {
    return ((axis * 2 + type) * 7 + comp) * per_axis + bin;
}

__device__ __forceinline__ uint32_t empty_bin(uint32_t index, uint32_t per_axis) {
    uint32_t const comp = index / per_axis % 7;
    return 0 == comp ? 0u : (comp < 4 ? key(Flt_max) : key(-Flt_max));
}

// Adds one reference to the bins (LDS).  The bin of v among the planes is the
// number of planes with !(v < plane): a reference is on side 0 of plane k
// (hi < plane) when its bin is at most k.  A NaN bound enters no box.
__device__ __forceinline__ void bin_ref(Planes const& p, Ref const& r, uint32_t* bins,
                                        uint32_t per_axis) {
    for (uint32_t a = 0; a < 3; ++a) {
        uint32_t const m  = p.count[a];
        uint32_t       bh = 0, bl = 0;
        for (uint32_t k = 0; k < m; ++k) {
            float const d = p.d[a][k];
            bh += r.hi[a] < d ? 0u : 1u;
            bl += r.lo[a] < d ? 0u : 1u;
        }
        bl = min(bl, bh);
        for (uint32_t type = 0; type < 2; ++type) {
            uint32_t const bin = type ? bl : bh;
            uint32_t*      at  = bins + bin_index(a, type, 0, bin, per_axis);
            atomicAdd(at, 1u);
            for (uint32_t k = 0; k < 3; ++k) {
                if (r.lo[k] == r.lo[k]) {
                    atomicMin(at + (1 + k) * per_axis, key(r.lo[k]));
                }
                if (r.hi[k] == r.hi[k]) {
                    atomicMax(at + (4 + k) * per_axis, key(r.hi[k]));
                }
            }
        }
    }
}

// Counts and boxes of both sides of a candidate plane (classify's over all
// references): side 0 holds bins 0 .. plane, side 1 (max bounds) the rest.
__device__ __forceinline__ void merge_bins(uint32_t const* bins, uint32_t per_axis, uint32_t axis,
                                           uint32_t plane, uint32_t planes, bool spatial, uint32_t n,
                                           Partial& p) {
    partial_init(p);
    uint32_t lo0[3], hi0[3], lo1[3], hi1[3];
    for (int k = 0; k < 3; ++k) {
        lo0[k] = lo1[k] = key(Flt_max);
        hi0[k] = hi1[k] = key(-Flt_max);
    }
    uint32_t const* s0 = bins + bin_index(axis, spatial ? 1 : 0, 0, 0, per_axis);
    uint32_t const* s1 = bins + bin_index(axis, 0, 0, 0, per_axis);
    for (uint32_t i = 0; i <= plane; ++i) {
        p.n0 += s0[i];
        for (int k = 0; k < 3; ++k) {
            lo0[k] = min(lo0[k], s0[(1 + k) * per_axis + i]);
            hi0[k] = max(hi0[k], s0[(4 + k) * per_axis + i]);
        }
    }
    for (uint32_t i = plane + 1; i <= planes; ++i) {
        p.n1 += s1[i];
        for (int k = 0; k < 3; ++k) {
            lo1[k] = min(lo1[k], s1[(1 + k) * per_axis + i]);
            hi1[k] = max(hi1[k], s1[(4 + k) * per_axis + i]);
        }
    }
    for (int k = 0; k < 3; ++k) {
        p.lo0[k] = unkey(lo0[k]);
        p.hi0[k] = unkey(hi0[k]);
        p.lo1[k] = unkey(lo1[k]);
        p.hi1[k] = unkey(hi1[k]);
    }
    p.used = spatial && p.n0 + p.n1 > n ? 1u : 0u;
}

// SAH cost of a candidate's counts and boxes, the straddling sides clipped
__device__ __forceinline__ float candidate_cost(Partial const& p, uint32_t axis, float d,
                                                bool spatial, uint32_t n, float sa) {
    float hi0[3], lo1[3];
    for (int k = 0; k < 3; ++k) {
        bool const clip = spatial && p.used && int(axis) == k;
        hi0[k]          = clip ? stdmin(d, p.hi0[k]) : p.hi0[k];
        lo1[k]          = clip ? stdmax(d, p.lo1[k]) : p.lo1[k];
    }
    return sah_cost(p.n0, p.n1, n, p.lo0, hi0, lo1, p.hi1, sa);
}

// ---- places of a decided node's children ------------------------------------

enum Need { Need_nodes, Need_leafs, Need_refs, Need_wave, Need_block, Need_big, Need_chunks, Num_needs };

enum List { List_leaf, List_wave, List_block, List_big };

__device__ __forceinline__ List list_of(Settings const& s, uint32_t n) {
    return n <= s.max_primitives                          ? List_leaf
           : n <= min(Wave_refs, s.sweep_threshold) ? List_wave
           : n <= Chunk                                   ? List_block
                                                          : List_big;
}

__device__ __forceinline__ uint32_t chunks_of(uint32_t n) {
    return (n + Chunk - 1) / Chunk;
}

// What a decided task takes from each counter.
__device__ __forceinline__ void needs_of(Settings const& s, Task const& t, Decision const& d,
                                         uint32_t need[Num_needs]) {
    for (int k = 0; k < Num_needs; ++k) {
        need[k] = 0;
    }
    if (Kind_leaf == d.kind) {
        need[Need_leafs] = t.count;
    } else if (Kind_split == d.kind) {
        need[Need_nodes] = 2;
        for (int c = 0; c < 2; ++c) {
            uint32_t const n = c ? d.n1 : d.n0;
            List const     l = list_of(s, n);
            need[List_leaf == l ? Need_leafs : Need_refs] += n;
            need[Need_wave] += List_wave == l;
            need[Need_block] += List_block == l;
            need[Need_big] += List_big == l;
            need[Need_chunks] += List_big == l ? chunks_of(n) : 0;
        }
    }
}

__device__ __forceinline__ uint32_t* need_counter(Build const& b, uint32_t level, uint32_t k) {
    return Need_nodes == k   ? counter(b, Counter_nodes)
           : Need_leafs == k ? counter(b, Counter_leafs)
                             : counter(b, level + 1,
                                       Need_refs == k    ? Lc_refs
                                       : Need_wave == k  ? Lc_wave
                                       : Need_block == k ? Lc_block
                                       : Need_big == k   ? Lc_big
                                                         : Lc_chunks);
}

__device__ __forceinline__ uint32_t need_capacity(Build const& b, uint32_t k) {
    return Need_nodes == k                     ? b.cap_nodes
           : Need_leafs == k || Need_refs == k ? b.cap_refs
           : Need_wave == k                    ? b.cap_wave
           : Need_block == k                   ? b.cap_block
           : Need_big == k                     ? b.cap_big
                                               : b.cap_chunks;
}

// Takes `amount` from counter k; the offset, and in *full whether it is past
// the capacity (the error word then says so and nothing may be written there).
__device__ __forceinline__ uint32_t take(Build const& b, uint32_t level, uint32_t k, uint32_t amount,
                                         bool* full) {
    uint32_t o = 0;
    if (amount) {
        o = atomicAdd(need_counter(b, level, k), amount);
        if (uint64_t(o) + amount > need_capacity(b, k)) {
            *full = true;
            atomicOr(counter(b, Counter_error), Err_capacity);
        }
    }
    return o;
}

// Where the references of a decided task go: {child 0's first place, child
// 1's, flags}: bit c: child c is a leaf (the place is in leaf_refs, else in
// the next level's references); bit 2: the task itself is a leaf.
struct Place {
    uint32_t dst[2];
    uint32_t leaf;
};

// Where the references of a decided task go, from its offsets.
__device__ __forceinline__ Place places(Settings const& s, Task const& t, Decision const& d,
                                        uint32_t const at[Num_needs]) {
    Place p;
    if (Kind_leaf == d.kind) {
        p.dst[0] = p.dst[1] = at[Need_leafs];
        p.leaf              = 4;
        return p;
    }
    uint32_t leafs = at[Need_leafs], refs = at[Need_refs];
    p.leaf         = 0;
    for (uint32_t c = 0; c < 2; ++c) {
        uint32_t const n = c ? d.n1 : d.n0;
        if (List_leaf == list_of(s, n)) {
            p.leaf |= 1u << c;
            p.dst[c] = leafs;
            leafs += n;
        } else {
            p.dst[c] = refs;
            refs += n;
        }
    }
    return p;
}

// Writes the node of a decided task and its children's nodes or tasks (one
// thread).  at: the task's offsets of every need.
__device__ __forceinline__ void emit(Build const& b, uint32_t level, Task const& t, Decision const& d,
                                      uint32_t const at[Num_needs]) {
    Node n;
    for (int a = 0; a < 3; ++a) {
        n.lo[a] = t.lo[a];
        n.hi[a] = t.hi[a];
    }
    if (Kind_leaf == d.kind) {
        n.data          = at[Need_leafs];
        n.meta          = t.count << 8;
        b.nodes[t.node] = n;
        return;
    }
    Place const    p     = places(b.s, t, d, at);
    uint32_t const child = at[Need_nodes];
    n.data               = child;
    n.meta               = d.axis;
    b.nodes[t.node]      = n;
    b.sums[t.node]       = 0;
    *counter(b, level, Lc_split) = 1;
    uint32_t const next  = (level + 1) & 1;
    uint32_t       off[Num_needs];
    for (int k = 0; k < Num_needs; ++k) {
        off[k] = at[k];
    }
    for (uint32_t c = 0; c < 2; ++c) {
        uint32_t const count = c ? d.n1 : d.n0;
        List const     l     = list_of(b.s, count);
        Task           x;
        x.count = count;
        x.node  = child + c;
        x.depth = t.depth + 1;
        for (int a = 0; a < 3; ++a) {
            x.lo[a] = c ? d.lo1[a] : d.lo0[a];
            x.hi[a] = c ? d.hi1[a] : d.hi0[a];
        }
        b.parent[child + c] = t.node;
        if (List_leaf == l) {
            Node m;
            for (int a = 0; a < 3; ++a) {
                m.lo[a] = x.lo[a];
                m.hi[a] = x.hi[a];
            }
            m.data             = p.dst[c];
            m.meta             = count << 8;
            b.nodes[child + c] = m;
            continue;
        }
        x.begin = p.dst[c];
        if (List_wave == l) {
            b.wave_tasks[next][off[Need_wave]++] = x;
        } else if (List_block == l) {
            b.block_tasks[next][off[Need_block]++] = x;
        } else {
            b.big_tasks[next][off[Need_big]] = x;
            b.big_chunk[next][off[Need_big]] = off[Need_chunks];
            ++off[Need_big];
            off[Need_chunks] += chunks_of(count);
        }
    }
}

// Puts a reference on child c's place (clipped already); true when it fits
// the child's segment, which the counts guarantee.
__device__ __forceinline__ void put(Build const& b, uint32_t level, Place const& p, uint32_t c,
                                    uint32_t rank, Ref const& r) {
    uint32_t const at = p.dst[c] + rank;
    if (p.leaf & (1u << c)) {
        b.leaf_refs[at] = r.prim;
    } else {
        b.refs[(level + 1) & 1][at] = r;
    }
}

__device__ __forceinline__ void put_sides(Build const& b, uint32_t level, Place const& p,
                                          Decision const& d, Ref const& r, bool go0, bool go1,
                                          uint32_t rank0, uint32_t rank1) {
    if (go0 && rank0 < d.n0) {
        Ref x = r;
        if (go1) {
            for (int a = 0; a < 3; ++a) {
                x.hi[a] = int(d.axis) == a ? stdmin(d.d, x.hi[a]) : x.hi[a];
            }
        }
        put(b, level, p, 0, rank0, x);
    }
    if (go1 && rank1 < d.n1) {
        Ref y = r;
        if (go0) {
            for (int a = 0; a < 3; ++a) {
                y.lo[a] = int(d.axis) == a ? stdmax(d.d, y.lo[a]) : y.lo[a];
            }
        }
        put(b, level, p, 1, rank1, y);
    }
}

// ---- kernels ----------------------------------------------------------------

__global__ void clear_counters(uint32_t* counters, uint32_t* root_keys) {
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < Build_words) {
        counters[i] = Counter_nodes == i ? 1u : 0u;  // the root is node 0
    }
    if (i < 6) {
        root_keys[i * Line] = key(i < 3 ? Flt_max : -Flt_max);
    }
}

// References of the triangles and the root box, one atomic per workgroup and
// coordinate on lines of their own (one per wave on one line took 380 us of
// 352 k triangles' build).
// A mesh's triangle with a vertex that is not finite has an infinite or NaN
// determinant with every ray, which makes its inverse NaN and the triangle a
// miss: its box is that of its finite coordinates, per axis, or 0.  Boxes of
// instances (boxes set) stand for what is inside and stay as they are.
__global__ void __launch_bounds__(256)
make_refs(float const* __restrict__ positions, uint32_t stride, uint32_t num_vertices,
          uint32_t const* __restrict__ indices, uint32_t num_triangles, uint32_t boxes,
          Ref* __restrict__ refs, uint32_t* __restrict__ root_keys, uint32_t* __restrict__ error) {
    __shared__ float wave_lo[4][3];
    __shared__ float wave_hi[4][3];

    float lo[3] = {Flt_max, Flt_max, Flt_max};
    float hi[3] = {-Flt_max, -Flt_max, -Flt_max};

    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < num_triangles;
         t += gridDim.x * blockDim.x) {
        uint32_t ia = indices[3 * size_t(t) + 0];
        uint32_t ib = indices[3 * size_t(t) + 1];
        uint32_t ic = indices[3 * size_t(t) + 2];
        if (ia >= num_vertices || ib >= num_vertices || ic >= num_vertices) {
            atomicOr(error, Err_index);
            ia = ib = ic = 0;
        }
        float const* pa = positions + size_t(ia) * stride;
        float const* pb = positions + size_t(ib) * stride;
        float const* pc = positions + size_t(ic) * stride;

        Ref  r;
        bool finite = true;
        for (int i = 0; i < 3; ++i) {
            // triangle_bvh_helper.cpp:15-21: min(a, min(b, c))
            r.lo[i] = smin(pa[i], smin(pb[i], pc[i]));
            r.hi[i] = smax(pa[i], smax(pb[i], pc[i]));
            finite  = finite && isfinite(pa[i]) && isfinite(pb[i]) && isfinite(pc[i]);
        }
        if (!finite && boxes) {
            atomicOr(error, Not_finite);
            for (int i = 0; i < 3; ++i) {  // one NaN, which sorts last (wave_sweep)
                r.lo[i] = r.lo[i] != r.lo[i] ? __builtin_nanf("") : r.lo[i];
                r.hi[i] = r.hi[i] != r.hi[i] ? __builtin_nanf("") : r.hi[i];
            }
        } else if (!finite) {
            for (int i = 0; i < 3; ++i) {
                float const v[3] = {pa[i], pb[i], pc[i]};
                r.lo[i]          = Flt_max;
                r.hi[i]          = -Flt_max;
                for (int k = 0; k < 3; ++k) {
                    r.lo[i] = isfinite(v[k]) ? smin(r.lo[i], v[k]) : r.lo[i];
                    r.hi[i] = isfinite(v[k]) ? smax(r.hi[i], v[k]) : r.hi[i];
                }
                if (r.lo[i] > r.hi[i]) {
                    r.lo[i] = r.hi[i] = 0.f;
                }
            }
        }
        for (int i = 0; i < 3; ++i) {
            lo[i] = fminf(lo[i], r.lo[i]);
            hi[i] = fmaxf(hi[i], r.hi[i]);
        }
        r.prim  = t;
        r.pad   = 0;
        refs[t] = r;
    }

    for (int i = 0; i < 3; ++i) {
        for (int off = 32; off > 0; off >>= 1) {
            lo[i] = fminf(lo[i], __shfl_xor(lo[i], off));
            hi[i] = fmaxf(hi[i], __shfl_xor(hi[i], off));
        }
        if (0 == (threadIdx.x & 63)) {
            wave_lo[threadIdx.x >> 6][i] = lo[i];
            wave_hi[threadIdx.x >> 6][i] = hi[i];
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        uint32_t const i = threadIdx.x;
        float          l = wave_lo[0][i];
        float          h = wave_hi[0][i];
        for (int w = 1; w < 4; ++w) {
            l = fminf(l, wave_lo[w][i]);
            h = fmaxf(h, wave_hi[w][i]);
        }
        atomicMin(&root_keys[i * Line], key(l));
        atomicMax(&root_keys[(3 + i) * Line], key(h));
    }
}

// Chunk records and empty bins of a big task; every thread of the workgroup.
__device__ __forceinline__ void start_big(Build const& b, uint32_t parity, uint32_t index,
                                          uint32_t begin, uint32_t count, uint32_t first_chunk) {
    for (uint32_t k = threadIdx.x; k < chunks_of(count); k += blockDim.x) {
        uint32_t const c                   = begin + k * Chunk;
        b.chunks[parity][first_chunk + k] = Chunk_rec{index, c, min(c + Chunk, begin + count)};
    }
    uint32_t const words = bin_words(b);
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) {
        b.big_bins[parity][size_t(index) * words + i] = empty_bin(i, b.bins_per_axis);
    }
}

// The root: a task of its list, or the only leaf.  One workgroup.
__global__ void __launch_bounds__(256)
init_root(Build b, uint32_t const* __restrict__ root_keys, uint32_t num_triangles) {
    Task t;
    t.begin = 0;
    t.count = num_triangles;
    t.node  = 0;
    t.depth = 0;
    for (int i = 0; i < 3; ++i) {
        t.lo[i] = unkey(root_keys[i * Line]);
        t.hi[i] = unkey(root_keys[(3 + i) * Line]);
    }
    List const l = list_of(b.s, num_triangles);
    if (0 == threadIdx.x) {
        b.parent[0]             = dev::Null;
        *counter(b, 0, Lc_refs) = num_triangles;
        if (List_leaf == l) {
            Node n;
            for (int i = 0; i < 3; ++i) {
                n.lo[i] = t.lo[i];
                n.hi[i] = t.hi[i];
            }
            n.data     = 0;
            n.meta     = num_triangles << 8;
            b.nodes[0] = n;
            *counter(b, Counter_leafs) = num_triangles;
        } else if (List_wave == l) {
            b.wave_tasks[0][0]      = t;
            *counter(b, 0, Lc_wave) = 1;
        } else if (List_block == l) {
            b.block_tasks[0][0]      = t;
            *counter(b, 0, Lc_block) = 1;
        } else {
            b.big_tasks[0][0]         = t;
            b.big_chunk[0][0]         = 0;
            *counter(b, 0, Lc_big)    = 1;
            *counter(b, 0, Lc_chunks) = chunks_of(num_triangles);
        }
    }
    if (List_leaf == l) {
        for (uint32_t i = threadIdx.x; i < num_triangles; i += blockDim.x) {
            b.leaf_refs[i] = i;
        }
    } else if (List_big == l) {
        start_big(b, 0, 0, 0, num_triangles, 0);
    }
}

// Sweep candidate c over n references in LDS: the three centre planes, then
// every reference's max bound on each axis (scene_bvh_builder_base.cpp:106-114)
__device__ __forceinline__ void sweep_candidate(Task const& t, Ref const* refs, uint32_t c,
                                                uint32_t& axis, float& d, bool& spatial) {
    if (c < 3) {
        axis    = c;
        d       = (pick(t.lo, c) + pick(t.hi, c)) * 0.5f;
        spatial = true;
    } else {
        uint32_t const r = (c - 3) / 3;
        axis             = (c - 3) % 3;
        d                = pick(refs[r].hi, axis);
        spatial          = false;
    }
}

__device__ __forceinline__ Partial sweep_sides(Ref const* refs, uint32_t n, uint32_t axis, float d,
                                               bool spatial) {
    Partial p;
    partial_init(p);
    for (uint32_t i = 0; i < n; ++i) {
        classify(p, refs[i], axis, d, spatial);
    }
    return p;
}

// The best sweep candidate of a node by one wave, lane i holding reference i.
// Up to Direct_refs references every candidate has a lane that goes through
// them all.  Above that the sides come from sorted order: on each axis the
// references of side 0 of a max-bound candidate are the ones sorted before
// it, so its counts and boxes are a prefix and a suffix of the references in
// that order (min / max, so the same values in any order).  64 references:
// about 2 500 instructions where lane-by-lane folding takes 11 500.
constexpr uint32_t Direct_refs = 20;  // 3 + 3 * 20 candidates fit a wave's lanes

__device__ __forceinline__ Best wave_sweep(Task const& t, Ref const* refs, uint16_t* order) {
    uint32_t const lane = threadIdx.x & 63;
    uint32_t const n    = t.count;
    float const    sa   = surface_area(t.lo, t.hi);
    Best           mine = {__builtin_nanf(""), 0xFFFFFFFFu};
    if (n <= Direct_refs) {
        if (lane < 3 + 3 * n) {
            uint32_t axis;
            float    x;
            bool     spatial;
            sweep_candidate(t, refs, lane, axis, x, spatial);
            Partial const q = sweep_sides(refs, n, axis, x, spatial);
            mine            = {candidate_cost(q, axis, x, spatial, n, sa), lane};
        }
        return wave_best(mine);
    }

    // the centre planes: every lane classifies its reference
    for (uint32_t a = 0; a < 3; ++a) {
        float const x = (t.lo[a] + t.hi[a]) * 0.5f;
        Partial     q;
        partial_init(q);
        if (lane < n) {
            classify(q, refs[lane], a, x, true);
        }
        wave_merge(q);
        if (lane == a) {
            mine = {candidate_cost(q, a, x, true, n, sa), a};
        }
    }

    // each reference's place in the order of its max bound: (bound, index)
    // ascending, -0 as +0, NaN (without a sign, make_refs) last
    uint32_t own[3], rank[3] = {0, 0, 0}, less[3] = {0, 0, 0};
    for (int a = 0; a < 3; ++a) {
        own[a] = lane < n ? key(refs[lane].hi[a] + 0.f) : 0u;
    }
    for (uint32_t j = 0; j < n; ++j) {
        for (int a = 0; a < 3; ++a) {
            uint32_t const k = key(refs[j].hi[a] + 0.f);
            less[a] += k < own[a] ? 1u : 0u;
            rank[a] += k < own[a] || (k == own[a] && j < lane) ? 1u : 0u;
        }
    }
    if (lane < n) {
        for (int a = 0; a < 3; ++a) {
            // the reference at a place, and how many are before its bound
            order[a * Wave_refs + rank[a]] = uint16_t(lane | (less[a] << 8));
        }
    }
    wave_sync();
    for (uint32_t a = 0; a < 3; ++a) {
        uint32_t const o = lane < n ? order[a * Wave_refs + lane] : 0u;
        uint32_t const i = o & 0xFFu;
        Ref            r = refs[i];
        float          lo[3], hi[3], plo[3], phi[3];
        for (int k = 0; k < 3; ++k) {
            lo[k] = plo[k] = lane < n ? r.lo[k] : Flt_max;
            hi[k] = phi[k] = lane < n ? r.hi[k] : -Flt_max;
        }
        // inclusive prefix (plo, phi) and suffix (lo, hi) over the lanes
        for (uint32_t off = 1; off < 64; off <<= 1) {
            for (int k = 0; k < 3; ++k) {
                float const x = __shfl_up(plo[k], off);
                float const y = __shfl_up(phi[k], off);
                float const u = __shfl_down(lo[k], off);
                float const v = __shfl_down(hi[k], off);
                plo[k]        = lane >= off ? fminf(plo[k], x) : plo[k];
                phi[k]        = lane >= off ? fmaxf(phi[k], y) : phi[k];
                lo[k]         = lane + off < 64 ? fminf(lo[k], u) : lo[k];
                hi[k]         = lane + off < 64 ? fmaxf(hi[k], v) : hi[k];
            }
        }
        // candidate: the max bound d of the reference at this place; nothing
        // is below a NaN bound
        float const    d  = pick(r.hi, a);
        uint32_t const n0 = d == d ? o >> 8 : 0u;
        Partial        q;
        partial_init(q);
        q.n0 = n0;
        q.n1 = n - n0;
        for (int k = 0; k < 3; ++k) {
            float const x = __shfl(plo[k], int(n0) - 1);
            float const y = __shfl(phi[k], int(n0) - 1);
            float const u = __shfl(lo[k], int(n0));
            float const v = __shfl(hi[k], int(n0));
            q.lo0[k]      = n0 ? x : Flt_max;
            q.hi0[k]      = n0 ? y : -Flt_max;
            q.lo1[k]      = u;
            q.hi1[k]      = v;
        }
        if (lane < n) {
            Best const c = {candidate_cost(q, a, d, false, n, sa), 3 + 3 * i + a};
            if (better(c, mine)) {
                mine = c;
            }
        }
    }
    return wave_best(mine);
}

// One wave a node; a workgroup of eight waves decides sixteen nodes, two a
// wave, before they take their places with one atomic per counter (an atomic
// per node serializes at 12 ns on each counter), then moves their references.
constexpr uint32_t Node_waves = 8;
constexpr uint32_t Node_round = 2 * Node_waves;

__global__ void __launch_bounds__(Node_waves * 64) __attribute__((amdgpu_waves_per_eu(6)))
wave_nodes(Build b, uint32_t level) {
    __shared__ Ref      lds_refs[Node_round][Wave_refs];
    __shared__ Decision decision_s[Node_round];
    __shared__ uint16_t order_s[Node_waves][3 * Wave_refs];
    __shared__ uint32_t need_s[Node_round][4];
    __shared__ uint32_t base_s[4];
    __shared__ uint32_t full_s;

    if (stopped(b)) {
        return;
    }
    // a wave's node only has leaves and wave nodes below it
    uint32_t const kinds[4] = {Need_nodes, Need_leafs, Need_refs, Need_wave};
    uint32_t const total    = min(*counter(b, level, Lc_wave), b.cap_wave);
    uint32_t const lane     = threadIdx.x & 63;
    uint32_t const wave     = threadIdx.x >> 6;

    for (uint32_t base = blockIdx.x * Node_round; base < total; base += gridDim.x * Node_round) {
        if (0 == threadIdx.x) {
            full_s = 0;
        }
        for (uint32_t i = wave; i < Node_round; i += Node_waves) {
            bool const have = base + i < total;
            uint32_t   need[Num_needs];
            for (int k = 0; k < Num_needs; ++k) {
                need[k] = 0;
            }
            if (have) {
                Task const     t    = b.wave_tasks[level & 1][base + i];
                uint32_t const n    = t.count;
                Ref* const     refs = lds_refs[i];
                if (lane < n) {
                    refs[lane] = b.refs[level & 1][t.begin + lane];
                }
                wave_sync();
                Best const mine = wave_sweep(t, refs, order_s[wave]);
                uint32_t axis;
                float    x;
                bool     spatial;
                sweep_candidate(t, refs, mine.index, axis, x, spatial);
                Partial p;
                partial_init(p);
                if (lane < n) {
                    classify(p, refs[lane], axis, x, spatial);
                }
                wave_merge(p);
                Decision d;
                decide(t, axis, x, spatial, p, mine.cost, d);
                needs_of(b.s, t, d, need);
                if (0 == lane) {
                    decision_s[i] = d;  // a leaf or a split: up to 255 references are never unsplittable
                }
            }
            if (0 == lane) {
                for (int k = 0; k < 4; ++k) {
                    need_s[i][k] = need[kinds[k]];
                }
            }
        }
        __syncthreads();
        if (threadIdx.x < 4) {
            uint32_t sum = 0;
            for (uint32_t w = 0; w < Node_round; ++w) {
                uint32_t const x       = need_s[w][threadIdx.x];
                need_s[w][threadIdx.x] = sum;
                sum += x;
            }
            bool full           = false;
            base_s[threadIdx.x] = take(b, level, kinds[threadIdx.x], sum, &full);
            if (full) {
                full_s = 1;
            }
        }
        __syncthreads();
        for (uint32_t i = wave; i < Node_round; i += Node_waves) {
            if (base + i >= total || full_s) {
                continue;
            }
            Decision const d = decision_s[i];
            Task const     t = b.wave_tasks[level & 1][base + i];
            uint32_t const n = t.count;
            uint32_t       at[Num_needs];
            for (int k = 0; k < Num_needs; ++k) {
                at[k] = 0;
            }
            for (int k = 0; k < 4; ++k) {
                at[kinds[k]] = base_s[k] + need_s[i][k];
            }
            // every lane forms the places; lane 0 writes the nodes and tasks
            Place const p = places(b.s, t, d, at);
            if (0 == lane) {
                emit(b, level, t, d, at);
            }
            Ref const r = lds_refs[i][lane];
            if (Kind_leaf == d.kind) {
                if (lane < n) {
                    b.leaf_refs[p.dst[0] + lane] = r.prim;
                }
            } else {
                bool go0 = false, go1 = false;
                if (lane < n) {
                    side_flags(r, d, go0, go1);
                }
                uint64_t const below = (uint64_t(1) << lane) - 1;
                uint32_t const r0    = uint32_t(__popcll(__ballot(go0) & below));
                uint32_t const r1    = uint32_t(__popcll(__ballot(go1) & below));
                put_sides(b, level, p, d, r, go0, go1, r0, r1);
            }
        }
        __syncthreads();  // the next round reuses the LDS
    }
}

struct Block_lds {
    Planes   planes;
    Best     best[4];
    Partial  sides;
    Best     winner;
    uint32_t at[Num_needs];
    uint32_t full;
    uint32_t scan[8];
};

// Takes the places of one decided task; every thread of the workgroup calls
// it, lanes 0..6 one counter each.  False when something is full.
__device__ __forceinline__ bool take_places(Build const& b, uint32_t level, Task const& t,
                                            Decision const& d, Block_lds& s) {
    if (0 == threadIdx.x) {
        s.full = 0;
    }
    __syncthreads();
    if (threadIdx.x < Num_needs) {
        uint32_t need[Num_needs];
        needs_of(b.s, t, d, need);
        uint32_t mine = 0;
        for (uint32_t k = 0; k < Num_needs; ++k) {
            mine = threadIdx.x == k ? need[k] : mine;
        }
        bool full         = false;
        s.at[threadIdx.x] = take(b, level, threadIdx.x, mine, &full);
        if (full) {
            s.full = 1;
        }
        if (0 == threadIdx.x && Kind_error == d.kind) {
            unsplittable(b, level);
        }
    }
    __syncthreads();
    return 0 == s.full && (Kind_leaf == d.kind || Kind_split == d.kind);
}

// The winning candidate of a workgroup's node in s.winner, its sides in
// s.sides: cost(c, p) fills p and returns the cost of candidate c.
template <typename Cost>
__device__ __forceinline__ void block_winner(uint32_t candidates, Block_lds& s, Cost const& cost) {
    Best    mine = {__builtin_nanf(""), 0xFFFFFFFFu};
    Partial sides;
    partial_init(sides);
    for (uint32_t c = threadIdx.x; c < candidates; c += blockDim.x) {
        Partial    p;
        Best const o = {cost(c, p), c};
        if (better(o, mine)) {
            mine  = o;
            sides = p;
        }
    }
    Best const best = block_best(mine, s.best);
    if (mine.index == best.index) {
        s.sides  = sides;
        s.winner = best;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(256) block_nodes(Build b, uint32_t level) {
    extern __shared__ Ref lds_refs[];  // Chunk references, then the bins
    __shared__ Block_lds  s;
    uint32_t* const       bins = reinterpret_cast<uint32_t*>(lds_refs + Chunk);

    if (stopped(b)) {
        return;
    }
    uint32_t const total = min(*counter(b, level, Lc_block), b.cap_block);
    uint32_t const per   = b.bins_per_axis;
    for (uint32_t ti = blockIdx.x; ti < total; ti += gridDim.x) {
        Task const     t     = b.block_tasks[level & 1][ti];
        uint32_t const n     = t.count;
        bool const     sweep = n <= b.s.sweep_threshold;
        float const    sa    = surface_area(t.lo, t.hi);
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
            lds_refs[i] = b.refs[level & 1][t.begin + i];
        }
        uint32_t axis = 0;
        float    x    = 0.f;
        bool     spatial;
        if (sweep) {
            __syncthreads();
            block_winner(3 + 3 * n, s, [&](uint32_t c, Partial& p) {
                sweep_candidate(t, lds_refs, c, axis, x, spatial);
                p = sweep_sides(lds_refs, n, axis, x, spatial);
                return candidate_cost(p, axis, x, spatial, n, sa);
            });
            sweep_candidate(t, lds_refs, s.winner.index, axis, x, spatial);
        } else {
            uint32_t const per_slice = t.depth < b.s.spatial_split_threshold ? 2 : 1;
            make_planes(t, b.s, s.planes);
            for (uint32_t i = threadIdx.x; i < 42 * per; i += blockDim.x) {
                bins[i] = empty_bin(i, per);
            }
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
                bin_ref(s.planes, lds_refs[i], bins, per);
            }
            __syncthreads();
            uint32_t plane = 0;
            block_winner(grid_candidates(s.planes, per_slice), s, [&](uint32_t c, Partial& p) {
                grid_candidate(s.planes, per_slice, c, axis, plane, spatial);
                merge_bins(bins, per, axis, plane, s.planes.count[axis], spatial, n, p);
                return candidate_cost(p, axis, s.planes.d[axis][plane], spatial, n, sa);
            });
            grid_candidate(s.planes, per_slice, s.winner.index, axis, plane, spatial);
            x = s.planes.d[axis][plane];
        }
        Decision d;
        decide(t, axis, x, spatial, s.sides, s.winner.cost, d);
        if (take_places(b, level, t, d, s)) {
            Place const p = places(b.s, t, d, s.at);
            if (0 == threadIdx.x) {
                emit(b, level, t, d, s.at);
            }
            if (Kind_leaf == d.kind) {
                for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
                    b.leaf_refs[p.dst[0] + i] = lds_refs[i].prim;
                }
            } else {
                constexpr uint32_t Per_thread = Chunk / 256;
                uint32_t const     first      = threadIdx.x * Per_thread;
                bool               g0[Per_thread], g1[Per_thread];
                uint32_t           c0 = 0, c1 = 0;
                for (uint32_t k = 0; k < Per_thread; ++k) {
                    g0[k] = g1[k] = false;
                    if (first + k < n) {
                        side_flags(lds_refs[first + k], d, g0[k], g1[k]);
                    }
                    c0 += g0[k];
                    c1 += g1[k];
                }
                uint32_t r0 = block_exclusive(c0, s.scan);
                uint32_t r1 = block_exclusive(c1, s.scan + 4);
                for (uint32_t k = 0; k < Per_thread; ++k) {
                    if (g0[k] || g1[k]) {
                        put_sides(b, level, p, d, lds_refs[first + k], g0[k], g1[k], r0, r1);
                        r0 += g0[k];
                        r1 += g1[k];
                    }
                }
            }
        }
        __syncthreads();  // the next task reuses the LDS
    }
}

// Bins the chunks of the big tasks and merges them into the tasks' bins.  A
// chunk of a mesh is one patch of it, so its references fall into few bins
// and LDS atomics on one word serialize: the lanes spread over `copies` sets of
// bins, added up at the end (80 us for the root of 352 k triangles with one).
constexpr uint32_t Bin_threads = 512;

__global__ void __launch_bounds__(Bin_threads) big_bins(Build b, uint32_t level, uint32_t copies) {
    extern __shared__ uint32_t bins[];
    __shared__ Planes          planes;

    if (stopped(b)) {
        return;
    }
    uint32_t const total = min(*counter(b, level, Lc_chunks), b.cap_chunks);
    uint32_t const per   = b.bins_per_axis;
    uint32_t const words = bin_words(b);
    for (uint32_t ci = blockIdx.x; ci < total; ci += gridDim.x) {
        Chunk_rec const ch = b.chunks[level & 1][ci];
        make_planes(b.big_tasks[level & 1][ch.task], b.s, planes);
        for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) {
            uint32_t const v = empty_bin(i, per);
            for (uint32_t k = 0; k < copies; ++k) {
                bins[k * words + i] = v;
            }
        }
        __syncthreads();
        for (uint32_t i = ch.begin + threadIdx.x; i < ch.end; i += blockDim.x) {
            bin_ref(planes, b.refs[level & 1][i], bins + threadIdx.x % copies * words, per);
        }
        __syncthreads();
        uint32_t* const out = b.big_bins[level & 1] + size_t(ch.task) * words;
        for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) {
            uint32_t const comp = i / per % 7;
            uint32_t       v    = bins[i];
            for (uint32_t k = 1; k < copies; ++k) {
                uint32_t const x = bins[k * words + i];
                v                = 0 == comp ? v + x : comp < 4 ? min(v, x) : max(v, x);
            }
            if (v != empty_bin(i, per)) {
                if (0 == comp) {
                    atomicAdd(out + i, v);
                } else if (comp < 4) {
                    atomicMin(out + i, v);
                } else {
                    atomicMax(out + i, v);
                }
            }
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) big_select(Build b, uint32_t level) {
    extern __shared__ uint32_t bins[];
    __shared__ Block_lds       s;

    if (stopped(b)) {
        return;
    }
    uint32_t const total = min(*counter(b, level, Lc_big), b.cap_big);
    uint32_t const per   = b.bins_per_axis;
    uint32_t const words = bin_words(b);
    for (uint32_t ti = blockIdx.x; ti < total; ti += gridDim.x) {
        Task const     t         = b.big_tasks[level & 1][ti];
        uint32_t const n         = t.count;
        float const    sa        = surface_area(t.lo, t.hi);
        uint32_t const per_slice = t.depth < b.s.spatial_split_threshold ? 2 : 1;
        make_planes(t, b.s, s.planes);
        for (uint32_t i = threadIdx.x; i < words; i += blockDim.x) {
            bins[i] = b.big_bins[level & 1][size_t(ti) * words + i];
        }
        __syncthreads();
        uint32_t axis = 0, plane = 0;
        bool     spatial;
        block_winner(grid_candidates(s.planes, per_slice), s, [&](uint32_t c, Partial& p) {
            grid_candidate(s.planes, per_slice, c, axis, plane, spatial);
            merge_bins(bins, per, axis, plane, s.planes.count[axis], spatial, n, p);
            return candidate_cost(p, axis, s.planes.d[axis][plane], spatial, n, sa);
        });
        grid_candidate(s.planes, per_slice, s.winner.index, axis, plane, spatial);
        Decision d;
        decide(t, axis, s.planes.d[axis][plane], spatial, s.sides, s.winner.cost, d);
        bool const placed = take_places(b, level, t, d, s);
        if (!placed) {
            d.kind = Kind_error;  // nothing moves
        } else {
            Place const p = places(b.s, t, d, s.at);
            if (0 == threadIdx.x) {
                emit(b, level, t, d, s.at);
                b.big_place[ti] = make_uint4(p.dst[0], p.dst[1], p.leaf, b.big_chunk[level & 1][ti]);
            }
            if (Kind_split == d.kind) {
                uint32_t big = s.at[Need_big], chunk = s.at[Need_chunks];
                for (uint32_t c = 0; c < 2; ++c) {
                    uint32_t const count = c ? d.n1 : d.n0;
                    if (List_big == list_of(b.s, count)) {
                        start_big(b, (level + 1) & 1, big++, p.dst[c], count, chunk);
                        chunk += chunks_of(count);
                    }
                }
            }
        }
        if (0 == threadIdx.x) {
            b.big_decision[ti] = d;
        }
        __syncthreads();
    }
}

// References of every chunk on each side.
__global__ void __launch_bounds__(256) big_count(Build b, uint32_t level) {
    __shared__ uint32_t s0[4];
    __shared__ uint32_t s1[4];

    if (stopped(b)) {
        return;
    }
    uint32_t const total = min(*counter(b, level, Lc_chunks), b.cap_chunks);
    for (uint32_t ci = blockIdx.x; ci < total; ci += gridDim.x) {
        Chunk_rec const ch = b.chunks[level & 1][ci];
        Decision const& d  = b.big_decision[ch.task];
        uint32_t        c0 = 0, c1 = 0;
        if (Kind_split == d.kind) {
            for (uint32_t i = ch.begin + threadIdx.x; i < ch.end; i += blockDim.x) {
                bool go0, go1;
                side_flags(b.refs[level & 1][i], d, go0, go1);
                c0 += go0;
                c1 += go1;
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            c0 += __shfl_xor(c0, off);
            c1 += __shfl_xor(c1, off);
        }
        if (0 == (threadIdx.x & 63)) {
            s0[threadIdx.x >> 6] = c0;
            s1[threadIdx.x >> 6] = c1;
        }
        __syncthreads();
        if (0 == threadIdx.x) {
            b.side0[ci] = (s0[0] + s0[1]) + (s0[2] + s0[3]);
            b.side1[ci] = (s1[0] + s1[1]) + (s1[2] + s1[3]);
        }
        __syncthreads();
    }
}

// Stable partition of the big tasks' references into the two children
// (Split_candidate::distribute, scene_bvh_split_candidate.inl:125-151); a
// chunk starts after what its task's earlier chunks send to each side.
__global__ void __launch_bounds__(256) big_move(Build b, uint32_t level) {
    __shared__ uint32_t scan[8];
    __shared__ uint32_t before[2];

    if (stopped(b)) {
        return;
    }
    uint32_t const total = min(*counter(b, level, Lc_chunks), b.cap_chunks);
    for (uint32_t ci = blockIdx.x; ci < total; ci += gridDim.x) {
        Chunk_rec const ch = b.chunks[level & 1][ci];
        Decision const  d  = b.big_decision[ch.task];
        if (Kind_split != d.kind) {
            continue;  // a big node is never a leaf (255 references at most)
        }
        uint4 const pl = b.big_place[ch.task];
        Place       p;
        p.dst[0] = pl.x;
        p.dst[1] = pl.y;
        p.leaf   = pl.z;
        uint32_t q0 = 0, q1 = 0;
        for (uint32_t k = pl.w + threadIdx.x; k < ci; k += blockDim.x) {
            q0 += b.side0[k];
            q1 += b.side1[k];
        }
        uint32_t const e0 = block_exclusive(q0, scan);
        uint32_t const e1 = block_exclusive(q1, scan + 4);
        if (blockDim.x - 1 == threadIdx.x) {
            before[0] = e0 + q0;
            before[1] = e1 + q1;
        }
        __syncthreads();

        constexpr uint32_t Per_thread = Chunk / 256;
        uint32_t const     first      = ch.begin + threadIdx.x * Per_thread;
        Ref                local[Per_thread];
        bool               g0[Per_thread], g1[Per_thread];
        uint32_t           c0 = 0, c1 = 0;
        for (uint32_t k = 0; k < Per_thread; ++k) {
            g0[k] = g1[k] = false;
            if (first + k < ch.end) {
                local[k] = b.refs[level & 1][first + k];
                side_flags(local[k], d, g0[k], g1[k]);
            }
            c0 += g0[k];
            c1 += g1[k];
        }
        uint32_t r0 = before[0] + block_exclusive(c0, scan);
        uint32_t r1 = before[1] + block_exclusive(c1, scan + 4);
        for (uint32_t k = 0; k < Per_thread; ++k) {
            if (g0[k] || g1[k]) {
                put_sides(b, level, p, d, local[k], g0[k], g1[k], r0, r1);
                r0 += g0[k];
                r1 += g1[k];
            }
        }
        __syncthreads();
    }
}

// ---- depth-first serialization ----------------------------------------------

// sums word: arrived children (2 bits) | inner nodes below (30) | slots below (32)
constexpr uint32_t Sum_inner  = 32;
constexpr uint32_t Sum_arrive = 62;

__device__ __forceinline__ uint32_t sum_inner(unsigned long long v) {
    return uint32_t(v >> Sum_inner) & 0x3FFFFFFFu;
}

// Every leaf adds its slots to its ancestors: the second child to arrive at a
// node carries the node's total on.  The totals travel in the atomics alone.
__global__ void __launch_bounds__(256)
count_subtrees(Node const* __restrict__ nodes, uint32_t num_nodes,
               uint32_t const* __restrict__ parent, unsigned long long* sums) {
    uint32_t const x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= num_nodes) {
        return;
    }
    uint32_t const num = (nodes[x].meta >> 8) & 0xFF;
    if (0 == num) {
        return;
    }
    unsigned long long v = (1ull << Sum_arrive) | num;
    for (uint32_t p = parent[x]; dev::Null != p; p = parent[p]) {
        unsigned long long const old = atomicAdd(&sums[p], v);
        if (0 == (old >> Sum_arrive)) {
            return;
        }
        // both children: one more inner node, arriving once
        v = ((old + v) & ((1ull << Sum_arrive) - 1)) + (1ull << Sum_inner) + (1ull << Sum_arrive);
    }
}

// A node's depth-first index, where an inner node's children go (pair) and a
// sub-tree's first slot (serialize(), triangle_bvh_builder_sah.cpp:129-164),
// from the second children on the way to the root: a second child comes after
// its sibling's sub-tree.
__global__ void __launch_bounds__(256)
place_nodes(Node const* __restrict__ nodes, uint32_t num_nodes, uint32_t const* __restrict__ parent,
            unsigned long long const* __restrict__ sums, uint32_t const* __restrict__ leaf_refs,
            uint32_t num_slots, Node* __restrict__ out_nodes, uint32_t* __restrict__ out_slots,
            uint32_t* __restrict__ error) {
    uint32_t const x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= num_nodes) {
        return;
    }
    Node           n    = nodes[x];
    uint32_t const num  = (n.meta >> 8) & 0xFF;
    uint32_t       pair = 1;  // of x
    uint32_t       slot = 0;
    uint32_t       own  = 0;  // what x itself adds to pair
    uint32_t       side = 0;
    uint32_t       up   = 0;
    for (uint32_t a = x, p = parent[x]; dev::Null != p; a = p, p = parent[p]) {
        uint32_t add    = 2;
        uint32_t second = 0;
        if (a != nodes[p].data) {
            second             = 1;
            uint32_t const sib = (nodes[a - 1].meta >> 8) & 0xFF;
            if (sib) {
                slot += sib;
            } else {
                unsigned long long const v = sums[a - 1];
                add += 2 * (sum_inner(v) + 1);
                slot += uint32_t(v);
            }
        }
        pair += add;
        if (a == x) {
            own  = add;
            side = second;
        }
        ++up;
    }
    uint32_t const dest = up ? pair - own + side : 0;
    if (dest >= num_nodes || (num && (uint64_t(slot) + num > num_slots ||
                                      uint64_t(n.data) + num > num_slots))) {
        atomicOr(error, Err_layout);
        return;
    }
    if (num) {
        for (uint32_t k = 0; k < num; ++k) {
            out_slots[slot + k] = leaf_refs[n.data + k];
        }
        n.data = slot;
    } else {
        n.data = pair;
    }
    out_nodes[dest] = n;
}

// ---- host side --------------------------------------------------------------

uint32_t blocks_for(uint64_t n, uint32_t block) {
    uint64_t const b = (n + block - 1) / block;
    return uint32_t(b > 0 ? b : 1);
}

// A build's workspace (one device allocation) and the page-locked words its
// counters are read into.  The last build's are kept for the next one on
// the same device, up to Keep_bytes, until mi_release or until the device's
// memory is used up (device_malloc): allocating and freeing took about as long
// as a small build.  A build that finds them in use by
// another thread has its own; one that ends early gives its own back, since
// its kernels may still run.
constexpr size_t Keep_bytes = size_t(1) << 30;

struct Kept {
    std::mutex lock;
    int        device = -1;
    char*      base   = nullptr;
    size_t     bytes  = 0;
    uint32_t*  words  = nullptr;
};

Kept kept;

struct Workspace {
    int       device = -1;
    char*     base   = nullptr;
    size_t    bytes  = 0;
    size_t    size   = 0;  // placed so far
    uint32_t* words  = nullptr;
    bool      idle   = false;  // the build's stream has been waited for

    Workspace() {
        if (hipGetDevice(&device) != hipSuccess) {
            device = -1;
        }
        std::lock_guard<std::mutex> guard(kept.lock);
        if (device == kept.device) {
            std::swap(base, kept.base);
            std::swap(bytes, kept.bytes);
            std::swap(words, kept.words);
        }
    }

    ~Workspace() {
        if (idle && bytes <= Keep_bytes) {
            std::lock_guard<std::mutex> guard(kept.lock);
            if (kept.device != device || bytes >= kept.bytes) {
                std::swap(device, kept.device);
                std::swap(base, kept.base);
                std::swap(bytes, kept.bytes);
                std::swap(words, kept.words);
            }
        }
        (void)hipFree(base);
        if (words) {
            (void)hipHostFree(words);
        }
    }

    hipError_t reserve(size_t n) {
        hipError_t e = hipSuccess;
        if (!words) {
            e = hipHostMalloc(&words, Build_words * sizeof(uint32_t));
        }
        if (!e && n > bytes) {
            (void)hipFree(base);
            base  = nullptr;
            bytes = 0;
            e     = device_malloc(&base, n);
            if (!e) {
                bytes = n;
            }
        }
        return e;
    }

    template <typename T>
    void place(T** p, size_t n) {
        *p = reinterpret_cast<T*>(base + size);
        size += (n * sizeof(T) + 255) / 256 * 256;
    }
};

}  // namespace

#define MI_TRY(expr)                                                                  \
    do {                                                                              \
        hipError_t const e_ = (expr);                                                 \
        if (e_ != hipSuccess) {                                                       \
            return fail(MI_ERR_HIP, "bvh build: %s: %s", #expr, hipGetErrorString(e_)); \
        }                                                                             \
    } while (0)

#define MI_LAUNCHED()                                                                   \
    do {                                                                                \
        hipError_t const e_ = hipGetLastError();                                        \
        if (e_ != hipSuccess) {                                                         \
            return fail(MI_ERR_HIP, "bvh build launch: %s", hipGetErrorString(e_));     \
        }                                                                               \
    } while (0)

int32_t build_bvh(float const* positions, uint32_t num_vertices, uint32_t position_stride,
                  uint32_t const* indices, uint32_t num_triangles, mi_bvh_settings const& settings,
                  hipStream_t stream, DeviceBvh& out, bool boxes) {
    if (settings.sweep_threshold > 1024 || settings.num_slices > 64) {
        return fail(MI_ERR_ARGS, "mi_bvh_build: sweep_threshold <= 1024 and num_slices <= 64");
    }

    auto const        start = std::chrono::steady_clock::now();
    hipStream_t const st    = stream;

    Build b;
    std::memset(&b, 0, sizeof(b));
    b.s.num_slices      = settings.num_slices;
    b.s.sweep_threshold = settings.sweep_threshold;
    b.s.max_primitives  = settings.max_primitives;
    // Builder_base::split, scene_bvh_builder_base.cpp:271-276
    b.s.spatial_split_threshold = uint32_t(std::lrint(std::log2(float(num_triangles)) / 2.f));
    // num_slices + 1 steps at most: num_slices slice planes and the centre
    b.bins_per_axis             = settings.num_slices + 3;

    // Straddling references are in both children, so a level can hold more
    // references than triangles (2.6 % more slots on the 1.41 M-triangle
    // benchmark mesh): room for a quarter more, and a fresh start with twice
    // as much if that is not enough.
    uint64_t const n64 = num_triangles;
    Workspace      arena;
    for (uint64_t room = n64 + n64 / 4 + 1024;; room *= 2) {
        if (room > 0xF0000000ull) {
            return fail(MI_ERR_HIP, "mi_bvh_build: more than %llu references on a level",
                        (unsigned long long)(room / 2));
        }
        b.cap_refs       = uint32_t(room);
        b.cap_wave       = uint32_t(room / (b.s.max_primitives + 1) + 1);
        b.cap_block      = uint32_t(room / (std::max(b.s.max_primitives, std::min(Wave_refs, b.s.sweep_threshold)) + 1) + 1);
        b.cap_big        = uint32_t(room / Chunk + 1);
        b.cap_chunks     = uint32_t(room / Chunk + b.cap_big);
        // up to twice the slots with one primitive a leaf; 0.65 a triangle with four
        b.cap_nodes      = uint32_t(std::min<uint64_t>(b.s.max_primitives < 3 ? 2 * room : room, 0xFFFFFFF0u));
        uint32_t const words = 6 * 7 * b.bins_per_axis;

        uint32_t* root_keys = nullptr;
        for (int pass = 0; pass < 2; ++pass) {
            arena.size = 0;
            arena.place(&b.counters, Build_words);
            arena.place(&root_keys, 6 * Line);
            for (int k = 0; k < 2; ++k) {
                arena.place(&b.refs[k], b.cap_refs);
                arena.place(&b.wave_tasks[k], b.cap_wave);
                arena.place(&b.block_tasks[k], b.cap_block);
                arena.place(&b.big_tasks[k], b.cap_big);
                arena.place(&b.big_chunk[k], b.cap_big);
                arena.place(&b.chunks[k], b.cap_chunks);
                arena.place(&b.big_bins[k], size_t(b.cap_big) * words);
            }
            arena.place(&b.big_decision, b.cap_big);
            arena.place(&b.big_place, b.cap_big);
            arena.place(&b.side0, b.cap_chunks);
            arena.place(&b.side1, b.cap_chunks);
            arena.place(&b.nodes, b.cap_nodes);
            arena.place(&b.parent, b.cap_nodes);
            arena.place(&b.sums, b.cap_nodes);
            arena.place(&b.leaf_refs, b.cap_refs);
            if (0 == pass) {
                MI_TRY(arena.reserve(arena.size));
            }
        }
        uint32_t* const error = b.counters + Counter_error;

        hipLaunchKernelGGL(clear_counters, dim3(blocks_for(Build_words, 256)), dim3(256), 0, st,
                           b.counters, root_keys);
        MI_LAUNCHED();
        hipLaunchKernelGGL(make_refs, dim3(std::min(blocks_for(num_triangles, 256), 512u)), dim3(256),
                           0, st, positions, position_stride, num_vertices, indices, num_triangles,
                           boxes ? 1u : 0u, b.refs[0], root_keys, error);
        MI_LAUNCHED();
        hipLaunchKernelGGL(init_root, dim3(1), dim3(256), 0, st, b, root_keys, num_triangles);
        MI_LAUNCHED();

        size_t const bins_lds  = size_t(words) * sizeof(uint32_t);
        size_t const block_lds = Chunk * sizeof(Ref) + bins_lds;
        // sets of bins of a workgroup within 48 KB: fifteen with 16 slices
        uint32_t const copies  = uint32_t(std::clamp<size_t>(48 * 1024 / bins_lds, 1, 16));

        // The host reads the lists' lengths once every few levels; until then
        // it launches for what may be there.  A list's nodes only come from
        // longer nodes' lists and its own, so one that is empty with those
        // stays so.
        constexpr uint32_t Read_every = 3;
        bool               big = num_triangles > Chunk, block = num_triangles > 64 || num_triangles > b.s.sweep_threshold;
        uint32_t           level = 0, err = 0, deepest = 0;
        uint32_t* const host = arena.words;
        auto value = [host](uint32_t l, uint32_t which) { return host[which * Kind_words + l]; };
        bool more = num_triangles > b.s.max_primitives;
        while (more && level < Max_levels) {
            uint32_t const from = level;
            uint32_t const to   = std::min(level + Read_every, Max_levels);
            for (; level < to; ++level) {
                uint32_t const width = level < 20 ? 1u << level : 1u << 20;  // nodes of a level
                if (big) {
                    uint32_t const chunks = std::min(b.cap_chunks, 2048u);
                    hipLaunchKernelGGL(big_bins, dim3(chunks), dim3(Bin_threads), copies * bins_lds, st,
                                       b, level, copies);
                    hipLaunchKernelGGL(big_select, dim3(std::min({b.cap_big, width, 512u})), dim3(256),
                                       bins_lds, st, b, level);
                    hipLaunchKernelGGL(big_count, dim3(chunks), dim3(256), 0, st, b, level);
                    hipLaunchKernelGGL(big_move, dim3(chunks), dim3(256), 0, st, b, level);
                }
                if (block) {
                    hipLaunchKernelGGL(block_nodes, dim3(std::min({b.cap_block, width, 1024u})),
                                       dim3(256), block_lds, st, b, level);
                }
                hipLaunchKernelGGL(wave_nodes,
                                   dim3(std::min(blocks_for(std::min(b.cap_wave, width), Node_round), 768u)),
                                   dim3(Node_waves * 64), 0, st, b, level);
                MI_LAUNCHED();
            }
            MI_TRY(hipMemcpyAsync(host, b.counters, Build_words * sizeof(uint32_t),
                                  hipMemcpyDeviceToHost, st));
            MI_TRY(hipStreamSynchronize(st));
            err = host[Counter_error];
            if (err & Err_stop) {
                break;
            }
            for (uint32_t l = from; l < level; ++l) {
                deepest = value(l, Lc_split) ? l + 1 : deepest;
            }
            big   = 0 != value(level, Lc_big);
            block = big || 0 != value(level, Lc_block);
            more  = block || 0 != value(level, Lc_wave);
        }
        if (err & Err_index) {
            return fail(MI_ERR_ARGS, "mi_bvh_build: vertex index out of range");
        }
        if (err & Err_unsplittable) {
            return fail(MI_ERR_UNSPLITTABLE,
                        "mi_bvh_build: a node of more than 255 references cannot be split "
                        "(level %u)",
                        err >> Err_level);
        }
        if (err & Err_capacity) {
            continue;
        }
        if (deepest > Reference_stack_size) {
            return fail(MI_ERR_STACK, "mi_bvh_build: tree deeper than %u levels",
                        Reference_stack_size);
        }
        if (num_triangles <= b.s.max_primitives) {
            MI_TRY(hipMemcpyAsync(host, b.counters, Build_words * sizeof(uint32_t),
                                  hipMemcpyDeviceToHost, st));
            MI_TRY(hipStreamSynchronize(st));
            if (host[Counter_error] & Err_index) {
                return fail(MI_ERR_ARGS, "mi_bvh_build: vertex index out of range");
            }
        }

        DeviceBvh bvh;
        bvh.num_nodes     = host[Counter_nodes];
        bvh.num_slots     = host[Counter_leafs];
        bvh.num_triangles = num_triangles;
        bvh.max_depth     = deepest;

        hipError_t e = device_malloc(&bvh.nodes_alloc, size_t(bvh.num_nodes + 1) * 32);
        if (e == hipSuccess) {
            e = device_malloc(&bvh.tris, size_t(std::max(1u, bvh.num_slots)) * 48);
        }
        if (e == hipSuccess) {
            e = device_malloc(&bvh.slots, size_t(std::max(1u, bvh.num_slots)) * 4);
        }
        if (e != hipSuccess) {
            bvh.release();
            return fail(MI_ERR_HIP, "bvh build: %s", hipGetErrorString(e));
        }
        bvh.nodes = reinterpret_cast<float4*>(static_cast<char*>(bvh.nodes_alloc) + 32);

        uint32_t const grid = blocks_for(bvh.num_nodes, 256);
        hipLaunchKernelGGL(count_subtrees, dim3(grid), dim3(256), 0, st, b.nodes, bvh.num_nodes,
                           b.parent, b.sums);
        hipLaunchKernelGGL(place_nodes, dim3(grid), dim3(256), 0, st, b.nodes, bvh.num_nodes, b.parent,
                           b.sums, b.leaf_refs, bvh.num_slots, reinterpret_cast<Node*>(bvh.nodes),
                           bvh.slots, error);
        if (hipError_t const le = hipGetLastError(); le != hipSuccess) {
            bvh.release();
            return fail(MI_ERR_HIP, "bvh build launch: %s", hipGetErrorString(le));
        }
        if (int32_t const r = fill_triangles(bvh, positions, position_stride, indices, st); r) {
            bvh.release();
            return r;
        }

        float* const root = reinterpret_cast<float*>(host);  // the counters have been read
        e = hipMemcpyAsync(root, bvh.nodes, 32, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) {
            e = hipMemcpyAsync(host + 8, error, 4, hipMemcpyDeviceToHost, st);
        }
        if (e == hipSuccess) {
            e = hipStreamSynchronize(st);
        }
        if (e != hipSuccess) {
            bvh.release();
            return fail(MI_ERR_HIP, "bvh build: %s", hipGetErrorString(e));
        }
        arena.idle = true;
        err        = host[8];
        if (err & Err_layout) {
            bvh.release();
            return fail(MI_ERR_HIP, "mi_bvh_build: internal error (layout %u)", err);
        }
        bvh.nan_bounds = 0 != (err & Not_finite);
        for (int a = 0; a < 3; ++a) {
            bvh.aabb_min[a] = root[a];
            bvh.aabb_max[a] = root[4 + a];
        }
        bvh.build_ms =
            std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - start).count();

        out = bvh;
        return MI_OK;
    }
}

bool release_build_workspace() {
    std::lock_guard<std::mutex> guard(kept.lock);
    bool const any = nullptr != kept.base;
    (void)hipFree(kept.base);
    if (kept.words) {
        (void)hipHostFree(kept.words);
    }
    kept.device = -1;
    kept.base   = nullptr;
    kept.bytes  = 0;
    kept.words  = nullptr;
    return any;
}

}  // namespace mi
