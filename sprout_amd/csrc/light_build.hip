// Light trees built on the device: sprout's Tree_builder
// (core/scene/light/light_tree_builder.cpp:436-760) for the scene tree over
// a scene's lights and for the Primitive_trees of its emissive parts, so a
// scene whose emitters move rebuilds its trees without a host round trip
// (Scene::compile rebuilds the light tree every frame, scene.cpp:216-267).
//
// The host builder (light_tree.cpp) recurses depth first; this one splits a
// whole level of nodes at a time.  It gives the same tree bit for bit:
//   * the arithmetic is light_build.hpp's, shared with the host builder;
//   * a candidate's sums and cone merges run over the node's lights in the
//     order the host's recursion leaves them, a wave per candidate: the sums
//     one light after the other, the cones only for the lights outside of
//     what is merged so far (the lanes test 64 at once);
//   * the cheapest candidate is the first of equal costs;
//   * the partition ends as libstdc++'s std::partition for bidirectional
//     iterators does: with k lights passing, the i-th failing light from the
//     left among the first k places and the i-th passing one from the right
//     among the others change places, all pairs at once;
//   * nodes are numbered as the recursion numbers them: the children of the
//     inner node with pre-order rank r among inner nodes are 2r + 1, 2r + 2
//     (counts added up by the leaves, ranks summed on the way to the root);
//   * a light's order is its final position (leaves are assigned left to
//     right), a node's variance runs over its final order.
// A scene-tree node whose every candidate leaves one side empty (the
// reference recurses forever there; the host builder falls back to a
// median split) makes the build report it, and the caller builds on the
// host instead.
//
// Several trees ("roots") over disjoint light ranges build in one pass:
// every part's Primitive_tree at once.

#include "light_build.hip.hpp"

#include "light_build.hpp"
#include "device_memory.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace mi {

namespace {

constexpr uint32_t Null = 0xFFFFFFFFu;

// A node of the level-by-level build, in creation order (level by level).
struct Tnode {
    lb::Box  bounds;
    lb::Cone cone;
    float    power;
    uint32_t begin, end;  // light positions (global)
    uint32_t root;
    uint32_t parent;      // temp id, or Null (a root)
    uint32_t left;        // temp id of the first child, or Null (a leaf)
    uint32_t mid;         // first position of the second child
    uint32_t two_sided;
    uint32_t closed;      // a part's leaf of more lights than a leaf takes
    uint32_t sum;         // arrived children (2 bits) | inner nodes below (30)
};

// Levels are started without waiting for their sizes: bounds[l] .. bounds[l +
// 1] are level l's nodes (l starts over when Max_levels are kept).
constexpr uint32_t Max_levels = 64;

// A light where the partitions have moved it, 64 bytes.
struct alignas(16) Rec {
    float    lo[3];
    float    power;
    float    hi[3];
    uint32_t light;  // global
    float    cone[4];
    float    angle, sine;  // lb::Wide's
    uint32_t two;
    uint32_t pad;

    __device__ lb::Wide wide() const {
        lb::Wide w;
        for (int k = 0; k < 4; ++k) {
            w.cone.v[k] = cone[k];
        }
        w.angle = angle;
        w.sine  = sine;
        return w;
    }
};

struct Forest {
    lb::Light_set    set;
    uint32_t const*  first;      // R + 1 light offsets of the roots
    float const*     part_cones; // 4 per root (parts)
    uint32_t         num_roots;
    uint32_t         num_lights;
    uint32_t         part;       // Primitive_trees (else the scene tree)
    Rec*             recs;       // per position
    uint32_t*        owner;      // per position: its deepest node
    lb::Sides*       sides;      // per candidate: candidate k of a node at 3 begin + k
    Tnode*           nodes;
    uint32_t*        counters;   // [0] nodes made, [1] failed, then the bounds
    uint32_t*        swap_left;  // per light: positions a partition exchanges
    uint32_t*        swap_right;

    __device__ uint32_t* bounds() const { return counters + 4; }
    // root r owns nodes [2 first_r - r, + 2 n_r - 1) and cdfs [2 first_r, + 2 n_r)
    __device__ uint32_t node_base(uint32_t r) const { return 2 * first[r] - r; }
};

__device__ uint32_t leaf_size(Forest const& f, uint32_t root) {
    if (!f.part) {
        return 4;
    }
    uint32_t const n = f.first[root + 1] - f.first[root];
    return n / 64 > 4 ? n / 64 : 4;
}

__device__ uint32_t sweep_threshold(Forest const& f) {
    return f.part ? lb::Part_sweep_threshold : lb::Scene_sweep_threshold;
}

// Candidates of a node that is no leaf.  A grid has 48 (denormal
// extents: up to 69) and its node 32 lights or more: never above the 3 a
// light that Forest::sides holds.
__device__ uint32_t num_candidates(Forest const& f, Tnode const& t) {
    uint32_t const len = t.end - t.begin;
    return len < sweep_threshold(f) ? 3 * len : lb::grid_candidates(t.bounds);
}

__device__ void make_candidate(Forest const& f, Tnode const& t, uint32_t k, lb::Candidate& c) {
    c = lb::Candidate();
    if (t.end - t.begin < sweep_threshold(f)) {
        c.axis = int(k % 3);
        c.d    = f.recs[t.begin + k / 3].hi[c.axis];
    } else {
        lb::grid_candidate(t.bounds, k, c);
    }
}

// Every light starts in its own place.
__global__ void make_recs(Forest f) {
    uint32_t const l = blockIdx.x * blockDim.x + threadIdx.x;
    if (0 == l) {
        f.counters[0] = f.num_roots;  // the roots are nodes 0 .. R - 1
        f.counters[1] = 0;
        f.bounds()[0] = 0;
    }
    if (l >= f.num_lights) {
        return;
    }
    uint32_t lo = 0, hi = f.num_roots;  // the root r with first[r] <= l < first[r + 1]
    while (hi - lo > 1) {
        uint32_t const mid = (lo + hi) / 2;
        if (f.first[mid] <= l) {
            lo = mid;
        } else {
            hi = mid;
        }
    }
    f.owner[l] = lo;
    Rec            r;
    lb::Wide const w = lb::wide(f.set.cone(l));
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = f.set.lo[3 * size_t(l) + k];
        r.hi[k] = f.set.hi[3 * size_t(l) + k];
    }
    for (int k = 0; k < 4; ++k) {
        r.cone[k] = w.cone.v[k];
    }
    r.power   = f.set.powers[l];
    r.light   = l;
    r.angle   = w.angle;
    r.sine    = w.sine;
    r.two     = f.set.two(l) ? 1u : 0u;
    r.pad     = 0;
    f.recs[l] = r;
}

__device__ __forceinline__ float lane_value(float v, uint32_t lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

__device__ __forceinline__ lb::Wide lane_value(lb::Wide const& w, uint32_t lane) {
    lb::Wide r;
    for (int k = 0; k < 4; ++k) {
        r.cone.v[k] = lane_value(w.cone.v[k], lane);
    }
    r.angle = lane_value(w.angle, lane);
    r.sine  = lane_value(w.sine, lane);
    return r;
}

// lb::smin (of lo) / lb::smax (of hi) over the lanes; count lanes matter
template <bool Low>
__device__ __forceinline__ float wave_edge(float v, uint32_t count) {
    for (uint32_t off = 1; off < 64 && off < count; off <<= 1) {
        float const o = __shfl_xor(v, int(off));
        v             = Low ? lb::smin(v, o) : lb::smax(v, o);
    }
    return v;
}

// b ? x : y by components (a choice between the structs is one of addresses)
__device__ __forceinline__ lb::Wide pick(bool b, lb::Wide const& x, lb::Wide const& y) {
    lb::Wide r;
    for (int k = 0; k < 4; ++k) {
        float const u = x.cone.v[k], v = y.cone.v[k];
        r.cone.v[k]   = b ? u : v;
    }
    float const xa = x.angle, ya = y.angle, xs = x.sine, ys = y.sine;
    r.angle = b ? xa : ya;
    r.sine  = b ? xs : ys;
    return r;
}

// The fold of positions [begin, end) by one wave: the lights `member` takes,
// onto s0 where `behind` holds, else onto s1, as lb::Sides::add in order.
//   * Powers are added one by one (a lane's value by v_readlane; the other
//     side adds 0, which changes no sum that began at 0).
//   * Boxes: minima are the same in any order, but for the sign of a zero,
//     which is the first zero's; it is looked up when a bound is zero.
//   * Cones: all lanes test their light against their side's cone; the first
//     one in order that may not lie inside is merged, and the test repeated
//     for the lights after it.
// Bound by the chain of the power sums, 16 cycles a light and side, and the
// loads of the records.  The 45 candidates of a root of 4000 lights: 169 us;
// a thread per candidate over lights in LDS took 1.62 ms.
template <bool Cones, class Member, class Behind>
__device__ __forceinline__ void fold_wave(Forest const& f, uint32_t begin, uint32_t end,
                                          Member member, Behind behind, lb::Side& s0,
                                          lb::Side& s1) {
    uint32_t const lane  = threadIdx.x & 63;
    uint32_t const count = min(64u, end - begin);
    for (uint32_t base = begin; base < end; base += 64) {
        bool const     in   = base + lane < end;
        Rec const      r    = f.recs[in ? base + lane : base];
        bool const     take = in && member(r);
        bool const     side = take && behind(r);
        uint64_t const m    = __ballot(take);
        uint64_t const m0   = __ballot(side);
        s0.n += uint32_t(__popcll(m0));
        s1.n += uint32_t(__popcll(m & ~m0));
        uint64_t const t = __ballot(take && r.two);
        s0.two           = s0.two || (t & m0);
        s1.two           = s1.two || (t & ~m0);
        for (int k = 0; k < 3; ++k) {
            s0.box.lo[k] = side ? lb::smin(s0.box.lo[k], r.lo[k]) : s0.box.lo[k];
            s0.box.hi[k] = side ? lb::smax(s0.box.hi[k], r.hi[k]) : s0.box.hi[k];
            s1.box.lo[k] = take && !side ? lb::smin(s1.box.lo[k], r.lo[k]) : s1.box.lo[k];
            s1.box.hi[k] = take && !side ? lb::smax(s1.box.hi[k], r.hi[k]) : s1.box.hi[k];
        }
        float const p0 = side ? r.power : 0.f;
        float const p1 = take && !side ? r.power : 0.f;
        for (uint32_t i = 0, n = min(64u, end - base); i < n; i += 8) {
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                s0.power += lane_value(p0, i + j);
                s1.power += lane_value(p1, i + j);
            }
        }
        if (Cones) {
            lb::Wide const w       = r.wide();
            uint64_t       pending = m;
            while (pending) {
                uint64_t const go = pending & __ballot(!lb::inside(pick(side, s0.cone, s1.cone), w));
                if (!go) {
                    break;
                }
                uint32_t const k = uint32_t(__ffsll(static_cast<unsigned long long>(go))) - 1;
                lb::Wide const o = lane_value(w, k);
                bool const     b = 0 != ((m0 >> k) & 1);
                lb::Wide const c = lb::merge(pick(b, s0.cone, s1.cone), o);
                s0.cone          = pick(b, c, s0.cone);
                s1.cone          = pick(b, s1.cone, c);
                pending &= k < 63 ? ~uint64_t(0) << (k + 1) : uint64_t(0);
            }
        }
    }
    // the first zero in order of bound `at` (0-2 lo, 3-5 hi) of a side
    auto const first_zero = [&](int at, bool of0) -> float {
        for (uint32_t base = begin; base < end; base += 64) {
            bool const     in = base + lane < end;
            Rec const      r  = f.recs[in ? base + lane : base];
            float const    l  = 0 == at ? r.lo[0] : 1 == at ? r.lo[1] : r.lo[2];
            float const    h  = 3 == at ? r.hi[0] : 4 == at ? r.hi[1] : r.hi[2];
            float const    v  = at < 3 ? l : h;
            uint64_t const m  = __ballot(in && member(r) && behind(r) == of0 && 0.f == v);
            if (m) {
                return lane_value(v, uint32_t(__ffsll(static_cast<unsigned long long>(m))) - 1);
            }
        }
        return 0.f;
    };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        s0.box.lo[k] = wave_edge<true>(s0.box.lo[k], count);
        s0.box.hi[k] = wave_edge<false>(s0.box.hi[k], count);
        s1.box.lo[k] = wave_edge<true>(s1.box.lo[k], count);
        s1.box.hi[k] = wave_edge<false>(s1.box.hi[k], count);
        if (0.f == s0.box.lo[k]) s0.box.lo[k] = first_zero(k, true);
        if (0.f == s0.box.hi[k]) s0.box.hi[k] = first_zero(3 + k, true);
        if (0.f == s1.box.lo[k]) s1.box.lo[k] = first_zero(k, false);
        if (0.f == s1.box.hi[k]) s1.box.hi[k] = first_zero(3 + k, false);
    }
}

// The roots' bounds, cones, powers and sidedness (build_light_tree /
// build_part_tree's first loop), a wave each.
__global__ void __launch_bounds__(64) init_roots(Forest f) {
    for (uint32_t r = blockIdx.x; r < f.num_roots; r += gridDim.x) {
        Tnode t;
        t.begin     = f.first[r];
        t.end       = f.first[r + 1];
        t.root      = r;
        t.parent    = Null;
        t.left      = Null;
        t.mid       = 0;
        t.closed    = 0;
        t.two_sided = 0;
        t.sum       = 0;
        lb::Side       s, none;
        auto const     all = [](Rec const&) { return true; };
        if (f.part) {
            fold_wave<false>(f, t.begin, t.end, [](Rec const& x) { return x.power > 0.f; }, all, s, none);
            for (int k = 0; k < 4; ++k) {
                t.cone.v[k] = f.part_cones[4 * size_t(r) + k];
            }
        } else {
            fold_wave<true>(f, t.begin, t.end, all, all, s, none);
            t.cone      = s.cone.cone;
            t.two_sided = s.two ? 1u : 0u;
        }
        t.bounds = s.box;
        t.power  = s.power;
        if (0 == threadIdx.x) {
            f.nodes[r] = t;
        }
    }
}

// Both sides of every candidate of the level's nodes, a wave each: wave
// 3 p + a has candidate 3 (p - begin) + a of the node that owns position p,
// if there is one.  Bound by the chains of a wave (powers, cones); the waves
// of a level are all independent.
constexpr uint32_t Evaluate_waves = 4;

__global__ void __launch_bounds__(Evaluate_waves * 64) evaluate_level(Forest f, uint32_t level) {
    if (0 == blockIdx.x && 0 == threadIdx.x) {
        f.bounds()[level + 1] = f.counters[0];
    }
    uint32_t const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint64_t const all  = 3 * uint64_t(f.num_lights);
    for (uint64_t w = uint64_t(blockIdx.x) * Evaluate_waves + wave; w < all;
         w += uint64_t(gridDim.x) * Evaluate_waves) {
        uint32_t const p = uint32_t(w / 3);
        Tnode const&   t = f.nodes[f.owner[p]];
        uint32_t const b = t.begin, e = t.end;
        if (t.closed || e - b <= leaf_size(f, t.root)) {
            continue;
        }
        uint32_t const k = uint32_t(w - 3 * uint64_t(b));
        if (k >= num_candidates(f, t)) {
            continue;
        }
        lb::Candidate c;
        make_candidate(f, t, k, c);
        int const   axis = c.axis;
        float const d    = c.d;
        lb::Sides   s;
        fold_wave<true>(
            f, b, e, [](Rec const& x) { return 0.f != x.power; },
            [=](Rec const& x) {
                return (0 == axis ? x.hi[0] : 1 == axis ? x.hi[1] : x.hi[2]) < d;
            },
            s.s0, s.s1);
        if (0 == (threadIdx.x & 63)) {
            f.sides[w] = s;
        }
    }
}

// Every node of the level that is no leaf splits by its first cheapest
// candidate into two children; one workgroup a node.  The partition takes
// three passes over the node's records, ranks by ballot: 32 us for 4000
// lights (one thread's walk over the lights, with the winner evaluated once
// more: 3 ms).
constexpr uint32_t Split_threads = 256;

__global__ void __launch_bounds__(Split_threads) split_level(Forest f, uint32_t level) {
    __shared__ float    cost_s[Split_threads / 64];
    __shared__ uint32_t index_s[Split_threads / 64];
    __shared__ uint32_t scan_s[Split_threads / 64];
    __shared__ uint32_t child_s;
    __shared__ alignas(16) unsigned char best_raw[sizeof(lb::Candidate)];
    lb::Candidate& best_s = *reinterpret_cast<lb::Candidate*>(best_raw);

    uint32_t const level_begin = f.bounds()[level];
    uint32_t const level_end   = f.bounds()[level + 1];
    uint32_t const lane        = threadIdx.x & 63;
    uint32_t const wave        = threadIdx.x >> 6;
    uint64_t const below       = (uint64_t(1) << lane) - 1;

    // rank of `flag` among the workgroup's threads, and their number
    auto const block_rank = [&](bool flag, uint32_t& total) -> uint32_t {
        uint64_t const m = __ballot(flag);
        __syncthreads();
        if (0 == lane) {
            scan_s[wave] = uint32_t(__popcll(m));
        }
        __syncthreads();
        uint32_t before = 0;
        total           = 0;
        for (uint32_t w = 0; w < Split_threads / 64; ++w) {
            before += w < wave ? scan_s[w] : 0u;
            total += scan_s[w];
        }
        return before + uint32_t(__popcll(m & below));
    };

    for (uint32_t a = level_begin + blockIdx.x; a < level_end; a += gridDim.x) {
        Tnode const    t   = f.nodes[a];
        uint32_t const len = t.end - t.begin;
        if (len <= leaf_size(f, t.root)) {
            continue;
        }
        uint32_t const n = num_candidates(f, t);
        if (0 == n) {
            // no candidate: a part's node is a leaf, a scene's the host's median split
            if (0 == threadIdx.x) {
                f.nodes[a].closed = 1;
                if (!f.part) {
                    atomicOr(&f.counters[1], 1u);
                }
            }
            continue;
        }
        float const   weight = lb::cone_cost(t.cone.v[3]);
        lb::Candidate mine;
        uint32_t      mine_k = Null;
        for (uint32_t k = threadIdx.x; k < n; k += Split_threads) {
            lb::Candidate   c;
            lb::Sides const s = f.sides[3 * size_t(t.begin) + k];
            make_candidate(f, t, k, c);
            s.finish(len, t.bounds, weight, c);
            // a later candidate replaces an earlier one when strictly
            // cheaper; a NaN cost stands only at candidate 0
            if (Null == mine_k || c.cost < mine.cost || (mine_k && mine.cost != mine.cost)) {
                mine   = c;
                mine_k = k;
            }
        }
        // the first cheapest: candidate 0 unless one is strictly cheaper
        // (which none is than a NaN there)
        bool const nan  = mine.cost != mine.cost;
        bool const none = Null == mine_k || (nan && mine_k);
        float      cost = none ? __builtin_huge_valf() : nan ? -__builtin_huge_valf() : mine.cost;
        uint32_t   idx  = none ? Null : mine_k;
        auto const first_cheapest = [](float& c0, uint32_t& i0, float c1, uint32_t i1) {
            if (c1 < c0 || (c1 == c0 && i1 < i0)) {
                c0 = c1;
                i0 = i1;
            }
        };
        for (int off = 32; off > 0; off >>= 1) {
            float const    c1 = __shfl_xor(cost, off);
            uint32_t const i1 = __shfl_xor(idx, off);
            first_cheapest(cost, idx, c1, i1);
        }
        __syncthreads();
        if (0 == lane) {
            cost_s[wave]  = cost;
            index_s[wave] = idx;
        }
        __syncthreads();
        cost = cost_s[0];
        idx  = index_s[0];
        for (uint32_t w = 1; w < Split_threads / 64; ++w) {
            first_cheapest(cost, idx, cost_s[w], index_s[w]);
        }
        if (mine_k == idx) {
            best_s = mine;
        }
        __syncthreads();
        int const   axis = best_s.axis;
        float const d    = best_s.d;
        if (f.part && best_s.exhausted) {
            // Tree_builder::split of a part: an exhausted node is a leaf
            if (0 == threadIdx.x) {
                f.nodes[a].closed = 1;
            }
            continue;
        }
        auto const behind = [&](uint32_t position) { return f.recs[position].hi[axis] < d; };
        // std::partition over [begin, end) by behind(box max)
        uint32_t passing = 0;
        for (uint32_t base = t.begin; base < t.end; base += Split_threads) {
            uint32_t const p = base + threadIdx.x;
            uint32_t       total;
            block_rank(p < t.end && behind(p), total);
            passing += total;
        }
        uint32_t const split = t.begin + passing;
        if (split == t.begin || split == t.end) {
            // the host builder's median fallback: not built here
            if (0 == threadIdx.x) {
                atomicOr(&f.counters[1], 1u);
            }
            continue;
        }
        uint32_t moves = 0;
        for (uint32_t base = t.begin; base < split; base += Split_threads) {
            uint32_t const p    = base + threadIdx.x;
            bool const     fail = p < split && !behind(p);
            uint32_t       total;
            uint32_t const rank = block_rank(fail, total);
            if (fail) {
                f.swap_left[t.begin + moves + rank] = p;
            }
            moves += total;
        }
        uint32_t found = 0;
        for (uint32_t base = split; base < t.end; base += Split_threads) {
            uint32_t const p    = base + threadIdx.x;
            bool const     pass = p < t.end && behind(p);
            uint32_t       total;
            uint32_t const rank = block_rank(pass, total);
            if (pass && found + rank < moves) {
                f.swap_right[t.begin + (moves - 1 - (found + rank))] = p;
            }
            found += total;
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < moves; i += Split_threads) {
            uint32_t const p = f.swap_left[t.begin + i];
            uint32_t const q = f.swap_right[t.begin + i];
            Rec const      x = f.recs[p];
            f.recs[p]        = f.recs[q];
            f.recs[q]        = x;
        }
        if (0 == threadIdx.x) {
            uint32_t const c = atomicAdd(&f.counters[0], 2u);
            child_s          = c;
            Tnode l = t, r = t;
            l.end = r.begin = split;
            l.bounds = best_s.box0, l.cone = best_s.cone0, l.power = best_s.power0;
            r.bounds = best_s.box1, r.cone = best_s.cone1, r.power = best_s.power1;
            l.parent = r.parent = a;
            l.two_sided = (!f.part && best_s.two0) ? 1u : 0u;
            r.two_sided = (!f.part && best_s.two1) ? 1u : 0u;
            f.nodes[c]     = l;
            f.nodes[c + 1] = r;
            f.nodes[a].left = c;
            f.nodes[a].mid  = split;
        }
        __syncthreads();
        for (uint32_t p = t.begin + threadIdx.x; p < t.end; p += Split_threads) {
            f.owner[p] = p < split ? child_s : child_s + 1;
        }
        __syncthreads();  // the next node reuses the LDS
    }
}

constexpr uint32_t Sum_mask = 0x3FFFFFFFu;

__device__ __forceinline__ uint32_t inner_count(Tnode const& t) {
    return Null == t.left ? 0u : 1u + (t.sum & Sum_mask);
}

// Inner nodes per subtree: every leaf goes up, the second child to arrive at
// a node carries its count on (in the atomics alone).
__global__ void count_inner(Forest f, uint32_t num_temp) {
    uint32_t const i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_temp || Null != f.nodes[i].left) {
        return;
    }
    uint32_t v = 1u << 30;
    for (uint32_t p = f.nodes[i].parent; Null != p; p = f.nodes[p].parent) {
        uint32_t const old = atomicAdd(&f.nodes[p].sum, v);
        if (0 == (old >> 30)) {
            return;
        }
        v = (((old + v) & Sum_mask) + 1u) | (1u << 30);
    }
}

// The serialized nodes (serialize, light_tree_builder.cpp:712-733), one wave
// a node: its pre-order rank among the root's inner nodes, summed on the way
// up, and its variance.  The variance's recurrence takes the lights in order:
// lanes fetch 64 at a time with their 1 / n, and every lane then folds the
// values handed round by v_readlane.  121 us over 4000 lights, the root's
// chain; a thread a node gathering from memory took 0.7 ms.
__global__ void __launch_bounds__(256) write_nodes(Forest f, uint32_t num_temp, mi_light_node* out,
                                                   uint32_t* middles, uint32_t* num_nodes) {
    uint32_t const i = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    if (i >= num_temp) {
        return;
    }
    uint32_t const lane  = threadIdx.x & 63;
    Tnode const    t     = f.nodes[i];
    uint32_t const first = f.first[t.root];
    uint32_t       rank = 0, own = 0;  // own: what i itself adds to its rank
    uint32_t       second = 0;
    for (uint32_t a = i, p = t.parent; Null != p; a = p, p = f.nodes[p].parent) {
        uint32_t const l   = f.nodes[p].left;
        uint32_t const add = a == l ? 1u : 1u + inner_count(f.nodes[l]);
        rank += add;
        if (a == i) {
            own    = add;
            second = a == l ? 0u : 1u;
        }
    }
    uint32_t const id = Null == t.parent ? 0u : 1u + second + 2 * (rank - own);

    // lb::variance over the node's lights
    float    ap = 0.f, aps = 0.f;
    uint32_t seen = 0;
    bool     two  = false;
    for (uint32_t base = t.begin; base < t.end; base += 64) {
        bool const     in  = base + lane < t.end;
        Rec const&     r   = f.recs[in ? base + lane : base];
        float const    p   = in ? r.power : 0.f;
        uint64_t       m   = __ballot(p > 0.f);
        uint32_t const n   = seen + uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1))) + 1;
        float const    inv = 1.f / float(n);
        auto const     add = [&](uint32_t k) {
            float const x = lane_value(p, k);
            float const w = lane_value(inv, k);
            ap += (x - ap) * w;
            aps += (x * x - aps) * w;
        };
        two = two || (in && r.two);
        seen += uint32_t(__popcll(m));
        if (~uint64_t(0) == m) {
#pragma unroll 16
            for (uint32_t k = 0; k < 64; ++k) {
                add(k);
            }
        } else {
            while (m) {
                add(uint32_t(__ffsll(static_cast<unsigned long long>(m))) - 1);
                m &= m - 1;
            }
        }
    }
    // a scene leaf is two-sided if any of its lights is
    bool const any = 0 != __ballot(two);
    two            = Null == t.left && !f.part ? any : 0 != t.two_sided;
    if (lane) {
        return;
    }
    mi_light_node d;
    float const   e[3] = {t.bounds.extent(0), t.bounds.extent(1), t.bounds.extent(2)};
    d.center[0]        = t.bounds.position(0);
    d.center[1]        = t.bounds.position(1);
    d.center[2]        = t.bounds.position(2);
    d.radius           = 0.5f * sqrtf(lb::dot3(e, e));
    for (int k = 0; k < 4; ++k) {
        d.cone[k] = t.cone.v[k];
    }
    d.power    = t.power;
    d.variance = fabsf(aps - ap * ap);
    uint32_t const inner    = Null != t.left ? 1u : 0u;
    uint32_t const children = inner ? 1u + 2u * rank : t.begin - first;
    d.bits       = inner | (two ? 2u : 0u) | (children << 2);
    d.num_lights = t.end - t.begin;
    uint32_t const at = f.node_base(t.root) + id;
    out[at]           = d;
    middles[at]       = inner ? t.mid - first : 0u;
    if (Null == t.parent) {
        num_nodes[t.root] = 2 * inner_count(t) + 1;
    }
}

__global__ void write_lights(Forest f, uint32_t* mapping_out, uint32_t* orders_out) {
    uint32_t const p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= f.num_lights) {
        return;
    }
    uint32_t const first = f.first[f.nodes[f.owner[p]].root];
    uint32_t const l     = f.recs[p].light;
    mapping_out[p]       = l - first;
    orders_out[l]        = p - first;
}

// Leaf distributions of the parts (light_tree_builder.cpp:760-795,
// distribution_1d.cpp:42-82): per part, over its nodes in id order, leaves
// of more than 4 lights get num + 1 cdf values (2 when their power is 0).
__global__ void part_cdfs(Forest f, mi_light_node const* nodes, uint32_t const* num_nodes,
                          uint32_t* cdf_offset, float* cdfs, uint32_t* num_cdfs) {
    uint32_t const r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= f.num_roots) {
        return;
    }
    uint32_t const first = f.first[r];
    uint32_t const base  = 2 * first;
    uint32_t       c     = base;
    for (uint32_t i = f.node_base(r), e = f.node_base(r) + num_nodes[r]; i < e; ++i) {
        mi_light_node const& nd = nodes[i];
        cdf_offset[i]           = Null;
        if ((nd.bits & 1u) || nd.num_lights <= 4) {
            continue;
        }
        uint32_t const b        = first + (nd.bits >> 2);
        uint32_t const num      = nd.num_lights;
        float          integral = 0.f;
        for (uint32_t t = 0; t < num; ++t) {
            integral += f.recs[b + t].power;
        }
        cdf_offset[i] = c - base;
        if (0.f == integral) {
            cdfs[c++] = 1.f;
            cdfs[c++] = 1.f;
            continue;
        }
        float const ii = 1.f / integral;
        float       v  = 0.f;
        cdfs[c++]      = v;
        for (uint32_t t = 1; t < num; ++t) {
            v         = __builtin_fmaf(f.recs[b + t - 1].power, ii, v);
            cdfs[c++] = v;
        }
        cdfs[c++] = 1.f;
    }
    num_cdfs[r] = c - base;
}

uint32_t blocks(uint64_t n, uint32_t b) {
    return uint32_t(std::max<uint64_t>(1, (n + b - 1) / b));
}

}  // namespace

void Light_forest_scratch::release() {
    (void)hipFree(recs);
    (void)hipFree(owner);
    (void)hipFree(sides);
    (void)hipFree(nodes);
    (void)hipFree(counters);
    (void)hipFree(swap_left);
    (void)hipFree(swap_right);
    (void)hipFree(num_nodes);
    (void)hipFree(first);
    if (host) {
        (void)hipHostFree(host);
    }
    *this = Light_forest_scratch();
}

int32_t Light_forest_scratch::reserve(uint32_t lights, uint32_t roots) {
    if (lights <= light_capacity && roots <= root_capacity) {
        return MI_OK;
    }
    uint32_t const nl = std::max(lights, light_capacity);
    uint32_t const nr = std::max(roots, root_capacity);
    release();
    size_t const counter_words = 4 + Max_levels + 2;
    hipError_t   e = device_malloc(&recs, size_t(nl) * sizeof(Rec));
    if (!e) e = device_malloc(&owner, size_t(nl) * sizeof(uint32_t));
    if (!e) e = device_malloc(&sides, 3 * size_t(nl) * sizeof(lb::Sides));
    if (!e) e = device_malloc(&nodes, (2 * size_t(nl) + 1) * sizeof(Tnode));
    if (!e) e = device_malloc(&counters, counter_words * sizeof(uint32_t));
    if (!e) e = device_malloc(&swap_left, size_t(nl) * sizeof(uint32_t));
    if (!e) e = device_malloc(&swap_right, size_t(nl) * sizeof(uint32_t));
    if (!e) e = device_malloc(&num_nodes, size_t(nr + 1) * sizeof(uint32_t));
    if (!e) e = device_malloc(&first, size_t(nr + 1) * sizeof(uint32_t));
    // page-locked: the counters, then the roots' offsets and node counts
    if (!e) e = hipHostMalloc(&host, (counter_words + size_t(nr + 1)) * sizeof(uint32_t));
    if (e) {
        release();
        return MI_ERR_HIP;
    }
    light_capacity = nl;
    root_capacity  = nr;
    return MI_OK;
}

int32_t build_light_forest(Light_forest const& in, Light_forest_scratch& s, Light_forest_out& out,
                           hipStream_t stream) {
    uint32_t const R = in.num_roots;
    uint32_t const N = in.num_lights;
    if (0 == R || 0 == N) {
        return MI_OK;
    }
    if (int32_t const st = s.reserve(N, R); st) {
        return st;
    }
    uint32_t const  counter_words = 4 + Max_levels + 2;
    uint32_t* const counters      = s.host;
    uint32_t* const per_root      = s.host + counter_words;
    std::copy(in.first, in.first + R + 1, per_root);
    hipError_t e = hipMemcpyAsync(s.first, per_root, (R + 1) * sizeof(uint32_t), hipMemcpyHostToDevice, stream);
    if (e) {
        return MI_ERR_HIP;
    }

    Forest f;
    f.set        = in.set;
    f.first      = s.first;
    f.part_cones = in.part_cones;
    f.num_roots  = R;
    f.num_lights = N;
    f.part       = in.part ? 1u : 0u;
    f.recs       = static_cast<Rec*>(s.recs);
    f.owner      = s.owner;
    f.sides      = static_cast<lb::Sides*>(s.sides);
    f.nodes      = static_cast<Tnode*>(s.nodes);
    f.counters   = s.counters;
    f.swap_left  = s.swap_left;
    f.swap_right = s.swap_right;

    hipLaunchKernelGGL(make_recs, dim3(blocks(N, 256)), dim3(256), 0, stream, f);
    hipLaunchKernelGGL(init_roots, dim3(std::min(R, 1u << 20)), dim3(64), 0, stream, f);
    uint32_t largest = 0;
    for (uint32_t r = 0; r < R; ++r) {
        largest = std::max(largest, in.first[r + 1] - in.first[r]);
    }
    uint32_t const evaluate_blocks =
        uint32_t(std::min<uint64_t>(blocks(3 * uint64_t(N), Evaluate_waves), 1u << 20));
    // Levels until one makes no nodes; the host looks once every few levels.
    // A root of at most four lights is a leaf.
    constexpr uint32_t Read_every = 4;
    uint32_t           num_temp   = R;
    uint64_t           widest     = R;  // nodes of the level, at most
    for (uint32_t level = 0; largest > 4;) {
        for (uint32_t k = 0; k < Read_every; ++k, ++level) {
            hipLaunchKernelGGL(evaluate_level, dim3(evaluate_blocks), dim3(Evaluate_waves * 64), 0,
                               stream, f, level);
            hipLaunchKernelGGL(split_level, dim3(uint32_t(std::min<uint64_t>(widest, 4096))),
                               dim3(Split_threads), 0, stream, f, level);
            // a node that splits holds five lights or more
            widest = std::max<uint64_t>(std::min<uint64_t>(2 * widest, 2 * (N / 5)), 1);
        }
        e = hipMemcpyAsync(counters, s.counters, (4 + level + 1) * sizeof(uint32_t), hipMemcpyDeviceToHost,
                           stream);
        if (!e) e = hipStreamSynchronize(stream);
        if (e) {
            return MI_ERR_HIP;
        }
        if (counters[1]) {
            return MI_ERR_UNSPLITTABLE;
        }
        num_temp = counters[0];
        widest   = num_temp - counters[4 + level];
        if (0 == widest) {
            break;  // no nodes on the level to come
        }
        if (level + Read_every > Max_levels) {
            e = hipMemcpyAsync(s.counters + 4, s.counters + 4 + level, sizeof(uint32_t),
                               hipMemcpyDeviceToDevice, stream);
            if (e) {
                return MI_ERR_HIP;
            }
            level = 0;
        }
    }
    hipLaunchKernelGGL(count_inner, dim3(blocks(num_temp, 256)), dim3(256), 0, stream, f, num_temp);
    hipLaunchKernelGGL(write_nodes, dim3(blocks(num_temp, 4)), dim3(256), 0, stream, f, num_temp, out.nodes,
                       out.middles, s.num_nodes);
    hipLaunchKernelGGL(write_lights, dim3(blocks(N, 256)), dim3(256), 0, stream, f, out.mapping, out.orders);
    if (in.part && out.cdf_offset) {
        hipLaunchKernelGGL(part_cdfs, dim3(blocks(R, 64)), dim3(64), 0, stream, f, out.nodes, s.num_nodes,
                           out.cdf_offset, out.cdfs, out.num_cdfs);
    }
    e = hipGetLastError();
    if (!e) e = hipMemcpyAsync(per_root, s.num_nodes, R * sizeof(uint32_t), hipMemcpyDeviceToHost, stream);
    if (!e) e = hipStreamSynchronize(stream);
    if (!e && out.num_nodes_host) {
        std::copy(per_root, per_root + R, out.num_nodes_host);
    }
    return e ? MI_ERR_HIP : MI_OK;
}

}  // namespace mi
