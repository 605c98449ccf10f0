// The arithmetic of sprout's light-tree builder (Tree_builder,
// core/scene/light/light_tree_builder.cpp:18-760), shared by the host
// builder (light_tree.cpp) and the device builder (light_build.hip) so that
// both produce the same tree bit for bit:
//
//   cone_cost                  light_tree_builder.cpp:74-83
//   variance                   light_tree_builder.cpp:85-101
//   Split_candidate::evaluate  light_tree_builder.cpp:149-234 (scene variant)
//   cone::merge                base/math/cone.inl:17-60
//   set_rotation, transform    base/math/matrix3x3.inl:49-53, 106-132
//
// min / max keep std::min / std::max's comparisons.  The trigonometry is
// evaluated in double and rounded to float: the host's libm and the device's
// give the same float there (their double results lie within an ulp of the
// exact value, so they round alike except when that value sits within an
// ulp of a float rounding boundary), where their float functions differ in
// one result out of ten.  Against sprout's float std::acos / cos / sin the
// values move by at most an ulp.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

namespace mi::lb {

inline constexpr float    Pi                    = 3.14159265358979323846f;
inline constexpr uint32_t Scene_sweep_threshold = 128;
inline constexpr uint32_t Part_sweep_threshold  = 32;
inline constexpr uint32_t Num_slices            = 16;

__host__ __device__ inline float acos_r(float x) {
    return float(::acos(double(x)));
}
__host__ __device__ inline float cos_r(float x) {
    return float(::cos(double(x)));
}
__host__ __device__ inline float sin_r(float x) {
    return float(::sin(double(x)));
}

// std::min / std::max
__host__ __device__ inline float smin(float a, float b) {
    return (b < a) ? b : a;
}
__host__ __device__ inline float smax(float a, float b) {
    return (a < b) ? b : a;
}

__host__ __device__ inline float dot3(float const* a, float const* b) {
    return (a[0] * b[0] + a[1] * b[1]) + a[2] * b[2];
}

struct Box {
    float lo[3] = {3.40282347e+38f, 3.40282347e+38f, 3.40282347e+38f};
    float hi[3] = {-3.40282347e+38f, -3.40282347e+38f, -3.40282347e+38f};

    __host__ __device__ void merge(float const* blo, float const* bhi) {
        for (int k = 0; k < 3; ++k) {
            lo[k] = smin(lo[k], blo[k]);
            hi[k] = smax(hi[k], bhi[k]);
        }
    }
    __host__ __device__ void merge(Box const& b) { merge(b.lo, b.hi); }
    __host__ __device__ float extent(int k) const { return hi[k] - lo[k]; }
    __host__ __device__ float position(int k) const { return 0.5f * (lo[k] + hi[k]); }
    __host__ __device__ float surface_area() const {
        float const d0 = extent(0), d1 = extent(1), d2 = extent(2);
        return 2.f * (d0 * d1 + d0 * d2 + d1 * d2);
    }
};

struct Cone {
    float v[4] = {1.f, 1.f, 1.f, 1.f};  // float4(1) is the empty cone
};

__host__ __device__ inline bool same_bits(Cone const& a, Cone const& b) {
    for (int k = 0; k < 4; ++k) {
        uint32_t x, y;
        __builtin_memcpy(&x, &a.v[k], 4);
        __builtin_memcpy(&y, &b.v[k], 4);
        if (x != y) {
            return false;
        }
    }
    return true;
}

__host__ __device__ inline bool empty(Cone const& a) {
    return 1.f == a.v[0] && 1.f == a.v[1] && 1.f == a.v[2] && 1.f == a.v[3];
}

// A cone with the angle of its cosine (acos_r) and a sine of that angle.
struct Wide {
    Cone  cone;
    float angle = 0.f;
    float sine  = 0.f;
};

__host__ __device__ inline Wide wide(Cone const& c) {
    return {c, acos_r(c.v[3]), sqrtf((1.f - c.v[3]) * (1.f + c.v[3]))};
}

// Whether cone b lies inside cone a for certain, so that merge gives a; told
// from the cosines alone.  The axes' angle d fits d + b <= a where cos d >=
// cos(a - b); as cosine is no steeper than 1, a cosine larger by Margin means
// an angle smaller by at least Margin, more than the rounding of the float
// angles and of this expression (under 2e-6 together).  With b = 0 (a flat
// light's cone) or d = 0 the float angles order as their cosines do, without
// a margin.  Cones nearer the edge, and NaNs, are left to the angles.
__host__ __device__ inline bool inside(Wide const& a, Wide const& b) {
    constexpr float Margin = 1e-5f;
    float const     ca = a.cone.v[3], cb = b.cone.v[3];
    float const     edge = 0.f == b.angle ? ca : ca * cb + a.sine * b.sine + Margin;
    float const     x    = dot3(a.cone.v, b.cone.v);
    return !empty(a.cone) && ((b.angle <= a.angle && smin(x, 1.f) >= smin(edge, 1.f)) ||
                              same_bits(a.cone, b.cone));
}

// cone::merge, base/math/cone.inl:17-60, of cones whose angles are known
__host__ __device__ inline Wide merge(Wide wa, Wide const& wb) {
    if (empty(wa.cone)) {
        return wb;
    }
    if (inside(wa, wb)) {
        return wa;
    }
    Cone  a = wa.cone, b = wb.cone;
    float a_angle = wa.angle;
    float b_angle = wb.angle;
    if (b_angle > a_angle) {
        a       = wb.cone;
        b       = wa.cone;
        a_angle = wb.angle;
        b_angle = wa.angle;
        wa      = wb;
    }
    float const d_angle = acos_r(smin(smax(dot3(a.v, b.v), -1.f), 1.f));
    if (smin(d_angle + b_angle, Pi) <= a_angle) {
        return wa;
    }
    float const o_angle = (a_angle + d_angle + b_angle) / 2.f;
    // (the reference computes, and drops, a full-sphere cone when o_angle >= pi)
    float const r_angle = o_angle - a_angle;

    float c[3] = {a.v[1] * b.v[2] - a.v[2] * b.v[1], a.v[2] * b.v[0] - a.v[0] * b.v[2],
                  a.v[0] * b.v[1] - a.v[1] * b.v[0]};
    float const cc = dot3(c, c);
    if (!(cc > 0.f)) {
        // opposite axes: the reference normalizes a zero vector here and gets
        // a NaN cone; the cone that bounds both is the whole sphere
        a.v[3] = -1.f;
        return wide(a);
    }
    float const cl = 1.f / sqrtf(cc);
    for (float& x : c) {
        x *= cl;
    }
    // set_rotation(rot, c, r_angle)
    float const cs = cos_r(r_angle);
    float const sn = sin_r(r_angle);
    float const t  = 1.f - cs;
    float       m[3][3];
    m[0][0]    = cs + c[0] * c[0] * t;
    m[1][1]    = cs + c[1] * c[1] * t;
    m[2][2]    = cs + c[2] * c[2] * t;
    float tmp1 = c[0] * c[1] * t;
    float tmp2 = c[2] * sn;
    m[1][0]    = tmp1 + tmp2;
    m[0][1]    = tmp1 - tmp2;
    tmp1       = c[0] * c[2] * t;
    tmp2       = c[1] * sn;
    m[2][0]    = tmp1 - tmp2;
    m[0][2]    = tmp1 + tmp2;
    tmp1       = c[1] * c[2] * t;
    tmp2       = c[0] * sn;
    m[2][1]    = tmp1 + tmp2;
    m[1][2]    = tmp1 - tmp2;
    // transform_vector(rot, a.xyz): row vector times matrix
    float ax[3];
    for (int j = 0; j < 3; ++j) {
        ax[j] = a.v[0] * m[0][j] + a.v[1] * m[1][j] + a.v[2] * m[2][j];
    }
    float const al = 1.f / sqrtf(dot3(ax, ax));
    Cone        r;
    r.v[0] = ax[0] * al;
    r.v[1] = ax[1] * al;
    r.v[2] = ax[2] * al;
    r.v[3] = cos_r(o_angle);
    return wide(r);
}

__host__ __device__ inline Cone merge(Cone const& a, Cone const& b) {
    if (empty(a)) {
        return b;
    }
    return merge(wide(a), wide(b)).cone;
}

__host__ __device__ inline float cone_cost(float cos) {
    float const o   = acos_r(cos);
    float const w   = smin(o + (Pi / 2.f), Pi);
    float const sin = sin_r(o);
    float const b   = (Pi / 2.f) * (2.f * w * sin - cos_r(o - 2.f * w) - 2.f * o * sin + cos);
    return (2.f * Pi) * (1.f - cos) + b;
}

// The lights as the builder reads them: box, cone, power, two-sidedness.
struct Light_set {
    float const*   lo;         // 3 per light
    float const*   hi;         // 3 per light
    float const*   cones;      // 4 per light
    float const*   powers;
    uint8_t const* two_sided;  // or null (one-sided)

    __host__ __device__ Cone cone(uint32_t l) const {
        Cone c;
        for (int k = 0; k < 4; ++k) {
            c.v[k] = cones[4 * size_t(l) + k];
        }
        return c;
    }
    __host__ __device__ bool two(uint32_t l) const { return two_sided && 0 != two_sided[l]; }
};

// variance over mapping[begin, end) of the lights with power
__host__ __device__ inline float variance(uint32_t const* mapping, uint32_t begin, uint32_t end,
                                          Light_set const& set) {
    float ap  = 0.f;
    float aps = 0.f;
    for (uint32_t i = begin, n = 0; i < end; ++i) {
        float const p = set.powers[mapping[i]];
        if (p > 0.f) {
            float const in = 1.f / float(++n);
            ap += (p - ap) * in;
            aps += (p * p - aps) * in;
        }
    }
    return fabsf(aps - ap * ap);
}

// A split plane and what it makes of a node's lights.
struct Candidate {
    Box   box0, box1;
    Cone  cone0, cone1;
    float power0 = 0.f, power1 = 0.f;
    float d      = 0.f;
    float cost   = 0.f;
    int   axis   = 0;
    bool  two0 = false, two1 = false;
    bool  exhausted = false;

    __host__ __device__ bool behind(float const* hi) const { return hi[axis] < d; }

    // Split_candidate::evaluate over mapping[begin, end) of a node with
    // the given bounds and cone weight
    __host__ __device__ void evaluate(uint32_t begin, uint32_t end, uint32_t const* mapping,
                                      Box const& bounds, float cone_weight, Light_set const& set);
};

// One side of a split: its lights added in order, one by one.
struct Side {
    uint32_t n = 0;
    Box      box;
    Wide     cone;
    float    power = 0.f;
    bool     two   = false;
};

// Both sides of a split: Split_candidate::evaluate's fold over a node's lights
// and the cost it comes to.
struct Sides {
    Side s0, s1;

    __host__ __device__ static void add(Side& s, float light_power, float const* lo,
                                        float const* hi, Wide const& light_cone, bool light_two) {
        if (0.f == light_power) {
            return;
        }
        ++s.n;
        s.box.merge(lo, hi);
        s.cone = merge(s.cone, light_cone);
        s.two  = s.two || light_two;
        s.power += light_power;
    }

    // the candidate's sides and cost, for a node of len lights
    __host__ __device__ void finish(uint32_t len, Box const& bounds, float cone_weight,
                                    Candidate& c) const {
        float const e0  = bounds.extent(0), e1 = bounds.extent(1), e2 = bounds.extent(2);
        float const reg = smax(smax(e0, e1), e2) / bounds.extent(c.axis);
        float const sa  = bounds.surface_area();
        c.box0 = s0.box, c.cone0 = s0.cone.cone, c.power0 = s0.power, c.two0 = s0.two;
        c.box1 = s1.box, c.cone1 = s1.cone.cone, c.power1 = s1.power, c.two1 = s1.two;
        if (0 == s0.n || 0 == s1.n) {
            c.cost      = 2.f * reg * (s0.power + s1.power) * (4.f * Pi) * sa * float(len);
            c.exhausted = true;
        } else {
            float const wa = cone_cost(s0.cone.cone.v[3]) * (s0.two ? 2.f : 1.f);
            float const wb = cone_cost(s1.cone.cone.v[3]) * (s1.two ? 2.f : 1.f);
            c.cost         = reg * (((s0.power * wa * s0.box.surface_area()) +
                             (s1.power * wb * s1.box.surface_area())) /
                            (sa * cone_weight));
            c.exhausted = false;
        }
    }
};

__host__ __device__ inline void Candidate::evaluate(uint32_t begin, uint32_t end,
                                                    uint32_t const* mapping, Box const& bounds,
                                                    float cone_weight, Light_set const& set) {
    Sides s;
    for (uint32_t i = begin; i < end; ++i) {
        uint32_t const l  = mapping[i];
        float const*   hi = set.hi + 3 * size_t(l);
        Sides::add(behind(hi) ? s.s0 : s.s1, set.powers[l], set.lo + 3 * size_t(l), hi,
                   wide(set.cone(l)), set.two(l));
    }
    s.finish(end - begin, bounds, cone_weight, *this);
}

// The number of split candidates of a node of len lights (sweep below the
// threshold: three per light; else the 16-slice grid of
// evaluate_splits, light_tree_builder.cpp:346-420).
// A node whose lights all sit at one point has no grid step: no candidates.
__host__ __device__ inline uint32_t grid_steps(Box const& bounds, int a) {
    float const e0 = bounds.extent(0), e1 = bounds.extent(1), e2 = bounds.extent(2);
    int const   la = e0 >= e1 ? (e0 >= e2 ? 0 : 2) : (e1 >= e2 ? 1 : 2);
    float const step = bounds.extent(la) / float(Num_slices);
    if (!(step > 0.f)) {
        return 0;
    }
    return uint32_t(ceilf(bounds.extent(a) / step));
}

__host__ __device__ inline uint32_t grid_candidates(Box const& bounds) {
    uint32_t n = 0;
    for (int a = 0; a < 3; ++a) {
        uint32_t const s = grid_steps(bounds, a);
        n += s > 0 ? s - 1 : 0;
    }
    return n;
}

// Candidate k of the grid (k counts the slices of axis 0, then 1, then 2).
__host__ __device__ inline void grid_candidate(Box const& bounds, uint32_t k, Candidate& c) {
    for (int a = 0; a < 3; ++a) {
        uint32_t const num_steps = grid_steps(bounds, a);
        uint32_t const n         = num_steps > 0 ? num_steps - 1 : 0;
        if (k < n) {
            float const step_a = bounds.extent(a) / float(num_steps);
            c.d                = bounds.lo[a] + float(k + 1) * step_a;
            c.axis             = a;
            return;
        }
        k -= n;
    }
}

// Candidate k of a node's sweep: light mapping[begin + k / 3]'s box max on axis k % 3.
__host__ __device__ inline void sweep_candidate(uint32_t const* mapping, uint32_t begin,
                                                uint32_t k, Light_set const& set, Candidate& c) {
    uint32_t const l = mapping[begin + k / 3];
    c.axis           = int(k % 3);
    c.d              = set.hi[3 * size_t(l) + c.axis];
}

// One emissive triangle as a light (a, b, c its vertices): its box, centre,
// half diagonal, unit normal and area.  False for a triangle of no area.
struct Tri_light {
    float lo[3], hi[3], center[3], n[3];
    float radius, area;
};

__host__ __device__ inline bool triangle_light(float const* a, float const* b, float const* c,
                                               Tri_light& t) {
    float const e1[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    float const e2[3] = {c[0] - a[0], c[1] - a[1], c[2] - a[2]};
    float       n[3]  = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2],
                         e1[0] * e2[1] - e1[1] * e2[0]};
    float const len   = sqrtf((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2]);
    t.area            = 0.5f * len;
    if (!(t.area > 0.f)) {
        return false;
    }
    for (int k = 0; k < 3; ++k) {
        t.n[k]      = n[k] / len;
        t.lo[k]     = smin(smin(a[k], b[k]), c[k]);
        t.hi[k]     = smax(smax(a[k], b[k]), c[k]);
        t.center[k] = 0.5f * (t.lo[k] + t.hi[k]);
    }
    float const ext[3] = {t.hi[0] - t.lo[0], t.hi[1] - t.lo[1], t.hi[2] - t.lo[2]};
    t.radius           = 0.5f * sqrtf((ext[0] * ext[0] + ext[1] * ext[1]) + ext[2] * ext[2]);
    return true;
}

// Part::init (triangle_mesh.cpp:177-239) over a part's triangles in order:
// the box, the power-weighted dominant axis, the widest angle from it
// (its cosine closes the cone) and the total power (area).
struct Part_light {
    float lo[3], hi[3];
    float cone[4];
    float total;
};

template <class Tri>  // tri(i) -> Tri_light of the part's i-th triangle
__host__ __device__ inline void part_light(uint32_t n, Tri tri, Part_light& p) {
    float axis[3] = {0.f, 0.f, 0.f};
    p.total       = 0.f;
    for (int k = 0; k < 3; ++k) {
        p.lo[k] = __builtin_huge_valf();
        p.hi[k] = -__builtin_huge_valf();
    }
    for (uint32_t i = 0; i < n; ++i) {
        Tri_light const t = tri(i);
        for (int k = 0; k < 3; ++k) {
            p.lo[k] = smin(p.lo[k], t.lo[k]);
            p.hi[k] = smax(p.hi[k], t.hi[k]);
            axis[k] += t.area * t.n[k];
        }
        p.total += t.area;
    }
    float ax[3] = {axis[0] / p.total, axis[1] / p.total, axis[2] / p.total};
    float const al = sqrtf((ax[0] * ax[0] + ax[1] * ax[1]) + ax[2] * ax[2]);
    for (float& x : ax) {
        x /= al;
    }
    float angle = 0.f;
    for (uint32_t i = 0; i < n; ++i) {
        Tri_light const t  = tri(i);
        float const     cc = (ax[0] * t.n[0] + ax[1] * t.n[1]) + ax[2] * t.n[2];
        angle              = smax(angle, acos_r(smin(smax(cc, -1.f), 1.f)));
    }
    p.cone[0] = ax[0];
    p.cone[1] = ax[1];
    p.cone[2] = ax[2];
    p.cone[3] = cos_r(angle);
}

}  // namespace mi::lb
