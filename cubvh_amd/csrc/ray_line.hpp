// ray_line.hpp -- a ray's line against the bounding sphere of a face.
//
// A face of a fine mesh covers one or two of a camera tile's rays, so a packet's (ray, face)
// pairs pass this test (some 20 instructions) before the exact intersection (60).  It may
// only drop pairs that tri_ray answers with a miss.
//
// With u = 2^-24, s the sine of the angle at a between e1 = b - a and e2 = c - a, c the cosine
// between the ray and the face's normal, and p = o - a, the roundings of tri_ray add up to
//   |error of n|        <= 4 u |e1| |e2|       (edges u each, cross product 2 u)
//   |error of q|        <= 3 u |p| |d|
//   |error of den|      <= 7 u |d| |e1| |e2|,  so den is off by a factor 1 +- 7 u / (s c)
//   |error of q . e|    <= 7 u |p| |d| |e|
// A hit's u and v therefore place it within 14 u |p| / (s c) of the line's true point in the
// plane, up to a scaling by 1 +- 10 u / (s c) about a.  Faces with s < 1/16, or with edges so
// short or long that products under- or overflow, are marked by the builders and never
// rejected; neither are faces seen at c < 1/20.  For the others the scaling is below 4e-4
// (1/64 of the radius is allowed for) and 14 u |p| / s below 1.34e-5 of the distance to the
// farthest vertex (2^-16 = 1.53e-5 is; the test's own roundings take 4e-7).
#pragma once

#include "geom.hpp"

namespace cubvh_amd {
namespace dev {

struct RayLine {
    f3 o, dn;      // origin, unit direction
    float margin;  // what tri_ray's rounding adds to a sphere's radius times c
};

// reach: no vertex is farther from o.  Directions whose length under- or overflows when
// squared get no test (an infinite margin).
__device__ __forceinline__ RayLine ray_line(f3 o, f3 d, float reach) {
    const float n2 = dot3(d, d), s = 1.0f / sqrtf(n2);
    RayLine r;
    r.o = o;
    r.dn = mk3(d.x * s, d.y * s, d.z * s);
    r.margin = n2 > 1e-12f && n2 < 1e12f ? reach * 1.52587890625e-05f : INFINITY;
    return r;
}

// True when the line passes the sphere around a face's disk (bvh.hpp: tbnd) so far out that
// tri_ray gives a miss; never with NaN anywhere.
__device__ __forceinline__ bool line_rejects(const RayLine& r, float4 cb, float4 nb) {
    const f3 x = cross3(mk3(cb.x - r.o.x, cb.y - r.o.y, cb.z - r.o.z), r.dn);
    const float c = fabsf(dot3(mk3(nb.x, nb.y, nb.z), r.dn));
    const float reach = (cb.w + nb.w) * 1.015625f * c + r.margin;
    return dot3(x, x) * (c * c) > reach * reach && c > 0.05f && nb.w > 0.0f;
}

}  // namespace dev
}  // namespace cubvh_amd
