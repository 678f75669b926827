// Host build of the rays' line test (csrc/ray_line.hpp), the face intersector (csrc/geom.hpp)
// and the host builder's face disks, for tests/test_ray_line_host.py.
#include <hip/hip_runtime.h>

#include <cstring>

// device functions that the headers use
inline int __float_as_int(float x) {
    int i;
    std::memcpy(&i, &x, 4);
    return i;
}
inline float __uint_as_float(unsigned x) {
    float f;
    std::memcpy(&f, &x, 4);
    return f;
}

#include "bvh.hpp"
#include "ray_line.hpp"

using namespace cubvh_amd;
using namespace cubvh_amd::dev;

// Face i (tris [n, 9]) against ray i (o, d [n, 3]): bit 0 of out[i] is set when tri_ray hits
// it, bit 1 when the line test rejects it, bit 2 when the face is one it never rejects.
extern "C" void ray_line_check(int64_t n, const float* tris, const float* o, const float* d, uint8_t* out) {
    HostBvh h;
    h.n_faces = n;
    h.tris.assign(12 * (size_t)n, 0.0f);
    for (int64_t i = 0; i < n; ++i)
        for (int k = 0; k < 9; ++k) h.tris[12 * i + k / 3 * 4 + k % 3] = tris[9 * i + k];
    compute_face_bounds(h);
    for (int64_t i = 0; i < n; ++i) {
        f3 v[3];
        for (int k = 0; k < 3; ++k) v[k] = mk3(tris[9 * i + 3 * k], tris[9 * i + 3 * k + 1], tris[9 * i + 3 * k + 2]);
        const f3 ro = mk3(o[3 * i], o[3 * i + 1], o[3 * i + 2]), rd = mk3(d[3 * i], d[3 * i + 1], d[3 * i + 2]);
        float reach = 0.0f;  // the farthest vertex: the least a caller may pass
        for (int k = 0; k < 3; ++k) reach = fmaxf(reach, sqrtf(dot3(sub3(v[k], ro), sub3(v[k], ro))));
        const float* t = &h.tbnd[8 * i];
        const bool rejects = line_rejects(ray_line(ro, rd, reach), make_float4(t[0], t[1], t[2], t[3]),
                                          make_float4(t[4], t[5], t[6], t[7]));
        out[i] = (uint8_t)((tri_ray(v[0], v[1], v[2], ro, rd) < 1e6f ? 1 : 0) | (rejects ? 2 : 0) | (t[7] > 0.0f ? 0 : 4));
    }
}
