// query.hpp -- host-side launch interface of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bvh.hpp"

namespace cubvh_amd {

// Device arrays of one tree (or of a forest's concatenated trees); layouts in bvh.hpp.
struct TreeArrays {
    const WideNode* nodes = nullptr;
    const float4* tris = nullptr;  // leaf-ordered triangles
    const float4* tbnd = nullptr;  // per-face bounding disks
    const float4* lbnd = nullptr;  // per-leaf bounding disks at leaf-start slots
    const float4* cbnd = nullptr;  // per-child bounding disks of internal subtrees
    const float4* tpre = nullptr;  // per-face constants of the distance formula
};

// How a call walks: lanes one query each, waves one query each in the caller's order, or
// packets of 64 queries, ordered first.
enum class Walk { lanes, waves, packets };

// Overrides for tests and measurements, per tree or forest (cubvh_bvh_walk_control).
struct WalkControl {
    int32_t route = 0;  // 1 waves, 2 packets, 0 by the rules below
    int32_t cap = -1;   // places of the hand-over's list; -1 by the rules, which may mean none
    int32_t first = 0;  // steps of a walk before it may be handed over; 0: the default
    int32_t factor = -1;  // sixteenths of the average walk's steps; -1: the default
    bool active() const { return route != 0 || cap >= 0 || first > 0 || factor >= 0; }
};

struct QueryArgs {
    int64_t n = 0;
    const float* in0 = nullptr;  // positions or ray origins [n,3]
    const float* in1 = nullptr;  // ray directions [n,3]
    const uint32_t* order = nullptr;  // optional query permutation [n] (lane i handles query order[i])
    bool permutation = false;    // order holds every query (a caller's may not)
    float* out_f = nullptr;      // distances or depth [n]
    int64_t* out_id = nullptr;   // face ids [n]
    float* out_v = nullptr;      // uvw or hit positions [n,3]
    TreeArrays tree;
    int64_t face0_slot = 0;
    int64_t n_faces = 0;
    int32_t stack_need = 0;
    Walk walk = Walk::packets;
    WalkControl control;
    void* rest = nullptr;  // packets: rest_bytes(n) bytes for the queries of given-up walks, or null: none is
    void* stream = nullptr;
};

// Small calls walk one wave per query in the caller's order, larger ones are ordered first
// and walk as packets of 64: a packet shares each fetch and test among its queries, but the
// ordering takes 60 to 120 us and a call lasts as long as its slowest tile, the more faces the
// longer.  Where both take the same time, in thousands of queries (points uniform, near the
// surface, normal, on a grid; smooth, jittered and soup meshes):
//   faces                    20   320  1,280  5,120  20,480  81,920  327,680  1.3 M
//   unsigned, raystab    95-340   120    130    170     190     220  240-300  360-500
//   watertight              150    90    105    140     170     190  200-300  330-450
//   rays, scattered         680   400    390    410     570     520      900    950
//   rays, camera            800   520    510    500     520     600      880   1,200
// 250,000 points near 320 faces, packets and waves: 208 / 387 us, 5,120 faces 273 / 511;
// below 2^18 rays waves always win.
constexpr int64_t kWaveMax = (int64_t)1 << 18;
inline bool waves_pay(int64_t n, int64_t n_faces, int mode) {  // mode as launch_distance's
    if (n_faces >= (int64_t)1 << 18) return n < kWaveMax;
    int64_t most = n_faces < 4096 ? (int64_t)1 << 17 : (int64_t)3 << 16;
    if (n_faces < 64 && mode != 2) most = kWaveMax;  // one node: a wave's round tests most of the mesh
    if (n_faces >= (int64_t)1 << 16 && mode == 2) most = kWaveMax;  // 76,377 loose faces: 250,000 points 1.35 ms by waves, 1.52 else
    if (mode == 1) most -= most / 4;                 // a packet's lanes search their normals at once
    return n < most;
}
inline bool ray_waves_pay(int64_t n) { return n < kWaveMax; }
// Never more waves than this: a launch has fewer than 2^32 threads.
constexpr int64_t kWaveMost = (int64_t)1 << 24;
inline Walk walk_of(const WalkControl& c, int64_t n, bool waves) {
    if (n >= (int64_t)1 << 31) return Walk::lanes;
    if (c.route == 1 && n < kWaveMost) return Walk::waves;
    return c.route == 2 || !waves ? Walk::packets : Walk::waves;
}

// Stack capacity instantiated for a tree that needs `need` entries (-1 if none).
int stack_capacity_for(int need);

// Queries one call's packet walks may hand on to waves of their own (query.hip); the
// walks past that many run to their end.
constexpr int64_t kRestMax = 1 << 19;
// Distance calls hand over below kRestLast queries, and from 16,384 on (walks end by the
// average of every 16th tile's, and fewer tiles never report enough), on trees of kRestFaces
// faces and more that have at most kRestQueries queries per face.  On smaller trees no walk is
// long and the two launches cost 3 to 8%: 2,000,000 points 371 us with, 356 without on 320
// faces, 425 and 410 on 1,280, but 600,000 near 5,120 jittered faces 479 and 655; many rounds
// of tiles cover the long walks: 7,000,000 points on 5,120 faces 1,340 us with, 1,305 without,
// on 20,480 1,742 and 1,680, on 81,920 2,482 and 2,415, but near 327,680 1,836 and 2,705; 2^24
// grid points on 1.3 M faces 12.76 and 12.45 ms.
constexpr int64_t kRestFaces = (int64_t)1 << 11;
constexpr int64_t kRestQueries = (int64_t)1 << 8;
constexpr int64_t kRestFirst = (int64_t)1 << 14;
constexpr int64_t kRestLast = (int64_t)1 << 23;
// Ray calls, whose walks are shorter: on 1.3 M faces 307,200 camera rays 455 us with, 692
// without, 8.3 M 1,148 and 1,195; 263,000 scattered ones 754 and 880, 7,000,000 5,575 and
// 5,627; on 81,920 faces 566 and 559.  Very many rays cover their long walks as above.
constexpr int64_t kRayRestFaces = (int64_t)1 << 18;
constexpr int64_t kRayRestLast = (int64_t)1 << 24;
inline bool hands_over(int64_t n, int64_t n_faces) {
    return n >= kRestFirst && n < kRestLast && n_faces >= kRestFaces && n / kRestQueries < n_faces;
}
size_t rest_bytes(int64_t n);
inline size_t rest_bytes(int64_t n, int64_t n_faces, const WalkControl& c) {
    return c.cap >= 0 || hands_over(n, n_faces) ? rest_bytes(n) : 0;
}
inline size_t ray_rest_bytes(int64_t n, int64_t n_faces, const WalkControl& c) {
    return c.cap >= 0 || (n < kRayRestLast && n_faces >= kRayRestFaces) ? rest_bytes(n) : 0;
}
// Queries handed over by the walks of a launch with this list so far (synchronizes).
hipError_t rest_count(const void* rest, hipStream_t s, uint32_t* count);

// Packets seed their walks (query.hip) while a face has fewer queries than this: with more,
// a walk finds its first face at once.  Seeded against not: 320 faces 263,000 points 180 / 201
// us, 2,000,000 353 / 337, 7,000,000 918 / 834; 5,120 faces 2,000,000 546 / 633, 16,000,000
// 2,866 / 2,775; 20,480 faces 7,000,000 1,684 / 1,858, 16,000,000 3,515 / 3,581.
constexpr int64_t kSeedQueries = 1 << 10;

// mode 0 unsigned distance, 1 signed (watertight), 2 signed (raystab)
hipError_t launch_distance(const QueryArgs& q, int mode);
hipError_t launch_ray(const QueryArgs& q);
// Negates q.out_f[i] of every query whose 64 raystab rays all hit (distances from mode 0),
// walking the queries of q.order (required by packets, n < 2^31) in passes over the undecided ones;
// ws holds stab_workspace_bytes(q.n) bytes.
size_t stab_workspace_bytes(int64_t n);
hipError_t launch_stab_sign(const QueryArgs& q, void* ws);
// The same for fewer than kStabFew queries, without scratch.
constexpr int64_t kStabFew = 1 << 11;
hipError_t launch_stab_few(const QueryArgs& q);

// The VALU issue-ceiling probe (probe.hip): `blocks` workgroups of 256 threads, each
// thread kValuProbeChains independent fp32 fma chains of `iters` steps; form 0 = VGPR
// and literal operands, 1 = one SGPR operand; out holds blocks x 256 floats.
constexpr int kValuProbeChains = 16;
hipError_t launch_valu_probe(int form, int blocks, int32_t iters, float* out, hipStream_t s);

// Morton permutation of point queries (order.hip).
size_t morton_workspace_bytes(int64_t n);
hipError_t morton_order(int64_t n, const float* positions, void* ws, uint32_t* order_out, hipStream_t s);
// Permutation of rays that puts rays of close origins and directions together (order.hip);
// ws holds morton_workspace_bytes(n) bytes.
hipError_t ray_order(int64_t n, const float* rays_o, const float* rays_d, void* ws, uint32_t* order_out, hipStream_t s);

// Static per-device scratch of the allocation-free distance call (order.hip): room for
// the Morton order and ordering workspace of kNoAllocMaxQueries queries.
constexpr int64_t kNoAllocMaxQueries = (int64_t)1 << 20;
constexpr size_t kNoAllocScratchBytes = (size_t)40 << 20;
constexpr int kNoAllocDevices = 64;
// Device address of the scratch on `device` (the current device); looked up once per device.
hipError_t noalloc_scratch(int device, void** ptr);

hipError_t launch_floodfill(const uint8_t* grid, int32_t B, int32_t H, int32_t W, int32_t D, int32_t* labels,
                            hipStream_t stream);

// Backward of the unsigned distance (grad.hip).  With grad_vertices, `ws` holds
// udf_backward_workspace_bytes(...) bytes of device scratch (sorts and per-face sums);
// point gradients alone need none.  corners / corner_begin / corner_end: the mesh's
// vertex -> corners table (launch_vertex_corners), or all null to build it in `ws`.
size_t udf_backward_workspace_bytes(int64_t n, int64_t n_vertices, int64_t n_faces, bool have_grad_points,
                                    bool have_tables);
hipError_t launch_udf_backward(int64_t n, const float* grad_dist, const float* positions, const int64_t* face_id,
                               const float* uvw, const float* vertices, int64_t n_vertices, const int32_t* faces,
                               int64_t n_faces, float* grad_points, float* grad_vertices, const uint32_t* corners,
                               const uint32_t* corner_begin, const uint32_t* corner_end, void* ws, hipStream_t stream);
// The vertex -> corners table of a mesh: corners (3 n_faces) = the corners 3 f + k grouped
// by vertex, ascending inside a vertex (corners of out-of-range indices last); vertex v
// owns corners[begin[v] .. end[v]).  ws holds vertex_corners_workspace_bytes(...) bytes.
size_t vertex_corners_workspace_bytes(int64_t n_vertices, int64_t n_faces);
hipError_t launch_vertex_corners(const int32_t* faces, int64_t n_faces, int64_t n_vertices, uint32_t* corners,
                                 uint32_t* begin, uint32_t* end, void* ws, hipStream_t stream);

}  // namespace cubvh_amd
