// wave_walk.hpp -- one wave per query: the walks of small calls.
//
// A call of few queries cannot fill the chip with one lane per query, and each lane's
// walk is one chain of dependent loads; a packet of queries that lie far apart walks the
// union of unlike paths, one load after another.  Here the 64 lanes of a wave share one
// query: a node round tests up to 16 nodes (one child per lane: box, then the child's
// bounding disk), a face round up to 4 leaves (one face per lane), so that a round costs
// one or two memory latencies for 64 tests.  Results do not depend on the order of the
// walk, the work does: until a first face is known only the nearest 4 nodes are opened
// (every box is in reach then; opening 16 let the pending nodes pile up to where they were
// taken one by one: 117 node rounds a query on 1.3 M faces, now 12), and the leaves are
// always taken nearest first (640 exact face tests a query, now 143).
//
// What bounds it: instruction issue.  A query on 81,920 faces takes 8 node, 5 face and 2
// exact rounds, some 1,730 vector instructions (57% of their lanes active) and as many scalar
// ones: 0.17 of each per SIMD-cycle, where the fma probe reads 0.42 with vector operands and
// 0.22 with a scalar one; the bytes (about 20 KB a query) come out of L2 and the Infinity
// Cache.  Exact tests recompute the face's terms from its 48-byte record: the 144-byte
// record that packets read made 250,000 points on 1.3 M faces 1.48 ms instead of 1.19.
// Measured: 777 points on 5,120 faces 16 us (351 us with a lane each); 50,003 on 81,920
// 0.21 ms (3.8 ms as packets, before their seeds and hand-over; query.hpp has both routes'
// times now); 1,501 rays on 81,920 14 us (146).  Not taken: 16 lanes per
// query, four walks a wave (0.9-1.4 times as long), and queries in Morton order (5%, less
// than the ordering costs).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "query.hpp"

namespace cubvh_amd {
namespace dev {

// Pending nodes of a wave's walk.  A node round replaces t entries by at most 4 t; t > 1
// only below kWaveChunk entries, and one node at a time adds at most STACK_TOTAL more.
constexpr int kWaveStack = 256;
constexpr int kWaveChunk = kWaveStack - STACK_TOTAL - 48;
constexpr int kWaveNodes = 16;   // nodes of a round
constexpr int kWaveDive = 4;     // the same until a first face is known
constexpr int kWaveLeaves = 4;   // leaves of a face round (16 lanes each)
static_assert(MAX_LEAF_SIZE == 16, "a face round gives a leaf 16 lanes");
struct alignas(8) WaveLists {
    int32_t ref[kWaveStack];
    float key[kWaveStack];
    int32_t leaf[64];
    float lkey[64];
    uint32_t face[128];  // faces that wait for the exact test: under 64, and one round's more
};

template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_min(uint32_t x) {
    return min(x, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)x, CTRL, ROWS, 0xf, false));
}
// Minimum over the wave's 64 lanes (row shifts, then the rows' totals broadcast on).
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
    x = dpp_min<0x111, 0xf>(x);
    x = dpp_min<0x112, 0xf>(x);
    x = dpp_min<0x114, 0xf>(x);
    x = dpp_min<0x118, 0xf>(x);
    x = dpp_min<0x142, 0xa>(x);
    x = dpp_min<0x143, 0xc>(x);
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// Lanes of m (not empty) with the smallest keys (non-negative floats): at most k of them,
// as many as eight bisections of the keys' range can tell apart, or the smallest alone.
// (Taking the keys within 3% of the smallest instead costs a third of the instructions but
// 38% more time on 1.3 M faces, where it tells far points' leaves apart too coarsely.)
__device__ __forceinline__ uint64_t nearest_lanes(uint64_t m, float key, int k) {
    const bool in = (m >> (threadIdx.x & 63)) & 1;
    const uint32_t bits = __float_as_uint(key);
    const uint32_t least = wave_min(in ? bits : 0xffffffffu);
    uint32_t lo = least, hi = ~wave_min(in ? ~bits : 0xffffffffu);
    for (int i = 0; i < 8; ++i) {
        const uint32_t mid = lo + (hi - lo + 1) / 2;
        if (__builtin_popcountll(ballot(bits < mid) & m) <= k) lo = mid;
        else hi = mid - 1;
    }
    const uint64_t near = ballot(bits < lo) & m;
    return near ? near : ballot(bits == least) & m;
}

// Appends (ref, key) of the lanes in m to a list at `at`, those of `last` after the rest.
__device__ __forceinline__ void append_ordered(int32_t* ref, float* key, int at, uint64_t m, uint64_t last, int32_t r,
                                               float k) {
    const int lane = (int)(threadIdx.x & 63);
    const uint64_t first = m & ~last;
    if ((m >> lane) & 1) {
        const int i = ((last >> lane) & 1) ? at + __builtin_popcountll(first) + (int)lanes_below(last)
                                           : at + (int)lanes_below(first);
        ref[i] = r;
        key[i] = k;
    }
}

// One child of a node, by the lane that tests it.
struct LaneChild {
    float lx, hx, ly, hy, lz, hz;
    int32_t ref;
};
__device__ __forceinline__ LaneChild load_child(const WideNode* __restrict__ nodes, int32_t node, int j) {
    const float* f = reinterpret_cast<const float*>(nodes + node) + j;
    LaneChild c;
    c.lx = f[0];
    c.hx = f[4];
    c.ly = f[8];
    c.hy = f[12];
    c.lz = f[16];
    c.hz = f[20];
    c.ref = __float_as_int(f[24]);
    return c;
}

// The pending work of one wave's walk (wave-uniform counts).
struct WaveWork {
    WaveLists& L;
    int sp = 0, nl = 0, nf = 0;

    __device__ __forceinline__ void start(int32_t root) {
        L.ref[0] = root;  // every lane the same value
        L.key[0] = 0.0f;
        sp = 1;
        nl = nf = 0;
        wave_fence();
    }
    // Takes nodes off the stack, one per quad of lanes: false for lanes without one (or
    // with one that the bound has passed).
    __device__ __forceinline__ bool take_nodes(float bound, int most, int32_t& node) {
        const int quad = (int)(threadIdx.x & 63) >> 2;
        const int want = sp > kWaveChunk ? 1 : min(most, (64 - nl) >> 2);
        const int take = min(want, sp);
        bool on = quad < take;
        node = 0;
        if (on) {
            const int e = sp - 1 - quad;
            node = L.ref[e];
            on = L.key[e] <= bound;
        }
        sp -= take;
        wave_fence();
        return on;
    }
    // Files the surviving children; of more than `most` nodes the nearest go on top.
    __device__ __forceinline__ void add_children(bool on, int32_t ref, float key, int most) {
        const uint64_t lm = ballot(on && ref < 0), im = ballot(on && ref >= 0);
        append_ordered(L.leaf, L.lkey, nl, lm, 0, ref, key);
        nl += __builtin_popcountll(lm);
        const int c = __builtin_popcountll(im);
        const uint64_t top = c > most ? nearest_lanes(im, key, most) : 0;
        append_ordered(L.ref, L.key, sp, im, top, ref, key);
        sp += c;
        wave_fence();
    }
    // Drops the stacked nodes that the bound has passed.
    __device__ __forceinline__ void prune(float bound) {
        const int lane = (int)(threadIdx.x & 63);
        int kept = 0;
        for (int at = 0; at < sp; at += 64) {
            int32_t r = 0;
            float k = INFINITY;
            if (at + lane < sp) {
                r = L.ref[at + lane];
                k = L.key[at + lane];
            }
            const uint64_t m = ballot(at + lane < sp && k <= bound);
            wave_fence();
            append_ordered(L.ref, L.key, kept, m, 0, r, k);
            kept += __builtin_popcountll(m);
            wave_fence();
        }
        sp = kept;
    }
    // Takes leaves, one per 16 lanes, after dropping those the bound has passed: the
    // lane's face slot, or -1.
    __device__ __forceinline__ int32_t take_leaves(float bound, bool nearest) {
        const int lane = (int)(threadIdx.x & 63);
        int32_t r = 0;
        float k = INFINITY;
        if (lane < nl) {
            r = L.leaf[lane];
            k = L.lkey[lane];
        }
        const uint64_t m = ballot(lane < nl && k <= bound);
        nl = __builtin_popcountll(m);
        const uint64_t top = nearest && nl > kWaveLeaves ? nearest_lanes(m, k, kWaveLeaves) : 0;
        wave_fence();
        append_ordered(L.leaf, L.lkey, 0, m, top, r, k);
        wave_fence();
        const int take = min(kWaveLeaves, nl), g = lane >> 4;
        int32_t slot = -1;
        if (g < take) {
            const int32_t leaf = L.leaf[nl - 1 - g];
            if ((lane & 15) < leaf_ref_count(leaf)) slot = leaf_ref_first(leaf) + (lane & 15);
        }
        nl -= take;
        wave_fence();
        return slot;
    }
};

// Nearest face to p in the tree below `root` (wave-uniform arguments and results), as
// closest_face; best_d2 / bslot / bid hold a candidate or the unset values.
__device__ void closest_face_wave(const Tree& T, int32_t root, f3 p, WaveLists& L, float& best_d2, int32_t& bslot,
                                  uint32_t& bid) {
    const int lane = (int)(threadIdx.x & 63);
    uint32_t best = __float_as_uint(best_d2);
    float bound = best_d2 * BOUND_SLACK;
    WaveWork w{L};
    w.start(root);
    if (has_nan(p)) w.sp = 0;
    for (;;) {
        const bool unset = bslot < 0;
        if (w.sp > 0 && w.nl < kWaveLeaves && !(unset && w.nl > 0)) {
            int32_t node, ref = CHILD_EMPTY;
            float key = INFINITY;
            // until a first face is known every box is in reach: the nearest few nodes only
            const int most = unset ? kWaveDive : kWaveNodes;
            bool on = w.take_nodes(bound, most, node);
            if (on) {
                const LaneChild c = load_child(T.nodes, node, lane & 3);
                key = box_d2(c.lx, c.hx, c.ly, c.hy, c.lz, c.hz, p);
                ref = c.ref;
                on = ref != CHILD_EMPTY && key <= bound;
                if (on) {
                    const float4* d = ref >= 0 ? T.cbnd + 8 * node + 2 * (lane & 3) : T.lbnd + 2 * leaf_ref_first(ref);
                    key = fmaxf(key, disk_bound(p, d[0], d[1]));
                    on = key <= bound;
                }
            }
            w.add_children(on, ref, key, unset ? most : 64);
        } else if (w.nl > 0) {
            const int32_t slot = w.take_leaves(bound, true);
            bool on = slot >= 0;
            if (on) on = !disk_rejects(p, T.tbnd[2 * slot], T.tbnd[2 * slot + 1], bound);
            const uint64_t m = ballot(on);
            if (on) L.face[w.nf + (int)lanes_below(m)] = (uint32_t)slot;
            w.nf += __builtin_popcountll(m);
            wave_fence();
        } else if (w.nf == 0) {
            break;
        }
        const bool last = w.sp == 0 && w.nl == 0;
        if (w.nf >= 64 || (w.nf > 0 && (last || bslot < 0))) {
            const int take = min(w.nf, 64);
            uint32_t bits = 0xffffffffu, id = 0xffffffffu;
            int32_t slot = 0;
            if (lane < take) {
                slot = (int32_t)L.face[w.nf - take + lane];
                f3 a, b, c;
                int32_t i;
                load_tri(T.tris, slot, a, b, c, i);
                bits = __float_as_uint(tri_dist2(a, b, c, p));  // >= 0, or a NaN that orders last
                id = (uint32_t)i;
            }
            w.nf -= take;
            const uint32_t m = wave_min(bits);
            if (m < best || (m == best && bslot >= 0)) {
                const uint32_t i = wave_min(bits == m ? id : 0xffffffffu);
                if (m < best || i < bid) {
                    best = m;
                    bid = i;
                    bslot = __builtin_amdgcn_readlane(slot, (int)__builtin_ctzll(ballot(bits == m && id == i)));
                    bound = __uint_as_float(best) * BOUND_SLACK;
                    if (w.sp > kWaveNodes) w.prune(bound);
                }
            }
            wave_fence();
        }
    }
    best_d2 = __uint_as_float(best);
}

// add_normals over one wave (c and sum wave-uniform).
template <class Sum>
__device__ __forceinline__ void add_normals_wave(const Tree& T, f3 c, WaveLists& L, Sum& sum) {
    const int lane = (int)(threadIdx.x & 63);
    WaveWork w{L};
    w.start(0);
    if (has_nan(c)) w.sp = 0;
    for (;;) {
        if (w.sp > 0 && w.nl < kWaveLeaves) {
            int32_t node, ref = CHILD_EMPTY;
            float key = INFINITY;
            bool on = w.take_nodes(NORMAL_EPS, kWaveNodes, node);
            if (on) {
                const LaneChild ch = load_child(T.nodes, node, lane & 3);
                key = box_d2(ch.lx, ch.hx, ch.ly, ch.hy, ch.lz, ch.hz, c);
                ref = ch.ref;
                on = ref != CHILD_EMPTY && key < NORMAL_EPS;
                if (on && ref < 0) {
                    const float4* d = T.lbnd + 2 * leaf_ref_first(ref);
                    on = !disk_rejects(c, d[0], d[1], NORMAL_EPS);
                }
            }
            w.add_children(on, ref, key, 64);
        } else if (w.nl > 0) {
            const int32_t slot = w.take_leaves(NORMAL_EPS, false);
            bool on = slot >= 0;
            if (on) on = !disk_rejects(c, T.tbnd[2 * slot], T.tbnd[2 * slot + 1], NORMAL_EPS);
            f3 n = mk3(0.0f, 0.0f, 0.0f);
            if (on) {
                f3 a, b, cc;
                int32_t id;
                load_tri(T.tris, slot, a, b, cc, id);
                on = tri_dist2(a, b, cc, c) < NORMAL_EPS;
                if (on) n = tri_normal(a, b, cc);
            }
            for (uint64_t m = ballot(on); m != 0; m &= m - 1) {
                const int l = (int)__builtin_ctzll(m);
                sum.add(mk3(lane_value(n.x, l), lane_value(n.y, l), lane_value(n.z, l)));
            }
        } else {
            break;
        }
    }
}

// avg_normal over one wave (c wave-uniform).
__device__ f3 avg_normal_wave(const Tree& T, f3 c, WaveLists& L) {
    NormalSum sum;
    add_normals_wave(T, c, L, sum);
    if (sum.exact()) return sum.mean();
    NormalParts parts{reinterpret_cast<double*>(L.face)};  // no faces wait here
    do {
        parts.start();
        add_normals_wave(T, c, L, parts);
        wave_fence();
    } while (parts.next());
    wave_fence();
    return parts.mean();
}

// Closest hit of the ray (wave-uniform arguments and results), as closest_hit; best / bslot
// hold a candidate or the unset values.
__device__ void closest_hit_wave(const Tree& T, f3 o, f3 d, WaveLists& L, float& best, int32_t& bslot, uint32_t& bid) {
    const int lane = (int)(threadIdx.x & 63);
    const f3 inv = ray_inverse(d);
    float bound = best * BOUND_SLACK + 1e-30f;
    WaveWork w{L};
    w.start(0);
    for (;;) {
        const bool unset = bslot < 0;
        if (w.sp > 0 && w.nl < kWaveLeaves && !(unset && w.nl > 0)) {
            int32_t node, ref = CHILD_EMPTY;
            float key = INFINITY;
            bool on = w.take_nodes(bound, kWaveNodes, node);
            if (on) {
                const LaneChild c = load_child(T.nodes, node, lane & 3);
                ref = c.ref;
                // a box around the origin enters at a negative t: ordered as 0
                key = fmaxf(slab_entry(c.lx, c.hx, c.ly, c.hy, c.lz, c.hz, o, inv), 0.0f);
                on = ref != CHILD_EMPTY && key <= bound;
            }
            w.add_children(on, ref, key, kWaveNodes);
        } else if (w.nl > 0) {
            const int32_t slot = w.take_leaves(bound, true);
            float t = INFINITY;
            uint32_t id = 0xffffffffu;
            if (slot >= 0) {
                f3 a, b, c;
                int32_t i;
                load_tri(T.tris, slot, a, b, c, i);
                t = tri_ray(a, b, c, o, d);
                id = (uint32_t)i;
            }
            const uint32_t bits = t == 0.0f ? 0u : __float_as_uint(t);  // t >= 0, -0 as 0
            const uint32_t m = wave_min(bits), cur = best == 0.0f ? 0u : __float_as_uint(best);
            if (m < cur || (m == cur && bslot >= 0)) {
                const uint32_t i = wave_min(bits == m ? id : 0xffffffffu);
                if (m < cur || i < bid) {
                    const int l = (int)__builtin_ctzll(ballot(bits == m && id == i));
                    best = lane_value(t, l);
                    bid = i;
                    bslot = __builtin_amdgcn_readlane(slot, l);
                    bound = best * BOUND_SLACK + 1e-30f;
                    if (w.sp > kWaveNodes) w.prune(bound);
                }
            }
        } else {
            break;
        }
    }
}

// any_hit_line over one wave (wave-uniform arguments and result).  A pending entry's key
// holds the directions it is open for in its two low bits; open1 / open2 count the entries
// open for +d / -d: the pair is decided when a direction not hit yet has none left.
__device__ int any_hit_line_wave(const Tree& T, f3 o, f3 d, WaveLists& L) {
    const int lane = (int)(threadIdx.x & 63);
    const f3 inv = ray_inverse(d);
    const float limit = MAX_DIST * BOUND_SLACK;
    int found = 0, open1 = 1, open2 = 1;
    WaveWork w{L};
    w.start(0);
    L.key[0] = __uint_as_float(3u);
    wave_fence();
    for (;;) {
        const uint32_t want = 3u & ~(uint32_t)found;
        if (w.sp > 0 && w.nl < kWaveLeaves) {
            const int quad = lane >> 2;
            const int take = min(w.sp > kWaveChunk ? 1 : min(kWaveNodes, (64 - w.nl) >> 2), w.sp);
            bool on = quad < take;
            int32_t node = 0, ref = CHILD_EMPTY;
            uint32_t dirs = 0;
            if (on) {
                node = L.ref[w.sp - 1 - quad];
                dirs = __float_as_uint(L.key[w.sp - 1 - quad]) & 3u;
            }
            w.sp -= take;
            const bool first = (lane & 3) == 0;  // one lane of the quad accounts for the entry
            open1 -= __builtin_popcountll(ballot(first && (dirs & 1u)));
            open2 -= __builtin_popcountll(ballot(first && (dirs & 2u)));
            wave_fence();
            on = on && (dirs & want) != 0;
            uint32_t m = 0;
            if (on) {
                const LaneChild c = load_child(T.nodes, node, lane & 3);
                ref = c.ref;
                const float tx0 = (c.lx - o.x) * inv.x, tx1 = (c.hx - o.x) * inv.x;
                const float ty0 = (c.ly - o.y) * inv.y, ty1 = (c.hy - o.y) * inv.y;
                const float tz0 = (c.lz - o.z) * inv.z, tz1 = (c.hz - o.z) * inv.z;
                const float tn = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fminf(tz0, tz1));
                const float tf = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fmaxf(tz0, tz1));
                if (ref != CHILD_EMPTY && tn <= tf)
                    m = ((tf >= 0.0f && tn <= limit ? 1u : 0u) | (tn <= 0.0f && tf >= -limit ? 2u : 0u)) & want & dirs;
            }
            on = m != 0;
            open1 += __builtin_popcountll(ballot(m & 1u));
            open2 += __builtin_popcountll(ballot(m & 2u));
            const uint64_t lm = ballot(on && ref < 0), im = ballot(on && ref >= 0);
            append_ordered(L.leaf, L.lkey, w.nl, lm, 0, ref, __uint_as_float(m));
            append_ordered(L.ref, L.key, w.sp, im, 0, ref, __uint_as_float(m));
            w.nl += __builtin_popcountll(lm);
            w.sp += __builtin_popcountll(im);
            wave_fence();
        } else {  // leaves: one of the two lists has an entry, or a count would be zero
            const int take = min(kWaveLeaves, w.nl), g = lane >> 4;
            int32_t slot = -1;
            uint32_t dirs = 0;
            if (g < take) {
                const int32_t leaf = L.leaf[w.nl - 1 - g];
                dirs = __float_as_uint(L.lkey[w.nl - 1 - g]) & 3u;
                if ((lane & 15) < leaf_ref_count(leaf)) slot = leaf_ref_first(leaf) + (lane & 15);
            }
            w.nl -= take;
            const bool first = (lane & 15) == 0;
            open1 -= __builtin_popcountll(ballot(first && (dirs & 1u)));
            open2 -= __builtin_popcountll(ballot(first && (dirs & 2u)));
            uint32_t hit = 0;
            if (slot >= 0 && (dirs & want) != 0) {
                f3 a, b, c;
                int32_t id;
                load_tri(T.tris, slot, a, b, c, id);
                hit = (uint32_t)tri_line(a, b, c, o, d, MAX_DIST) & dirs;
            }
            found |= (ballot(hit & 1u) != 0 ? 1 : 0) | (ballot(hit & 2u) != 0 ? 2 : 0);
            wave_fence();
        }
        if (found == 3) return 3;
        if ((!(found & 1) && open1 == 0) || (!(found & 2) && open2 == 0)) return found;
    }
}

// Query q at p from a candidate (d2, slot; slot < 0: none) to its outputs, by one wave.
template <int MODE>
__device__ __forceinline__ void wave_query(const Tree& T, int32_t root, int32_t face0_slot, int64_t q, f3 p, float d2,
                                           int32_t slot, WaveLists& L, float* __restrict__ distances,
                                           int64_t* __restrict__ face_id, float* __restrict__ uvw) {
    uint32_t bid = slot >= 0 ? (uint32_t)__float_as_int(T.tris[3 * slot].w) : 0u;
    closest_face_wave(T, root, p, L, d2, slot, bid);
    if (slot < 0) {  // nothing within MAX_DIST: distance 0 and face 0
        slot = face0_slot;
        d2 = 0.0f;
    }
    f3 a, b, c;
    int32_t id;
    load_tri(T.tris, slot, a, b, c, id);
    float dist = sqrtf(d2);
    f3 cp = mk3(0.0f, 0.0f, 0.0f);
    if (MODE == 1 || uvw) cp = tri_closest_pt(a, b, c, p);
    if constexpr (MODE == 1) dist = copysignf(dist, dot3(avg_normal_wave(T, cp, L), sub3(p, cp)));
    if ((threadIdx.x & 63) == 0) {
        distances[q] = dist;
        face_id[q] = (int64_t)id;
        if (uvw) store_pt(uvw, q, tri_barycentric(a, b, c, cp));
    }
}

// Unsigned (MODE 0) and watertight signed (MODE 1) distance, one wave per query.
template <int MODE>
__global__ __launch_bounds__(64) void distance_wave_kernel(const float* __restrict__ positions,
                                                           float* __restrict__ distances,
                                                           int64_t* __restrict__ face_id, float* __restrict__ uvw,
                                                           Tree T) {
    __shared__ WaveLists lists;
    const int64_t q = blockIdx.x;
    wave_query<MODE>(T, 0, (int32_t)T.face0_slot, q, load_pt(positions, q), MAX_DIST_SQ, -1, lists, distances, face_id,
                     uvw);
}

// The queries that packet walks gave up (see PacketRest), a wave each.
template <int MODE>
__global__ __launch_bounds__(64) void distance_rest_kernel(const PacketRest* __restrict__ rest,
                                                           const float* __restrict__ positions,
                                                           float* __restrict__ distances,
                                                           int64_t* __restrict__ face_id, float* __restrict__ uvw,
                                                           Tree T) {
    __shared__ WaveLists lists;
    const uint32_t total = min(rest->count, rest->cap);
    for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int4 e = rest->list()[t];
        if (uniform(e.x) == -1) continue;  // an empty place
        const int64_t q = (int64_t)(uint32_t)uniform(e.x);
        const int32_t slot = uniform(e.z);
        wave_query<MODE>(T, uniform(e.w), ~slot, q, load_pt(positions, q), __int_as_float(uniform(e.y)), slot, lists,
                         distances, face_id, uvw);
        __builtin_amdgcn_wave_barrier();  // one back edge: every lane starts the next walk together
    }
}

// Ray q from a candidate (t, slot; slot < 0: none) to its outputs, by one wave.
__device__ __forceinline__ void wave_ray(const Tree& T, int64_t q, f3 o, f3 d, float t, int32_t slot, WaveLists& L,
                                         float* __restrict__ positions, int64_t* __restrict__ face_id,
                                         float* __restrict__ depth) {
    uint32_t id = slot >= 0 ? (uint32_t)__float_as_int(T.tris[3 * slot].w) : 0u;
    closest_hit_wave(T, o, d, L, t, slot, id);
    if ((threadIdx.x & 63) == 0) {
        depth[q] = t;
        store_pt(positions, q,
                 mk3(__builtin_fmaf(t, d.x, o.x), __builtin_fmaf(t, d.y, o.y), __builtin_fmaf(t, d.z, o.z)));
        face_id[q] = slot >= 0 ? (int64_t)id : -1;
    }
}

// Rays, one wave per ray.
__global__ __launch_bounds__(64) void ray_wave_kernel(const float* __restrict__ rays_o, const float* __restrict__ rays_d,
                                                      float* __restrict__ positions, int64_t* __restrict__ face_id,
                                                      float* __restrict__ depth, Tree T) {
    __shared__ WaveLists lists;
    const int64_t q = blockIdx.x;
    wave_ray(T, q, load_pt(rays_o, q), load_pt(rays_d, q), MAX_DIST, -1, lists, positions, face_id, depth);
}

// The rays that packet and lane walks gave up, a wave each.
__global__ __launch_bounds__(64) void ray_rest_kernel(const PacketRest* __restrict__ rest,
                                                      const float* __restrict__ rays_o, const float* __restrict__ rays_d,
                                                      float* __restrict__ positions, int64_t* __restrict__ face_id,
                                                      float* __restrict__ depth, Tree T) {
    __shared__ WaveLists lists;
    const uint32_t total = min(rest->count, rest->cap);
    for (uint32_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int4 e = rest->list()[t];
        if (uniform(e.x) == -1) continue;  // an empty place
        const int64_t q = (int64_t)(uint32_t)uniform(e.x);
        wave_ray(T, q, load_pt(rays_o, q), load_pt(rays_d, q), __int_as_float(uniform(e.y)), uniform(e.z), lists,
                 positions, face_id, depth);
        __builtin_amdgcn_wave_barrier();  // one back edge: every lane starts the next walk together
    }
}

}  // namespace dev
}  // namespace cubvh_amd
