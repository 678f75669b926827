// smc.hip -- sparse marching cubes.
//
// Output contract of the reference's GPU extraction (include/gpu/spcumc.cuh:631-868):
//   * one vertex per lattice edge that carries a sign change in some cell, numbered in
//     ascending order of (lowest lattice point x, y, z, axis); its position is linear
//     interpolation of the iso level along the edge, from the values of the first cell
//     (input order) that has the edge;
//   * per cell in input order, the case's triangles in table order with the second and
//     third vertex exchanged.
// With ensure_consistency the corner values are first replaced by the mean over every
// cell that shares the lattice point, summed in double in cell order (the reference's
// CPU path, include/cpu/spmc.h:408-433; its GPU path sums in fp32 in an order that its
// library reduction leaves open).
//
// Pipeline: bounds (per-block partials, one fold) -> [corner keys, radix sort, run
// means] -> classify (case, counts) -> exclusive scan -> one synchronization (bounds and
// totals) -> edge keys in cell order -> stable radix sort -> inclusive scan of run
// starts (vertex ids) -> one synchronization (vertex count) -> [caller's buffers]
// vertices from the first cell of each run and a raw -> vertex map -> triangles.  Edge
// and corner keys pack the lattice point relative to the minimum with B bits per axis
// (B from the measured span), so the sorts run over 3B + 2 and 3B bits, with 32-bit
// edge keys whenever 3B + 2 <= 32 (spans up to 1022).
//
// Cells in strictly ascending order of (x, y, z), as a lattice scan lists them, need no
// sort when their bounding lattice is not too sparse (dense_words_most): a bit per lattice
// cell and a prefix count per 32 of them find a cell's neighbours and count the cells before
// any place.  An edge is owned by its first cell; edges of one (dx, dy) of their lowest
// point in the owner's cell ("stream") ascend with the cells, up to the neighbours along z,
// so a vertex's number is, over the four streams, the owned edges of the cells before its
// place and a few bits of the two cells there.  Only owners compute it; the other cells of
// an edge keep the owner's slot.  Latency of the gathers bounds these kernels.  Cut cells of
// a lattice: 742,270 307 -> 198 us (257 with every cell computing the numbers of all its
// edges), 174,056 231 -> 116, 3,850 142 -> 115; with averaged corners 454,180 515 -> 208.
// Cells in random order are sorted as before: 742,270 340 -> 345, 25,542 158 -> 156.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>
#include <stdint.h>

#include <algorithm>
#include <climits>
#include <cstring>
#include <mutex>
#include <vector>

#include "mc_table.hpp"
#include "smc.hpp"

namespace cubvh_amd {

namespace {

__constant__ uint64_t c_triangles[256] = {CUBVH_MC_TRIANGLES};

constexpr int kBlock = 256;

unsigned blocks_for(int64_t n) { return (unsigned)std::max<int64_t>(1, (n + kBlock - 1) / kBlock); }

__device__ __forceinline__ uint32_t edge_mask_of(uint32_t c) {
    const uint32_t lo = c & 15u, hi = c >> 4;
    const uint32_t rlo = ((lo >> 1) | (lo << 3)) & 15u, rhi = ((hi >> 1) | (hi << 3)) & 15u;
    return (lo ^ rlo) | ((hi ^ rhi) << 4) | ((lo ^ hi) << 8);
}

// info: [0..2] min x y z, [3..5] max x y z (int32), [6] 1 unless the cells ascend strictly.
constexpr int kBounds = 7;

// Bounds in two steps without same-address atomics: each block writes its six extremes
// to part[kBounds * block], one block folds them into info.
__device__ __forceinline__ void block_extremes(int32_t (&lo)[3], int32_t (&hi)[3]) {
    __shared__ int32_t sh[6][kBlock / 64];
    for (int o = 32; o > 0; o >>= 1)
        for (int k = 0; k < 3; ++k) {
            lo[k] = min(lo[k], __shfl_xor(lo[k], o));
            hi[k] = max(hi[k], __shfl_xor(hi[k], o));
        }
    const int w = (int)(threadIdx.x >> 6);
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 3; ++k) {
            sh[k][w] = lo[k];
            sh[3 + k][w] = hi[k];
        }
    __syncthreads();
    for (int k = 0; k < 3; ++k) {
        lo[k] = sh[k][0];
        hi[k] = sh[3 + k][0];
        for (int j = 1; j < kBlock / 64; ++j) {
            lo[k] = min(lo[k], sh[k][j]);
            hi[k] = max(hi[k], sh[3 + k][j]);
        }
    }
}

__global__ __launch_bounds__(kBlock) void smc_bounds(const int32_t* __restrict__ coords, int64_t n,
                                                     int32_t* __restrict__ part) {
    int32_t lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
    int mixed = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        int32_t v[3], order = i == 0 ? -1 : 0;  // of the cell before against this one
        for (int k = 0; k < 3; ++k) {
            v[k] = coords[3 * i + k];
            lo[k] = min(lo[k], v[k]);
            hi[k] = max(hi[k], v[k]);
            if (i > 0 && order == 0) {
                const int32_t u = coords[3 * (i - 1) + k];
                order = u < v[k] ? -1 : (u > v[k] ? 1 : 0);
            }
        }
        mixed |= order >= 0;
    }
    block_extremes(lo, hi);
    mixed = __syncthreads_or(mixed);
    if (threadIdx.x < 3) {
        part[kBounds * blockIdx.x + threadIdx.x] = lo[threadIdx.x];
        part[kBounds * blockIdx.x + 3 + threadIdx.x] = hi[threadIdx.x];
    }
    if (threadIdx.x == 0) part[kBounds * blockIdx.x + 6] = mixed;
}

__global__ __launch_bounds__(kBlock) void smc_fold_bounds(const int32_t* __restrict__ part, int n_part,
                                                          int32_t* __restrict__ info) {
    int32_t lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {INT_MIN, INT_MIN, INT_MIN};
    int mixed = 0;
    for (int b = (int)threadIdx.x; b < n_part; b += kBlock) {
        for (int k = 0; k < 3; ++k) {
            lo[k] = min(lo[k], part[kBounds * b + k]);
            hi[k] = max(hi[k], part[kBounds * b + 3 + k]);
        }
        mixed |= part[kBounds * b + 6];
    }
    block_extremes(lo, hi);
    mixed = __syncthreads_or(mixed);
    if (threadIdx.x == 0) info[6] = mixed;
    if (threadIdx.x < 3) {
        info[threadIdx.x] = lo[threadIdx.x];
        info[3 + threadIdx.x] = hi[threadIdx.x];
    }
}

// Lattice point packed relative to the minimum, B bits per axis.
__device__ __forceinline__ uint64_t pack_point(int64_t x, int64_t y, int64_t z, const int32_t* mn, int B) {
    return ((uint64_t)(x - mn[0]) << (2 * B)) | ((uint64_t)(y - mn[1]) << B) | (uint64_t)(z - mn[2]);
}

// ---- corner consistency
template <typename K>
__global__ __launch_bounds__(kBlock) void smc_corner_keys(const int32_t* __restrict__ coords, int64_t n,
                                                          const int32_t* __restrict__ info, int B,
                                                          K* __restrict__ keys, uint32_t* __restrict__ vals) {
    const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (j >= 8 * n) return;
    const int64_t i = j >> 3;
    const int k = (int)(j & 7);
    keys[j] = (K)pack_point((int64_t)coords[3 * i] + mc::corner_dx(k), (int64_t)coords[3 * i + 1] + mc::corner_dy(k),
                            (int64_t)coords[3 * i + 2] + mc::corner_dz(k), info, B);
    vals[j] = (uint32_t)j;
}

// Run of equal keys starting at s: mean of the corner values in cell order (the sort is
// stable and the values were laid out in cell order), written to every member.
template <typename K>
__global__ __launch_bounds__(kBlock) void smc_corner_mean(const K* __restrict__ keys,
                                                          const uint32_t* __restrict__ vals, int64_t m,
                                                          const float* __restrict__ corners,
                                                          float* __restrict__ out) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (s >= m || (s > 0 && keys[s - 1] == keys[s])) return;
    const K key = keys[s];
    double sum = 0.0;
    int64_t e = s;
    for (; e < m && keys[e] == key; ++e) sum += (double)corners[vals[e]];
    const float mean = (float)(sum / (double)(e - s));
    for (int64_t j = s; j < e; ++j) out[vals[j]] = mean;
}

// ---- classification
__global__ __launch_bounds__(kBlock) void smc_classify(const float* __restrict__ corners, int64_t n, float iso,
                                                       uint8_t* __restrict__ cases, uint64_t* __restrict__ counts) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t c = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) c |= (corners[8 * i + k] < iso ? 1u : 0u) << k;
    cases[i] = (uint8_t)c;
    const uint32_t nv = (uint32_t)__popc(edge_mask_of(c));
    const uint32_t nt = (uint32_t)mc::triangle_count(c_triangles[c]);
    counts[i] = ((uint64_t)nv << 32) | nt;
}

// offsets = exclusive scan of counts; totals = last offset + last count.
__global__ void smc_totals(const uint64_t* __restrict__ counts, const uint64_t* __restrict__ offsets, int64_t n,
                           uint64_t* __restrict__ totals) {
    if (threadIdx.x == 0 && blockIdx.x == 0) totals[0] = offsets[n - 1] + counts[n - 1];
}

// ---- edge vertices
// Edge keys (lowest lattice point relative to the minimum, then the axis) and
// (cell, edge) values, laid out in cell order at each cell's first raw slot.
template <typename K>
__global__ __launch_bounds__(kBlock) void smc_edge_keys(const int32_t* __restrict__ coords,
                                                        const uint8_t* __restrict__ cases,
                                                        const uint64_t* __restrict__ offsets, int64_t n,
                                                        const int32_t* __restrict__ info, int B,
                                                        K* __restrict__ keys, uint32_t* __restrict__ vals) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t m = edge_mask_of(cases[i]);
    if (!m) return;
    uint64_t r = offsets[i] >> 32;
    const int64_t x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
    while (m) {
        const int e = __ffs(m) - 1;
        m &= m - 1;
        const int a = mc::edge_a(e), b = mc::edge_b(e);
        const uint64_t p = pack_point(x + min(mc::corner_dx(a), mc::corner_dx(b)),
                                      y + min(mc::corner_dy(a), mc::corner_dy(b)),
                                      z + min(mc::corner_dz(a), mc::corner_dz(b)), info, B);
        keys[r] = (K)((p << 2) | (uint64_t)mc::edge_axis(e));
        vals[r] = (uint32_t)(i * 16 + e);
        ++r;
    }
}

// 1 where sorted position s starts a run of equal keys (read by the id scan).
template <typename K>
struct RunStart {
    const K* keys;
    __host__ __device__ uint32_t operator()(int64_t s) const { return (s == 0 || keys[s - 1] != keys[s]) ? 1u : 0u; }
};

// Raw vertex slot of edge e in cell i: the cell's first slot + the crossing edges below e.
__device__ __forceinline__ uint32_t raw_slot(uint64_t offset, uint32_t mask, int e) {
    return (uint32_t)(offset >> 32) + (uint32_t)__popc(mask & ((1u << e) - 1u));
}

// Vertex on edge e of cell i.
// include/gpu/spcumc.cuh:455-471: t = (iso - va) / (vb - va) clamped to [0, 1] (0.5
// on a flat edge), p = pA + t (pB - pA); t (pB - pA) is exact for lattice points
__device__ __forceinline__ void store_vertex(const int32_t* __restrict__ coords, const float* __restrict__ corners,
                                             int64_t i, int e, float iso, float* __restrict__ out) {
    const int a = mc::edge_a(e), b = mc::edge_b(e);
    const float va = corners[8 * i + a], vb = corners[8 * i + b];
    const float denom = vb - va;
    float t;
    if (fabsf(denom) < 1e-30f) {
        t = 0.5f;
    } else {
        t = (iso - va) / denom;
        t = fminf(fmaxf(t, 0.0f), 1.0f);
    }
    const int64_t x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
    const float ax = (float)(x + mc::corner_dx(a)), ay = (float)(y + mc::corner_dy(a)),
                az = (float)(z + mc::corner_dz(a));
    const float bx = (float)(x + mc::corner_dx(b)), by = (float)(y + mc::corner_dy(b)),
                bz = (float)(z + mc::corner_dz(b));
    out[0] = ax + t * (bx - ax);
    out[1] = ay + t * (by - ay);
    out[2] = az + t * (bz - az);
}

template <typename K>
__global__ __launch_bounds__(kBlock) void smc_vertices(const K* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                       const uint32_t* __restrict__ ids, int64_t m,
                                                       const int32_t* __restrict__ coords,
                                                       const float* __restrict__ corners,
                                                       const uint8_t* __restrict__ cases,
                                                       const uint64_t* __restrict__ offsets, float iso,
                                                       float* __restrict__ verts, int32_t* __restrict__ map) {
    const int64_t s = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (s >= m) return;
    const uint32_t id = ids[s] - 1u;
    const uint32_t v = vals[s];
    const int64_t i = v >> 4;
    const int e = (int)(v & 15u);
    map[raw_slot(offsets[i], edge_mask_of(cases[i]), e)] = (int32_t)id;
    if (s > 0 && keys[s - 1] == keys[s]) return;
    store_vertex(coords, corners, i, e, iso, verts + 3 * (int64_t)id);
}

__global__ __launch_bounds__(kBlock) void smc_triangles(const uint8_t* __restrict__ cases,
                                                        const uint64_t* __restrict__ offsets, int64_t n,
                                                        const int32_t* __restrict__ map,
                                                        int32_t* __restrict__ tris) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = cases[i];
    const uint64_t packed = c_triangles[c];
    const int nt = mc::triangle_count(packed);
    if (!nt) return;
    const uint32_t mask = edge_mask_of(c);
    const uint64_t off = offsets[i];
    int32_t* o = tris + 3 * (int64_t)(uint32_t)off;
    for (int t = 0; t < nt; ++t) {
        const int e0 = mc::triangle_edge(packed, 3 * t), e1 = mc::triangle_edge(packed, 3 * t + 1),
                  e2 = mc::triangle_edge(packed, 3 * t + 2);
        o[3 * t] = map[raw_slot(off, mask, e0)];
        o[3 * t + 1] = map[raw_slot(off, mask, e2)];
        o[3 * t + 2] = map[raw_slot(off, mask, e1)];
    }
}

// ---- ascending cells: no sort
// The cells' bounding lattice, one cell wider on every side: bits[w] holds a bit per cell
// of 32 along z, before[w] the cells in the words below w.
struct Lattice {
    int32_t mn[3];
    int32_t ny, zw;  // rows per x, words per row
    const uint32_t* bits;
    const uint32_t* before;
};

// Row of (x, y) and place along z, x .. z within one cell of the bounds.
__device__ __forceinline__ uint32_t lattice_row(const Lattice& L, int64_t x, int64_t y) {
    return (uint32_t)(x - L.mn[0] + 1) * (uint32_t)L.ny + (uint32_t)(y - L.mn[1] + 1);
}
__device__ __forceinline__ uint32_t lattice_z(const Lattice& L, int64_t z) { return (uint32_t)(z - L.mn[2] + 1); }

// Cells before place z of a row, whether that place holds one, and whether the next does.
struct Place {
    uint32_t at;
    bool here, next;
};
__device__ __forceinline__ Place place_of(const Lattice& L, uint32_t row, uint32_t z) {
    const uint32_t w = row * (uint32_t)L.zw + (z >> 5), b = z & 31u, m = L.bits[w];
    Place p;
    p.at = L.before[w] + (uint32_t)__popc(m & ((1u << b) - 1u));
    p.here = (m >> b) & 1u;
    p.next = b < 31u ? (m >> (b + 1u)) & 1u : (z + 1u < 32u * (uint32_t)L.zw ? L.bits[w + 1] & 1u : 0u);
    return p;
}

// A cell's edges as 4 bits per axis (x, y, z from the least significant): bit u + 2 v for
// the edge whose lowest point lies (u, v) along the other two axes in their order.
__host__ __device__ constexpr int edge_bit(int e) {
    const int a = mc::edge_a(e), b = mc::edge_b(e), axis = mc::edge_axis(e);
    const int x = mc::corner_dx(a) & mc::corner_dx(b), y = mc::corner_dy(a) & mc::corner_dy(b),
              z = mc::corner_dz(a) & mc::corner_dz(b);
    return 4 * axis + (axis == 0 ? y : x) + 2 * (axis == 2 ? y : z);
}
// Edge bits of the 12 edges, and edges of the 12 bits, 4 bits each.
constexpr uint64_t edge_table(bool inverse) {
    uint64_t t = 0;
    for (int e = 0; e < 12; ++e) t |= (uint64_t)(inverse ? e : edge_bit(e)) << (4 * (inverse ? edge_bit(e) : e));
    return t;
}
constexpr uint64_t kBitOfEdge = edge_table(false), kEdgeOfBit = edge_table(true);
__device__ __forceinline__ int nibble(uint64_t table, int k) { return (int)((table >> (4 * k)) & 15u); }
__device__ __forceinline__ uint32_t bits_below(uint32_t m, int k) { return (uint32_t)__popc(m & ((1u << k) - 1u)); }

// Streams s = dx + 2 dy, and the edges whose lowest point is at dz = 0 / 1.
__device__ __forceinline__ uint32_t stream_mask(int s) { return s == 0 ? 0x155u : s == 1 ? 0x2a0u : s == 2 ? 0x40au : 0x800u; }
constexpr uint32_t kLowZ = 0xf33u, kHighZ = 0x0ccu;

// Owned edges per stream before a cell: `base` before its block of kBlock cells, and four
// 16-bit counts inside the block (at most 5 kBlock each).
static_assert(5 * kBlock < 1 << 16, "block counts fit 16 bits");
struct OwnSums {
    const uint4* base;
    const uint64_t* local;
};
__device__ __forceinline__ uint32_t own_before(const OwnSums& t, uint32_t cell, int s) {
    const uint32_t* b = reinterpret_cast<const uint32_t*>(t.base + cell / kBlock);
    return b[s] + (uint32_t)((t.local[cell] >> (16 * s)) & 0xffffu);
}
struct WordCells {
    const uint32_t* bits;
    __device__ uint32_t operator()(int64_t w) const { return (uint32_t)__popc(bits[w]); }
};

__global__ __launch_bounds__(kBlock) void smc_clear(uint32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// The first cell of each word writes the word.
__global__ __launch_bounds__(kBlock) void smc_mark(const int32_t* __restrict__ coords, int64_t n, Lattice L,
                                                   uint32_t* __restrict__ bits) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    auto word = [&](int64_t j, uint32_t& b) {
        const uint32_t z = lattice_z(L, coords[3 * j + 2]);
        b = z & 31u;
        return lattice_row(L, coords[3 * j], coords[3 * j + 1]) * (uint32_t)L.zw + (z >> 5);
    };
    uint32_t b, u;
    const uint32_t w = word(i, b);
    if (i > 0 && word(i - 1, u) == w) return;
    uint32_t m = 1u << b;
    for (int64_t j = i + 1; j < n && word(j, u) == w; ++j) m |= 1u << u;
    bits[w] = m;
}

// Corner means: the up to eight cells around a lattice point in ascending order.
__global__ __launch_bounds__(kBlock) void smc_dense_mean(const int32_t* __restrict__ coords, int64_t n, Lattice L,
                                                         const float* __restrict__ corners, float* __restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (j >= 8 * n) return;
    const int64_t i = j >> 3;
    const int k = (int)(j & 7);
    const int64_t x = (int64_t)coords[3 * i] + mc::corner_dx(k), y = (int64_t)coords[3 * i + 1] + mc::corner_dy(k),
                  z = (int64_t)coords[3 * i + 2] + mc::corner_dz(k);
    double sum = 0.0;
    int cnt = 0;
    for (int dx = 1; dx >= 0; --dx)
        for (int dy = 1; dy >= 0; --dy) {
            const Place p = place_of(L, lattice_row(L, x - dx, y - dy), lattice_z(L, z - 1));
            const int c = dy ? (dx ? 2 : 3) : dx;  // the point's corner of a cell at dz = 0
            if (p.here) {
                sum += (double)corners[8 * (int64_t)p.at + 4 + c];
                ++cnt;
            }
            if (p.next) {
                sum += (double)corners[8 * ((int64_t)p.at + p.here) + c];
                ++cnt;
            }
        }
    out[j] = (float)(sum / (double)cnt);
}

// own[i]: the edge bits of cell i that no earlier cell has; ref of each raw slot (a cell's
// edges by edge bit, from its first slot on): the owner's slot; local and block: the owned
// edges per stream, of the cells before in the block and of the whole block.
__global__ __launch_bounds__(kBlock) void smc_own_edges(const int32_t* __restrict__ coords,
                                                        const uint8_t* __restrict__ cases,
                                                        const uint64_t* __restrict__ offsets, int64_t n, Lattice L,
                                                        uint16_t* __restrict__ own, uint32_t* __restrict__ ref,
                                                        uint64_t* __restrict__ local, uint4* __restrict__ block) {
    __shared__ uint16_t bits_of[256];  // edge bits of every case
    __shared__ uint64_t wave_sum[kBlock / 64];
    static_assert(kBlock == 256, "one case per thread");
    uint32_t of = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e)
        of |= (((threadIdx.x >> mc::edge_a(e)) ^ (threadIdx.x >> mc::edge_b(e))) & 1u) << edge_bit(e);
    bits_of[threadIdx.x] = (uint16_t)of;
    __syncthreads();
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    uint32_t m = 0;
    if (i < n) {
        const uint32_t mask = bits_of[cases[i]];
        m = mask;
        if (m) {
            const uint32_t slot = (uint32_t)(offsets[i] >> 32);
            const int64_t x = coords[3 * i], y = coords[3 * i + 1];
            const uint32_t z = lattice_z(L, coords[3 * i + 2]);
            // the edges of `shared` that cell j has too, as its edge bits `shift` higher
            auto claim = [&](uint32_t j, int shift, uint32_t shared) {
                const uint32_t nb = bits_of[cases[j]];
                uint32_t t = m & shared & (shift > 0 ? nb >> shift : nb << -shift);
                if (!t) return;
                m &= ~t;
                const uint32_t first = (uint32_t)(offsets[j] >> 32);
                for (; t; t &= t - 1) {
                    const int k = __ffs(t) - 1;
                    ref[slot + bits_below(mask, k)] = first + bits_below(nb, k + shift);
                }
            };
            // the earlier cells that share edges, in their order
            uint32_t r = lattice_row(L, x - 1, y - 1);
            Place p = place_of(L, r, z);
            if (p.here) claim(p.at, 3, 0x100u);   // one z edge
            r = lattice_row(L, x - 1, y);
            p = place_of(L, r, z - 1);
            const bool top = (L.bits[r * (uint32_t)L.zw + ((z + 1) >> 5)] >> ((z + 1) & 31u)) & 1u;
            if (p.here) claim(p.at, 3, 0x010u);   // one y edge
            if (p.next) claim(p.at + p.here, 1, 0x550u);  // a face: y and z edges at dx = 0
            if (top) claim(p.at + p.here + p.next, -1, 0x040u);
            p = place_of(L, lattice_row(L, x - 1, y + 1), z);
            if (p.here) claim(p.at, -1, 0x400u);
            r = lattice_row(L, x, y - 1);
            p = place_of(L, r, z - 1);
            const bool top2 = (L.bits[r * (uint32_t)L.zw + ((z + 1) >> 5)] >> ((z + 1) & 31u)) & 1u;
            if (p.here) claim(p.at, 3, 0x001u);   // one x edge
            if (p.next) {                         // a face: x and z edges at dy = 0
                claim(p.at + p.here, 1, 0x005u);
                claim(p.at + p.here, 2, 0x300u);
            }
            if (top2) claim(p.at + p.here + p.next, -1, 0x004u);
            p = place_of(L, lattice_row(L, x, y), z - 1);
            if (p.here) claim(p.at, 2, 0x033u);   // a face: x and y edges at dz = 0
            for (uint32_t t = m; t; t &= t - 1) {
                const uint32_t k = slot + bits_below(mask, __ffs(t) - 1);
                ref[k] = k;
            }
        }
        own[i] = (uint16_t)m;
    }
    uint64_t sum = 0;
#pragma unroll
    for (int s = 0; s < 4; ++s) sum |= (uint64_t)__popc(m & stream_mask(s)) << (16 * s);
    const uint64_t mine = sum;
    const int lane = (int)(threadIdx.x & 63);
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t u = __shfl_up((unsigned long long)sum, o);
        if (lane >= o) sum += u;
    }
    if (lane == 63) wave_sum[threadIdx.x >> 6] = sum;
    __syncthreads();
    for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) sum += wave_sum[w];
    if (i <= n) local[i] = sum - mine;
    if (threadIdx.x == kBlock - 1)
        block[blockIdx.x] = make_uint4((uint32_t)(sum & 0xffffu), (uint32_t)((sum >> 16) & 0xffffu),
                                       (uint32_t)((sum >> 32) & 0xffffu), (uint32_t)(sum >> 48));
}

// base[b]: the sums of the blocks before b, b = 0 .. nb, by one workgroup: a run of blocks
// per thread.
constexpr int kBaseBlock = 1024;
__global__ __launch_bounds__(kBaseBlock) void smc_own_base(const uint4* __restrict__ block, int64_t nb,
                                                           uint4* __restrict__ base) {
    __shared__ uint32_t wave_sum[4][kBaseBlock / 64];
    const int64_t run = (nb + kBaseBlock - 1) / kBaseBlock;
    const int64_t b0 = min((int64_t)threadIdx.x * run, nb), b1 = min(b0 + run, nb);
    uint32_t t[4] = {0u, 0u, 0u, 0u};
    for (int64_t b = b0; b < b1; ++b) {
        const uint4 v = block[b];
        t[0] += v.x;
        t[1] += v.y;
        t[2] += v.z;
        t[3] += v.w;
    }
    const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6);
    uint32_t at[4];
    for (int k = 0; k < 4; ++k) {
        uint32_t sum = t[k];
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = __shfl_up(sum, o);
            if (lane >= o) sum += u;
        }
        if (lane == 63) wave_sum[k][w] = sum;
        at[k] = sum - t[k];
    }
    __syncthreads();
    for (int k = 0; k < 4; ++k)
        for (int j = 0; j < w; ++j) at[k] += wave_sum[k][j];
    for (int64_t b = b0; b < b1; ++b) {
        const uint4 v = block[b];
        base[b] = make_uint4(at[0], at[1], at[2], at[3]);
        at[0] += v.x;
        at[1] += v.y;
        at[2] += v.z;
        at[3] += v.w;
    }
    if (threadIdx.x == kBaseBlock - 1) base[nb] = make_uint4(at[0], at[1], at[2], at[3]);
}

// Number of the vertex of the edge along `axis` from lattice point (x, y, z).
__device__ __forceinline__ uint32_t vertex_number(const Lattice& L, const uint16_t* __restrict__ own,
                                                  const OwnSums& sums, int64_t x, int64_t y, int64_t z, int axis) {
    const uint32_t lower = (1u << (4 * axis)) - 1u;  // the axes before
    uint32_t id = 0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const Place p = place_of(L, lattice_row(L, x - (s & 1), y - (s >> 1)), lattice_z(L, z - 1));
        id += own_before(sums, p.at, s);
        if (p.here) id += (uint32_t)__popc(own[p.at] & stream_mask(s) & (kLowZ | (kHighZ & lower)));
        if (p.next) id += (uint32_t)__popc(own[p.at + p.here] & stream_mask(s) & kLowZ & lower);
    }
    return id;
}

// A thread per cell: the vertices of the edges it owns, and their numbers at their slots.
__global__ __launch_bounds__(kBlock) void smc_own_vertices(const int32_t* __restrict__ coords,
                                                           const float* __restrict__ corners,
                                                           const uint8_t* __restrict__ cases,
                                                           const uint64_t* __restrict__ offsets, int64_t n, Lattice L,
                                                           const uint16_t* __restrict__ own, OwnSums sums, float iso,
                                                           float* __restrict__ verts, int32_t* __restrict__ map) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t mine = own[i];
    if (!mine) return;
    uint32_t mask = 0;
    const uint32_t c = cases[i], slot = (uint32_t)(offsets[i] >> 32);
#pragma unroll
    for (int e = 0; e < 12; ++e) mask |= (((c >> mc::edge_a(e)) ^ (c >> mc::edge_b(e))) & 1u) << edge_bit(e);
    const int64_t x = coords[3 * i], y = coords[3 * i + 1], z = coords[3 * i + 2];
    for (uint32_t m = mine; m; m &= m - 1) {
        const int k = __ffs(m) - 1, axis = k >> 2, u = k & 1, v = (k >> 1) & 1;
        const uint32_t id = vertex_number(L, own, sums, x + (axis == 0 ? 0 : u), y + (axis == 0 ? u : axis == 2 ? v : 0),
                                          z + (axis == 2 ? 0 : v), axis);
        map[slot + bits_below(mask, k)] = (int32_t)id;
        store_vertex(coords, corners, i, nibble(kEdgeOfBit, k), iso, verts + 3 * (int64_t)id);
    }
}

__global__ __launch_bounds__(kBlock) void smc_own_triangles(const uint8_t* __restrict__ cases,
                                                            const uint64_t* __restrict__ offsets, int64_t n,
                                                            const uint32_t* __restrict__ ref,
                                                            const int32_t* __restrict__ map, int32_t* __restrict__ tris) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t c = cases[i];
    const uint64_t packed = c_triangles[c];
    const int nt = mc::triangle_count(packed);
    if (!nt) return;
    uint32_t mask = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e) mask |= (((c >> mc::edge_a(e)) ^ (c >> mc::edge_b(e))) & 1u) << edge_bit(e);
    const uint64_t off = offsets[i];
    const uint32_t* r = ref + (uint32_t)(off >> 32);
    auto vertex = [&](int j) { return map[r[bits_below(mask, nibble(kBitOfEdge, mc::triangle_edge(packed, j)))]]; };
    int32_t* o = tris + 3 * (int64_t)(uint32_t)off;
    for (int t = 0; t < nt; ++t) {
        o[3 * t] = vertex(3 * t);
        o[3 * t + 1] = vertex(3 * t + 2);
        o[3 * t + 2] = vertex(3 * t + 1);
    }
}

int bits_for(int64_t span) {  // bits to hold 0..span
    int b = 1;
    while (((int64_t)1 << b) <= span) ++b;
    return b;
}

}  // namespace

// Scratch of the extractions on one device, kept between calls and grown when a larger
// one arrives, so that steady-state calls allocate nothing: region A holds the per-cell
// arrays, region B the per-edge arrays (sized once the edge count is known).  One
// extraction at a time owns it (from smc_extract to smc_release); a concurrent one
// allocates its own blocks from the stream-ordered pool.  The next owner's stream waits
// for the event the previous owner recorded at release.
struct Region {
    char* base = nullptr;
    size_t cap = 0;
};

struct DeviceScratch {
    std::mutex mu;
    bool busy = false;
    Region a, b;
    hipEvent_t done = nullptr;
    uint64_t* readback = nullptr;  // pinned host words for the small readbacks
};

namespace {

constexpr int kScratchDevices = 64;
DeviceScratch g_scratch[kScratchDevices];

size_t align_up(size_t b) { return (b + 255) & ~(size_t)255; }

// Bump allocation over one block; with base == nullptr it only measures.
struct Carve {
    char* base = nullptr;
    size_t used = 0;
    template <typename T>
    T* take(int64_t count) {
        T* p = base ? reinterpret_cast<T*>(base + used) : nullptr;
        used += align_up((size_t)std::max<int64_t>(count, 1) * sizeof(T));
        return p;
    }
};

hipError_t reserve(Region& r, size_t need) {
    if (need <= r.cap) return hipSuccess;
    if (r.base) {
        hipError_t e = hipFree(r.base);  // synchronizes the device: nothing uses the old block
        r.base = nullptr;
        r.cap = 0;
        if (e != hipSuccess) return e;
    }
    need += need / 4;
    hipError_t e = hipMalloc((void**)&r.base, need);
    if (e != hipSuccess) {
        r.base = nullptr;
        return e;
    }
    r.cap = need;
    return hipSuccess;
}

}  // namespace

// State of one extraction between its two phases.
struct SmcState {
    int64_t n = 0, m_raw = 0, m = 0, t = 0;
    float iso = 0.0f;
    bool wide = false;  // 64-bit edge keys (more than 32 key bits)
    const int32_t* coords = nullptr;
    const float* corners = nullptr;  // the caller's, or the averaged copy
    int device = -1;
    DeviceScratch* shared = nullptr;  // the device's scratch, or null for private blocks
    std::vector<void*> blocks;        // private blocks (stream-ordered)
    int32_t* info = nullptr;          // [0..5] bounds, [8..9] totals (uint64)
    uint8_t* cases = nullptr;
    uint64_t* offsets = nullptr;
    void* keys = nullptr;      // sorted edge keys (uint32 or uint64)
    uint32_t* vals = nullptr;  // sorted (cell, edge)
    uint32_t* ids = nullptr;   // vertex id + 1 per sorted position
    int32_t* map = nullptr;    // raw slot -> vertex id
    // ascending cells
    bool dense = false;
    Lattice lattice = {};
    uint16_t* own = nullptr;   // edge bits owned
    uint32_t* ref = nullptr;   // raw slot -> the owner's raw slot
    uint64_t* local = nullptr;
    uint4* block = nullptr;
    uint4* base = nullptr;
};

namespace {

SmcStatus hip_status(hipError_t e, const char* what) {
    SmcStatus st;
    if (e != hipSuccess) {
        st.code = -2;
        st.message = std::string(what) + ": " + hipGetErrorString(e);
    }
    return st;
}

// A block of `bytes` for region `which` (0 = A, 1 = B): the shared scratch, or a private
// stream-ordered allocation.
hipError_t region(SmcState* st, int which, size_t bytes, hipStream_t s, char** out) {
    if (st->shared) {
        Region& r = which == 0 ? st->shared->a : st->shared->b;
        hipError_t e = reserve(r, bytes);
        *out = r.base;
        return e;
    }
    void* q = nullptr;
    hipError_t e = hipMallocAsync(&q, std::max<size_t>(bytes, 1), s);
    if (e != hipSuccess) return e;
    st->blocks.push_back(q);
    *out = (char*)q;
    return hipSuccess;
}

template <typename K>
size_t sort_bytes(int64_t m) {
    size_t b = 0;
    hipcub::DeviceRadixSort::SortPairs(nullptr, b, (const K*)nullptr, (K*)nullptr, (const uint32_t*)nullptr,
                                       (uint32_t*)nullptr, (int)m, 0, (int)(8 * sizeof(K)));
    return b;
}

template <typename K>
using StartIter = hipcub::TransformInputIterator<uint32_t, RunStart<K>, hipcub::CountingInputIterator<int64_t>>;

template <typename K>
size_t id_scan_bytes(int64_t m) {
    size_t b = 0;
    StartIter<K> it(hipcub::CountingInputIterator<int64_t>(0), RunStart<K>{nullptr});
    hipcub::DeviceScan::InclusiveSum(nullptr, b, it, (uint32_t*)nullptr, (int)m);
    return b;
}

// Corner means: keys of the 8 n corners, stable sort, run means into `mean`.
template <typename K>
hipError_t average_corners(SmcState* st, Carve& c, int B, float* mean, hipStream_t s) {
    const int64_t m = 8 * st->n;
    K* ck = c.take<K>(m);
    uint32_t* cv = c.take<uint32_t>(m);
    K* ck2 = c.take<K>(m);
    uint32_t* cv2 = c.take<uint32_t>(m);
    size_t bytes = sort_bytes<K>(m);
    char* tmp = c.take<char>((int64_t)bytes);
    hipLaunchKernelGGL(smc_corner_keys<K>, dim3(blocks_for(m)), dim3(kBlock), 0, s, st->coords, st->n, st->info, B,
                       ck, cv);
    hipError_t e = hipcub::DeviceRadixSort::SortPairs(tmp, bytes, ck, ck2, cv, cv2, (int)m, 0, 3 * B, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(smc_corner_mean<K>, dim3(blocks_for(m)), dim3(kBlock), 0, s, ck2, cv2, m, st->corners, mean);
    return hipGetLastError();
}

// Region B: edge keys in cell order, their stable sort, the vertex ids (inclusive scan
// of run starts) and the raw -> vertex map used by the triangles.
template <typename K>
hipError_t order_edges(SmcState* st, int B, hipStream_t s) {
    const int64_t m = st->m_raw;
    const size_t sbytes = sort_bytes<K>(m), ibytes = id_scan_bytes<K>(m);
    auto lay = [&](Carve& c, K** k1, K** k2, uint32_t** v1, uint32_t** v2, char** t1, char** t2) {
        *k1 = c.take<K>(m);
        *k2 = c.take<K>(m);
        *v1 = c.take<uint32_t>(m);
        *v2 = c.take<uint32_t>(m);
        st->ids = c.take<uint32_t>(m);
        st->map = c.take<int32_t>(m);
        *t1 = c.take<char>((int64_t)sbytes);
        *t2 = c.take<char>((int64_t)ibytes);
    };
    K *k1, *k2;
    uint32_t *v1, *v2;
    char *t1, *t2;
    Carve size;
    lay(size, &k1, &k2, &v1, &v2, &t1, &t2);
    Carve c;
    hipError_t e = region(st, 1, size.used, s, &c.base);
    if (e != hipSuccess) return e;
    lay(c, &k1, &k2, &v1, &v2, &t1, &t2);
    hipLaunchKernelGGL(smc_edge_keys<K>, dim3(blocks_for(st->n)), dim3(kBlock), 0, s, st->coords, st->cases,
                       st->offsets, st->n, st->info, B, k1, v1);
    size_t bytes = sbytes;
    e = hipcub::DeviceRadixSort::SortPairs(t1, bytes, k1, k2, v1, v2, (int)m, 0, 3 * B + 2, s);
    if (e != hipSuccess) return e;
    st->keys = k2;
    st->vals = v2;
    StartIter<K> starts(hipcub::CountingInputIterator<int64_t>(0), RunStart<K>{k2});
    bytes = ibytes;
    return hipcub::DeviceScan::InclusiveSum(t2, bytes, starts, st->ids, (int)m, s);
}

template <typename K>
void launch_vertices(const SmcState* st, float* verts, hipStream_t s) {
    hipLaunchKernelGGL(smc_vertices<K>, dim3(blocks_for(st->m_raw)), dim3(kBlock), 0, s, (const K*)st->keys,
                       st->vals, st->ids, st->m_raw, st->coords, st->corners, st->cases, st->offsets, st->iso, verts,
                       st->map);
}

// Words of the bounding lattice's bits up to which ascending cells go without the sort (a
// word costs some 12 bytes of traffic, the sort's passes over a cell's edges about 300).
int64_t dense_words_most(int64_t n) { return std::min<int64_t>(8 * n + (1 << 14), INT32_MAX); }

using WordIter = hipcub::TransformInputIterator<uint32_t, WordCells, hipcub::CountingInputIterator<int64_t>>;

size_t word_scan_bytes(int64_t words) {
    size_t b = 0;
    WordIter it(hipcub::CountingInputIterator<int64_t>(0), WordCells{nullptr});
    hipcub::DeviceScan::ExclusiveSum(nullptr, b, it, (uint32_t*)nullptr, (int)words);
    return b;
}

// Region B of ascending cells (with the arrays per edge where m_raw is known), and their
// lattice's bits and prefix counts.
hipError_t dense_lattice(SmcState* st, int64_t words, hipStream_t s) {
    const int64_t n = st->n, nb = n / kBlock + 1;
    const size_t wbytes = word_scan_bytes(words);
    uint32_t *bits, *before;
    char* tmp;
    auto lay = [&](Carve& c) {
        bits = c.take<uint32_t>(words);
        before = c.take<uint32_t>(words);
        st->own = c.take<uint16_t>(n);
        st->local = c.take<uint64_t>(n + 1);
        st->block = c.take<uint4>(nb);
        st->base = c.take<uint4>(nb + 1);
        tmp = c.take<char>((int64_t)wbytes);
        if (st->m_raw > 0) {
            st->ref = c.take<uint32_t>(st->m_raw);
            st->map = c.take<int32_t>(st->m_raw);
        }
    };
    Carve size;
    lay(size);
    Carve c;
    hipError_t e = region(st, 1, size.used, s, &c.base);
    if (e != hipSuccess) return e;
    lay(c);
    st->lattice.bits = bits;
    st->lattice.before = before;
    hipLaunchKernelGGL(smc_clear, dim3(blocks_for(words)), dim3(kBlock), 0, s, bits, words);
    hipLaunchKernelGGL(smc_mark, dim3(blocks_for(n)), dim3(kBlock), 0, s, st->coords, n, st->lattice, bits);
    WordIter it(hipcub::CountingInputIterator<int64_t>(0), WordCells{bits});
    size_t bytes = wbytes;
    return hipcub::DeviceScan::ExclusiveSum(tmp, bytes, it, before, (int)words, s);
}

// The owned edges of ascending cells (classified) and their sums.
hipError_t dense_edges(SmcState* st, hipStream_t s) {
    const int64_t n = st->n, nb = n / kBlock + 1;
    hipLaunchKernelGGL(smc_own_edges, dim3((unsigned)nb), dim3(kBlock), 0, s, st->coords, st->cases, st->offsets, n,
                       st->lattice, st->own, st->ref, st->local, st->block);
    hipLaunchKernelGGL(smc_own_base, dim3(1), dim3(kBaseBlock), 0, s, st->block, nb, st->base);
    return hipGetLastError();
}

// Copies `bytes` from the device once the stream's work is done (through pinned memory
// when the extraction owns the shared scratch).
hipError_t read_back(SmcState* st, const void* src, size_t bytes, void* dst, hipStream_t s) {
    void* host = dst;
    if (st->shared && st->shared->readback) host = st->shared->readback;
    hipError_t e = hipMemcpyAsync(host, src, bytes, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e == hipSuccess && host != dst) std::memcpy(dst, host, bytes);
    return e;
}

}  // namespace

void smc_release(SmcState* st, hipStream_t s) {
    if (!st) return;
    for (void* p : st->blocks) (void)hipFreeAsync(p, s);
    if (st->shared) {
        std::lock_guard<std::mutex> lock(st->shared->mu);
        if (!st->shared->done) (void)hipEventCreateWithFlags(&st->shared->done, hipEventDisableTiming);
        if (st->shared->done) (void)hipEventRecord(st->shared->done, s);
        st->shared->busy = false;
    }
    delete st;
}

SmcStatus smc_extract(const int32_t* coords, const float* corners, int64_t n, float iso, bool consistent,
                      hipStream_t s, SmcState** out, int64_t* n_verts, int64_t* n_tris) {
    *out = nullptr;
    *n_verts = *n_tris = 0;
    SmcState* st = new SmcState();
    st->n = n;
    st->iso = iso;
    st->coords = coords;
    st->corners = corners;
    auto bail = [&](SmcStatus r) {
        smc_release(st, s);
        return r;
    };
    auto arg_error = [&](const std::string& msg) {
        SmcStatus r;
        r.code = -1;
        r.message = msg;
        return bail(r);
    };
    if (n == 0) {
        *out = st;
        return SmcStatus();
    }
    hipError_t e = hipGetDevice(&st->device);
    if (e != hipSuccess) return bail(hip_status(e, "hipGetDevice"));
    if (st->device >= 0 && st->device < kScratchDevices) {
        DeviceScratch& d = g_scratch[st->device];
        std::lock_guard<std::mutex> lock(d.mu);
        if (!d.busy) {
            d.busy = true;
            st->shared = &d;
            if (!d.readback) (void)hipHostMalloc((void**)&d.readback, 64, hipHostMallocDefault);
            if (d.done) e = hipStreamWaitEvent(s, d.done, 0);
        }
    }
    if (e != hipSuccess) return bail(hip_status(e, "hipStreamWaitEvent"));

    // region A: per-cell arrays (and the corner averaging, sized for 64-bit keys)
    const unsigned nb = std::min<unsigned>(blocks_for(n), 1024);
    size_t scan_bytes = 0;
    hipcub::DeviceScan::ExclusiveSum(nullptr, scan_bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr, (int)n);
    int32_t* part = nullptr;
    uint64_t* counts = nullptr;
    float* mean = nullptr;
    char* scan_tmp = nullptr;
    Carve corner_area;
    auto lay_a = [&](Carve& c) {
        st->info = c.take<int32_t>(16);
        part = c.take<int32_t>(kBounds * (int64_t)nb);
        st->cases = c.take<uint8_t>(n);
        counts = c.take<uint64_t>(n);
        st->offsets = c.take<uint64_t>(n);
        scan_tmp = c.take<char>((int64_t)scan_bytes);
        if (consistent) {
            mean = c.take<float>(8 * n);
            corner_area.base = c.base ? c.base + c.used : nullptr;
            const size_t need = 2 * align_up(8 * n * sizeof(uint64_t)) + 2 * align_up(8 * n * sizeof(uint32_t)) +
                                align_up(std::max(sort_bytes<uint64_t>(8 * n), sort_bytes<uint32_t>(8 * n)));
            c.take<char>((int64_t)need);
        }
    };
    Carve size_a;
    lay_a(size_a);
    Carve ca;
    e = region(st, 0, size_a.used, s, &ca.base);
    if (e != hipSuccess) return bail(hip_status(e, "scratch allocation"));
    lay_a(ca);

    // bounds of the cell coordinates
    hipLaunchKernelGGL(smc_bounds, dim3(nb), dim3(kBlock), 0, s, coords, n, part);
    hipLaunchKernelGGL(smc_fold_bounds, dim3(1), dim3(kBlock), 0, s, part, (int)nb, st->info);
    int32_t info[10];
    int B = 0;
    auto read_bounds = [&]() -> SmcStatus {
        int64_t span = 0;
        for (int k = 0; k < 3; ++k) span = std::max<int64_t>(span, (int64_t)info[3 + k] - info[k]);
        if (span > kSmcMaxSpan) {
            SmcStatus r;
            r.code = -1;
            r.message = "cell coordinates span " + std::to_string(span) + " lattice steps on one axis; at most " +
                        std::to_string(kSmcMaxSpan) + " are supported";
            return r;
        }
        B = bits_for(span + 1);  // lattice points min .. max + 1
        return SmcStatus();
    };
    // ascending cells whose bounding lattice is dense enough need no sort
    auto try_dense = [&]() {
        const int64_t nx = (int64_t)info[3] - info[0] + 3, ny = (int64_t)info[4] - info[1] + 3,
                      zw = ((int64_t)info[5] - info[2] + 3 + 31) / 32;
        const int64_t most = dense_words_most(n);
        if (info[6] != 0 || nx * ny > most || nx * ny * zw > most) return hipSuccess;
        st->dense = true;
        for (int k = 0; k < 3; ++k) st->lattice.mn[k] = info[k];
        st->lattice.ny = (int32_t)ny;
        st->lattice.zw = (int32_t)zw;
        return dense_lattice(st, nx * ny * zw, s);
    };
    if (consistent) {
        // the corners' means need the lattice or the key width before the cells are classified
        e = read_back(st, st->info, kBounds * sizeof(int32_t), info, s);
        if (e != hipSuccess) return bail(hip_status(e, "cell bounds"));
        SmcStatus r = read_bounds();
        if (r.code) return bail(r);
        e = try_dense();
        if (e != hipSuccess) return bail(hip_status(e, "cell lattice"));
        if (st->dense) {
            // the corner sort's room holds the arrays per edge
            st->ref = corner_area.take<uint32_t>(12 * n);
            st->map = corner_area.take<int32_t>(12 * n);
            hipLaunchKernelGGL(smc_dense_mean, dim3(blocks_for(8 * n)), dim3(kBlock), 0, s, coords, n, st->lattice, corners,
                               mean);
            e = hipGetLastError();
        } else {
            e = 3 * B <= 32 ? average_corners<uint32_t>(st, corner_area, B, mean, s)
                            : average_corners<uint64_t>(st, corner_area, B, mean, s);
        }
        if (e != hipSuccess) return bail(hip_status(e, "corner averaging"));
        st->corners = mean;
    }

    // cases and per-cell counts, their exclusive scan and the totals
    hipLaunchKernelGGL(smc_classify, dim3(blocks_for(n)), dim3(kBlock), 0, s, st->corners, n, iso, st->cases, counts);
    e = hipcub::DeviceScan::ExclusiveSum(scan_tmp, scan_bytes, counts, st->offsets, (int)n, s);
    if (e != hipSuccess) return bail(hip_status(e, "count scan"));
    uint64_t* totals = reinterpret_cast<uint64_t*>(st->info + 8);
    hipLaunchKernelGGL(smc_totals, dim3(1), dim3(64), 0, s, counts, st->offsets, n, totals);
    e = read_back(st, st->info, sizeof info, info, s);
    if (e != hipSuccess) return bail(hip_status(e, "bounds and totals"));
    if (!consistent) {
        SmcStatus r = read_bounds();
        if (r.code) return bail(r);
    }
    uint64_t tot = 0;
    std::memcpy(&tot, info + 8, sizeof tot);
    st->m_raw = (int64_t)(tot >> 32);
    st->t = (int64_t)(uint32_t)tot;
    if (st->m_raw >= (int64_t)INT32_MAX) return arg_error("more than 2^31 - 1 edge vertices");
    if (st->m_raw == 0) {
        *out = st;
        *n_tris = st->t;
        return SmcStatus();
    }

    if (!consistent) {
        e = try_dense();
        if (e != hipSuccess) return bail(hip_status(e, "cell lattice"));
    }
    if (st->dense) {
        e = dense_edges(st, s);
        if (e != hipSuccess) return bail(hip_status(e, "edge numbering"));
        uint4 all;
        e = read_back(st, st->base + (n / kBlock + 1), sizeof all, &all, s);
        if (e != hipSuccess) return bail(hip_status(e, "vertex count"));
        st->m = (int64_t)all.x + all.y + all.z + all.w;
        *out = st;
        *n_verts = st->m;
        *n_tris = st->t;
        return SmcStatus();
    }

    // region B: edge keys in cell order, stable sort, vertex ids from run starts
    st->wide = 3 * B + 2 > 32;
    e = st->wide ? order_edges<uint64_t>(st, B, s) : order_edges<uint32_t>(st, B, s);
    if (e != hipSuccess) return bail(hip_status(e, "edge ordering"));
    uint32_t m = 0;
    e = read_back(st, st->ids + (st->m_raw - 1), sizeof m, &m, s);
    if (e != hipSuccess) return bail(hip_status(e, "vertex count"));
    st->m = m;
    *out = st;
    *n_verts = st->m;
    *n_tris = st->t;
    return SmcStatus();
}

SmcStatus smc_write(SmcState* st, float* verts, int32_t* tris, hipStream_t s) {
    SmcStatus r;
    if (st->dense) {
        if (st->m > 0)
            hipLaunchKernelGGL(smc_own_vertices, dim3(blocks_for(st->n)), dim3(kBlock), 0, s, st->coords, st->corners, st->cases,
                               st->offsets, st->n, st->lattice, st->own, OwnSums{st->base, st->local}, st->iso, verts, st->map);
        if (st->t > 0)
            hipLaunchKernelGGL(smc_own_triangles, dim3(blocks_for(st->n)), dim3(kBlock), 0, s, st->cases, st->offsets, st->n,
                               st->ref, st->map, tris);
        r = hip_status(hipGetLastError(), "marching cubes kernel launch");
    } else if (st->m_raw > 0) {
        if (st->wide)
            launch_vertices<uint64_t>(st, verts, s);
        else
            launch_vertices<uint32_t>(st, verts, s);
        if (st->t > 0)
            hipLaunchKernelGGL(smc_triangles, dim3(blocks_for(st->n)), dim3(kBlock), 0, s, st->cases, st->offsets,
                               st->n, st->map, tris);
        r = hip_status(hipGetLastError(), "marching cubes kernel launch");
    }
    return r;
}

}  // namespace cubvh_amd
