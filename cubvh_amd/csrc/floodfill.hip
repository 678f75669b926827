// floodfill.hip -- 6-connected labelling of the free voxels of [B,H,W,D] grids.
//
// Replaces the reference's host-driven loop of hook and pointer-jump kernels
// (include/gpu/floodfill.cuh:157-272: up to ~500 iterations at 256^3, each with a
// device synchronization and a 4-byte copy back to the host) by a fixed sequence of
// three kernels with no host round trip, working in place in the output array:
//
//   1. tiles  : each workgroup labels one tile of 64 x 8 x 8 voxels (64 along the last
//               axis: one row per wave, a lane per voxel, so that occupancy is one ballot,
//               loads and stores are whole lines, and runs are bit arithmetic), or of
//               16 x 16 x 16, four rows per wave, where the last axis has at most 16 and the
//               grids are many or large.
//               Union-find in LDS between overlapping runs of neighbouring rows; every
//               free voxel gets the global index of its tile-local root, others -1.
//   2. merge  : voxels on a tile's low faces union themselves with their free
//               neighbour in the adjacent tile, one wave per face, whose pairs with the
//               same two labels are united once.  Union-find over the label
//               array: a node's parent is always a smaller index of the same component,
//               roots are linked smaller-under-larger with atomicMin and the link is
//               retried until it lands on a root, so concurrent unions never lose an
//               edge.
//   3. flatten: label[i] = root(i).  Since parents only ever point to smaller
//               indices, the root of each component is its minimum linear index.
//
// At 256^3 (a shell; 67 MB of labels, written, read at the faces, read and written): tiles
// 57 us, merge 66 us, flatten 21 us, bound by latency (chains of dependent loads of a few
// lanes) and for flatten by its 134 MB.  With tiles of 16^3 loaded a byte per lane, a
// union per row of every face and a root search per voxel these were 118, 287 and 54 us.
// A third of the voxels occupied at random: 760 -> 187 us; 64^3: 78 -> 38 us.
// Axes of one voxel do not matter to the labels: a last axis of 1 is dropped, so that the
// next one takes its place.
//
// The result equals the reference's converged output (the minimum linear index of
// each free component, -1 for occupied voxels, indices global across the batch)
// for cubic grids.  Connectivity is tensor-order (last axis fastest) for every grid
// shape; the reference decodes coordinates as if H == W == D.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "query.hpp"

namespace cubvh_amd {
namespace dev {

__device__ __forceinline__ int32_t ld_parent(const int32_t* L, int32_t x) {
    return __hip_atomic_load(L + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int32_t find_root(const int32_t* L, int32_t x) {
    int32_t p = ld_parent(L, x);
    while (p != x) {
        x = p;
        p = ld_parent(L, x);
    }
    return x;
}

// find_root that points every node it passes at its grandparent.  A store may undo a
// concurrent link of a node that was no root any more; unite goes on from the value that
// link replaced, so no edge is lost.
__device__ __forceinline__ int32_t find_root_halving(int32_t* L, int32_t x) {
    int32_t p = ld_parent(L, x);
    while (p != x) {
        const int32_t g = ld_parent(L, p);
        if (g != p) __hip_atomic_store(L + x, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = p;
        p = g;
    }
    return x;
}

__device__ __forceinline__ void unite(int32_t* L, int32_t a, int32_t b) {
    for (;;) {
        a = find_root_halving(L, a);
        b = find_root_halving(L, b);
        if (a == b) return;
        if (a > b) {
            int32_t t = a; a = b; b = t;
        }
        // link root b under a; succeeds only if b is still a root
        int32_t old = atomicMin(L + b, a);
        if (old == b) return;
        b = old;
    }
}

// A tile has TD x TW x TH voxels along the last, middle and first axis; 64 / TD rows along the
// last axis share a wave pass.
constexpr int TILE_WAVES = 4;
constexpr int TILE_PASSES = 64;  // 4,096 voxels
constexpr int WAVE_PASSES = TILE_PASSES / TILE_WAVES;
template <int TD>
struct Tile {
    static_assert(TD == 64 || TD == 16, "cubic but for the order of the lanes");
    static constexpr int TW = TD == 64 ? 8 : 16, TH = TW;
    static constexpr int ROWS = TW * TH, PER_PASS = 64 / TD;  // rows, and those of a pass
    static constexpr uint64_t ROW = TD == 64 ? ~0ull : (1ull << (TD & 63)) - 1ull;
    static constexpr int HALVES = TD == 64 ? 2 : 1;  // threads for a pair of neighbouring rows
    static_assert(ROWS * TD == 64 * TILE_PASSES, "a lane per voxel");
    int32_t d0, w0, h0, base;  // the tile's first voxel; of its grid (the whole has fewer than 2^31)
    __device__ __forceinline__ Tile(uint32_t tile, int32_t H, int32_t W, int32_t D) {
        const uint32_t nd = (D + TD - 1) / TD, nw = (W + TW - 1) / TW, nh = (H + TH - 1) / TH;
        d0 = (int32_t)(tile % nd) * TD;
        w0 = (int32_t)((tile / nd) % nw) * TW;
        const uint32_t rest = tile / (nd * nw);
        h0 = (int32_t)(rest % nh) * TH;
        base = (int32_t)(rest / nh) * H * W * D;
    }
};

__device__ __forceinline__ int32_t lds_parent(const int32_t* L, int32_t x) {
    return __hip_atomic_load(L + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int32_t lds_root(const int32_t* L, int32_t x) {
    int32_t p = lds_parent(L, x);
    while (p != x) {
        x = p;
        p = lds_parent(L, x);
    }
    return x;
}
__device__ __forceinline__ void lds_unite(int32_t* L, int32_t a, int32_t b) {
    for (;;) {
        a = lds_root(L, a);
        b = lds_root(L, b);
        if (a == b) return;
        if (a > b) {
            int32_t t = a; a = b; b = t;
        }
        int32_t old = atomicMin(L + b, a);
        if (old == b) return;
        b = old;
    }
}

// First voxel of the run of set bits of `free` that holds bit `lane` (which is set).
__device__ __forceinline__ int run_start(uint64_t free, int lane) {
    const uint64_t gaps = ~free & ((1ull << lane) - 1ull);
    return gaps ? 64 - __builtin_clzll(gaps) : 0;
}

// One workgroup per tile (from tile `first` on); tiles numbered along the last axis fastest,
// then w, h, b.  Voxel c of row r (w = r % TW, h = r / TW) has the local index TD r + c, which
// orders voxels like the tile's linear index; only the first voxel of a run is a union-find
// node.
template <int TD>
__global__ __launch_bounds__(64 * TILE_WAVES) void ff_tiles(const uint8_t* __restrict__ grid, int32_t* __restrict__ out,
                                                            uint32_t first, int32_t H, int32_t W, int32_t D) {
    using T = Tile<TD>;
    constexpr int TW = T::TW, TH = T::TH;
    __shared__ int32_t L[64 * TILE_PASSES];
    __shared__ uint64_t rows[TILE_PASSES];
    const T t(first + blockIdx.x, H, W, D);
    const int lane = (int)threadIdx.x & 63, p0 = ((int)threadIdx.x >> 6) * WAVE_PASSES, c = lane % TD;
    const int32_t d = t.d0 + c;
    uint8_t occ[WAVE_PASSES];
#pragma unroll
    for (int k = 0; k < WAVE_PASSES; ++k) {
        const int r = (p0 + k) * T::PER_PASS + lane / TD, h = t.h0 + r / TW, w = t.w0 + r % TW;
        occ[k] = 1;  // outside the grid counts as occupied
        if (h < H && w < W && d < D) occ[k] = grid[t.base + (h * W + w) * D + d];
    }
    uint64_t free[WAVE_PASSES];
#pragma unroll
    for (int k = 0; k < WAVE_PASSES; ++k) {
        free[k] = __builtin_amdgcn_ballot_w64(occ[k] == 0);
        rows[p0 + k] = free[k];  // every lane the same value
        L[64 * (p0 + k) + lane] = 64 * (p0 + k) + lane;
    }
    __syncthreads();
    auto row = [&](int r) { return (rows[r / T::PER_PASS] >> (TD * (r % T::PER_PASS))) & T::ROW; };
    // a thread (two, one per half of the row, where rows are long) for each pair of neighbouring
    // rows: two runs meet in one contiguous segment, united at its first voxel
    for (int pt = (int)threadIdx.x; pt < T::HALVES * (2 * T::ROWS - TW - TH); pt += 64 * TILE_WAVES) {
        const int pr = pt / T::HALVES;
        const bool along_w = pr < T::ROWS - TH;
        const int r = along_w ? pr / (TW - 1) * TW + pr % (TW - 1) + 1 : pr - (T::ROWS - TH) + TW;
        const int o = along_w ? r - 1 : r - TW;  // the row at w - 1, or at h - 1
        const uint64_t mine = row(r), other = row(o), both = mine & other;
        uint64_t segments = both & ~(both << 1);
        if (T::HALVES == 2) segments &= 0xffffffffull << (32 * (pt & 1));
        for (; segments != 0; segments &= segments - 1) {
            const int l = __builtin_ctzll(segments);
            lds_unite(L, TD * r + run_start(mine, l), TD * o + run_start(other, l));
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < WAVE_PASSES; ++k) {
        const int r = (p0 + k) * T::PER_PASS + lane / TD, h = t.h0 + r / TW, w = t.w0 + r % TW;
        if (h >= H || w >= W || d >= D) continue;
        int32_t lab = -1;
        if ((free[k] >> lane) & 1) {
            const uint64_t mine = (free[k] >> (TD == 64 ? 0 : lane - c)) & T::ROW;
            const int32_t root = lds_root(L, TD * r + run_start(mine, c)), rr = root / TD;
            lab = t.base + ((t.h0 + rr / TW) * W + (t.w0 + rr % TW)) * D + t.d0 + root % TD;
        }
        out[t.base + (h * W + w) * D + d] = lab;
    }
}

// Unions across the tile faces: the voxels on a tile's low faces with their neighbour one
// step back, one wave per face normal to the middle or the first axis (8 passes of 64 pairs,
// or 4 of 4 rows),
// and per 512 pairs of the faces normal to the last axis.  Pairs with the same two labels
// are the same union: a pair that repeats the one before it in its lane is dropped, the
// others leave their number in a small table, and one that finds another pair's number
// there with the same labels is done (a pair whose entry was taken by different labels is
// united as often as it occurs).  A wave per face and not a workgroup: the unions are
// chains of dependent loads by a few lanes, so what counts is the faces in flight.
constexpr uint32_t MERGE_SLOTS = 1024;
template <int TD>
__global__ __launch_bounds__(64) void ff_merge(int32_t* L, int32_t B, int32_t H, int32_t W, int32_t D, uint32_t b0,
                                               uint32_t b1) {
    using T = Tile<TD>;
    constexpr int TW = T::TW, TH = T::TH, MERGE_ROWS = TW / T::PER_PASS;  // one wave per face
    __shared__ int32_t low[64 * MERGE_ROWS], high[64 * MERGE_ROWS];
    __shared__ uint16_t owner[MERGE_SLOTS];
    const int t = (int)threadIdx.x;
    const uint32_t nd = (D + TD - 1) / TD, nw = (W + TW - 1) / TW, nh = (H + TH - 1) / TH;
    int32_t li[MERGE_ROWS], lj[MERGE_ROWS];
#pragma unroll
    for (int r = 0; r < MERGE_ROWS; ++r) li[r] = lj[r] = -1;
    if (blockIdx.x < b0) {  // the last axis: w fastest, then the boundary, then h, then b
#pragma unroll
        for (int r = 0; r < MERGE_ROWS; ++r) {
            const uint32_t k = (blockIdx.x * MERGE_ROWS + r) * 64 + t, q = k / W, q2 = q / (nd - 1);
            const int32_t b = (int32_t)(q2 / H);
            if (b >= B) continue;
            const int32_t i = ((b * H + (int32_t)(q2 % H)) * W + (int32_t)(k % W)) * D + (int32_t)(q % (nd - 1) + 1) * TD;
            li[r] = L[i];
            lj[r] = L[i - 1];
        }
    } else {
        const bool middle = blockIdx.x < b0 + b1;
        const uint32_t k = blockIdx.x - b0 - (middle ? 0 : b1), q = k / nd;
        const int32_t d = (int32_t)(k % nd) * TD + t % TD;
        const uint32_t cw = middle ? nw - 1 : nw, ch = middle ? nh : nh - 1;  // faces along w and h
        const int32_t w0 = (int32_t)(q % cw + (middle ? 1 : 0)) * TW, h0 = (int32_t)(q / cw % ch + (middle ? 0 : 1)) * TH;
        const int32_t b = (int32_t)(q / cw / ch), step = middle ? D : D * W;
#pragma unroll
        for (int r = 0; r < MERGE_ROWS; ++r) {
            const int32_t o = r * T::PER_PASS + t / TD, w = middle ? w0 : w0 + o, h = middle ? h0 + o : h0;
            if (d >= D || w >= W || h >= H) continue;
            const int32_t i = ((b * H + h) * W + w) * D + d;
            li[r] = L[i];
            lj[r] = L[i - step];
        }
    }
    uint32_t todo = 0;
#pragma unroll
    for (int r = 0; r < MERGE_ROWS; ++r) {
        if (li[r] < 0 || lj[r] < 0 || (r > 0 && li[r] == li[r - 1] && lj[r] == lj[r - 1])) continue;
        const int at = 64 * r + t;
        low[at] = lj[r];
        high[at] = li[r];
        owner[(((uint32_t)li[r] * 0x9e3779b1u) ^ ((uint32_t)lj[r] * 0x85ebca77u)) >> 22] = (uint16_t)at;
        todo |= 1u << r;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < MERGE_ROWS; ++r) {
        if (!((todo >> r) & 1u)) continue;
        const int o = owner[(((uint32_t)li[r] * 0x9e3779b1u) ^ ((uint32_t)lj[r] * 0x85ebca77u)) >> 22];
        if (o != 64 * r + t && low[o] == lj[r] && high[o] == li[r]) continue;
        unite(L, li[r], lj[r]);
    }
}

// label[i] = root(i), a workgroup per tile.  A tile's voxels have few distinct labels (its
// local roots), whose roots are kept in a table: most voxels find theirs there.
constexpr uint32_t FLAT_SLOTS = 512;
template <int TD>
__global__ __launch_bounds__(64 * TILE_WAVES) void ff_flatten(int32_t* L, uint32_t first, int32_t H, int32_t W, int32_t D) {
    using T = Tile<TD>;
    __shared__ unsigned long long known[FLAT_SLOTS];  // (label, root)
    const T t(first + blockIdx.x, H, W, D);
    const int lane = (int)threadIdx.x & 63, p0 = ((int)threadIdx.x >> 6) * WAVE_PASSES;
    const int32_t d = t.d0 + lane % TD;
    for (int k = (int)threadIdx.x; k < (int)FLAT_SLOTS; k += 64 * TILE_WAVES) known[k] = ~0ull;
    int32_t lab[WAVE_PASSES];
#pragma unroll
    for (int k = 0; k < WAVE_PASSES; ++k) {
        const int r = (p0 + k) * T::PER_PASS + lane / TD, h = t.h0 + r / T::TW, w = t.w0 + r % T::TW;
        lab[k] = -1;
        if (h < H && w < W && d < D) lab[k] = L[t.base + (h * W + w) * D + d];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < WAVE_PASSES; ++k) {
        if (lab[k] < 0) continue;  // occupied, or outside the grid
        unsigned long long* at = known + (((uint32_t)lab[k] * 0x9e3779b1u) >> 23);
        const unsigned long long e = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        int32_t root = (int32_t)(uint32_t)e;
        if ((uint32_t)(e >> 32) != (uint32_t)lab[k]) {
            root = find_root(L, lab[k]);
            __hip_atomic_store(at, ((unsigned long long)(uint32_t)lab[k] << 32) | (uint32_t)root, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        const int r = (p0 + k) * T::PER_PASS + lane / TD, h = t.h0 + r / T::TW, w = t.w0 + r % T::TW;
        if (root != lab[k]) L[t.base + (h * W + w) * D + d] = root;
    }
}

}  // namespace dev

namespace {

// A launch has fewer than 2^32 threads: tiles in runs of 2^23 workgroups.
constexpr int64_t kTileRun = (int64_t)1 << 23;
constexpr int64_t kNarrowTiles = 1024;

template <int TD>
hipError_t launch_tiles(const uint8_t* grid, int32_t B, int32_t H, int32_t W, int32_t D, int32_t* labels, hipStream_t stream) {
    using T = dev::Tile<TD>;
    const int64_t nd = (D + TD - 1) / TD, nw = (W + T::TW - 1) / T::TW, nh = (H + T::TH - 1) / T::TH;
    const int64_t n_tiles = B * nh * nw * nd;
    for (int64_t at = 0; at < n_tiles; at += kTileRun)
        hipLaunchKernelGGL(dev::ff_tiles<TD>, dim3((unsigned)std::min(n_tiles - at, kTileRun)), dim3(64 * dev::TILE_WAVES), 0,
                           stream, grid, labels, (uint32_t)at, H, W, D);
    // waves of the faces normal to the last, the middle and the first axis: at most an eighth of
    // the voxels each, a wave to 64 of the first and 16 or more of the others
    constexpr int64_t pairs = 64 * T::TW / T::PER_PASS;
    const uint32_t b0 = (uint32_t)((B * (nd - 1) * W * H + pairs - 1) / pairs);
    const uint32_t b1 = (uint32_t)(B * nh * (nw - 1) * nd), b2 = (uint32_t)(B * (nh - 1) * nw * nd);
    if (b0 + b1 + b2 > 0) {  // labels of one tile are final already
        hipLaunchKernelGGL(dev::ff_merge<TD>, dim3(b0 + b1 + b2), dim3(64), 0, stream, labels, B, H, W, D, b0, b1);
        for (int64_t at = 0; at < n_tiles; at += kTileRun)
            hipLaunchKernelGGL(dev::ff_flatten<TD>, dim3((unsigned)std::min(n_tiles - at, kTileRun)), dim3(64 * dev::TILE_WAVES),
                               0, stream, labels, (uint32_t)at, H, W, D);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_floodfill(const uint8_t* grid, int32_t B, int32_t H, int32_t W, int32_t D, int32_t* labels,
                            hipStream_t stream) {
    if ((int64_t)B * H * W * D <= 0) return hipSuccess;
    for (int k = 0; k < 2 && D == 1; ++k) {
        D = W;
        W = H;
        H = 1;
    }
    // Rows of 64 leave three lanes of four idle when the last axis has at most 16, but while
    // they make fewer than four workgroups a CU there is room for them: 64 grids of 16^3
    // (256 workgroups, or 64 of narrow tiles) 26-36 and 28-42 us, 512 of them 47-63 and 31-48.
    const int64_t wide = (int64_t)B * ((H + 7) / 8) * ((W + 7) / 8);
    return D <= 16 && wide >= kNarrowTiles ? launch_tiles<16>(grid, B, H, W, D, labels, stream)
                                           : launch_tiles<64>(grid, B, H, W, D, labels, stream);
}

}  // namespace cubvh_amd
