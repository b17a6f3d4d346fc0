// PLOC BVH2 construction on gfx950.
//
// Restates PlocBuilder::build_ploc / build_ploc_from_leaves (ploc/mod.rs:169-503) as a sequence of data-parallel
// passes whose outputs are bit-identical to the reference's serial loop:
//   k_leaf_init_*  : leaf Bvh2Node per primitive (ploc/mod.rs:187-243) + scene bounds (atomic min/max on
//                    order-preserving keys; the zero sign of the bounds cannot change a Morton code)
//   k_morton       : 63-bit Morton code of the f32 centre normalised in f64 (ploc/mod.rs:287-288, 782-785;
//                    morton.rs:35-58), or the 126-bit code of SortPrecision::U128 (morton.rs:63-89) as two words
//   radix sort     : stable (sort.hip), by the code's top 32 bits
//   k_gather       : sorted leaves become the first cluster array (ploc/mod.rs:829-846)
//   per pass       : k_ploc_search_count (ploc/mod.rs:329-419, window in LDS, and the per-tile counts of emitted
//                    clusters and merges), their prefix sums in two launches over chunks for the largest passes,
//                    k_ploc_compact (ploc/mod.rs:420-487: the parent of a mutual pair is emitted at the higher
//                    index, its children go to nodes[insert - 2(s+1)] and [+1] where s is the merge's rank in the
//                    pass); passes of at most 1,024 tiles are one launch each (k_ploc_pass)
//   k_ploc_tail    : once at most 2048 clusters remain, one workgroup finishes every remaining pass with the
//                    clusters resident in LDS and writes the root (ploc/mod.rs:499), then evaluates the cost-table
//                    entries of its merges by height (tail.hpp)
// Pass state (cluster count, insert index, depth) lives on the device so passes are enqueued without host syncs;
// the host only reads the count every few passes to shrink the grids.
//
// ploc_rebuild runs the same passes over clusters taken from an existing tree (rebuild_from_leaves,
// ploc/rebuild.rs:136-183).  For a partial rebuild the children of the g-th merge (counted over all passes in the
// serial loop's order) go to the g-th freed sibling pair from the top (`slot_map`, the REBUILD placement of
// ploc/mod.rs:449-462); the plain placement is the special case slot_map[g] = 2n-3-2g.
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

#include "common.hpp"
#include "cwdp.hpp"
#include "device_util.hpp"
#include "internal.hpp"
#include "tail.hpp"

namespace obvhs {

namespace {

constexpr int T256 = 256;
constexpr uint32_t TAIL_MAX = 2048;  // 4096 measured 5% slower per build (the tail's passes are LDS and ALU bound)
constexpr int TAIL_THREADS = 1024;
// Passes enqueued between host reads of the cluster count (1.29M-triangle build: 4 -> 1.97 ms, 8 -> 1.92, 16 -> 1.93).
constexpr int PASSES_PER_SYNC = 8;

// Passes of at most GROUP_MAX_TILES tiles need no scan between search and compaction: a tile's place is the sum of the
// groups before its own and of the tiles before it in its group (k_ploc_compact).  Eight passes of up to 5,033 tiles:
// the scans took 46 us; the search's atomics cost 8 of them with 16 tiles to a group, 46 with 64.
constexpr uint32_t GROUP_TILES = 16;
constexpr uint32_t TILE_GROUPS = 1024;
constexpr uint32_t GROUP_MAX_TILES = GROUP_TILES * TILE_GROUPS;

struct Misc {
    uint32_t bounds[6];  // order keys: min x,y,z (atomicMin) then max x,y,z (atomicMax)
    uint32_t err;
    uint32_t pad;
    PlocState state[2];
    CwRootInfo info;  // written by the tail of a build that evaluates the cost table
    // Sums of the tiles' counts (emits in the low word, merges in the high one) by GROUP_TILES tiles, by slot; zero
    // before a pass, the other slot's cleared by the pass's compaction.
    unsigned long long groups[2][TILE_GROUPS];
};

__device__ __forceinline__ void clear_groups(Misc* misc) {
    for (uint32_t g = threadIdx.x; g < 2u * TILE_GROUPS; g += blockDim.x) (&misc->groups[0][0])[g] = 0ull;
}

__global__ void k_init_misc(Misc* misc, uint32_t n, uint32_t* hist) {
    if (threadIdx.x == 0) {
        hist[0] = 2u * n - 1u;
        for (int a = 0; a < 3; ++a) {
            misc->bounds[a] = 0xffffffffu;
            misc->bounds[3 + a] = 0u;
        }
        misc->err = 0u;
        misc->state[0] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
        misc->state[1] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
    }
    clear_groups(misc);
}

// Reduces the leaf bounds of one block into the scene bounds.  Both the min and the max corner of every leaf go
// into both reductions, like `local_aabb.extend(aabb.min); local_aabb.extend(aabb.max)` (ploc/mod.rs:189-190).
__device__ __forceinline__ void reduce_scene_bounds(bool valid, const Box& b, bool nan, Misc* misc,
                                                    uint32_t* __restrict__ partials) {
    __shared__ uint32_t red[6][T256 / 64];
    uint32_t k[6];
    if (valid) {
        uint32_t kl[3] = {f32_order_key(b.lx), f32_order_key(b.ly), f32_order_key(b.lz)};
        uint32_t kh[3] = {f32_order_key(b.hx), f32_order_key(b.hy), f32_order_key(b.hz)};
        for (int a = 0; a < 3; ++a) {
            k[a] = min(kl[a], kh[a]);
            k[3 + a] = max(kl[a], kh[a]);
        }
    } else {
        for (int a = 0; a < 3; ++a) {
            k[a] = 0xffffffffu;
            k[3 + a] = 0u;
        }
    }
    for (int a = 0; a < 3; ++a) {
        k[a] = wave_min_u32(k[a]);
        k[3 + a] = wave_max_u32(k[3 + a]);
    }
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (lane == 0)
        for (int a = 0; a < 6; ++a) red[a][wave] = k[a];
    if (__ballot(nan) != 0ull && lane == 0) atomicOr(&misc->err, DERR_NAN_INPUT);
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        uint32_t v = red[a][0];
        for (int w = 1; w < T256 / 64; ++w) v = a < 3 ? min(v, red[a][w]) : max(v, red[a][w]);
        partials[blockIdx.x * 6 + a] = v;
    }
}

// Final reduction of the per-block scene bounds (one workgroup).
__global__ void __launch_bounds__(1024) k_reduce_bounds(const uint32_t* __restrict__ partials, uint32_t nblocks,
                                                        Misc* misc) {
    __shared__ uint32_t red[6][16];
    uint32_t k[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
    for (uint32_t b = threadIdx.x; b < nblocks; b += 1024) {
        for (int a = 0; a < 3; ++a) {
            k[a] = min(k[a], partials[b * 6 + a]);
            k[3 + a] = max(k[3 + a], partials[b * 6 + 3 + a]);
        }
    }
    for (int a = 0; a < 3; ++a) {
        k[a] = wave_min_u32(k[a]);
        k[3 + a] = wave_max_u32(k[3 + a]);
    }
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (lane == 0)
        for (int a = 0; a < 6; ++a) red[a][wave] = k[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        uint32_t v = red[a][0];
        for (int w = 1; w < 16; ++w) v = a < 3 ? min(v, red[a][w]) : max(v, red[a][w]);
        misc->bounds[a] = v;
    }
}

// Triangle::aabb = Aabb::from_points([v0, v1, v2]) (triangle.rs:28-30; aabb.rs:59-66).
__device__ __forceinline__ Box tri_box(const float4& v0, const float4& v1, const float4& v2) {
    const Box b{smin(v0.x, v1.x), smin(v0.y, v1.y), smin(v0.z, v1.z), smax(v0.x, v1.x), smax(v0.y, v1.y),
                smax(v0.z, v1.z)};
    return Box{smin(b.lx, v2.x), smin(b.ly, v2.y), smin(b.lz, v2.z), smax(b.hx, v2.x), smax(b.hy, v2.y),
               smax(b.hz, v2.z)};
}

// iota_out (when the caller gave no indices): primitive_indices = 0..n-1, written here instead of by a launch of its own.
__global__ void __launch_bounds__(T256) k_leaf_init_tris(const float4* __restrict__ tris,
                                                         const uint32_t* __restrict__ indices, uint32_t n,
                                                         Node32* __restrict__ leaves, Misc* misc,
                                                         uint32_t* __restrict__ partials,
                                                         uint32_t* __restrict__ iota_out) {
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    const bool valid = i < n;
    if (iota_out && valid) iota_out[i] = i;
    Box b{0, 0, 0, 0, 0, 0};
    bool nan = false;
    if (valid) {
        float4 v0 = tris[3 * (size_t)i], v1 = tris[3 * (size_t)i + 1], v2 = tris[3 * (size_t)i + 2];
        b = tri_box(v0, v1, v2);
        nan = box_has_nan(b);
        store_node(&leaves[i], make_node(b, 1u, indices ? indices[i] : i));
    }
    reduce_scene_bounds(valid, b, nan, misc, partials);
}

// T = Aabb: the leaf box is the input box (aabb.rs:209-214).
__global__ void __launch_bounds__(T256) k_leaf_init_aabbs(const float4* __restrict__ aabbs,
                                                          const uint32_t* __restrict__ indices, uint32_t n,
                                                          Node32* __restrict__ leaves, Misc* misc,
                                                          uint32_t* __restrict__ partials,
                                                          uint32_t* __restrict__ iota_out) {
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    const bool valid = i < n;
    if (iota_out && valid) iota_out[i] = i;
    Box b{0, 0, 0, 0, 0, 0};
    bool nan = false;
    if (valid) {
        float4 lo = aabbs[2 * (size_t)i], hi = aabbs[2 * (size_t)i + 1];
        b = Box{lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
        nan = box_has_nan(b);
        store_node(&leaves[i], make_node(b, 1u, indices ? indices[i] : i));
    }
    reduce_scene_bounds(valid, b, nan, misc, partials);
}

// rebuild_from_leaves takes the root's stored box as the scene box (ploc/rebuild.rs:154).
__global__ void k_bounds_from_node(Misc* misc, const Node32* __restrict__ nodes) {
    if (threadIdx.x == 0) {
        const Node32 r = load_node(&nodes[0]);
        misc->bounds[0] = f32_order_key(r.minx);
        misc->bounds[1] = f32_order_key(r.miny);
        misc->bounds[2] = f32_order_key(r.minz);
        misc->bounds[3] = f32_order_key(r.maxx);
        misc->bounds[4] = f32_order_key(r.maxy);
        misc->bounds[5] = f32_order_key(r.maxz);
    }
}

// The scene's normalisation to the unit cube (ploc/mod.rs:287-288 and 782-785) from the bounds' order keys.
struct SceneMap {
    double sx, sy, sz, ox, oy, oz;
    __device__ __forceinline__ void point(const Box& b, double& px, double& py, double& pz) const {
        const float cx = (b.hx + b.lx) * 0.5f, cy = (b.hy + b.ly) * 0.5f, cz = (b.hz + b.lz) * 0.5f;
        px = (double)cx * sx + ox;
        py = (double)cy * sy + oy;
        pz = (double)cz * sz + oz;
    }
};
__device__ __forceinline__ SceneMap scene_map(const uint32_t* bounds) {
    const float mnx = f32_from_order_key(bounds[0]), mny = f32_from_order_key(bounds[1]),
                mnz = f32_from_order_key(bounds[2]);
    const float mxx = f32_from_order_key(bounds[3]), mxy = f32_from_order_key(bounds[4]),
                mxz = f32_from_order_key(bounds[5]);
    SceneMap m;
    m.sx = 1.0 / (double)(mxx - mnx);
    m.sy = 1.0 / (double)(mxy - mny);
    m.sz = 1.0 / (double)(mxz - mnz);
    m.ox = -(double)mnx * m.sx;
    m.oy = -(double)mny * m.sy;
    m.oz = -(double)mnz * m.sz;
    return m;
}

// The 63-bit Morton code of a unit-cube point (morton.rs:35-58).
__device__ __forceinline__ uint64_t morton64_of_point(double px, double py, double pz) {
    const double s = 2097152.0;  // 2^21
    return split_by_3_u64(f64_as_u32(px * s)) | split_by_3_u64(f64_as_u32(py * s)) << 1 |
           split_by_3_u64(f64_as_u32(pz * s)) << 2;
}

// The top 32 bits of a 63-bit code, or of a 126-bit code's 62-bit high word.
__device__ __forceinline__ uint32_t top_of_u64(uint64_t code) { return (uint32_t)(code >> 31); }
__device__ __forceinline__ uint32_t top_of_u128(uint64_t hi) { return (uint32_t)(hi >> 30); }

// keys_hi = NULL: U64 codes into keys.  Otherwise U128 codes, low words into keys and high words into keys_hi.
// tops: the codes' top 32 bits (the first sort key).
__global__ void __launch_bounds__(T256) k_morton(const Node32* __restrict__ leaves, uint32_t n,
                                                 const Misc* __restrict__ misc, uint64_t* __restrict__ keys,
                                                 uint64_t* __restrict__ keys_hi, uint32_t* __restrict__ tops) {
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    if (i >= n) return;
    const SceneMap map = scene_map(misc->bounds);
    double px, py, pz;
    map.point(node_box(load_node(&leaves[i])), px, py, pz);
    if (keys_hi) {
        uint64_t lo, hi;
        morton128_of_point(px, py, pz, lo, hi);
        keys[i] = lo;
        keys_hi[i] = hi;
        tops[i] = top_of_u128(hi);
        return;
    }
    const uint64_t code = morton64_of_point(px, py, pz);
    keys[i] = code;
    tops[i] = top_of_u64(code);
}

// `bits` bits of the codes' words from `shift` up, in the given order (NULL: leaf order).
__global__ void __launch_bounds__(T256) k_code_words(const uint64_t* __restrict__ src,
                                                     const uint32_t* __restrict__ order, uint32_t n, uint32_t shift,
                                                     uint32_t bits, uint32_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    if (i >= n) return;
    out[i] = (uint32_t)(src[order ? order[i] : i] >> shift) & (0xffffffffu >> (32u - bits));
}

__global__ void __launch_bounds__(T256) k_gather(const Node32* __restrict__ leaves,
                                                 const uint32_t* __restrict__ order, uint32_t n,
                                                 Node32* __restrict__ out) {
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    if (i >= n) return;
    store_node(&out[i], load_node(&leaves[order[i]]));
}

// The sorted leaves in cluster order from the sort by the codes' top 32 bits (tops and order, stable): a run of equal
// tops is put in the order of the codes' remaining bits, ties by position (the leaf order, the sort being stable), by
// ranking each of its members against the others from LDS, so that the result is the order of a stable sort of the
// whole codes.  Runs are short (the tops are cells of 10 or 11 bits per axis: 1 to 12 leaves a run on the benchmark's
// heightfields of 1.3M and 17.3M triangles).  A run longer than RUN_MAX (or that long on one side of a member) sets
// DERR_RESORT and leaves one cluster in the pass state, which turns the passes behind this launch into no-ops; the
// host then sorts the whole codes.  Such a scene (a dense object in a large extent, duplicated geometry) pays for the
// first sort, the launches without work and a host wait: 16.8M leaves in a 500th of their box 7.5 ms against 5.9 for
// an evenly filled one (20.1 when every member of a run set the flag by an atomic of its own, which a workgroup that
// finds it set now skips with all its work), 1M 1.24 ms, 65,536 0.68 (0.53 evenly filled).
// Bound by the random 32-byte leaf reads.  1,288,352 leaves: 23 us against the plain gather's 16, and with it the sort
// takes 4 passes of 20 bytes per key instead of 8 of 32 (198 -> 98 us).
// order_out (may be NULL): the final permutation.
constexpr uint32_t RUN_MAX = 64;

template <bool WIDE>
__global__ void __launch_bounds__(T256) k_gather_runs(const Node32* __restrict__ leaves,
                                                      const uint32_t* __restrict__ tops,
                                                      const uint32_t* __restrict__ order, uint32_t n,
                                                      const uint64_t* __restrict__ keys,
                                                      const uint64_t* __restrict__ keys_hi, Misc* misc,
                                                      Node32* __restrict__ out, uint32_t* __restrict__ order_out) {
    constexpr uint32_t WIN = T256 + 2 * RUN_MAX;
    __shared__ uint32_t tk[WIN];
    __shared__ uint32_t rest[WIN];                  // the bits below the top: 31, or 30 of the high word
    __shared__ uint64_t low[WIDE ? WIN : 1];        // the low word of a 126-bit code
    __shared__ bool flagged;
    const uint32_t base = xcd_tile() * T256;
    if (base >= n) return;
    // window slot w holds sorted position base - RUN_MAX + w
    const uint32_t w0 = base < RUN_MAX ? RUN_MAX - base : 0u;             // first slot inside the array
    const uint32_t w1 = min(WIN, n - base + RUN_MAX);                     // end of the slots inside it
    for (uint32_t w = w0 + threadIdx.x; w < w1; w += T256) tk[w] = tops[base + w - RUN_MAX];
    if (threadIdx.x == 0) flagged = resort_flagged(&misc->err);
    __syncthreads();
    if (flagged) return;  // the host sorts again
    for (uint32_t w = w0 + threadIdx.x; w < w1; w += T256) {
        const uint32_t t = tk[w];
        if ((w > w0 && tk[w - 1] == t) || (w + 1 < w1 && tk[w + 1] == t)) {
            const uint32_t leaf = order[base + w - RUN_MAX];
            if (WIDE) {
                rest[w] = (uint32_t)keys_hi[leaf] & 0x3fffffffu;
                low[w] = keys[leaf];
            } else {
                rest[w] = (uint32_t)keys[leaf] & 0x7fffffffu;
            }
        }
    }
    __syncthreads();
    const uint32_t i = base + threadIdx.x;
    if (i >= n) return;
    const uint32_t leaf = order[i], me = threadIdx.x + RUN_MAX, t = tk[me];
    uint32_t a = me, b = me;  // the run's first and last slot
    while (a > w0 && me - a < RUN_MAX && tk[a - 1] == t) --a;
    while (b + 1 < w1 && b - me < RUN_MAX && tk[b + 1] == t) ++b;
    if (flag_resort(me - a == RUN_MAX || b - me == RUN_MAX, &misc->err)) {
        misc->state[0].count = 1u;
        return;
    }
    uint32_t rank = 0u;
    if (a != b) {
        const uint32_t r = rest[me];
        const uint64_t l = WIDE ? low[me] : 0ull;
        for (uint32_t j = a; j <= b; ++j) {
            const bool same = rest[j] == r;
            const bool less = rest[j] < r || (same && WIDE && low[j] < l);
            const bool tie = same && (!WIDE || low[j] == l) && j < me;
            rank += (less || tie) ? 1u : 0u;
        }
    }
    const uint32_t pos = base + a - RUN_MAX + rank;
    store_node(&out[pos], load_node(&leaves[leaf]));
    if (order_out) order_out[pos] = leaf;
}

// State reset before a build repeats its passes (after DERR_RESORT); the bounds and the codes stay.
__global__ void k_reset_state(Misc* misc, uint32_t n) {
    if (threadIdx.x == 0) {
        misc->err &= ~DERR_RESORT;
        misc->state[0] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
        misc->state[1] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
    }
    clear_groups(misc);
}

// The front of a build of at most SMALL_MAX leaves in one workgroup and one launch: leaf boxes, scene bounds, Morton
// codes, the stable sort (four 8-bit LSD passes over the codes' top 32 bits in LDS, wave multisplit ranking as in
// sort.hip, then runs of equal tops ranked by the remaining bits) and the sorted leaves as the first clusters.  At
// these sizes the 29 launches it replaces are 2 to 7 us each whatever they hold (1,501 triangles: 109 us of kernels in
// 29 launches -> 20 us in one).
constexpr uint32_t SMALL_MAX = 2048;
constexpr int SMALL_THREADS = 1024;
constexpr int SMALL_ITEMS = (int)SMALL_MAX / SMALL_THREADS;
constexpr int SMALL_WAVES = SMALL_THREADS / 64;
constexpr uint32_t SMALL_RUN = 64;

template <bool WIDE>
__global__ void __launch_bounds__(SMALL_THREADS)
    k_front_small(const float4* __restrict__ tris, const float4* __restrict__ aabbs,
                  const uint32_t* __restrict__ indices, uint32_t n, Misc* misc, uint32_t* __restrict__ hist,
                  uint32_t* __restrict__ iota_out, uint64_t* __restrict__ codes_out,
                  uint64_t* __restrict__ codes_hi_out, uint32_t* __restrict__ order_out,
                  Node32* __restrict__ clusters) {
    __shared__ uint64_t low[SMALL_MAX];                // codes (the low words of 126-bit codes), leaf order
    __shared__ uint64_t high[WIDE ? SMALL_MAX : 1];
    __shared__ uint32_t tk[SMALL_MAX];                 // tops in sorted order
    __shared__ uint16_t tv[SMALL_MAX];                 // leaves in sorted order
    __shared__ uint32_t whist[SMALL_WAVES][256];
    __shared__ uint32_t red[6][SMALL_WAVES];
    __shared__ uint32_t wtot[4];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;

    // leaf boxes (as k_leaf_init_*) and scene bounds
    auto leaf_box = [&](uint32_t i) {
        if (tris) {
            const float4 v0 = tris[3 * (size_t)i], v1 = tris[3 * (size_t)i + 1], v2 = tris[3 * (size_t)i + 2];
            return tri_box(v0, v1, v2);
        }
        const float4 lo = aabbs[2 * (size_t)i], hi = aabbs[2 * (size_t)i + 1];
        return Box{lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
    };
    Box box[SMALL_ITEMS];
    uint32_t k[6] = {0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u};
    bool nan = false;
#pragma unroll
    for (int q = 0; q < SMALL_ITEMS; ++q) {
        const uint32_t i = (uint32_t)q * SMALL_THREADS + tid;
        box[q] = Box{0, 0, 0, 0, 0, 0};
        if (i < n) {
            box[q] = leaf_box(i);
            nan |= box_has_nan(box[q]);
            if (iota_out) iota_out[i] = i;
            const uint32_t kl[3] = {f32_order_key(box[q].lx), f32_order_key(box[q].ly), f32_order_key(box[q].lz)};
            const uint32_t kh[3] = {f32_order_key(box[q].hx), f32_order_key(box[q].hy), f32_order_key(box[q].hz)};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                k[a] = min(k[a], min(kl[a], kh[a]));
                k[3 + a] = max(k[3 + a], max(kl[a], kh[a]));
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        k[a] = wave_min_u32(k[a]);
        k[3 + a] = wave_max_u32(k[3 + a]);
        if (lane == 0) {
            red[a][wave] = k[a];
            red[3 + a][wave] = k[3 + a];
        }
    }
    const bool any_nan = __syncthreads_or(nan);
    if (tid == 0) {
        hist[0] = 2u * n - 1u;
        misc->err = any_nan ? DERR_NAN_INPUT : 0u;
        misc->state[0] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
        misc->state[1] = PlocState{n, 2u * n - 1u, 0u, 0u, 0ull};
    }
#pragma unroll
    for (int w = 0; w < SMALL_WAVES; ++w)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            k[a] = min(k[a], red[a][w]);
            k[3 + a] = max(k[3 + a], red[3 + a][w]);
        }
    const SceneMap map = scene_map(k);
#pragma unroll
    for (int q = 0; q < SMALL_ITEMS; ++q) {
        const uint32_t i = (uint32_t)q * SMALL_THREADS + tid;
        if (i >= n) continue;
        double px, py, pz;
        map.point(box[q], px, py, pz);
        if (WIDE) {
            uint64_t lo, hi;
            morton128_of_point(px, py, pz, lo, hi);
            low[i] = lo;
            high[i] = hi;
            tk[i] = top_of_u128(hi);
            if (codes_hi_out) codes_hi_out[i] = hi;
            if (codes_out) codes_out[i] = lo;
        } else {
            const uint64_t code = morton64_of_point(px, py, pz);
            low[i] = code;
            tk[i] = top_of_u64(code);
            if (codes_out) codes_out[i] = code;
        }
        tv[i] = (uint16_t)i;
    }
    __syncthreads();

    // Four LSD passes over the tops; wave w owns positions [w * 64 * ITEMS, (w + 1) * 64 * ITEMS).  If they leave a run
    // of more than SMALL_RUN equal ones, the leaves are sorted again by all words of the codes, the lowest first:
    // ranking a run's members against each other grows with its square (2,048 leaves in one cell: build 1,097 -> 254
    // us; the look for such a run costs an evenly filled build 0.6 us).
    constexpr uint32_t TOP = WIDE ? 3u : 1u;  // the words: 31 bits and the top, or 32, 32, 30 and the top
    auto word_of = [&](uint32_t leaf, uint32_t w) {
        if (!WIDE) return w == 0u ? (uint32_t)low[leaf] & 0x7fffffffu : top_of_u64(low[leaf]);
        if (w < 2u) return (uint32_t)(low[leaf] >> (32u * w));
        return w == 2u ? (uint32_t)high[leaf] & 0x3fffffffu : top_of_u128(high[leaf]);
    };
    const uint64_t lt = lanemask_lt();
    bool whole = false;
    for (uint32_t w = TOP;;) {
        for (uint32_t shift = 0; shift < 32u; shift += 8u) {
            uint32_t key[SMALL_ITEMS], rank[SMALL_ITEMS];
            uint16_t val[SMALL_ITEMS];
            for (uint32_t d = lane; d < 256u; d += 64u) whist[wave][d] = 0u;
            wave_lds_fence();
#pragma unroll
            for (int j = 0; j < SMALL_ITEMS; ++j) {
                const uint32_t p = wave * (64u * SMALL_ITEMS) + (uint32_t)j * 64u + lane;
                const bool valid = p < n;
                key[j] = valid ? tk[p] : 0u;
                val[j] = valid ? tv[p] : (uint16_t)0;
                const uint32_t d = (key[j] >> shift) & 0xffu;
                uint64_t peers = ballot64(valid);
#pragma unroll
                for (int b = 0; b < 8; ++b) {
                    const bool bit = (d >> b) & 1u;
                    const uint64_t bm = ballot64(bit);
                    peers &= bit ? bm : ~bm;
                }
                const uint32_t below = (uint32_t)__popcll(peers & lt);
                uint32_t at = 0u;
                if (valid) at = whist[wave][d];
                wave_lds_fence();
                if (valid && below == 0u) whist[wave][d] = at + (uint32_t)__popcll(peers);
                wave_lds_fence();
                rank[j] = at + below;
            }
            __syncthreads();
            uint32_t run = 0u, incl = 0u;
            if (tid < 256u) {  // thread d: prefix of digit d across the waves, then across the digits
#pragma unroll
                for (int w = 0; w < SMALL_WAVES; ++w) {
                    const uint32_t c = whist[w][tid];
                    whist[w][tid] = run;
                    run += c;
                }
                incl = wave_inclusive_scan(run);
                if (lane == 63u) wtot[wave] = incl;
            }
            __syncthreads();
            if (tid < 256u) {
                uint32_t before = incl - run;
                for (uint32_t w = 0; w < wave; ++w) before += wtot[w];
#pragma unroll
                for (int w = 0; w < SMALL_WAVES; ++w) whist[w][tid] += before;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < SMALL_ITEMS; ++j) {
                const uint32_t p = wave * (64u * SMALL_ITEMS) + (uint32_t)j * 64u + lane;
                if (p < n) {
                    const uint32_t to = whist[wave][(key[j] >> shift) & 0xffu] + rank[j];
                    tk[to] = key[j];
                    tv[to] = val[j];
                }
            }
            __syncthreads();
        }
        if (whole) {
            if (w == TOP) break;
            ++w;
        } else {
            bool long_run = false;
#pragma unroll
            for (int q = 0; q < SMALL_ITEMS; ++q) {
                const uint32_t p = (uint32_t)q * SMALL_THREADS + tid;
                long_run |= p + SMALL_RUN < n && tk[p] == tk[p + SMALL_RUN];
            }
            if (!__syncthreads_or(long_run)) break;
            whole = true;
            w = 0u;
        }
#pragma unroll
        for (int q = 0; q < SMALL_ITEMS; ++q) {
            const uint32_t p = (uint32_t)q * SMALL_THREADS + tid;
            if (p >= n) continue;
            if (w == 0u) tv[p] = (uint16_t)p;
            tk[p] = word_of(tv[p], w);
        }
        __syncthreads();
    }

    // runs of equal tops by the remaining bits, ties by position
#pragma unroll
    for (int q = 0; q < SMALL_ITEMS; ++q) {
        const uint32_t p = (uint32_t)q * SMALL_THREADS + tid;
        if (p >= n) continue;
        const uint32_t t = tk[p], leaf = tv[p];
        uint32_t at = p;
        if (!whole) {
            uint32_t a = p, rank = 0u;
            while (a > 0u && tk[a - 1] == t) --a;
            const uint64_t l = low[leaf], h = WIDE ? high[leaf] : 0ull;
            for (uint32_t j = a; j < n && tk[j] == t; ++j) {
                const uint64_t jl = low[tv[j]], jh = WIDE ? high[tv[j]] : 0ull;
                const bool less = jh < h || (jh == h && (jl < l || (jl == l && j < p)));
                rank += less ? 1u : 0u;
            }
            at = a + rank;
        }
        store_node(&clusters[at], make_node(leaf_box(leaf), 1u, indices ? indices[leaf] : leaf));
        if (order_out) order_out[at] = leaf;
    }
}

// The neighbour search of one pass (ploc/mod.rs:329-419) and the per-tile counts of emitted clusters and merges in
// one launch.  Each cluster's best neighbour is the LAST minimum over its window in ascending index order (`<=`,
// find_best_node_basic ploc/mod.rs:508-528, equal to the cached search).  Besides its 256 clusters, a workgroup
// searches the r clusters on either side of its tile (the halo) with threads of their own (SC_THREADS = 256 +
// 2 * MAX_RADIUS), so that it classifies each of its clusters against its neighbour's choice (ploc/mod.rs:423-439)
// without another launch; the window in LDS spans [base - 2r, base + 256 + 2r).  Every workgroup writes its (emit,
// merge) counts, zero beyond the cluster count.
constexpr int SC_THREADS = T256 + 2 * (int)MAX_RADIUS;
constexpr int SC_WINDOW = T256 + 4 * (int)MAX_RADIUS;

// Best neighbour offset of cluster c over a window starting at cluster wstart.
__device__ __forceinline__ int8_t cluster_merge(const float (*s)[SC_WINDOW], int wstart, uint32_t c, uint32_t count,
                                                uint32_t r, uint32_t dist1, bool nonan, uint32_t* __restrict__ err) {
    const int lc = (int)c - wstart;
    const Box me{s[0][lc], s[1][lc], s[2][lc], s[3][lc], s[4][lc], s[5][lc]};
    if (dist1) {
        if (c == count - 1) return (int8_t)-1;
        const float cost = half_area(box_union(me, Box{s[0][lc + 1], s[1][lc + 1], s[2][lc + 1], s[3][lc + 1],
                                                      s[4][lc + 1], s[5][lc + 1]}));
        float last = INFINITY;
        if (c > 0)
            last = half_area(box_union(Box{s[0][lc - 1], s[1][lc - 1], s[2][lc - 1], s[3][lc - 1], s[4][lc - 1],
                                           s[5][lc - 1]},
                                       me));
        return last < cost ? (int8_t)-1 : (int8_t)1;
    }
    const uint32_t begin = c - min(r, c);
    const uint32_t end = min(c + r + 1u, count);
    uint32_t best = c;
    float best_cost = INFINITY;
    for (uint32_t j = begin; j < end; ++j) {
        if (j == c) continue;
        const int o = (int)j - wstart;
        const Box ob{s[0][o], s[1][o], s[2][o], s[3][o], s[4][o], s[5][o]};
        const float cost = nonan ? union_area_nonan(me, ob) : half_area(box_union(me, ob));
        if (cost <= best_cost) {
            best = j;
            best_cost = cost;
        }
    }
    if (best == c) atomicOr(err, DERR_SELF_MERGE);
    return (int8_t)((int)best - (int)c);
}

// The same search for a distance R known at compile time, over a window whose slots outside [0, count) hold NaN
// boxes: a NaN cost never passes `cost <= best_cost`, so the unrolled offsets -R..R (ascending, as j ascends) pick
// what the bounded loop picks, with the LDS addresses as immediates and no per-neighbour bounds test.
template <int R, bool NONAN>
__device__ __forceinline__ int cluster_merge_unrolled(const float* __restrict__ x0, const float* __restrict__ y0,
                                                      const float* __restrict__ z0, const float* __restrict__ x1,
                                                      const float* __restrict__ y1, const float* __restrict__ z1,
                                                      int lc) {
    // U neighbours per unrolled block (U divides R); the blocks themselves stay a loop so that the compiler does
    // not hoist every neighbour's loads (2R boxes would not fit the registers).
    constexpr int U = R <= 8 ? R : (R % 8 == 0 ? 8 : (R % 7 == 0 ? 7 : 6));
    static_assert(R % U == 0, "block size must divide the distance");
    const Box me{x0[lc], y0[lc], z0[lc], x1[lc], y1[lc], z1[lc]};
    int best = 0;
    float best_cost = INFINITY;
    auto block = [&](int k0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u;
            const int o = lc + k;
            const Box ob{x0[o], y0[o], z0[o], x1[o], y1[o], z1[o]};
            const float cost = NONAN ? union_area_nonan(me, ob) : half_area(box_union(me, ob));
            if (cost <= best_cost) {
                best = k;
                best_cost = cost;
            }
        }
    };
#pragma unroll 1
    for (int k0 = -R; k0 < 0; k0 += U) block(k0);
#pragma unroll 1
    for (int k0 = 1; k0 <= R; k0 += U) block(k0);
    return best;
}

// Symmetric form of the unrolled search for a NaN-free window: union_area_nonan(a, b) == union_area_nonan(b, a) bit
// for bit (IEEE minimum / maximum are commutative, signed zeros included), so slot w computes its R right-hand pair
// costs once into pc[k - 1][w] and a cluster reads its left-hand costs from the slots before it.
template <int R>
__device__ __forceinline__ void pair_costs(const float (*s)[SC_WINDOW], float (*pc)[SC_WINDOW], int w) {
    constexpr int U = R <= 8 ? R : (R % 8 == 0 ? 8 : (R % 7 == 0 ? 7 : 6));
    const Box me{s[0][w], s[1][w], s[2][w], s[3][w], s[4][w], s[5][w]};
#pragma unroll 1
    for (int k0 = 1; k0 <= R; k0 += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u, o = w + k;
            pc[k - 1][w] = union_area_nonan(me, Box{s[0][o], s[1][o], s[2][o], s[3][o], s[4][o], s[5][o]});
        }
    }
}

// The pick over the pair costs: offsets -R..-1 then 1..R (j ascending), the last minimum, as cluster_merge_unrolled.
template <int R>
__device__ __forceinline__ int pick_from_pairs(const float (*pc)[SC_WINDOW], int lc) {
    int best = 0;
    float best_cost = INFINITY;
#pragma unroll
    for (int k = R; k >= 1; --k) {
        const float cost = pc[k - 1][lc - k];
        if (cost <= best_cost) {
            best = -k;
            best_cost = cost;
        }
    }
#pragma unroll
    for (int k = 1; k <= R; ++k) {
        const float cost = pc[k - 1][lc];
        if (cost <= best_cost) {
            best = k;
            best_cost = cost;
        }
    }
    return best;
}

// R > 0: the search distance r, known at compile time (unrolled search over a NaN-padded window); R = 0: any r.
template <int R>
__global__ void __launch_bounds__(SC_THREADS) k_ploc_search_count(const Node32* __restrict__ cur, Misc* misc,
                                                                  uint32_t slot, uint32_t r, uint32_t dist1,
                                                                  int8_t* __restrict__ merge,
                                                                  uint2* __restrict__ blocksums, uint32_t grouped) {
    __shared__ float s[6][SC_WINDOW];
    __shared__ int8_t mm[T256 + 2 * MAX_RADIUS];  // offsets of clusters [base - r, base + 256 + r)
    __shared__ uint32_t we[T256 / 64], wm[T256 / 64];
    const uint32_t count = misc->state[slot].count;
    const uint32_t base = blockIdx.x * T256;
    if (count <= 1 || base >= count) {  // workgroup-uniform
        if (threadIdx.x == 0)
            blocksums[blockIdx.x] = count == 1 && blockIdx.x == 0 ? make_uint2(1u, 0u) : make_uint2(0u, 0u);
        return;  // a single cluster's pass changes nothing: its group stays empty
    }
    const int wstart = (int)base - 2 * (int)r;
    const int wlen = T256 + 4 * (int)r;
    bool nan_here = false;
    for (int w = threadIdx.x; w < wlen; w += SC_THREADS) {
        const int g = wstart + w;
        if (g >= 0 && (uint32_t)g < count) {
            const Node32 nd = load_node(&cur[g]);
            s[0][w] = nd.minx;
            s[1][w] = nd.miny;
            s[2][w] = nd.minz;
            s[3][w] = nd.maxx;
            s[4][w] = nd.maxy;
            s[5][w] = nd.maxz;
            nan_here |= box_has_nan_any(node_box(nd));
        } else if (R > 0) {
#pragma unroll
            for (int a = 0; a < 6; ++a) s[a][w] = __builtin_nanf("");
        }
    }
    const bool nonan = !__syncthreads_or(nan_here);  // NaN-free window: costs from union_area_nonan
    // thread t < 256: cluster base + t; thread 256 + h, h < 2r: halo cluster base - r + h or base + 256 + h - r
    const uint32_t t = threadIdx.x;
    // NaN-free windows: every pair cost once (the searchers sit at slots [R, 256 + 3R), their partners below 256 + 4R)
    __shared__ float pcost[R > 0 ? R : 1][SC_WINDOW];
    const bool pairs = R > 0 && !dist1 && nonan;  // workgroup-uniform
    if constexpr (R > 0) {
        if (pairs) {
            for (int w = (int)t; w < T256 + 3 * R; w += SC_THREADS) pair_costs<R>(s, pcost, w);
            __syncthreads();
        }
    }
    int c = -1;
    if (t < (uint32_t)T256) c = (int)(base + t);
    else if (t - T256 < 2u * r) c = t - T256 < r ? (int)base - (int)r + (int)(t - T256) : (int)(base + t - r);
    if (c >= 0 && (uint32_t)c < count) {
        int8_t m = 0;
        bool unrolled = false;
        if constexpr (R > 0) {
            if (!dist1) {
                const int lc = c - wstart;
                const int b = pairs ? pick_from_pairs<R>(pcost, lc)
                                    : cluster_merge_unrolled<R, false>(s[0], s[1], s[2], s[3], s[4], s[5], lc);
                if (b == 0) atomicOr(&misc->err, DERR_SELF_MERGE);
                m = (int8_t)b;
                unrolled = true;
            }
        }
        if (!unrolled) m = cluster_merge(s, wstart, (uint32_t)c, count, r, dist1, nonan, &misc->err);
        mm[c - ((int)base - (int)r)] = m;
        if (t < (uint32_t)T256) merge[c] = m;
    }
    __syncthreads();
    // classify (ploc/mod.rs:423-439) the tile's clusters from the offsets in LDS
    bool emit = false, mrg = false;
    if (t < (uint32_t)T256 && base + t < count) {
        const int i = (int)(base + t);
        const int bi = i + (int)mm[i - ((int)base - (int)r)];
        const bool mutual = bi + (int)mm[bi - ((int)base - (int)r)] == i;
        if (!mutual || bi == i) {
            emit = true;
        } else if (bi < i) {
            emit = true;
            mrg = true;
        }
    }
    const uint64_t be = __ballot(emit), bm = __ballot(mrg);
    const uint32_t wave = t >> 6;
    if ((t & 63u) == 0 && wave < (uint32_t)(T256 / 64)) {
        we[wave] = (uint32_t)__popcll(be);
        wm[wave] = (uint32_t)__popcll(bm);
    }
    __syncthreads();
    if (t == 0) {
        uint32_t E = 0, M = 0;
        for (int w = 0; w < T256 / 64; ++w) {
            E += we[w];
            M += wm[w];
        }
        blocksums[blockIdx.x] = make_uint2(E, M);
        if (grouped) atomicAdd(&misc->groups[slot][blockIdx.x / GROUP_TILES], (unsigned long long)M << 32 | E);
    }
}

// Two-level scan of the tile counts for passes of more than GROUP_MAX_TILES tiles: k_ploc_scan_chunks sums SCAN_CHUNK
// counts per workgroup, k_ploc_scan_apply offsets each chunk by the chunks before it and scans it, and its workgroup 0
// writes the next pass's state.
__global__ void __launch_bounds__(1024) k_ploc_scan_chunks(const uint2* __restrict__ blocksums, uint32_t nblocks,
                                                           uint2* __restrict__ chunk_tot) {
    scan_chunk_total(blocksums, nblocks, chunk_tot);
}

__global__ void __launch_bounds__(1024) k_ploc_scan_apply(uint2* __restrict__ blocksums, uint32_t nblocks,
                                                          const uint2* __restrict__ chunk_tot, uint32_t nchunks,
                                                          Misc* misc, uint32_t slot, uint32_t* __restrict__ hist) {
    const uint2 all = scan_chunk_apply(blocksums, nblocks, chunk_tot, nchunks);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const PlocState st = misc->state[slot];
        PlocState nx = st;
        if (st.count > 1) {
            nx.count = all.x;
            nx.insert = st.insert - 2u * all.y;
            nx.depth = st.depth + 1u;
            nx.cluster_sum = st.cluster_sum + st.count;
            hist[nx.depth] = nx.insert;
        }
        misc->state[slot ^ 1u] = nx;
    }
}

// Merges of a tile: a merge is counted at its higher cluster; pairs inside the tile use two of its clusters, and at most
// r of its clusters pair with distinct clusters in [base - r, base): at most 128 + r / 2.
constexpr uint32_t MAX_TILE_MERGES = (T256 + MAX_RADIUS) / 2;

// Compaction of one 256-cluster tile (ploc/mod.rs:420-493): kept clusters and the parents of mutual pairs go to
// `next` in order; a merge's two children go to the slots below the pass's insert index in the serial loop's order
// (`pe0` / `pm0`: the emits and merges of the tiles before this one).  The tile's merges are then
// listed in LDS and their cost-table entries evaluated by consecutive threads, so that a pass where a fifth of the
// clusters merge runs the evaluation in about one wave per tile instead of in every wave with a few lanes active.
// The caller classifies its cluster and loads its node (`a`, for i < count) at the start of the kernel, so that
// those loads overlap the tile offsets' loads.  Called by every thread of the workgroup (it holds workgroup
// barriers, for LDS only: the clusters' stores are not waited for).
__device__ __forceinline__ void compact_tile(const Node32* __restrict__ cur, Node32* __restrict__ next,
                                             const Node32& a, bool emit, bool mrg, uint32_t b,
                                             const PlocState& st, uint32_t pe0, uint32_t pm0,
                                             Node32* __restrict__ bvh_nodes,
                                             const DpView& dp, uint32_t fused, const uint32_t* __restrict__ slot_map,
                                             uint32_t vtop, uint32_t map_len, uint32_t* __restrict__ err,
                                             uint32_t* we, uint32_t* wm) {
    __shared__ __align__(16) Node32 s_left[MAX_TILE_MERGES], s_right[MAX_TILE_MERGES];
    __shared__ uint32_t s_first[MAX_TILE_MERGES];
    const uint64_t be = __ballot(emit), bm = __ballot(mrg);
    const uint64_t lt = lanemask_lt();
    const uint32_t wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0) {
        we[wave] = (uint32_t)__popcll(be);
        wm[wave] = (uint32_t)__popcll(bm);
    }
    lds_barrier();
    if (emit) {
        uint32_t pe = pe0, pm = pm0;
        for (uint32_t w = 0; w < wave; ++w) {
            pe += we[w];
            pm += wm[w];
        }
        const uint32_t pos = pe + (uint32_t)__popcll(be & lt);
        if (mrg) {
            const uint32_t sq = pm + (uint32_t)__popcll(bm & lt);
            const Node32 c = load_node(&cur[b]);
            uint32_t first;
            const uint32_t q = sq - pm0;  // the merge's rank in this tile
            if (q >= MAX_TILE_MERGES || !child_slot(st.insert - 2u * (sq + 1u), slot_map, vtop, map_len, first)) {
                atomicOr(err, DERR_CAPACITY);
                if (q < MAX_TILE_MERGES) s_first[q] = UINT32_MAX;
            } else {
                store_node(&next[pos], make_node(box_union(node_box(a), node_box(c)), 0u, first));
                s_left[q] = a;
                s_right[q] = c;
                s_first[q] = first;
            }
        } else {
            store_node(&next[pos], a);
        }
    }
    lds_barrier();
    const uint32_t nm = min(wm[0] + wm[1] + wm[2] + wm[3], MAX_TILE_MERGES);
    if (wave * 64u >= nm) return;
    store_pairs(s_left, s_right, wave, nm, bvh_nodes,
                [&](uint32_t q) { return s_first[q] == UINT32_MAX ? SIZE_MAX : (size_t)s_first[q]; });
    if (!fused) return;  // uniform
    const bool entry = threadIdx.x < nm && s_first[threadIdx.x] != UINT32_MAX;
    Node32 l{}, r{};
    l.prim_count = r.prim_count = 1u;
    uint32_t first = 0u;
    if (entry) {
        l = s_left[threadIdx.x];
        r = s_right[threadIdx.x];
        first = s_first[threadIdx.x];
    }
    const Box box = box_union(node_box(l), node_box(r));
    uint32_t e;
    if (wave < 2u) {  // the wave's entries of s_left are in its lanes' registers now: 2 KB of LDS
        e = dp_evaluate_wave(dp, box, first, l, r, entry, reinterpret_cast<uint4*>(&s_left[wave * 64u]));
    } else {
        e = entry ? dp_evaluate(dp, box, first, l, r) : 0u;
    }
    if (e) atomicOr(err, e);
}

// Emits and merges of the first `n` groups, plus the lanes' own e and m, in every lane of the wave.
__device__ __forceinline__ uint2 group_sums(const unsigned long long* groups, uint32_t n, uint32_t e, uint32_t m) {
    for (uint32_t g = threadIdx.x & 63u; g < n; g += 64u) {
        const unsigned long long x = groups[g];
        e += (uint32_t)x;
        m += (uint32_t)(x >> 32);
    }
    e = wave_inclusive_scan_dpp(e);
    m = wave_inclusive_scan_dpp(m);
    return make_uint2((uint32_t)__builtin_amdgcn_readlane((int)e, 63), (uint32_t)__builtin_amdgcn_readlane((int)m, 63));
}

__global__ void __launch_bounds__(T256) k_ploc_compact(const Node32* __restrict__ cur, Node32* __restrict__ next,
                                                       const int8_t* __restrict__ merge, Misc* misc, uint32_t slot,
                                                       const uint2* __restrict__ counts, uint32_t grouped,
                                                       Node32* __restrict__ bvh_nodes, DpView dp, uint32_t fused,
                                                       const uint32_t* __restrict__ slot_map, uint32_t vtop,
                                                       uint32_t map_len, uint32_t* __restrict__ hist) {
    __shared__ uint32_t we[T256 / 64], wm[T256 / 64];
    const PlocState st = misc->state[slot];
    if (grouped && blockIdx.x == 0) {  // the state after the pass; the other slot's groups for the next one
        for (uint32_t g = threadIdx.x; g < TILE_GROUPS; g += T256) misc->groups[slot ^ 1u][g] = 0ull;
        if (threadIdx.x < 64u) {
            const uint2 all = group_sums(misc->groups[slot], (gridDim.x + GROUP_TILES - 1u) / GROUP_TILES, 0u, 0u);
            if (threadIdx.x == 0) {
                PlocState nx = st;
                if (st.count > 1u) {
                    nx.count = all.x;
                    nx.insert = st.insert - 2u * all.y;
                    nx.depth = st.depth + 1u;
                    nx.cluster_sum = st.cluster_sum + st.count;
                    hist[nx.depth] = nx.insert;
                }
                misc->state[slot ^ 1u] = nx;
            }
        }
    }
    if (blockIdx.x * T256 >= st.count) return;
    const uint32_t i = blockIdx.x * T256 + threadIdx.x;
    Node32 a{};
    if (i < st.count) a = load_node(&cur[i]);
    const Cls k = classify(merge, i, st.count);
    uint2 off;
    if (grouped) {  // in every wave by itself: no barrier
        const uint32_t g0 = blockIdx.x / GROUP_TILES, tile = g0 * GROUP_TILES + (threadIdx.x & 63u);  // those below its own
        uint2 v = make_uint2(0u, 0u);
        if (tile < blockIdx.x) v = counts[tile];
        off = group_sums(misc->groups[slot], g0, v.x, v.y);
    } else {
        off = counts[blockIdx.x];
    }
    compact_tile(cur, next, a, k.emit, k.mrg, k.b, st, off.x, off.y, bvh_nodes, dp, fused, slot_map, vtop, map_len,
                 &misc->err, we, wm);
}

// ---- passes of at most PASS_TILES tiles: one launch per pass ----
// A pass's compaction needs the emits and merges of every tile before a cluster's (a scan over the tiles), so it is a
// launch behind the search.  Here it is left to the next pass's launch: a tile leaves its emitted clusters at the front
// of its own 256 slots (with its counts) and its merges in a list, and the next launch starts with the scan of the
// counts (every workgroup scans them all, at most 1,024), finds its own 256 clusters and their window by it, and, with
// other waves than those that search, gives the listed merges of tile blockIdx.x their slots, writes their children
// and evaluates their cost-table entries.  A parent emitted by the pass before carries MERGE_RANK and its merge's rank
// in its tile in the place of its first_index until then.  k_ploc_flush ends a run of such passes: dense clusters, the
// last merges, the state.  The loads of a merge's entry are issued a barrier ahead of their use, so they run under the
// search.  Latency bounds these passes (2.5 us of each launch are the launch): 1.29M-triangle build, 675 tiles down
// to 26: 11.6 -> 9.0 us a pass (65,536 triangles, 256 tiles down to 9: 11.4 -> 7.8).
constexpr uint32_t PASS_TILES = 1024;
constexpr int PASS_THREADS = 512;
constexpr uint32_t MERGE_RANK = 0x80000000u;                       // prim_count of such a parent
constexpr uint32_t PASS_MERGE_THREAD0 = (uint32_t)SC_THREADS;      // threads from here on take a merge each
static_assert(PASS_THREADS - (int)PASS_MERGE_THREAD0 >= (int)MAX_TILE_MERGES, "a thread per merge");

struct PassMerge {
    Node32 left, right;
};

// The tiles' counts before a pass, scanned: for tile t the clusters and merges of the tiles before it.
struct PassScan {
    uint32_t emits[PASS_TILES + 1], merges[PASS_TILES + 1];
    uint32_t wave_e[PASS_THREADS / 64], wave_m[PASS_THREADS / 64];
};

// Fills ps for ntiles counts; ends with a barrier.  Every thread calls.
__device__ __forceinline__ void pass_scan(const uint2* __restrict__ counts, uint32_t ntiles, PassScan& ps) {
    const uint32_t tid = threadIdx.x, wave = tid >> 6, t = 2u * tid;
    const uint2 c0 = t < ntiles ? counts[t] : make_uint2(0u, 0u);
    const uint2 c1 = t + 1u < ntiles ? counts[t + 1u] : make_uint2(0u, 0u);
    const uint32_t ie = wave_inclusive_scan_dpp(c0.x + c1.x), im = wave_inclusive_scan_dpp(c0.y + c1.y);
    if ((tid & 63u) == 63u) {
        ps.wave_e[wave] = ie;
        ps.wave_m[wave] = im;
    }
    lds_barrier();
    uint32_t e = ie - (c0.x + c1.x), m = im - (c0.y + c1.y);
#pragma unroll
    for (uint32_t w = 0; w < PASS_THREADS / 64; ++w) {
        e += w < wave ? ps.wave_e[w] : 0u;
        m += w < wave ? ps.wave_m[w] : 0u;
    }
    ps.emits[t] = e;
    ps.merges[t] = m;
    ps.emits[t + 1u] = e + c0.x;
    ps.merges[t + 1u] = m + c0.y;
    if (tid == (uint32_t)PASS_THREADS - 1u) {
        ps.emits[t + 2u] = e + c0.x + c1.x;
        ps.merges[t + 2u] = m + c0.y + c1.y;
    }
    lds_barrier();
}

// The state after the pass that state `st` was before.
__device__ __forceinline__ PlocState pass_next(const PlocState& st, const PassScan& ps) {
    PlocState nx = st;
    if (st.count > 1u) {
        nx.count = ps.emits[PASS_TILES];
        nx.insert = st.insert - 2u * ps.merges[PASS_TILES];
        nx.depth = st.depth + 1u;
        nx.cluster_sum = st.cluster_sum + st.count;
    }
    return nx;
}

// A cluster of tile t as the pass before left it: a parent's rank becomes its first child slot.
__device__ __forceinline__ Node32 pass_cluster(Node32 c, uint32_t merges_before, const PlocState& st,
                                               const uint32_t* __restrict__ slot_map, uint32_t vtop, uint32_t map_len) {
    if (c.prim_count == MERGE_RANK) {
        uint32_t first = 0u;
        (void)child_slot(st.insert - 2u * (merges_before + c.first_index + 1u), slot_map, vtop, map_len, first);
        c.prim_count = 0u;
        c.first_index = first;
    }
    return c;
}

// One pass over the clusters in `cur`: dense (`ntiles` = 0) or as a pass left them in ntiles tiles with `counts`
// and `merges_in`; the result goes to next, counts_out and merges_out, a tile per workgroup.
template <int R>
__global__ void __launch_bounds__(PASS_THREADS)
    k_ploc_pass(const Node32* __restrict__ cur, Node32* __restrict__ next, const uint2* __restrict__ counts,
                uint32_t ntiles, uint2* __restrict__ counts_out, const PassMerge* __restrict__ merges_in,
                PassMerge* __restrict__ merges_out, Misc* misc, uint32_t slot, uint32_t r, uint32_t dist1,
                Node32* __restrict__ bvh_nodes, DpView dp, uint32_t fused, const uint32_t* __restrict__ slot_map,
                uint32_t vtop, uint32_t map_len, uint32_t* __restrict__ hist) {
    __shared__ PassScan ps;
    __shared__ float s[6][SC_WINDOW];
    __shared__ uint32_t w_pc[SC_WINDOW], w_fi[SC_WINDOW];  // of clusters from base - r on
    __shared__ int8_t mm[T256 + 2 * MAX_RADIUS];  // offsets of clusters [base - r, base + 256 + r)
    __shared__ float pcost[R > 0 ? R : 1][SC_WINDOW];
    __shared__ uint32_t we[T256 / 64], wm[T256 / 64], w_nan[PASS_THREADS / 64], s_tile0;
    const uint32_t t = threadIdx.x, base = blockIdx.x * T256;
    const PlocState st = misc->state[slot];
    const bool dense = ntiles == 0u;
    PlocState nx = st;
    const int wstart = (int)base - 2 * (int)r, wlen = T256 + 4 * (int)r;
    if (!dense) {
        pass_scan(counts, ntiles, ps);
        nx = pass_next(st, ps);
    }
    if (blockIdx.x == 0 && t == 0) {
        misc->state[slot ^ 1u] = nx;
        if (!dense && st.count > 1u) hist[nx.depth] = nx.insert;
    }
    const uint32_t count = nx.count;
    const bool search = count > 1u && base < count;  // workgroup-uniform
    // the merges of tile blockIdx.x of the pass before: their nodes are loaded now
    const uint32_t mj = t - PASS_MERGE_THREAD0;
    const uint32_t my_merges = !dense && blockIdx.x < ntiles ? ps.merges[blockIdx.x + 1u] - ps.merges[blockIdx.x] : 0u;
    const bool merging = t >= PASS_MERGE_THREAD0 && mj < my_merges;
    Node32 ml{}, mr{};
    if (merging) {
        const PassMerge* pm = &merges_in[(size_t)blockIdx.x * MAX_TILE_MERGES + mj];
        ml = load_node(&pm->left);
        mr = load_node(&pm->right);
    }
    if (!search) {  // beyond the clusters, or a lone cluster, which goes through
        if (t == 0) {
            const bool lone = count == 1u && blockIdx.x == 0;
            if (lone) {
                uint32_t tile = 0u;
                if (!dense)
                    while (ps.emits[tile + 1u] == 0u) ++tile;
                store_node(&next[0], pass_cluster(load_node(&cur[(size_t)tile * T256]), dense ? 0u : ps.merges[tile], st,
                                                  slot_map, vtop, map_len));
            }
            counts_out[blockIdx.x] = make_uint2(lone ? 1u : 0u, 0u);
        }
        if (my_merges == 0u) return;
    }
    bool nan_here = false;
    if (search) {
        auto put = [&](int w, const Node32& nd) {
            s[0][w] = nd.minx;
            s[1][w] = nd.miny;
            s[2][w] = nd.minz;
            s[3][w] = nd.maxx;
            s[4][w] = nd.maxy;
            s[5][w] = nd.maxz;
            w_pc[w] = nd.prim_count;
            w_fi[w] = nd.first_index;
            nan_here |= box_has_nan_any(node_box(nd));
        };
        for (int w = (int)t; w < wlen; w += PASS_THREADS) {
            const int g = wstart + w;
            if (g >= 0 && (uint32_t)g < count) {
                if (dense) put(w, load_node(&cur[g]));
            } else if (R > 0) {
#pragma unroll
                for (int a = 0; a < 6; ++a) s[a][w] = __builtin_nanf("");
            }
        }
        if (!dense) {
            // the tile that holds the window's first cluster, then the tiles up to its last, two at a time
            const uint32_t w0 = wstart > 0 ? (uint32_t)wstart : 0u, w1 = min(count, (uint32_t)(wstart + wlen));
#pragma unroll
            for (uint32_t k = 0; k < 2u; ++k) {
                const uint32_t tile = 2u * t + k;
                if (ps.emits[tile] <= w0 && ps.emits[tile + 1u] > w0) s_tile0 = tile;
            }
            lds_barrier();
            for (uint32_t tile = s_tile0 + (t >> 8); tile < ntiles && ps.emits[tile] < w1; tile += PASS_THREADS / T256) {
                const uint32_t first = ps.emits[tile], g = first + (t & 255u);
                if (g < ps.emits[tile + 1u] && g >= w0 && g < w1)
                    put((int)g - wstart, pass_cluster(load_node(&cur[(size_t)tile * T256 + (t & 255u)]),
                                                      ps.merges[tile], st, slot_map, vtop, map_len));
            }
        }
    }
    // the merges' slots, children and table records
    uint32_t mfirst = 0u;
    DpRaw raw_l, raw_r;
    if (merging) {
        if (!child_slot(st.insert - 2u * (ps.merges[blockIdx.x] + mj + 1u), slot_map, vtop, map_len, mfirst)) {
            atomicOr(&misc->err, DERR_CAPACITY);
            mfirst = UINT32_MAX;
        } else {
            store_node(&bvh_nodes[mfirst], ml);
            store_node(&bvh_nodes[mfirst + 1u], mr);
            if (fused) {
                raw_l = load_dp_raw(dp_child_record(dp, ml));
                raw_r = load_dp_raw(dp_child_record(dp, mr));
            }
        }
    }
    if ((t & 63u) == 0u) w_nan[t >> 6] = 0u;
    wave_lds_fence();
    if (nan_here) w_nan[t >> 6] = 1u;
    lds_barrier();
    uint32_t any_nan = 0u;
#pragma unroll
    for (uint32_t w = 0; w < PASS_THREADS / 64; ++w) any_nan |= w_nan[w];
    const bool nonan = any_nan == 0u;  // NaN-free window: costs from union_area_nonan
    const bool pairs = R > 0 && !dist1 && nonan;  // workgroup-uniform
    if constexpr (R > 0) {
        if (search && pairs) {
            if (t < PASS_MERGE_THREAD0)
                for (int w = (int)t; w < T256 + 3 * R; w += SC_THREADS) pair_costs<R>(s, pcost, w);
        }
    }
    if (search && pairs) lds_barrier();
    // thread t < 256: cluster base + t; thread 256 + h, h < 2r: halo cluster base - r + h or base + 256 + h - r
    int c = -1;
    if (t < (uint32_t)T256) c = (int)(base + t);
    else if (t - T256 < 2u * r) c = t - T256 < r ? (int)base - (int)r + (int)(t - T256) : (int)(base + t - r);
    if (search && c >= 0 && (uint32_t)c < count) {
        int8_t m = 0;
        bool unrolled = false;
        if constexpr (R > 0) {
            if (!dist1) {
                const int lc = c - wstart;
                const int b = pairs ? pick_from_pairs<R>(pcost, lc)
                                    : cluster_merge_unrolled<R, false>(s[0], s[1], s[2], s[3], s[4], s[5], lc);
                if (b == 0) atomicOr(&misc->err, DERR_SELF_MERGE);
                m = (int8_t)b;
                unrolled = true;
            }
        }
        if (!unrolled) m = cluster_merge(s, wstart, (uint32_t)c, count, r, dist1, nonan, &misc->err);
        mm[c - ((int)base - (int)r)] = m;
    }
    if (fused && merging && mfirst != UINT32_MAX) {
        const uint32_t e = dp_evaluate(dp, half_area(box_union(node_box(ml), node_box(mr))), mfirst,
                                       dp_child(ml), dp_child(mr), raw_l, raw_r);
        if (e) atomicOr(&misc->err, e);
    }
    lds_barrier();
    // classify (ploc/mod.rs:423-439) the tile's clusters from the offsets in LDS
    bool emit = false, mrg = false;
    int partner = 0;
    if (search && t < (uint32_t)T256 && base + t < count) {
        const int i = (int)(base + t);
        partner = i + (int)mm[i - ((int)base - (int)r)];
        const bool mutual = partner + (int)mm[partner - ((int)base - (int)r)] == i;
        emit = !mutual || partner <= i;
        mrg = mutual && partner < i;
    }
    const uint64_t be = __ballot(emit), bm = __ballot(mrg);
    const uint32_t wave = t >> 6;
    if ((t & 63u) == 0 && wave < (uint32_t)(T256 / 64)) {
        we[wave] = (uint32_t)__popcll(be);
        wm[wave] = (uint32_t)__popcll(bm);
    }
    lds_barrier();
    if (t == 0 && search) {
        uint32_t E = 0, M = 0;
        for (int w = 0; w < T256 / 64; ++w) {
            E += we[w];
            M += wm[w];
        }
        counts_out[blockIdx.x] = make_uint2(E, M);
    }
    if (!emit) return;
    uint32_t pe = 0u, pm = 0u;
    for (uint32_t w = 0; w < wave; ++w) {
        pe += we[w];
        pm += wm[w];
    }
    pe += (uint32_t)__popcll(be & lanemask_lt());
    auto cluster = [&](int g) {
        const int w = g - wstart;
        return Node32{s[0][w], s[1][w], s[2][w], w_pc[w], s[3][w], s[4][w], s[5][w], w_fi[w]};
    };
    Node32 out = cluster((int)(base + t));
    if (mrg) {
        pm += (uint32_t)__popcll(bm & lanemask_lt());
        if (pm < MAX_TILE_MERGES) {
            const Node32 b = cluster(partner);
            PassMerge* o = &merges_out[(size_t)blockIdx.x * MAX_TILE_MERGES + pm];
            store_node(&o->left, out);
            store_node(&o->right, b);
            out = make_node(box_union(node_box(out), node_box(b)), MERGE_RANK, pm);
        } else {
            atomicOr(&misc->err, DERR_CAPACITY);
        }
    }
    store_node(&next[(size_t)base + pe], out);
}

// The end of a run of k_ploc_pass launches: the clusters of the last one's tiles, dense, and its merges.
__global__ void __launch_bounds__(PASS_THREADS)
    k_ploc_flush(const Node32* __restrict__ cur, Node32* __restrict__ next, const uint2* __restrict__ counts,
                 uint32_t ntiles, const PassMerge* __restrict__ merges_in, Misc* misc, uint32_t slot,
                 Node32* __restrict__ bvh_nodes, DpView dp, uint32_t fused, const uint32_t* __restrict__ slot_map,
                 uint32_t vtop, uint32_t map_len, uint32_t* __restrict__ hist) {
    __shared__ PassScan ps;
    const uint32_t t = threadIdx.x, tile = blockIdx.x;
    const PlocState st = misc->state[slot];
    pass_scan(counts, ntiles, ps);
    const PlocState nx = pass_next(st, ps);
    if (tile == 0 && t == 0) {
        misc->state[slot ^ 1u] = nx;
        if (st.count > 1u) hist[nx.depth] = nx.insert;
    }
    const uint32_t mb = ps.merges[tile], nm = ps.merges[tile + 1u] - mb;
    if (t < T256 && ps.emits[tile] + t < ps.emits[tile + 1u])
        store_node(&next[ps.emits[tile] + t],
                   pass_cluster(load_node(&cur[(size_t)tile * T256 + t]), mb, st, slot_map, vtop, map_len));
    const uint32_t mj = t - PASS_MERGE_THREAD0;
    if (t < PASS_MERGE_THREAD0 || mj >= nm) return;
    const PassMerge* pm = &merges_in[(size_t)tile * MAX_TILE_MERGES + mj];
    const Node32 l = load_node(&pm->left), r = load_node(&pm->right);
    uint32_t first;
    if (!child_slot(st.insert - 2u * (mb + mj + 1u), slot_map, vtop, map_len, first)) {
        atomicOr(&misc->err, DERR_CAPACITY);
        return;
    }
    store_node(&bvh_nodes[first], l);
    store_node(&bvh_nodes[first + 1u], r);
    if (fused) {
        const uint32_t e = dp_evaluate(dp, box_union(node_box(l), node_box(r)), first, l, r);
        if (e) atomicOr(&misc->err, e);
    }
}

// The one-workgroup tail of a build (tail.hpp) once at most TAIL_MAX clusters remain.
template <int R>
__global__ void __launch_bounds__(TAIL_THREADS) k_ploc_tail(const Node32* __restrict__ cur, Misc* misc,
                                                            uint32_t slot, uint32_t first_pass, uint32_t r,
                                                            uint32_t sd_is_one, uint32_t depth_threshold,
                                                            Node32* __restrict__ bvh_nodes,
                                                            uint32_t* __restrict__ hist, DpView dp, uint32_t fused,
                                                            const uint32_t* __restrict__ slot_map, uint32_t vtop,
                                                            uint32_t map_len) {
    PlocState st = misc->state[slot];
    if (st.count > TAIL_MAX) {
        if (threadIdx.x == 0) atomicOr(&misc->err, DERR_CAPACITY);
        return;
    }
    ploc_tail<R, TAIL_MAX>(cur, st, first_pass, r, sd_is_one, depth_threshold, bvh_nodes, hist, dp, fused, slot_map,
                           vtop, map_len, &misc->err);
    if (threadIdx.x == 0) {
        misc->state[slot] = st;
        if (fused && st.insert == 1u) misc->info = root_info(bvh_nodes, dp);  // a finished tree
    }
}

}  // namespace

hipError_t DevBuf::ensure(size_t want) {
    if (want <= bytes && ptr) return hipSuccess;
    release();
    size_t sz = want < 256 ? 256 : want;
    hipError_t e = hipMalloc(&ptr, sz);
    if (e != hipSuccess) {
        ptr = nullptr;
        bytes = 0;
        return e;
    }
    bytes = sz;
    return hipSuccess;
}

void DevBuf::release() {
    if (ptr) (void)hipFree(ptr);
    ptr = nullptr;
    bytes = 0;
}

#define OBVHS_TRY(expr, where)                                              \
    do {                                                                    \
        hipError_t _e = (expr);                                             \
        if (_e != hipSuccess) return set_hip_error(ctx, _e, where);         \
    } while (0)

// Sorts the leaf indices vals[0..n) by their whole Morton codes, ties in leaf order (ploc/mod.rs:811-827): stable sorts
// by 32 bits of the code at a time, the lowest first, the words gathered in the order so far.  The codes stay in leaf
// order.  Eight passes of 20 bytes a key and two gathers (16.8M leaves: 1.23 ms) where a sort of 64-bit keys makes
// eight of 32 bytes.
static obvhs_status sort_codes(obvhs_context* ctx, const uint64_t* keys, const uint64_t* keys_hi, uint32_t* vals,
                               uint32_t n) {
    hipStream_t st = ctx->stream;
    BuildScratch& S = ctx->scratch;
    uint32_t* words = S.tops.as<uint32_t>();
    struct Word {
        const uint64_t* from;
        uint32_t shift, bits;
    };
    const Word u64[2] = {{keys, 0u, 31u}, {keys, 31u, 32u}};
    const Word u128[4] = {{keys, 0u, 32u}, {keys, 32u, 32u}, {keys_hi, 0u, 30u}, {keys_hi, 30u, 32u}};
    const Word* const w = keys_hi ? u128 : u64;
    for (int k = 0; k < (keys_hi ? 4 : 2); ++k) {
        k_code_words<<<(n + T256 - 1) / T256, T256, 0, st>>>(w[k].from, k ? vals : nullptr, n, w[k].shift, w[k].bits,
                                                             words);
        OBVHS_TRY(hipGetLastError(), "code words");
        OBVHS_TRY(radix_sort_pairs32(words, vals, k == 0, n, (int)w[k].bits, S.sort_scratch.ptr, st,
                                     sort_items_for(ctx, n)),
                  "radix sort (whole codes)");
    }
    return OBVHS_OK;
}

// Clusters in Morton order (ploc/mod.rs:811-846) from the codes: the top 32 bits sorted, the runs of equal tops
// ordered by the gather.  keys and keys_hi keep their leaf order.  order_out (may be NULL): the permutation.
static obvhs_status sort_gather(obvhs_context* ctx, const Node32* leaves, const uint64_t* keys,
                                const uint64_t* keys_hi, uint32_t n, Node32* cur, uint32_t* order_out) {
    hipStream_t st = ctx->stream;
    BuildScratch& S = ctx->scratch;
    uint32_t* tops = S.tops.as<uint32_t>();
    uint32_t* vals = S.vals.as<uint32_t>();
    Misc* misc = S.misc.as<Misc>();
    OBVHS_TRY(radix_sort_pairs32(tops, vals, true, n, 32, S.sort_scratch.ptr, st, sort_items_for(ctx, n)),
              "radix sort (top words)");
    const uint32_t nblk = (n + T256 - 1) / T256;
    if (keys_hi)
        k_gather_runs<true><<<xcd_grid(nblk), T256, 0, st>>>(leaves, tops, vals, n, keys, keys_hi, misc, cur,
                                                             order_out);
    else
        k_gather_runs<false><<<xcd_grid(nblk), T256, 0, st>>>(leaves, tops, vals, n, keys, keys_hi, misc, cur,
                                                              order_out);
    OBVHS_TRY(hipGetLastError(), "gather launch");
    return OBVHS_OK;
}

// The same by a sort of the whole codes, after sort_gather met a long run (DERR_RESORT): the pass state starts over.
static obvhs_status resort_gather(obvhs_context* ctx, const Node32* leaves, const uint64_t* keys,
                                  const uint64_t* keys_hi, uint32_t n, Node32* cur, uint32_t* order_out) {
    hipStream_t st = ctx->stream;
    BuildScratch& S = ctx->scratch;
    uint32_t* vals = S.vals.as<uint32_t>();
    k_reset_state<<<1, 64, 0, st>>>(S.misc.as<Misc>(), n);
    const obvhs_status ss = sort_codes(ctx, keys, keys_hi, vals, n);
    if (ss != OBVHS_OK) return ss;
    if (order_out)
        OBVHS_TRY(hipMemcpyAsync(order_out, vals, (size_t)n * 4, hipMemcpyDeviceToDevice, st), "copy sorted index");
    k_gather<<<(n + T256 - 1) / T256, T256, 0, st>>>(leaves, vals, n, cur);
    OBVHS_TRY(hipGetLastError(), "gather launch");
    return OBVHS_OK;
}

// The PLOC passes from the sorted clusters in `cur` to the root (ploc/mod.rs:327-499): grid passes while more than
// TAIL_MAX clusters remain, then the one-workgroup tail.  `fin`
// receives the final pass state; `resort` is set (and the passes did nothing) when the gather flagged DERR_RESORT.
// The error word and the pass state of `slot` with one copy (err, pad, state[0], state[1] are adjacent) into the
// pinned staging area, then a stream synchronisation.
static hipError_t read_state(const Misc* misc, uint32_t slot, void* pinned, hipStream_t st, PlocState& state,
                             uint32_t& err, CwRootInfo* info = nullptr) {
    const size_t lo = offsetof(Misc, err),
                 hi = info ? offsetof(Misc, info) + sizeof(CwRootInfo) : offsetof(Misc, state) + (slot + 1u) * sizeof(PlocState);
    hipError_t e = hipMemcpyAsync(pinned, reinterpret_cast<const char*>(misc) + lo, hi - lo, hipMemcpyDeviceToHost,
                                  st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    const char* h = static_cast<const char*>(pinned);
    memcpy(&err, h, 4);
    memcpy(&state, h + (offsetof(Misc, state) + slot * sizeof(PlocState) - lo), sizeof(PlocState));
    if (info) memcpy(info, h + (offsetof(Misc, info) - lo), sizeof(CwRootInfo));
    return hipSuccess;
}

// The search-and-count kernel for the search distance (each allowed distance has its unrolled instance).
static void launch_search_count(uint32_t blocks, hipStream_t st, const Node32* cur, Misc* misc, uint32_t slot,
                                uint32_t r, uint32_t dist1, int8_t* merge, uint2* blocksums, uint32_t grouped) {
    switch (r) {
        case 2: k_ploc_search_count<2><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
        case 6: k_ploc_search_count<6><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
        case 14: k_ploc_search_count<14><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
        case 24: k_ploc_search_count<24><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
        case 32: k_ploc_search_count<32><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
        default: k_ploc_search_count<0><<<blocks, SC_THREADS, 0, st>>>(cur, misc, slot, r, dist1, merge, blocksums, grouped); break;
    }
}

// The tail for the search distance (each allowed distance has its unrolled instance).
static void launch_tail(hipStream_t st, const Node32* cur, Misc* misc, uint32_t slot, uint32_t pass, uint32_t r,
                        uint32_t threshold, Node32* bvh_nodes, uint32_t* hist, const DpView& dp, uint32_t fused,
                        const uint32_t* slot_map, uint32_t vtop, uint32_t map_len) {
    const uint32_t one = r == 1 ? 1u : 0u;
#define OBVHS_TAIL(RR)                                                                                           \
    k_ploc_tail<RR><<<1, TAIL_THREADS, 0, st>>>(cur, misc, slot, pass, r, one, threshold, bvh_nodes, hist, dp, \
                                                fused, slot_map, vtop, map_len)
    switch (r) {
        case 2: OBVHS_TAIL(2); break;
        case 6: OBVHS_TAIL(6); break;
        case 14: OBVHS_TAIL(14); break;
        case 24: OBVHS_TAIL(24); break;
        case 32: OBVHS_TAIL(32); break;
        default: OBVHS_TAIL(0); break;
    }
#undef OBVHS_TAIL
}

// Working memory of the one-launch passes: two arrays of tile counts, two of merge lists (18.9 MB at most).
static size_t pass_tile_bytes(uint32_t n) {
    const size_t tiles = std::min<uint32_t>((n + T256 - 1) / T256, PASS_TILES);
    return 2 * PASS_TILES * sizeof(uint2) + 2 * tiles * MAX_TILE_MERGES * sizeof(PassMerge);
}

// The one-launch pass for the search distance (each allowed distance has its unrolled instance).
static void launch_pass(uint32_t blocks, hipStream_t st, const Node32* cur, Node32* next, const uint2* counts,
                        uint32_t ntiles, uint2* counts_out, const PassMerge* merges_in, PassMerge* merges_out,
                        Misc* misc, uint32_t slot, uint32_t r, uint32_t dist1, Node32* bvh_nodes, const DpView& dp,
                        uint32_t fused, const uint32_t* slot_map, uint32_t vtop, uint32_t map_len, uint32_t* hist) {
#define OBVHS_PASS(RR)                                                                                              \
    k_ploc_pass<RR><<<blocks, PASS_THREADS, 0, st>>>(cur, next, counts, ntiles, counts_out, merges_in, merges_out, \
                                                     misc, slot, r, dist1, bvh_nodes, dp, fused, slot_map, vtop,    \
                                                     map_len, hist)
    switch (r) {
        case 2: OBVHS_PASS(2); break;
        case 6: OBVHS_PASS(6); break;
        case 14: OBVHS_PASS(14); break;
        case 24: OBVHS_PASS(24); break;
        case 32: OBVHS_PASS(32); break;
        default: OBVHS_PASS(0); break;
    }
#undef OBVHS_PASS
}

static obvhs_status run_passes(obvhs_context* ctx, Node32* cur, Node32* nxt, uint32_t n, uint32_t r,
                               uint32_t search_depth_threshold, Node32* bvh_nodes, uint32_t* hist, DpView dp,
                               uint32_t fused, const uint32_t* slot_map, uint32_t vtop, uint32_t map_len,
                               PlocState& fin, bool& resort, CwRootInfo* info) {
    resort = false;
    hipStream_t st = ctx->stream;
    BuildScratch& S = ctx->scratch;
    Misc* misc = S.misc.as<Misc>();
    int8_t* merge = S.merge.as<int8_t>();
    uint2* blocksums = S.blocksums.as<uint2>();
    const uint32_t tiles = std::min<uint32_t>((n + T256 - 1) / T256, PASS_TILES);
    uint2* pass_counts[2] = {S.pass_tiles.as<uint2>(), S.pass_tiles.as<uint2>() + PASS_TILES};
    PassMerge* pass_merges[2];
    pass_merges[0] = reinterpret_cast<PassMerge*>(pass_counts[1] + PASS_TILES);
    pass_merges[1] = pass_merges[0] + (size_t)tiles * MAX_TILE_MERGES;
    uint32_t known = n;
    uint32_t pass = 0;
    uint32_t slot = 0;
    PlocState hstate{};
    while (known > TAIL_MAX) {
        const uint32_t blocks = (known + T256 - 1) / T256;
        if (blocks <= PASS_TILES) {
            // one launch per pass, then the flush; counts and merges double-buffered
            for (int k = 0; k < PASSES_PER_SYNC; ++k) {
                const uint32_t dist1 = (r == 1 || pass < search_depth_threshold) ? 1u : 0u;
                launch_pass(blocks, st, cur, nxt, pass_counts[k & 1], k == 0 ? 0u : blocks, pass_counts[(k & 1) ^ 1],
                            pass_merges[k & 1], pass_merges[(k & 1) ^ 1], misc, slot, r, dist1, bvh_nodes, dp, fused,
                            slot_map, vtop, map_len, hist);
                std::swap(cur, nxt);
                slot ^= 1u;
                pass++;
            }
            constexpr int last = PASSES_PER_SYNC & 1;
            k_ploc_flush<<<blocks, PASS_THREADS, 0, st>>>(cur, nxt, pass_counts[last], blocks, pass_merges[last], misc,
                                                          slot, bvh_nodes, dp, fused, slot_map, vtop, map_len, hist);
            std::swap(cur, nxt);
            slot ^= 1u;
        } else {
            for (int k = 0; k < PASSES_PER_SYNC; ++k) {
                const uint32_t dist1 = (r == 1 || pass < search_depth_threshold) ? 1u : 0u;
                const uint32_t grouped = blocks <= GROUP_MAX_TILES ? 1u : 0u;
                launch_search_count(blocks, st, cur, misc, slot, r, dist1, merge, blocksums, grouped);
                if (!grouped) {
                    // chunk totals after the counts, in the blocksums allocation's tail (dead during the passes)
                    uint2* chunk_tot = blocksums + blocks + 16;
                    const uint32_t nchunks = (blocks + SCAN_CHUNK - 1) / SCAN_CHUNK;
                    k_ploc_scan_chunks<<<nchunks, 1024, 0, st>>>(blocksums, blocks, chunk_tot);
                    k_ploc_scan_apply<<<nchunks, 1024, 0, st>>>(blocksums, blocks, chunk_tot, nchunks, misc, slot,
                                                                 hist);
                }
                k_ploc_compact<<<blocks, T256, 0, st>>>(cur, nxt, merge, misc, slot, blocksums, grouped, bvh_nodes, dp,
                                                       fused, slot_map, vtop, map_len, hist);
                std::swap(cur, nxt);
                slot ^= 1u;
                pass++;
            }
        }
        OBVHS_TRY(hipGetLastError(), "ploc pass launch");
        uint32_t herr_loop = 0u;
        OBVHS_TRY(read_state(misc, slot, ctx->pinned, st, hstate, herr_loop), "read ploc state");
        if (herr_loop & ~DERR_RESORT) return device_error_to_status(herr_loop);
        if (herr_loop) {
            resort = true;
            return OBVHS_OK;
        }
        // Every pass merges at least one pair unless costs are NaN; a batch without progress would never end.
        if (hstate.count >= known) return OBVHS_ERR_PLOC_SELF_MERGE;
        known = hstate.count;
        // The device depth counts real passes only; later enqueued passes may have been no-ops.
        pass = hstate.depth;
    }
    launch_tail(st, cur, misc, slot, pass, r, search_depth_threshold, bvh_nodes, hist, dp, fused, slot_map, vtop,
                map_len);
    OBVHS_TRY(hipGetLastError(), "ploc tail launch");
    uint32_t herr = 0u;
    OBVHS_TRY(read_state(misc, slot, ctx->pinned, st, hstate, herr, info), "read final ploc state");
    if (herr & ~DERR_RESORT) return device_error_to_status(herr);
    if (herr) {
        resort = true;
        return OBVHS_OK;
    }
    if (hstate.insert != 1u) return OBVHS_ERR_PLOC_SELF_MERGE;  // ploc/mod.rs:495-497
    fin = hstate;
    return OBVHS_OK;
}

obvhs_status ploc_build(obvhs_context* ctx, const obvhs_triangle* d_tris, const obvhs_aabb* d_aabbs,
                        const uint32_t* d_indices, uint32_t n, uint32_t search_distance, bool u128,
                        uint32_t search_depth_threshold, uint32_t fused_max_prims, obvhs_bvh2* bvh,
                        CwRootInfo* info) {
    if (!(search_distance == 1 || search_distance == 2 || search_distance == 6 || search_distance == 14 ||
          search_distance == 24 || search_distance == 32))
        return OBVHS_ERR_INVALID_ARG;  // ploc/mod.rs:550-561
    hipStream_t st = ctx->stream;
    bvh->prim_count = n;
    bvh->node_count = n == 0 ? 0u : 2u * n - 1u;
    bvh->max_depth = 96;
    bvh->ploc_iterations = 0;
    bvh->cluster_sum = 0;
    bvh->dp_max_prims = 0;
    bvh->pass_ordered = true;
    OBVHS_TRY(bvh->prim_indices.ensure((size_t)n * 4 + 4), "alloc primitive_indices");
    if (n == 0) return OBVHS_OK;
    OBVHS_TRY(bvh->hist.ensure((size_t)(n + 1) * 4), "alloc pass history");
    DpView dp{};
    if (fused_max_prims) {
        OBVHS_TRY(bvh_dp_alloc(bvh), "alloc cost table");
        dp = bvh_dp_view(bvh, fused_max_prims);
    }
    const uint32_t fused = fused_max_prims ? 1u : 0u;
    OBVHS_TRY(bvh->nodes.ensure((size_t)bvh->node_count * sizeof(Node32)), "alloc bvh2 nodes");
    BuildScratch& S = ctx->scratch;
    OBVHS_TRY(S.leaves.ensure((size_t)n * sizeof(Node32)), "alloc leaves");
    OBVHS_TRY(S.clusters_a.ensure(((size_t)n + T256) * sizeof(Node32)), "alloc clusters");  // whole tiles
    OBVHS_TRY(S.clusters_b.ensure(((size_t)n + T256) * sizeof(Node32)), "alloc clusters");
    OBVHS_TRY(S.keys.ensure((size_t)n * 8), "alloc keys");
    if (u128) OBVHS_TRY(S.keys_hi.ensure((size_t)n * 8), "alloc high key words");
    OBVHS_TRY(S.vals.ensure((size_t)n * 4), "alloc vals");
    OBVHS_TRY(S.tops.ensure((size_t)n * 4), "alloc top key words");
    OBVHS_TRY(S.merge.ensure((size_t)n + 64), "alloc merge");
    OBVHS_TRY(S.pass_tiles.ensure(pass_tile_bytes(n)), "alloc pass tiles");
    const uint32_t nblk = (n + T256 - 1) / T256;
    OBVHS_TRY(S.blocksums.ensure((size_t)nblk * sizeof(uint2) + 64 + (size_t)nblk * 6 * 4), "alloc blocksums");
    OBVHS_TRY(S.sort_scratch.ensure(radix_sort_scratch_bytes(n)), "alloc sort scratch");
    OBVHS_TRY(S.misc.ensure(sizeof(Misc)), "alloc misc");
    Misc* misc = S.misc.as<Misc>();
    Node32* leaves = S.leaves.as<Node32>();
    Node32* bvh_nodes = bvh->nodes.as<Node32>();
    uint64_t* keys = S.keys.as<uint64_t>();
    uint64_t* keys_hi = u128 ? S.keys_hi.as<uint64_t>() : nullptr;
    uint32_t* hist = bvh->hist.as<uint32_t>();
    // per-block bound partials share the blocksums allocation (they are dead before the first pass)
    uint32_t* partials = reinterpret_cast<uint32_t*>(S.blocksums.as<char>() + (size_t)nblk * sizeof(uint2) + 64);

    // primitive_indices = indices (Bvh2::reset_for_reuse, bvh2/mod.rs:106-121)
    if (d_indices) {
        OBVHS_TRY(hipMemcpyAsync(bvh->prim_indices.ptr, d_indices, (size_t)n * 4, hipMemcpyDeviceToDevice, st),
                  "copy indices");
    }
    uint32_t* iota_out = d_indices ? nullptr : bvh->prim_indices.as<uint32_t>();  // primitive_indices = 0..n-1
    bvh->code_words = u128 ? 2u : 1u;
    uint64_t *codes = nullptr, *codes_hi = nullptr;  // kept with the sort permutation for parity tests
    uint32_t* order_out = nullptr;
    if (ctx->keep_trace) {  // low words, then the high words of U128 codes
        OBVHS_TRY(bvh->codes.ensure((size_t)n * 8 * bvh->code_words), "alloc codes");
        OBVHS_TRY(bvh->sorted_index.ensure((size_t)n * 4), "alloc sorted index");
        codes = bvh->codes.as<uint64_t>();
        codes_hi = u128 ? codes + n : nullptr;
        order_out = bvh->sorted_index.as<uint32_t>();
    }
    const float4* tris = reinterpret_cast<const float4*>(d_tris);
    const float4* aabbs = d_tris ? nullptr : reinterpret_cast<const float4*>(d_aabbs);
    Node32* cur = S.clusters_a.as<Node32>();
    Node32* nxt = S.clusters_b.as<Node32>();
    if (n <= SMALL_MAX) {
        if (u128)
            k_front_small<true><<<1, SMALL_THREADS, 0, st>>>(tris, aabbs, d_indices, n, misc, hist, iota_out, codes,
                                                             codes_hi, order_out, cur);
        else
            k_front_small<false><<<1, SMALL_THREADS, 0, st>>>(tris, aabbs, d_indices, n, misc, hist, iota_out, codes,
                                                              codes_hi, order_out, cur);
        OBVHS_TRY(hipGetLastError(), "small build front launch");
    } else {
        k_init_misc<<<1, 64, 0, st>>>(misc, n, hist);
        if (d_tris)
            k_leaf_init_tris<<<nblk, T256, 0, st>>>(tris, d_indices, n, leaves, misc, partials, iota_out);
        else
            k_leaf_init_aabbs<<<nblk, T256, 0, st>>>(aabbs, d_indices, n, leaves, misc, partials, iota_out);
        k_reduce_bounds<<<1, 1024, 0, st>>>(partials, nblk, misc);
        k_morton<<<nblk, T256, 0, st>>>(leaves, n, misc, keys, keys_hi, S.tops.as<uint32_t>());
        OBVHS_TRY(hipGetLastError(), "leaf/morton launch");
        if (codes) OBVHS_TRY(hipMemcpyAsync(codes, keys, (size_t)n * 8, hipMemcpyDeviceToDevice, st), "copy codes");
        if (codes_hi)
            OBVHS_TRY(hipMemcpyAsync(codes_hi, keys_hi, (size_t)n * 8, hipMemcpyDeviceToDevice, st), "copy codes");
        const obvhs_status ss = sort_gather(ctx, leaves, keys, keys_hi, n, cur, order_out);
        if (ss != OBVHS_OK) return ss;
    }

    PlocState fin{};
    bool resort = false;
    obvhs_status ps = run_passes(ctx, cur, nxt, n, search_distance, search_depth_threshold, bvh_nodes, hist, dp,
                                 fused, nullptr, 0u, 0u, fin, resort, info);
    bvh->long_runs = resort;
    if (ps == OBVHS_OK && resort) {
        ps = resort_gather(ctx, leaves, keys, keys_hi, n, cur, order_out);
        if (ps == OBVHS_OK)
            ps = run_passes(ctx, cur, nxt, n, search_distance, search_depth_threshold, bvh_nodes, hist, dp, fused,
                            nullptr, 0u, 0u, fin, resort, info);
    }
    if (ps != OBVHS_OK) return ps;
    bvh->ploc_iterations = fin.depth;
    bvh->cluster_sum = fin.cluster_sum;
    bvh->max_depth = fin.depth + 1 > 96 ? fin.depth + 1 : 96;  // ploc/mod.rs:501
    bvh->dp_max_prims = fused_max_prims;
    return OBVHS_OK;
}

// rebuild_from_leaves (ploc/rebuild.rs:136-183) over the nodes at d_src_slots[0..k) of bvh->nodes, listed in slot
// order (the order that breaks Morton-code ties).  slot_map = NULL: full rebuild, the tree becomes 2k-1 nodes with
// the plain placement (children after parents).  Otherwise slot_map[g] (k-1 entries, descending) is the left slot
// of the g-th freed sibling pair; every other slot keeps its node.  The scene box is the root's stored box.
obvhs_status ploc_rebuild(obvhs_context* ctx, obvhs_bvh2* bvh, const uint32_t* d_src_slots, uint32_t k,
                          const uint32_t* d_slot_map, uint32_t search_distance, bool u128,
                          uint32_t search_depth_threshold) {
    if (!(search_distance == 1 || search_distance == 2 || search_distance == 6 || search_distance == 14 ||
          search_distance == 24 || search_distance == 32))
        return OBVHS_ERR_INVALID_ARG;
    if (k == 0) return OBVHS_OK;
    if (!d_slot_map && 2ull * k - 1ull > bvh->node_count) return OBVHS_ERR_INVALID_ARG;
    hipStream_t st = ctx->stream;
    BuildScratch& S = ctx->scratch;
    OBVHS_TRY(bvh->hist.ensure((size_t)(k + 1) * 4), "alloc pass history");
    OBVHS_TRY(S.leaves.ensure((size_t)k * sizeof(Node32)), "alloc leaves");
    OBVHS_TRY(S.clusters_a.ensure(((size_t)k + T256) * sizeof(Node32)), "alloc clusters");  // whole tiles
    OBVHS_TRY(S.clusters_b.ensure(((size_t)k + T256) * sizeof(Node32)), "alloc clusters");
    OBVHS_TRY(S.keys.ensure((size_t)k * 8), "alloc keys");
    if (u128) OBVHS_TRY(S.keys_hi.ensure((size_t)k * 8), "alloc high key words");
    OBVHS_TRY(S.vals.ensure((size_t)k * 4), "alloc vals");
    OBVHS_TRY(S.tops.ensure((size_t)k * 4), "alloc top key words");
    OBVHS_TRY(S.merge.ensure((size_t)k + 64), "alloc merge");
    OBVHS_TRY(S.pass_tiles.ensure(pass_tile_bytes(k)), "alloc pass tiles");
    const uint32_t nblk = (k + T256 - 1) / T256;
    OBVHS_TRY(S.blocksums.ensure((size_t)nblk * sizeof(uint2) + 64 + (size_t)nblk * 6 * 4), "alloc blocksums");
    OBVHS_TRY(S.sort_scratch.ensure(radix_sort_scratch_bytes(k)), "alloc sort scratch");
    OBVHS_TRY(S.misc.ensure(sizeof(Misc)), "alloc misc");
    Misc* misc = S.misc.as<Misc>();
    Node32* leaves = S.leaves.as<Node32>();
    Node32* bvh_nodes = bvh->nodes.as<Node32>();
    uint64_t* keys = S.keys.as<uint64_t>();
    uint64_t* keys_hi = u128 ? S.keys_hi.as<uint64_t>() : nullptr;
    uint32_t* hist = bvh->hist.as<uint32_t>();
    // From here on the nodes change: a rebuild that fails leaves no tree in pass order, and no cost table.
    bvh->pass_ordered = false;
    bvh->dp_max_prims = 0;
    // The clusters are copied out first: merges may overwrite the freed slots they came from.
    k_gather<<<nblk, T256, 0, st>>>(bvh_nodes, d_src_slots, k, leaves);
    k_init_misc<<<1, 64, 0, st>>>(misc, k, hist);
    k_bounds_from_node<<<1, 64, 0, st>>>(misc, bvh_nodes);
    k_morton<<<nblk, T256, 0, st>>>(leaves, k, misc, keys, keys_hi, S.tops.as<uint32_t>());
    OBVHS_TRY(hipGetLastError(), "rebuild morton launch");
    Node32* cur = S.clusters_a.as<Node32>();
    Node32* nxt = S.clusters_b.as<Node32>();
    // A tree that met long runs is not tried by its tops again: 1M leaves in a thousandth of their box, 2% of the
    // leaves rebuilt 884 -> 747 us, all 949 -> 757.
    const obvhs_status ss = bvh->long_runs ? resort_gather(ctx, leaves, keys, keys_hi, k, cur, nullptr)
                                           : sort_gather(ctx, leaves, keys, keys_hi, k, cur, nullptr);
    if (ss != OBVHS_OK) return ss;
    PlocState fin{};
    bool resort = false;
    obvhs_status ps = run_passes(ctx, cur, nxt, k, search_distance, search_depth_threshold, bvh_nodes, hist,
                                 DpView{}, 0u, d_slot_map, 2u * k - 3u, k - 1u, fin, resort, nullptr);
    if (ps == OBVHS_OK && resort) {
        bvh->long_runs = true;
        ps = resort_gather(ctx, leaves, keys, keys_hi, k, cur, nullptr);
        if (ps == OBVHS_OK)
            ps = run_passes(ctx, cur, nxt, k, search_distance, search_depth_threshold, bvh_nodes, hist, DpView{}, 0u,
                            d_slot_map, 2u * k - 3u, k - 1u, fin, resort, nullptr);
    }
    if (ps != OBVHS_OK) return ps;
    if (!d_slot_map) bvh->node_count = 2u * k - 1u;  // ploc/mod.rs:283-284 (nodes.resize)
    bvh->pass_ordered = d_slot_map == nullptr;    // ploc/mod.rs:502
    bvh->ploc_iterations = fin.depth;
    bvh->cluster_sum = fin.cluster_sum;
    bvh->max_depth = fin.depth + 1 > 96 ? fin.depth + 1 : 96;  // ploc/mod.rs:501
    bvh->dp_max_prims = 0;                                      // boxes changed: any cost table is stale
    return OBVHS_OK;
}

namespace {
__global__ void k_iota(uint32_t* p, uint32_t n) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}
}  // namespace

hipError_t launch_iota(uint32_t* p, uint32_t n, hipStream_t st) {
    k_iota<<<(n + 255) / 256, 256, 0, st>>>(p, n);
    return hipGetLastError();
}

}  // namespace obvhs
