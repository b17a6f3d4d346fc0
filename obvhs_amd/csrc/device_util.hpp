// Small device helpers shared by the PLOC kernels of the single and batched builds.
#pragma once

#include "common.hpp"

namespace obvhs {

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, off));
    return v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off));
    return v;
}
__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
    const int lane = (int)__lane_id();
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t t = (uint32_t)__shfl_up((int)v, off);
        if (lane >= off) v += t;
    }
    return v;
}

// The same for a full wave as DPP moves (row shifts, then the row totals broadcast), which stay in the VALU instead of
// six round trips through the LDS crossbar.  Every lane must be active.
__device__ __forceinline__ uint32_t wave_inclusive_scan_dpp(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
    return v;
}

__device__ __forceinline__ bool box_has_nan(const Box& b) {
    return isnan(b.lx) || isnan(b.ly) || isnan(b.lz) || isnan(b.hx) || isnan(b.hy) || isnan(b.hz);
}

// A workgroup barrier for data in LDS only: global loads and stores in flight are not waited for.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The same inside a wave, for lanes that read what other lanes of it wrote to LDS, or overwrite what they read: the
// hardware keeps a wave's LDS accesses in order, and this keeps the compiler's.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// morton.rs:35-43
__device__ __forceinline__ uint64_t split_by_3_u64(uint32_t a) {
    uint64_t x = (uint64_t)a & 0x1fffffull;
    x = (x | x << 32) & 0x1f00000000ffffull;
    x = (x | x << 16) & 0x1f0000ff0000ffull;
    x = (x | x << 8) & 0x100f00f00f00f00full;
    x = (x | x << 4) & 0x10c30c30c30c30c3ull;
    x = (x | x << 2) & 0x1249249249249249ull;
    return x;
}
// Rust `f64 as u32` (saturating, NaN -> 0).
__device__ __forceinline__ uint32_t f64_as_u32(double v) {
    if (!(v >= 1.0)) return 0u;
    if (v >= 4294967296.0) return 0xffffffffu;
    return (uint32_t)v;
}

// Rust `f64 as u64` (saturating, NaN -> 0).
__device__ __forceinline__ uint64_t f64_as_u64(double v) {
    if (!(v >= 1.0)) return 0u;
    if (v >= 18446744073709551616.0) return ~0ull;
    return (uint64_t)v;
}

// 126-bit Morton code of the unit-cube point (px, py, pz) (morton_encode_u128_unorm, morton.rs:63-89) as its low
// and high 64-bit words.  Each 42-bit coordinate is x = xh * 2^21 + xl; spreading puts bit i of x at 3i, so xl
// fills bits [0, 63) and xh bits [63, 126): the code is code64(xl, yl, zl) + code64(xh, yh, zh) * 2^63.
__device__ __forceinline__ void morton128_of_point(double px, double py, double pz, uint64_t& lo, uint64_t& hi) {
    const double s = 4398046511104.0;  // 2^42
    const uint64_t m = 0x3ffffffffffull;
    const uint64_t x = f64_as_u64(px * s) & m, y = f64_as_u64(py * s) & m, z = f64_as_u64(pz * s) & m;
    // split_by_3_u64 keeps the low 21 bits of its argument
    const uint64_t a = split_by_3_u64((uint32_t)x) | split_by_3_u64((uint32_t)y) << 1 |
                       split_by_3_u64((uint32_t)z) << 2;
    const uint64_t b = split_by_3_u64((uint32_t)(x >> 21)) | split_by_3_u64((uint32_t)(y >> 21)) << 1 |
                       split_by_3_u64((uint32_t)(z >> 21)) << 2;
    lo = a | b << 63;
    hi = b >> 1;
}

// Morton code of a leaf box under the scene normalisation (ploc/mod.rs:287-288, 782-785; morton.rs:55-58).
__device__ __forceinline__ uint64_t morton_of_box(const Box& b, double sx, double sy, double sz, double ox, double oy,
                                                  double oz) {
    const float cx = (b.hx + b.lx) * 0.5f, cy = (b.hy + b.ly) * 0.5f, cz = (b.hz + b.lz) * 0.5f;
    const double px = (double)cx * sx + ox, py = (double)cy * sy + oy, pz = (double)cz * sz + oz;
    const double s = 2097152.0;
    return split_by_3_u64(f64_as_u32(px * s)) | split_by_3_u64(f64_as_u32(py * s)) << 1 |
           split_by_3_u64(f64_as_u32(pz * s)) << 2;
}

// Exclusive scans over a 1024-thread workgroup of two u32 values at once; ta / tb receive the totals.  se / sm: 16
// words of LDS each (reused: the function ends with a barrier).
__device__ __forceinline__ void block_exscan2_1024(uint32_t a, uint32_t b, uint32_t* se, uint32_t* sm, uint32_t& ea,
                                                   uint32_t& eb, uint32_t& ta, uint32_t& tb) {
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t ia = wave_inclusive_scan(a), ib = wave_inclusive_scan(b);
    if (lane == 63u) {
        se[wave] = ia;
        sm[wave] = ib;
    }
    __syncthreads();
    uint32_t pa = 0u, pb = 0u;
    ta = 0u;
    tb = 0u;
#pragma unroll
    for (uint32_t w = 0; w < 16; ++w) {
        const uint32_t xa = se[w], xb = sm[w];
        if (w < wave) {
            pa += xa;
            pb += xb;
        }
        ta += xa;
        tb += xb;
    }
    ea = pa + ia - a;
    eb = pb + ib - b;
    __syncthreads();
}

// Two-level scan of per-tile (emit, merge) counts, SCAN_CHUNK counts (4 per thread) per 1,024-thread workgroup.
// scan_chunk_total: the chunk's totals into chunk_tot[blockIdx.x].  scan_chunk_apply: every count becomes its
// exclusive prefix over all tiles (the chunks before this one from chunk_tot); returns the totals of all chunks.
constexpr uint32_t SCAN_CHUNK = 4096;

__device__ __forceinline__ void scan_chunk_total(const uint2* __restrict__ counts, uint32_t n,
                                                 uint2* __restrict__ chunk_tot) {
    __shared__ uint32_t se[16], sm[16];
    const uint32_t b0 = blockIdx.x * SCAN_CHUNK + threadIdx.x * 4u;
    uint32_t E = 0u, M = 0u;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k)
        if (b0 + k < n) {
            const uint2 v = counts[b0 + k];
            E += v.x;
            M += v.y;
        }
    uint32_t ee, em, te, tm;
    block_exscan2_1024(E, M, se, sm, ee, em, te, tm);
    if (threadIdx.x == 0) chunk_tot[blockIdx.x] = make_uint2(te, tm);
}

__device__ __forceinline__ uint2 scan_chunk_apply(uint2* __restrict__ counts, uint32_t n,
                                                  const uint2* __restrict__ chunk_tot, uint32_t nchunks) {
    __shared__ uint32_t se[16], sm[16];
    uint32_t pe = 0u, pm = 0u, ae = 0u, am = 0u;
    for (uint32_t c = threadIdx.x; c < nchunks; c += 1024u) {
        const uint2 v = chunk_tot[c];
        if (c < blockIdx.x) {
            pe += v.x;
            pm += v.y;
        }
        ae += v.x;
        am += v.y;
    }
    uint32_t x0, x1, before_e, before_m, all_e, all_m;
    block_exscan2_1024(pe, pm, se, sm, x0, x1, before_e, before_m);
    block_exscan2_1024(ae, am, se, sm, x0, x1, all_e, all_m);
    const uint32_t b0 = blockIdx.x * SCAN_CHUNK + threadIdx.x * 4u;
    uint2 v[4];
    uint32_t E = 0u, M = 0u;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        v[k] = b0 + k < n ? counts[b0 + k] : make_uint2(0u, 0u);
        E += v[k].x;
        M += v[k].y;
    }
    uint32_t ee, em, te, tm;
    block_exscan2_1024(E, M, se, sm, ee, em, te, tm);
    ee += before_e;
    em += before_m;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k)
        if (b0 + k < n) {
            counts[b0 + k] = make_uint2(ee, em);
            ee += v[k].x;
            em += v[k].y;
        }
    return make_uint2(all_e, all_m);
}

// The children of a tile's merges [64 * wave, count) that are the wave's, 64 bytes each, from LDS to the child slots:
// four lanes to a pair.  (A lane that stores its own pair touches another line with every 16 bytes.)  offset(q): the
// slot of merge q's first child, SIZE_MAX for none.
template <class Offset>
__device__ __forceinline__ void store_pairs(const Node32* s_left, const Node32* s_right, uint32_t wave, uint32_t count,
                                            Node32* __restrict__ nodes, Offset offset) {
    const uint32_t lane = threadIdx.x & 63u, part = lane & 3u;
    const uint32_t end = min(count, wave * 64u + 64u);
    for (uint32_t q = wave * 64u + (lane >> 2); q < end; q += 16u) {
        const float4* from = reinterpret_cast<const float4*>(part < 2u ? &s_left[q] : &s_right[q]);
        const size_t at = offset(q);
        if (at != SIZE_MAX) reinterpret_cast<float4*>(&nodes[at])[part] = from[part & 1u];
    }
}

// Whether DERR_RESORT is set in the word (by some workgroup, as far as this one sees).
__device__ __forceinline__ bool resort_flagged(const uint32_t* err) {
    return (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & DERR_RESORT) != 0u;
}
// Sets it if one of the calling lanes asks for it (`mine`): one atomic a wave at most.  Returns `mine`.
__device__ __forceinline__ bool flag_resort(bool mine, uint32_t* err) {
    const uint64_t lanes = __ballot(mine);
    if (mine && (lanes & lanemask_lt()) == 0ull && !resort_flagged(err)) atomicOr(err, DERR_RESORT);
    return mine;
}

// Workgroups go round-robin to the 8 XCDs, each with its own L2.  The tile of a workgroup such that an XCD's
// workgroups take one contiguous eighth of the tiles: for kernels whose neighbouring tiles read the same lines at
// random (a 128-byte line holds four leaf records or parts of four triangles).  20M triangles in 4,096 meshes: leaf
// gather 502 -> 471 us; 17.3M-triangle build with reordering 29.96 -> 29.54 ms.  The grid is xcd_grid(tiles) workgroups;
// those that get a tile >= tiles have none.
constexpr uint32_t XCDS = 8;
inline uint32_t xcd_grid(uint32_t tiles) { return (tiles + XCDS - 1) / XCDS * XCDS; }
__device__ __forceinline__ uint32_t xcd_tile() {
    return (blockIdx.x % XCDS) * (gridDim.x / XCDS) + blockIdx.x / XCDS;
}

}  // namespace obvhs
