// PLOC passes inside one workgroup: the last passes of a build (ploc.hip) and of every mesh of a batch (batch.hip).
#pragma once

#include "common.hpp"
#include "cwdp.hpp"
#include "device_util.hpp"
#include "internal.hpp"

namespace obvhs {

constexpr uint32_t MAX_RADIUS = 32;  // the largest search distance

namespace {

// Child slot of a merge whose plain-placement left slot is v (see the header).  Returns false (and flags the error)
// when v is outside the map, which a well-formed pass sequence never produces.
__device__ __forceinline__ bool child_slot(uint32_t v, const uint32_t* __restrict__ slot_map, uint32_t vtop,
                                           uint32_t map_len, uint32_t& first) {
    if (!slot_map) {
        first = v;
        return true;
    }
    const uint32_t g = (vtop - v) >> 1;
    if (v > vtop || g >= map_len) return false;
    first = slot_map[g];
    return true;
}

// Classification of cluster i (ploc/mod.rs:423-439): `emit` when it goes to the next pass (kept, or the higher
// index of a mutual pair, which becomes the parent), `mrg` when it is the higher index of a mutual pair.
// A self-pair (no finite neighbour, already flagged as an error) is treated as kept so that no slot underflows.
struct Cls {
    bool emit, mrg;
    uint32_t b;  // the neighbour
};
__device__ __forceinline__ Cls classify(const int8_t* merge, uint32_t i, uint32_t count) {
    const bool valid = i < count, pair = valid && count > 1u;
    const int bi = pair ? (int)i + (int)merge[i] : (int)i;
    const bool mutual = pair && bi + (int)merge[bi] == (int)i;
    return Cls{valid && (!mutual || bi <= (int)i), mutual && bi < (int)i, (uint32_t)bi};
}

// A cluster in the tail's LDS arrays: lo = box minimum and prim_count, hi = box maximum and first_index.
__device__ __forceinline__ Box tail_box(const float4& lo, const float4& hi) {
    return Box{lo.x, lo.y, lo.z, hi.x, hi.y, hi.z};
}
__device__ __forceinline__ float4 nan4() {
    const float q = __builtin_nanf("");
    return make_float4(q, q, q, q);
}

// Best offset of the cluster with box me at slot lc among the N consecutive offsets from k0 (none of them 0): the last
// minimum, 0 if no cost passes `cost <= INFINITY`.
template <int N, bool NONAN>
__device__ __forceinline__ void search_part(const float4* __restrict__ lo, const float4* __restrict__ hi,
                                            const Box& me, int lc, int k0, int& best, float& best_cost) {
    constexpr int U = N <= 8 ? N : (N % 8 == 0 ? 8 : (N % 7 == 0 ? 7 : 6));
    static_assert(N % U == 0, "block size must divide the part");
#pragma unroll 1
    for (int b = 0; b < N; b += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + b + u;
            const Box ob = tail_box(lo[lc + k], hi[lc + k]);
            const float cost = NONAN ? union_area_nonan(me, ob) : half_area(box_union(me, ob));
            const bool take = cost <= best_cost;
            best = take ? k : best;
            best_cost = take ? cost : best_cost;
        }
    }
}

// cluster_merge_unrolled by G = 1, 2 or 4 adjacent lanes per cluster (lane % G takes its part of the 2R offsets in
// ascending order); every lane of the group gets the result.
template <int R, int G, bool NONAN>
__device__ __forceinline__ int search_group(const float4* __restrict__ lo, const float4* __restrict__ hi, int lc) {
    const Box me = tail_box(lo[lc], hi[lc]);
    int best = 0;
    float best_cost = INFINITY;
    if constexpr (G == 1) {
        search_part<R, NONAN>(lo, hi, me, lc, -R, best, best_cost);
        search_part<R, NONAN>(lo, hi, me, lc, 1, best, best_cost);
    } else {
        constexpr int N = 2 * R / G, H = G / 2;  // H parts on either side of the cluster
        const int part = (int)(threadIdx.x % G);
        search_part<N, NONAN>(lo, hi, me, lc, part < H ? -R + part * N : 1 + (part - H) * N, best, best_cost);
        // the higher part's offsets come later: its minimum wins a tie (lane moves inside a quad: DPP)
        auto combine = [&](int ob, float oc, bool other_later) {
            const bool take = ob != 0 && (best == 0 || (other_later ? oc <= best_cost : oc < best_cost));
            best = take ? ob : best;
            best_cost = take ? oc : best_cost;
        };
        constexpr int XOR1 = 0xB1, XOR2 = 0x4E;  // quad_perm [1, 0, 3, 2] and [2, 3, 0, 1]
        combine(__builtin_amdgcn_update_dpp(0, best, XOR1, 0xF, 0xF, true),
                __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(best_cost), XOR1, 0xF, 0xF, true)),
                (part & 1) == 0);
        if constexpr (G == 4)
            combine(__builtin_amdgcn_update_dpp(0, best, XOR2, 0xF, 0xF, true),
                    __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(best_cost), XOR2, 0xF, 0xF, true)),
                    (part & 2) == 0);
    }
    return best;
}

// The same with the number of lanes per cluster and the NaN choice at run time.
template <int R>
__device__ __forceinline__ int search_lanes(const float4* __restrict__ lo, const float4* __restrict__ hi, int lc,
                                            uint32_t g, bool nonan) {
    if (!nonan) return search_group<R, 1, false>(lo, hi, lc);
    if (g == 4u) return search_group<R, 4, true>(lo, hi, lc);
    if (g == 2u) return search_group<R, 2, true>(lo, hi, lc);
    return search_group<R, 1, true>(lo, hi, lc);
}

// The bounded search of a pass at distance 1 (dist1) or of a distance without an unrolled form.
__device__ __forceinline__ int search_bounded(const float4* __restrict__ lo, const float4* __restrict__ hi, uint32_t i,
                                              uint32_t count, uint32_t r, bool dist1, bool nonan) {
    const Box me = tail_box(lo[i], hi[i]);
    if (dist1) {
        if (i == count - 1) return -1;
        const float cost = half_area(box_union(me, tail_box(lo[i + 1], hi[i + 1])));
        float last = INFINITY;
        if (i > 0) last = half_area(box_union(tail_box(lo[i - 1], hi[i - 1]), me));
        return last < cost ? -1 : 1;
    }
    const uint32_t begin = i - min(r, i), end = min(i + r + 1u, count);
    uint32_t best = i;
    float best_cost = INFINITY;
    for (uint32_t j = begin; j < end; ++j) {
        if (j == i) continue;
        const Box o = tail_box(lo[j], hi[j]);
        const float c = nonan ? union_area_nonan(me, o) : half_area(box_union(me, o));
        if (c <= best_cost) {
            best = j;
            best_cost = c;
        }
    }
    return (int)best - (int)i;
}

// The merges of the tail (at most MAX - 1), listed in LDS for their cost-table entries: first child slot, the
// children's first_index and half area, the node's half area, and its height above the tail's first clusters with the
// children's prim_counts (0, 1, 2 = more) in the top bits.
template <int MAX>
struct TailMerges {
    uint32_t first[MAX], lf[MAX], rf[MAX];
    float ha[MAX], la[MAX], ra[MAX];
    uint16_t h[MAX], order[MAX];
    uint32_t at[MAX];  // merges per height, then where each height's merges begin
};

// The cost-table entries of the listed merges, by height: an entry needs only entries of lower height.  tm.at holds the
// merges per height on entry (after a barrier); MAX / 2 threads, wsum one word per wave.
template <int MAX>
__device__ __forceinline__ uint32_t entries_by_height(TailMerges<MAX>& tm, uint32_t* wsum, uint32_t merges,
                                                      const DpView& dp) {
    constexpr int THREADS = MAX / 2;
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    // The merges in the order of their heights (1 .. top): where each height begins, then the list.
    const uint32_t c0 = tm.at[2 * tid], c1 = tm.at[2 * tid + 1];
    const uint32_t incl = wave_inclusive_scan(c0 + c1);
    if ((tid & 63u) == 63u) wsum[wave] = incl;
    lds_barrier();
    uint32_t base = incl - (c0 + c1);
    for (uint32_t w = 0; w < wave; ++w) base += wsum[w];
    tm.at[2 * tid] = base;
    tm.at[2 * tid + 1] = base + c0;
    lds_barrier();
    for (uint32_t m = tid; m < merges; m += THREADS)
        tm.order[atomicAdd(&tm.at[tm.h[m] & 0xfffu], 1u)] = (uint16_t)m;
    lds_barrier();  // tm.at[h] is now where height h ends
    uint32_t err = 0u;
    for (uint32_t h = 1u; tm.at[h - 1] < merges; ++h) {
        for (uint32_t j = tm.at[h - 1] + tid; j < tm.at[h]; j += THREADS) {
            const uint32_t m = tm.order[j], c = tm.h[m];
            err |= dp_evaluate(dp, tm.ha[m], tm.first[m], DpChild{tm.lf[m], c >> 12 & 3u, tm.la[m]},
                               DpChild{tm.rf[m], c >> 14, tm.ra[m]});
        }
        __syncthreads();  // the next height reads this one's entries
    }
    return err;
}

// One merge of the tail: the children a (higher index) and b go to their slots, the merge to the list; returns the
// parent (and its height in h).  False slots are reported by the result.
template <int MAX>
__device__ __forceinline__ bool tail_merge(float4& alo, float4& ahi, uint32_t& h, const float4& blo, const float4& bhi,
                                           uint32_t bh, uint32_t v, const uint32_t* __restrict__ slot_map,
                                           uint32_t vtop, uint32_t map_len, Node32* __restrict__ bvh_nodes,
                                           TailMerges<MAX>& tm, uint32_t m, uint32_t fused) {
    uint32_t first = 0u;
    const bool ok = child_slot(v, slot_map, vtop, map_len, first);
    if (ok) {
        float4* q = reinterpret_cast<float4*>(&bvh_nodes[first]);
        q[0] = alo;
        q[1] = ahi;
        q[2] = blo;
        q[3] = bhi;
    }
    const Box a = tail_box(alo, ahi), b = tail_box(blo, bhi), u = box_union(a, b);
    h = 1u + max(h, bh);
    if (fused) {
        tm.first[m] = first;
        tm.lf[m] = __float_as_uint(ahi.w);
        tm.rf[m] = __float_as_uint(bhi.w);
        tm.ha[m] = half_area(u);
        tm.la[m] = half_area(a);
        tm.ra[m] = half_area(b);
        tm.h[m] = (uint16_t)(h | min(__float_as_uint(alo.w), 2u) << 12 | min(__float_as_uint(blo.w), 2u) << 14);
        atomicAdd(&tm.at[h], 1u);
    }
    alo = make_float4(u.lx, u.ly, u.lz, __uint_as_float(0u));
    ahi = make_float4(u.hx, u.hy, u.hz, __uint_as_float(first));
    return ok;
}

// Finishes a build inside one workgroup of MAX / 2 threads from its state (the same in every thread, count <= MAX)
// and the clusters in cur; hist may be NULL.  Clusters live in LDS as SoA.
// A pass is three steps between LDS barriers: the search (1, 2 or 4 lanes per cluster, so that a pass of few clusters
// does not wait for one lane's 2R neighbours), the classification with the reads of everything a thread will write
// (ballots give the positions), and the writes.  The nodes go out as plain stores that nothing waits for.  From 64
// clusters on one wave makes the passes alone, without barriers.  The merges are listed in LDS, and their cost-table
// entries are evaluated after the last pass by height above the tail's first clusters: an entry needs only entries of
// lower height, and there are fewer heights than passes (1,135 clusters: 14 against 29).
// A chain of passes and entries bounds the kernel, not any throughput.  1.29M-triangle build (1,135 clusters): 182 ->
// 114 us; of the 16.8K cycles of a late pass 9.7K had been the entries of the pass before it, 4.5K a lane's search,
// 2.9K the scan with a serial step and 3.4K a barrier that waited for the node stores.
// R > 0: the search distance, known at compile time (the unrolled search over NaN-padded arrays); R = 0: any r.
template <int R, int MAX>
__device__ __forceinline__ void ploc_tail(const Node32* __restrict__ cur, PlocState& state, uint32_t first_pass,
                                          uint32_t r, uint32_t sd_is_one, uint32_t depth_threshold,
                                          Node32* __restrict__ bvh_nodes, uint32_t* __restrict__ hist,
                                          const DpView& dp, uint32_t fused, const uint32_t* __restrict__ slot_map,
                                          uint32_t vtop, uint32_t map_len, uint32_t* err) {
    constexpr int ITEMS = 2, THREADS = MAX / ITEMS;
    // Cluster arrays with MAX_RADIUS slots on either side: NaN boxes before cluster 0 and after the last cluster, so
    // that the unrolled search needs no bounds test (refreshed after each pass's compaction).
    constexpr int PADDED = MAX + 2 * MAX_RADIUS;
    __shared__ float4 lo_p[PADDED], hi_p[PADDED];
    float4* const lo = lo_p + MAX_RADIUS;
    float4* const hi = hi_p + MAX_RADIUS;
    __shared__ uint16_t ht[MAX];  // height above the tail's first clusters
    __shared__ int8_t mg[MAX];
    __shared__ TailMerges<MAX> tm;
    __shared__ __align__(16) uint32_t wsum[THREADS / 64];
    __shared__ PlocState s_state;  // of the passes of one wave
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    uint32_t count = state.count;
    bool nan_here = false;
    for (uint32_t i = tid; i < count; i += THREADS) {
        const float4* q = reinterpret_cast<const float4*>(&cur[i]);
        const float4 a = q[0], b = q[1];
        lo[i] = a;
        hi[i] = b;
        ht[i] = 0;
        nan_here |= box_has_nan_any(tail_box(a, b));
    }
    for (uint32_t i = tid; i < MAX; i += THREADS) tm.at[i] = 0u;
    if (tid < 2u * MAX_RADIUS) {  // the pads: [-MAX_RADIUS, 0) and [count, count + MAX_RADIUS)
        const int p = tid < MAX_RADIUS ? -1 - (int)tid : (int)(count + tid - MAX_RADIUS);
        lo[p] = hi[p] = nan4();
    }
    // NaN-free clusters (merging keeps them so): search costs from union_area_nonan
    const bool nonan = !__syncthreads_or(nan_here);
    uint32_t insert = state.insert;
    uint32_t depth = state.depth;
    unsigned long long csum = state.cluster_sum;
    uint32_t pass = first_pass;
    bool self_merge = false;
    bool bad_slot = false;
    uint32_t merges = 0u;  // listed so far
    while (count > 64u) {
        csum += count;
        const bool dist1 = sd_is_one || pass < depth_threshold;
        // lanes per cluster: 4 for at most 256 clusters, 2 for at most 512
        const uint32_t g = R == 0 || dist1 ? 1u : (count <= THREADS / 4 ? 4u : (count <= THREADS / 2 ? 2u : 1u));
        for (uint32_t i = tid / g; i < count; i += THREADS / g) {  // the same i in a group's lanes
            int b;
            if (R == 0 || dist1)
                b = search_bounded(lo, hi, i, count, r, dist1, nonan);
            else
                b = search_lanes<R == 0 ? 2 : R>(lo, hi, (int)i, g, nonan);
            if (b == 0) self_merge = true;
            if (tid % g == 0u) mg[i] = (int8_t)b;
        }
        lds_barrier();
        // Thread t owns cluster t, or clusters 2t and 2t + 1 when there are more clusters than threads.
        const bool two = count > (uint32_t)THREADS;
        bool emit[ITEMS], mrg[ITEMS];
        uint64_t be[ITEMS], bm[ITEMS];
        float4 alo[ITEMS], ahi[ITEMS], blo[ITEMS], bhi[ITEMS];
        uint32_t ah[ITEMS], bh[ITEMS];
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            emit[q] = mrg[q] = false;
            be[q] = bm[q] = 0ull;
            if (q > 0 && !two) continue;  // uniform
            const uint32_t i = two ? tid * ITEMS + q : tid;
            const Cls k = classify(mg, i, count);
            const uint32_t b = k.b;
            emit[q] = k.emit;
            mrg[q] = k.mrg;
            be[q] = __ballot(emit[q]);
            bm[q] = __ballot(mrg[q]);
            // everything this thread writes is read before anyone overwrites the LDS arrays
            if (emit[q]) {
                alo[q] = lo[i];
                ahi[q] = hi[i];
                ah[q] = ht[i];
                if (mrg[q]) {
                    blo[q] = lo[b];
                    bhi[q] = hi[b];
                    bh[q] = ht[b];
                }
            }
        }
        if ((tid & 63u) == 0u)
            wsum[wave] = (uint32_t)(__popcll(be[0]) + __popcll(be[1])) |
                         (uint32_t)(__popcll(bm[0]) + __popcll(bm[1])) << 16;
        lds_barrier();
        uint32_t before = 0u, total = 0u;
#pragma unroll
        for (uint32_t w = 0; w < THREADS / 64; ++w) {
            const uint32_t x = wsum[w];
            before += w < wave ? x : 0u;
            total += x;
        }
        const uint64_t lt = lanemask_lt();
        uint32_t pe = (before & 0xffffu) + (uint32_t)(__popcll(be[0] & lt) + __popcll(be[1] & lt));
        uint32_t pm = (before >> 16) + (uint32_t)(__popcll(bm[0] & lt) + __popcll(bm[1] & lt));
#pragma unroll
        for (int q = 0; q < ITEMS; ++q) {
            if (!emit[q]) continue;
            if (mrg[q]) {
                bad_slot |= !tail_merge(alo[q], ahi[q], ah[q], blo[q], bhi[q], bh[q], insert - 2u * (pm + 1u), slot_map,
                                        vtop, map_len, bvh_nodes, tm, merges + pm, fused);
                pm++;
            }
            lo[pe] = alo[q];
            hi[pe] = ahi[q];
            ht[pe] = (uint16_t)ah[q];
            pe++;
        }
        if (tid < MAX_RADIUS)  // the pad after the new count (old clusters' slots, read before the last barrier)
            lo[(total & 0xffffu) + tid] = hi[(total & 0xffffu) + tid] = nan4();
        lds_barrier();
        merges += total >> 16;
        count = total & 0xffffu;
        insert -= 2u * (total >> 16);
        depth += 1u;
        pass += 1u;
        if (hist && tid == 0) hist[depth] = insert;
        if ((total >> 16) == 0u) {
            // No mutual pair in this pass: the reference would loop forever; report instead of hanging.
            self_merge = true;
            break;
        }
    }
    if (wave == 0u && count <= 64u) {
        const uint32_t lane = tid;
        const uint64_t lt = lanemask_lt();
        while (count > 1u) {
            csum += count;
            const bool dist1 = sd_is_one || pass < depth_threshold;
            const uint32_t g = R == 0 || dist1 ? 1u : (count <= 16u ? 4u : (count <= 32u ? 2u : 1u));
            int m = 0;
            if (lane / g < count) {
                if (R == 0 || dist1)
                    m = search_bounded(lo, hi, lane, count, r, dist1, nonan);
                else
                    m = search_lanes<R == 0 ? 2 : R>(lo, hi, (int)(lane / g), g, nonan);
                if (m == 0) self_merge = true;
            }
            if (g > 1u) m = __shfl(m, (int)(lane * g & 63u));  // lane i: cluster i's offset
            const bool valid = lane < count;
            const uint32_t b = valid ? (uint32_t)((int)lane + m) : lane;
            const bool mutual = (int)b + __shfl(m, (int)b) == (int)lane;
            // classify: a self-pair is kept, the higher index of a mutual pair becomes the parent
            const bool mrg = valid && mutual && b < lane, emit = valid && (!mutual || b <= lane);
            const uint64_t be = __ballot(emit), bm = __ballot(mrg);
            float4 alo = lo[lane], ahi = hi[lane];
            uint32_t ah = ht[lane];
            const float4 blo = lo[b], bhi = hi[b];
            const uint32_t bh = ht[b];
            wave_lds_fence();
            const uint32_t nm = (uint32_t)__popcll(bm);
            if (mrg) {
                const uint32_t pm = (uint32_t)__popcll(bm & lt);
                bad_slot |= !tail_merge(alo, ahi, ah, blo, bhi, bh, insert - 2u * (pm + 1u), slot_map, vtop, map_len,
                                        bvh_nodes, tm, merges + pm, fused);
            }
            count = (uint32_t)__popcll(be);
            if (emit) {
                const uint32_t pe = (uint32_t)__popcll(be & lt);
                lo[pe] = alo;
                hi[pe] = ahi;
                ht[pe] = (uint16_t)ah;
            }
            if (lane < MAX_RADIUS) lo[count + lane] = hi[count + lane] = nan4();
            wave_lds_fence();
            merges += nm;
            insert -= 2u * nm;
            depth += 1u;
            pass += 1u;
            if (hist && lane == 0u) hist[depth] = insert;
            if (nm == 0u) {
                self_merge = true;
                break;
            }
        }
        if (lane == 0u) s_state = PlocState{count, insert, depth, merges, csum};
    }
    lds_barrier();
    if (count <= 64u) {
        const PlocState x = s_state;
        count = x.count;
        insert = x.insert;
        depth = x.depth;
        merges = x.pad;
        csum = x.cluster_sum;
    }
    uint32_t dp_err = 0u;
    if (fused && merges != 0u) {
        dp_err = entries_by_height(tm, wsum, merges, dp);
    }
    if (self_merge) atomicOr(err, DERR_SELF_MERGE);
    if (bad_slot) atomicOr(err, DERR_CAPACITY);
    if (dp_err) atomicOr(err, dp_err);
    if (tid == 0) {
        float4* q = reinterpret_cast<float4*>(&bvh_nodes[0]);
        q[0] = lo[0];
        q[1] = hi[0];
    }
    state = PlocState{count, insert, depth, 0u, csum};
}

}  // namespace

}  // namespace obvhs
