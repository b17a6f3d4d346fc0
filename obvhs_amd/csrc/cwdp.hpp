// The BVH2 -> CWBVH cost table (calculate_cost_impl, cwbvh/bvh2_to_cwbvh.rs:220-344) and get_children
// (bvh2_to_cwbvh.rs:346-397) over a BVH2 whose internal nodes are identified by their first child slot.
//
// A PLOC internal node's children always exist before the node does, and the node's own array slot is assigned
// only later, when it is merged in turn.  Its first_index (the slot of its left child, always odd) is known at
// creation, so the table is keyed by first_index >> 1.  That lets the merge that creates a node evaluate the
// node's entry immediately (children finished earlier, no cross-workgroup synchronisation), and the same
// functions serve a standalone pass over a finished BVH2.  Leaves need no entry: all seven of their decisions are
// LEAF with cost half_area * 1 * 0.3 (bvh2_to_cwbvh.rs:249-256).
//
// Besides the reference's seven (cost, kind, distribute_left, distribute_right) decisions, each entry holds, per
// decision i, sub[i] = the number of CWBVH nodes in the subtrees of the INTERNAL children that get_children(node, i)
// would produce.  It obeys the same recurrence as the costs (children only), so no tree walk is needed, and
// cwsize = 1 + sub[0] is the size of the CWBVH subtree the node roots if it becomes a CWBVH node -- what the
// top-down pass needs to number nodes in the reference's pre-order (bvh2_to_cwbvh.rs:172-191).  The same
// recurrence with max instead of + gives the depth of that CWBVH subtree, so the top-down pass knows its level
// count without reading anything back.  Each entry also keeps the children's first_index words and, for a subtree
// of at most 3 primitives, its leaf list: the top-down pass walks get_children and collects a leaf child's
// primitives from the table, one dependent load per level instead of a node and then its decisions.
#pragma once

#include "common.hpp"
#include "device_util.hpp"
#include "internal.hpp"

namespace obvhs {

constexpr uint32_t KIND_LEAF = 0, KIND_INTERNAL = 1, KIND_DISTRIBUTE = 2;  // bvh2_to_cwbvh.rs:470-476
constexpr uint32_t DIDX_INVALID = 7u;      // distribute index "INVALID" (u8::MAX in the reference) in 3 bits
constexpr uint32_t SUB_INVALID = 0xffffffffu;
constexpr float PRIM_COST = 0.3f;  // bvh2_to_cwbvh.rs:30
constexpr uint32_t KID_LEAF = 0x80000000u;  // leaf flag in DpView::kids

// One table entry, a 128-byte cache line: every read of a node's entry (a parent's evaluation, a step of the
// get_children walk, the emit of a leaf list or a child's sizes) touches a single line.
// Decision byte: kind (2 bits) | distribute_left << 2 (3 bits) | distribute_right << 5 (3 bits).
struct __align__(128) DpRec {
    float cost[7];
    uint32_t nprims;    // primitives under the node
    uint32_t sub[7];
    uint32_t cwsize;    // 1 + sub[0], or 0 when the node's CWBVH subtree cannot be built
    uint2 meta;         // seven decision bytes (byte 7 unused)
    uint2 subdepth;     // seven bytes: CWBVH depth below the children get_children(node, i) produces
    uint2 kids;         // the children's first_index (bit 31 set for a leaf), left then right
    uint32_t cwdepth;   // 1 + subdepth[0]: levels of the CWBVH subtree the node roots
    uint32_t pad0;
    uint4 plist;        // for a subtree of at most 3 primitives: its leaves' first_index, left first, and count
    uint32_t pad1[4];
};
static_assert(sizeof(DpRec) == 128, "one cache line per entry");

struct DpView {
    DpRec* rec;         // [k]
    uint32_t max_prims; // max_prims_per_leaf the table was evaluated for
    uint32_t kbase;     // key offset of the BVH2 being processed (batched builds: the mesh's first primitive)
};

// One BVH of a batched build: slices of the shared node / primitive / cost-table / CWBVH arrays.
struct MeshDesc {
    uint32_t node_base;   // first BVH2 slot (2 * prim_base, so cost-table keys stay disjoint)
    uint32_t prim_base;   // first primitive; also the mesh's cost-table key base
    uint32_t prim_count;
    uint32_t cw_base;     // first CWBVH node
    uint32_t cw_count;
    uint32_t cw_depth;
    uint32_t radius;      // the mesh's PLOC search distance
    uint32_t pad;
};

// Table of k entries (the base must be 128-byte aligned; device allocations are 256-byte aligned).
__host__ __device__ __forceinline__ size_t dp_table_bytes(size_t k) { return k * sizeof(DpRec) + 1024; }
__host__ __device__ __forceinline__ DpView dp_view_at(char* base, size_t k, uint32_t max_prims) {
    (void)k;
    DpView v;
    v.rec = reinterpret_cast<DpRec*>(base);
    v.max_prims = max_prims;
    v.kbase = 0u;
    return v;
}

__host__ __device__ __forceinline__ uint32_t dkey(uint32_t first_index) { return first_index >> 1; }
__device__ __forceinline__ size_t dp_key(const DpView& dp, uint32_t first_index) {
    return (size_t)dp.kbase + (first_index >> 1);
}
__device__ __forceinline__ uint32_t dbyte(uint2 m, uint32_t i) {
    return ((i < 4u ? m.x : m.y) >> (8u * (i & 3u))) & 0xffu;
}
__device__ __forceinline__ uint32_t dkind(uint32_t b) { return b & 3u; }
__device__ __forceinline__ uint32_t dleft(uint32_t b) { return (b >> 2) & 7u; }
__device__ __forceinline__ uint32_t dright(uint32_t b) { return (b >> 5) & 7u; }
__device__ __forceinline__ uint32_t dpack(uint32_t k, uint32_t l, uint32_t r) { return k | (l << 2) | (r << 5); }

// What the evaluation reads of a child's node.
struct DpChild {
    uint32_t first_index, prim_count;
    float area;  // half area of its box
};

// Everything the parent's evaluation needs from one child, in registers.
struct ChildDp {
    float cost[7];
    uint32_t size[7];   // per decision, the CWBVH nodes the child contributes when taken through it
    uint32_t depth[7];  // per decision, the CWBVH levels below the parent through it
    uint32_t nprims;
    uint4 plist;        // leaf list (nprims <= 3)
};

// The first 112 bytes of a record, as loaded.
struct DpRaw {
    uint4 w[7];
};
__device__ __forceinline__ DpRaw load_dp_raw(const DpRec* rec) {
    const uint4* e = reinterpret_cast<const uint4*>(rec);
    DpRaw r;
#pragma unroll
    for (int k = 0; k < 7; ++k) r.w[k] = e[k];
    return r;
}

// The child's costs and contributions through each decision d: its own CWBVH subtree (size and depth) when it becomes
// a CWBVH child, those of its distributed descendants when it is DISTRIBUTE, nothing when it is a leaf child.
// SUB_INVALID marks a subtree that cannot be built.  raw: the child's record (any record for a leaf).
__device__ __forceinline__ ChildDp child_dp(const DpChild& c, const DpRaw& raw) {
    ChildDp o;
    const bool leaf = c.prim_count != 0u;
    const float leaf_cost = c.area * (float)c.prim_count * PRIM_COST;
    const uint4 c0 = raw.w[0], c1 = raw.w[1], s0 = raw.w[2], s1 = raw.w[3], m = raw.w[4], kc = raw.w[5], pl = raw.w[6];
    const uint32_t cost[7] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z}, sub[7] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z};
    const uint32_t cwsize = s1.w, cwdepth = kc.z;
    const uint2 meta = leaf ? make_uint2(0u, 0u) : make_uint2(m.x, m.y);  // a leaf's decisions are all LEAF
    const uint2 subdepth = make_uint2(m.z, m.w);
    const bool internal = dkind(dbyte(meta, 0u)) == KIND_INTERNAL;
    const uint32_t size0 = internal ? (cwsize == 0u ? SUB_INVALID : cwsize) : 0u, depth0 = internal ? cwdepth : 0u;
#pragma unroll
    for (uint32_t d = 0; d < 7u; ++d) {
        const bool dist = dkind(dbyte(meta, d)) == KIND_DISTRIBUTE;
        o.cost[d] = leaf ? leaf_cost : __uint_as_float(cost[d]);
        o.size[d] = dist ? sub[d] : size0;
        o.depth[d] = dist ? dbyte(subdepth, d) : depth0;
    }
    o.nprims = leaf ? c.prim_count : c1.w;
    o.plist = leaf ? make_uint4(c.first_index, 0u, 0u, 1u) : pl;
    return o;
}

// Evaluates the entry of the internal node of half area `ha` whose children are `l` and `r` (slots first, first + 1)
// and stores it under its key; raw_l and raw_r are the children's records (dp_child_record).  Returns a DERR_* bit or 0.
// One round of loads (both records at once, whatever the children are), selects without branches that carry the
// sizes and depths below the best pair of decisions along with its cost, one round of stores.  Where entries wait on
// each other the evaluation is a latency: in k_ploc_tail it took 9.7K cycles when the chosen pair's sizes were read
// from the records afterwards (up to 14 loads one after the other), 7.5K with the records loaded one after the other
// and a branch per candidate pair (1.29M-triangle build: the tail 215 -> 182 us, the grid passes' compactions 376 ->
// 338 us, the refit's table 792 -> 630 us).
__device__ __forceinline__ uint32_t dp_entry(const DpView& dp, float ha, const DpChild& l, const DpChild& r,
                                             const DpRaw& raw_l, const DpRaw& raw_r, uint4* e) {
    const bool ll = l.prim_count != 0u, rl = r.prim_count != 0u;
    const ChildDp L = child_dp(l, raw_l), R = child_dp(r, raw_r);
    const uint32_t num_primitives = L.nprims + R.nprims;
    const float cost_leaf = num_primitives <= dp.max_prims ? ((float)num_primitives) * ha * PRIM_COST : INFINITY;
    // aux: the pair's decision byte without its kind (dpack's distribute indices) and its depth from bit 8 up
    float cost[7];
    uint32_t meta[7], sub[7], sd[7];
    auto pick = [&](int last, float& best, uint32_t& size, uint32_t& aux) {  // pairs (k, last - k), first strict minimum
#pragma unroll
        for (int k = 0; k <= last; ++k) {
            const float c = L.cost[k] + R.cost[last - k];
            const uint32_t s = __builtin_elementwise_add_sat(L.size[k], R.size[last - k]);  // SUB_INVALID stays
            const uint32_t a = dpack(0u, (uint32_t)k, (uint32_t)(last - k)) | max(L.depth[k], R.depth[last - k]) << 8;
            const bool lower = c < best;
            best = lower ? c : best;
            size = lower ? s : size;
            aux = lower ? a : aux;
        }
    };
    constexpr uint32_t NONE = (DIDX_INVALID << 2) | (DIDX_INVALID << 5);  // no pair has a finite cost; depth 0
    float best = INFINITY;
    uint32_t size = SUB_INVALID, aux = NONE;
    pick(6, best, size, aux);
    const float cost_internal = best + ha;
    cost[0] = cost_leaf < cost_internal ? cost_leaf : cost_internal;
    meta[0] = (aux & 0xffu) | (cost_leaf < cost_internal ? KIND_LEAF : KIND_INTERNAL);
    sub[0] = size;
    sd[0] = aux >> 8;
#pragma unroll
    for (int i = 1; i < 7; ++i) {
        best = cost[i - 1];
        size = sub[i - 1];
        aux = NONE;
        pick(i - 1, best, size, aux);
        const bool found = (aux & 0xffu) != NONE;  // a pair's indices are below 7
        cost[i] = best;
        meta[i] = found ? ((aux & 0xffu) | KIND_DISTRIBUTE) : meta[i - 1];
        sub[i] = size;
        sd[i] = found ? aux >> 8 : sd[i - 1];
    }
#pragma unroll
    for (int i = 0; i < 7; ++i) sd[i] = min(255u, sd[i]);
    // The leaves count_primitives (bvh2_to_cwbvh.rs:197-211) visits, left subtree first.  Each child holds at least
    // one leaf, so the left list has one or two entries.
    const bool two = L.plist.w >= 2u, few = num_primitives <= 3u;
    const uint4 pl = make_uint4(few ? L.plist.x : 0u, few ? (two ? L.plist.y : R.plist.x) : 0u,
                                few ? (two ? R.plist.x : R.plist.y) : 0u, few ? num_primitives : 0u);
    // The whole 128-byte entry (the padding too, so that no 32-byte sector of the line is left partly written).
    e[0] = make_uint4(__float_as_uint(cost[0]), __float_as_uint(cost[1]), __float_as_uint(cost[2]),
                      __float_as_uint(cost[3]));
    e[1] = make_uint4(__float_as_uint(cost[4]), __float_as_uint(cost[5]), __float_as_uint(cost[6]), num_primitives);
    e[2] = make_uint4(sub[0], sub[1], sub[2], sub[3]);
    e[3] = make_uint4(sub[4], sub[5], sub[6], sub[0] == SUB_INVALID ? 0u : 1u + sub[0]);
    e[4] = make_uint4(meta[0] | meta[1] << 8 | meta[2] << 16 | meta[3] << 24, meta[4] | meta[5] << 8 | meta[6] << 16,
                      sd[0] | sd[1] << 8 | sd[2] << 16 | sd[3] << 24, sd[4] | sd[5] << 8 | sd[6] << 16);
    e[5] = make_uint4(l.first_index | (ll ? KID_LEAF : 0u), r.first_index | (rl ? KID_LEAF : 0u), 1u + sd[0], 0u);
    e[6] = pl;
    e[7] = make_uint4(0u, 0u, 0u, 0u);
    // checked last, so that the records' loads do not wait for the leaf counts (bvh2_to_cwbvh.rs:243-247)
    return l.prim_count > 1u || r.prim_count > 1u ? DERR_CW_NONUNIT_LEAF : 0u;
}

__device__ __forceinline__ uint32_t dp_evaluate(const DpView& dp, float ha, uint32_t first, const DpChild& l,
                                                const DpChild& r, const DpRaw& raw_l, const DpRaw& raw_r) {
    uint4 e[8];
    const uint32_t err = dp_entry(dp, ha, l, r, raw_l, raw_r, e);
    uint4* rec = reinterpret_cast<uint4*>(&dp.rec[dp_key(dp, first)]);
#pragma unroll
    for (int k = 0; k < 8; ++k) rec[k] = e[k];
    return err;
}

// The record to load for a child.  A leaf has none: the table's first is read in its place (a line every lane shares)
// and not used.
__device__ __forceinline__ const DpRec* dp_child_record(const DpView& dp, const DpChild& c) {
    return &dp.rec[c.prim_count != 0u ? (size_t)dp.kbase : dp_key(dp, c.first_index)];
}
__device__ __forceinline__ const DpRec* dp_child_record(const DpView& dp, const Node32& c) {
    return &dp.rec[c.prim_count != 0u ? (size_t)dp.kbase : dp_key(dp, c.first_index)];
}
__device__ __forceinline__ DpChild dp_child(const Node32& c) {
    return DpChild{c.first_index, c.prim_count, half_area(node_box(c))};
}

__device__ __forceinline__ uint32_t dp_evaluate(const DpView& dp, float ha, uint32_t first, const DpChild& l,
                                                const DpChild& r) {
    const DpRaw raw_l = load_dp_raw(dp_child_record(dp, l)), raw_r = load_dp_raw(dp_child_record(dp, r));
    // every load stays above this line: spread over the evaluation to save registers, each part waits on its own
    __builtin_amdgcn_sched_barrier(0);
    return dp_evaluate(dp, ha, first, l, r, raw_l, raw_r);
}

// The same for a node with box `box` and children `l` and `r`.
__device__ __forceinline__ uint32_t dp_evaluate(const DpView& dp, const Box& box, uint32_t first, const Node32& l,
                                                const Node32& r) {
    return dp_evaluate(dp, half_area(box), first, dp_child(l), dp_child(r));
}

// The same by a whole wave, the entries written eight lanes to a record through buf (2 KB of LDS of the wave's own): a
// lane that stores its own record touches another line with every 16 bytes, 64 requests of a store instruction where
// eight lanes a record make 16 (the batch's compactions 3.19 -> 2.65 ms at 20M triangles).  Lanes without an entry: valid
// false, any leaves.
__device__ __forceinline__ uint32_t dp_evaluate_wave(const DpView& dp, const Box& box, uint32_t first, const Node32& l,
                                                     const Node32& r, bool valid, uint4* buf) {
    const DpChild cl = dp_child(l), cr = dp_child(r);
    const DpRaw raw_l = load_dp_raw(dp_child_record(dp, cl)), raw_r = load_dp_raw(dp_child_record(dp, cr));
    __builtin_amdgcn_sched_barrier(0);
    uint4 e[8];
    const uint32_t err = dp_entry(dp, half_area(box), cl, cr, raw_l, raw_r, e);
    const uint32_t lane = __lane_id(), key = (uint32_t)dp_key(dp, first);
    const uint64_t entries = __ballot(valid);
    wave_lds_fence();  // buf may hold what lanes of the wave have just read as something else
#pragma unroll
    for (uint32_t q = 0; q < 4u; ++q) {  // 16 records at a time
        if (((entries >> (16u * q)) & 0xffffull) == 0ull) continue;
        if ((lane >> 4) == q) {
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) buf[(lane & 15u) * 8u + (k ^ (lane & 7u))] = e[k];
        }
        wave_lds_fence();
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h) {
            const uint32_t rec = h * 8u + (lane >> 3), from = 16u * q + rec, part = lane & 7u;
            const uint4 v = buf[rec * 8u + (part ^ (rec & 7u))];
            const uint32_t to = (uint32_t)__shfl((int)key, (int)from);
            if ((entries >> from) & 1ull) reinterpret_cast<uint4*>(&dp.rec[to])[part] = v;
        }
        wave_lds_fence();
    }
    return valid ? err : 0u;
}

// The root's part of the evaluated table (1 and 1 for a single-leaf BVH2).
__device__ __forceinline__ CwRootInfo root_info(const Node32* nodes, const DpView& dp) {
    const Node32 n = load_node(&nodes[0]);
    CwRootInfo r{{n.minx, n.miny, n.minz}, {n.maxx, n.maxy, n.maxz}, 1u, 1u};
    if (n.prim_count == 0u) {
        const DpRec& e = dp.rec[dkey(n.first_index)];
        r.size = e.cwsize;
        r.depth = e.cwdepth;
    }
    return r;
}

}  // namespace obvhs
