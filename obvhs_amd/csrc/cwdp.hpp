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

// Everything the parent's evaluation needs from one child, in registers: the whole record's loads go out together.
struct ChildDp {
    float cost[7];
    uint32_t size[7];   // per decision, the CWBVH nodes the child contributes when taken through it
    uint32_t depth[7];  // per decision, the CWBVH levels below the parent through it
    uint32_t nprims;
    uint4 plist;        // leaf list (nprims <= 3)
    bool leaf;
};

// Contributions of a child taken through decision d: its own CWBVH subtree (size and depth) when it becomes a CWBVH
// child, those of its distributed descendants when it is DISTRIBUTE, nothing when it is a leaf child.  SUB_INVALID
// marks a subtree that cannot be built.
__device__ __forceinline__ void load_child_dp(const DpView& dp, const Node32& c, ChildDp& o) {
    o.leaf = c.prim_count != 0u;
    if (o.leaf) {
        const float leaf = half_area(node_box(c)) * (float)c.prim_count * PRIM_COST;
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            o.cost[k] = leaf;
            o.size[k] = 0u;
            o.depth[k] = 0u;
        }
        o.nprims = c.prim_count;
        o.plist = make_uint4(c.first_index, 0u, 0u, 1u);
    } else {
        const uint4* e = reinterpret_cast<const uint4*>(&dp.rec[dp_key(dp, c.first_index)]);
        const uint4 c0 = e[0], c1 = e[1], s0 = e[2], s1 = e[3], m = e[4], kc = e[5];
        o.plist = e[6];
        o.cost[0] = __uint_as_float(c0.x);
        o.cost[1] = __uint_as_float(c0.y);
        o.cost[2] = __uint_as_float(c0.z);
        o.cost[3] = __uint_as_float(c0.w);
        o.cost[4] = __uint_as_float(c1.x);
        o.cost[5] = __uint_as_float(c1.y);
        o.cost[6] = __uint_as_float(c1.z);
        o.nprims = c1.w;
        const uint32_t sub[7] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z};
        const uint32_t cwsize = s1.w, cwdepth = kc.z;
        const uint2 meta = make_uint2(m.x, m.y), subdepth = make_uint2(m.z, m.w);
        const bool internal = dkind(dbyte(meta, 0u)) == KIND_INTERNAL;
        const uint32_t size0 = internal ? (cwsize == 0u ? SUB_INVALID : cwsize) : 0u, depth0 = internal ? cwdepth : 0u;
#pragma unroll
        for (uint32_t d = 0; d < 7u; ++d) {
            const bool dist = dkind(dbyte(meta, d)) == KIND_DISTRIBUTE;
            o.size[d] = dist ? sub[d] : size0;
            o.depth[d] = dist ? dbyte(subdepth, d) : depth0;
        }
    }
}

// Evaluates the entry of the internal node with box `box` whose children records are `l` and `r` (slots first,
// first + 1) and stores it under its key.  Returns a DERR_* bit or 0.
// The sizes and depths below the chosen pair of decisions are carried along with its cost, so the evaluation is one
// round of loads, arithmetic and one round of stores.  (Reading the chosen pair's sizes from the records afterwards
// took up to 14 loads one after the other, each behind its own branch: 9.7K of the 16.8K cycles of a pass of
// k_ploc_tail, where the entries wait on nothing else.)
__device__ __forceinline__ uint32_t dp_evaluate(const DpView& dp, const Box& box, uint32_t first, const Node32& l,
                                                const Node32& r) {
    if ((l.prim_count != 0u && l.prim_count != 1u) || (r.prim_count != 0u && r.prim_count != 1u))
        return DERR_CW_NONUNIT_LEAF;  // bvh2_to_cwbvh.rs:243-247
    ChildDp L, R;
    load_child_dp(dp, l, L);
    load_child_dp(dp, r, R);
    const uint32_t num_primitives = L.nprims + R.nprims;
    const float ha = half_area(box);
    float cost[7];
    uint32_t meta[7], sub[7], sd[7];
    {
        const float cost_leaf =
            num_primitives <= dp.max_prims ? ((float)num_primitives) * ha * PRIM_COST : INFINITY;
        float cost_distribute = INFINITY;
        uint32_t dl = DIDX_INVALID, dr = DIDX_INVALID;
        sub[0] = SUB_INVALID;
        sd[0] = 0u;
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            const float c = L.cost[k] + R.cost[6 - k];
            const uint32_t size = __builtin_elementwise_add_sat(L.size[k], R.size[6 - k]);  // SUB_INVALID stays
            const uint32_t depth = max(L.depth[k], R.depth[6 - k]);
            if (c < cost_distribute) {
                cost_distribute = c;
                dl = (uint32_t)k;
                dr = (uint32_t)(6 - k);
                sub[0] = size;
                sd[0] = depth;
            }
        }
        const float cost_internal = cost_distribute + ha;
        if (cost_leaf < cost_internal) {
            cost[0] = cost_leaf;
            meta[0] = dpack(KIND_LEAF, dl, dr);
        } else {
            cost[0] = cost_internal;
            meta[0] = dpack(KIND_INTERNAL, dl, dr);
        }
    }
#pragma unroll
    for (int i = 1; i < 7; ++i) {
        float cost_distribute = cost[i - 1];
        uint32_t dl = DIDX_INVALID, dr = DIDX_INVALID;
        sub[i] = sub[i - 1];
        sd[i] = sd[i - 1];
#pragma unroll
        for (int k = 0; k < i; ++k) {
            const float c = L.cost[k] + R.cost[i - k - 1];
            const uint32_t size = __builtin_elementwise_add_sat(L.size[k], R.size[i - k - 1]);
            const uint32_t depth = max(L.depth[k], R.depth[i - k - 1]);
            if (c < cost_distribute) {
                cost_distribute = c;
                dl = (uint32_t)k;
                dr = (uint32_t)(i - k - 1);
                sub[i] = size;
                sd[i] = depth;
            }
        }
        if (dl != DIDX_INVALID) {
            cost[i] = cost_distribute;
            meta[i] = dpack(KIND_DISTRIBUTE, dl, dr);
        } else {
            cost[i] = cost[i - 1];
            meta[i] = meta[i - 1];
        }
    }
#pragma unroll
    for (int i = 0; i < 7; ++i) sd[i] = min(255u, sd[i]);
    // The leaves count_primitives (bvh2_to_cwbvh.rs:197-211) visits, left subtree first.  Each child holds at least
    // one leaf, so the left list has one or two entries.
    uint4 pl = make_uint4(0u, 0u, 0u, 0u);
    if (num_primitives <= 3u)
        pl = L.plist.w >= 2u ? make_uint4(L.plist.x, L.plist.y, R.plist.x, num_primitives)
                             : make_uint4(L.plist.x, R.plist.x, R.plist.y, num_primitives);
    // The whole 128-byte entry in eight 16-byte stores (the padding too, so that no 32-byte sector of the line is
    // left partly written).
    uint4* e = reinterpret_cast<uint4*>(&dp.rec[dp_key(dp, first)]);
    e[0] = make_uint4(__float_as_uint(cost[0]), __float_as_uint(cost[1]), __float_as_uint(cost[2]),
                      __float_as_uint(cost[3]));
    e[1] = make_uint4(__float_as_uint(cost[4]), __float_as_uint(cost[5]), __float_as_uint(cost[6]), num_primitives);
    e[2] = make_uint4(sub[0], sub[1], sub[2], sub[3]);
    e[3] = make_uint4(sub[4], sub[5], sub[6], sub[0] == SUB_INVALID ? 0u : 1u + sub[0]);
    e[4] = make_uint4(meta[0] | meta[1] << 8 | meta[2] << 16 | meta[3] << 24, meta[4] | meta[5] << 8 | meta[6] << 16,
                      sd[0] | sd[1] << 8 | sd[2] << 16 | sd[3] << 24, sd[4] | sd[5] << 8 | sd[6] << 16);
    e[5] = make_uint4(l.first_index | (L.leaf ? KID_LEAF : 0u), r.first_index | (R.leaf ? KID_LEAF : 0u), 1u + sd[0],
                      0u);
    e[6] = pl;
    e[7] = make_uint4(0u, 0u, 0u, 0u);
    return 0u;
}

}  // namespace obvhs
