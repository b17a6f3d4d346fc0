// What the batched builder's translation units share: the passes' state and the one-workgroup tail of a mesh.
#pragma once

#include "common.hpp"
#include "cwdp.hpp"
#include "device_util.hpp"
#include "internal.hpp"
#include "tail.hpp"

namespace obvhs {

// Clusters of a mesh that one workgroup takes over (k_b_tail), and the sizes of the workgroups that do (half as many
// threads).
constexpr int B_TAIL_MAX = 1024;
constexpr int B_TAIL_CLASSES = 3;
constexpr uint32_t B_TAIL_SIZES[B_TAIL_CLASSES] = {128, 512, B_TAIL_MAX};
// Meshes of a class from which it gets a launch of its own beside the larger classes'.  Launches follow each other, so
// few small meshes cost more apart than among the larger ones (4,096 icospheres: build 8.32 ms with a launch for every
// class, 8.26 with two).
constexpr uint32_t B_TAIL_OWN = 4096;

struct SegState {
    uint32_t start;   // first cluster of the mesh in the current cluster array
    uint32_t count;   // clusters of the mesh
    uint32_t insert;  // next free child slot + 1 (mesh-local), ploc/mod.rs:283-284
    uint32_t mbase;   // global exclusive merge count at the segment's first cluster (current pass)
};

// The cluster count is double-buffered by pass parity q: pass p reads total[p & 1] and its scan writes the next
// pass's count into total[(p + 1) & 1], so no launch is needed between passes to move it.
struct BatchMisc {
    uint32_t err;
    uint32_t total[2];   // clusters in the current array (by pass parity)
    uint32_t large;      // 1 if a mesh has more than B_TAIL_MAX clusters after the last pass, else 0
    uint32_t totals[2];  // emits, merges of the pass
    uint32_t passes;     // of the mesh that took most
};

// A launch of the tail over all meshes: the workgroups of those not of (above, upto] triangles and distance r leave.
struct BatchTail {
    hipStream_t stream;
    const Node32* cur;
    const SegState* seg;
    BatchMisc* misc;
    const MeshDesc* meshes;
    uint32_t m, above, upto, r, pass, threshold;
    Node32* nodes;
    DpView dp;
    uint32_t q;
};

// The tail by workgroups for up to 128 clusters (c = 0) or 512 (c = 1).  Defined in batch_small.hip: beside it in one
// translation unit the compiler schedules the tail for 1,024 clusters 4% slower.
void launch_tail_small(int c, const BatchTail& t);

namespace {

// The remaining passes of every mesh of (above, upto] triangles and search distance r, one workgroup per mesh
// (tail.hpp), once no mesh has more than MAX clusters; its last cluster goes to the mesh's node 0
// (ploc/mod.rs:495-499).  R: r if that distance has an unrolled search, else 0.
// A mesh's chain of passes bounds a workgroup, not any throughput, so what counts is how many fit a CU's LDS: 2 for
// 1,024 clusters, 4 for 512, 14 for 128 (a wave each).  Builds of 1M meshes of 12 triangles 47.9 -> 19.0 ms against all
// of them in workgroups for 1,024, 50,000 of 64 4.5 -> 2.0, 50,000 of 200 8.3 -> 6.0; 4,096 icospheres of up to 20,480
// triangles make passes 16 to 48 in 353 us, about 0.8 ms as launches over all meshes.
template <int R, int MAX>
__global__ void __launch_bounds__(MAX / 2, 4) k_b_tail(const Node32* __restrict__ cur,
                                                       const SegState* __restrict__ seg, BatchMisc* misc,
                                                       const MeshDesc* __restrict__ meshes, uint32_t above,
                                                       uint32_t upto, uint32_t r, uint32_t first_pass,
                                                       uint32_t depth_threshold, Node32* __restrict__ nodes, DpView dp,
                                                       uint32_t q) {
    const MeshDesc md = meshes[blockIdx.x];
    const SegState sg = seg[blockIdx.x];
    const uint32_t total = misc->total[q];  // 0: DERR_RESORT
    // The greatest pass count so far, or an older one.  A mesh that does not raise it leaves the word alone: one atomic
    // per mesh on it takes 11 ns each.
    const uint32_t deepest = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(&misc->passes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (md.prim_count <= above || md.prim_count > upto || md.radius != r || total == 0u) return;
    if (sg.count == 0u || sg.count > (uint32_t)MAX) {
        if (threadIdx.x == 0) atomicOr(&misc->err, DERR_CAPACITY);
        return;
    }
    dp.kbase = md.prim_base;
    PlocState st{sg.count, sg.insert, first_pass, 0u, 0ull};
    ploc_tail<R, MAX>(cur + sg.start, st, first_pass, r, r == 1u ? 1u : 0u, depth_threshold,
                      nodes + md.node_base, nullptr, dp, 1u, nullptr, 0u, 0u, &misc->err);
    if (threadIdx.x == 0) {
        if (st.count != 1u || st.insert != 1u) atomicOr(&misc->err, DERR_SELF_MERGE);
        if (st.depth > deepest) atomicMax(&misc->passes, st.depth);
    }
}

// Each allowed distance has its unrolled instance.
template <int MAX>
static void launch_tail(const BatchTail& t) {
#define OBVHS_TAIL(RR)                                                                                             \
    k_b_tail<RR, MAX><<<t.m, MAX / 2, 0, t.stream>>>(t.cur, t.seg, t.misc, t.meshes, t.above, t.upto, t.r, t.pass, \
                                                     t.threshold, t.nodes, t.dp, t.q)
    switch (t.r) {
        case 2: OBVHS_TAIL(2); break;
        case 6: OBVHS_TAIL(6); break;
        case 14: OBVHS_TAIL(14); break;
        case 24: OBVHS_TAIL(24); break;
        case 32: OBVHS_TAIL(32); break;
        default: OBVHS_TAIL(0); break;
    }
#undef OBVHS_TAIL
}

}  // namespace

}  // namespace obvhs
