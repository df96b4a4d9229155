// bottomup.hpp -- bottom-up tree passes in one launch.
//
// A pass visits every internal node after both of its children, computing
// its payload (bounds, count, cost ...) from theirs.  Workgroup w owns leaf
// positions [w * 512, (w + 1) * 512) and the internal nodes with the same
// indices (for a Karras-ordered tree those below its own top nodes).  One lane
// per leaf climbs while the parent lies in the tile: arrivals are counted and
// payloads passed in LDS, and the completed nodes are written once, in index
// order.  Everything else (parents outside the tile, tile nodes whose other
// child is completed elsewhere) goes on through global memory, in the same
// launch: the payload is stored past the L2 caches, the arrival counted, and
// the lane that arrives second loads its sibling's payload past the caches and
// climbs on.  Children, parents and arrival counts are loaded two nodes ahead;
// a sibling seen to have arrived is loaded one ahead, and then nothing is
// published.  Nobody waits for anybody, and a payload is stored before its
// arrival is counted, so no order of the workgroups matters.
//
// Bound by latency: about 18 levels above the tiles of a 1 M-triangle LBVH,
// each a store, an atomic and a load through memory where the sibling was not
// seen (2.5 us), overlapped with the tiles still running.  Against three phases
// in three launches, arrivals and payloads through global memory from the
// leaves on: LBVH bounds of 1 M triangles 173 -> 85 us (92 without the loads
// ahead), final bounds and collapse marks of a 200 K ATRBVH 96 -> 42 and 105 ->
// 38 us.
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "obvh/obvh.h"

namespace obvh {

constexpr uint32_t kUpTile = 512;
constexpr uint32_t kUpNone = 0xFFFFFFFFu;

// 40 KB with the 32-byte payload of bounds: exactly four workgroups per CU (one
// word more and the LBVH build of 1 M triangles takes 229 us, 217 with four).
template <class Pay>
struct UpTile {
    Pay leaf[kUpTile];        // of the leaves
    Pay node[kUpTile];        // of the internal nodes completed here
    uint2 kids[kUpTile];
    uint32_t parent[kUpTile];
    uint32_t arrive[kUpTile];
};

// A node's children, parent and arrivals (none past the internal nodes).
struct UpTopo {
    uint2 kids;
    uint32_t parent, seen;
};
template <class Op>
__device__ __forceinline__ UpTopo up_topo(uint32_t p, uint32_t I, uint32_t* visit, const Op& op) {
    UpTopo T{make_uint2(0u, 0u), kUpNone, 0u};
    if (p < I) {
        T.kids = op.kids(p);
        T.parent = op.parent(p);
        T.seen = ld_agent(&visit[p]);
    }
    return T;
}

// Op provides
//   uint2 kids(uint32_t p), uint32_t parent(uint32_t node)
//   Pay leaf(uint32_t node)                    a leaf's payload; writes its outputs
//   Pay merge(p, l, r, const Pay&, const Pay&) an internal node's, from its children's; other outputs written here
//   void store(uint32_t node, const Pay&)      an internal node's payload to its outputs
//   void publish(node, const Pay&), Pay fetch(node)
//                                              the same outputs with agent-scope stores and loads
// visit: one zeroed counter per internal node.
template <class Pay, class Op>
__device__ __forceinline__ void bottom_up(uint32_t nf, uint32_t* visit, UpTile<Pay>& L, Op& op) {
    const uint32_t I = nf - 1, total = 2 * nf - 1, t = threadIdx.x;
    const uint32_t lo = blockIdx.x * kUpTile, pos = lo + t;
    uint32_t cur = I + pos, p = kUpNone;
    Pay pay{};
    bool climbing = pos < nf;
    if (climbing) {
        p = op.parent(cur);
        pay = op.leaf(cur);
        L.leaf[t] = pay;
    }
    if (pos < I) {
        L.kids[t] = op.kids(pos);
        L.parent[t] = op.parent(pos);
    }
    L.arrive[t] = 0;
    __syncthreads();

    const uint32_t nin = lo < I ? min(kUpTile, I - lo) : 0u;
    for (uint32_t step = 0; climbing && p - lo < nin && step < nf; ++step) {
        const uint32_t s = p - lo;
        const uint2 k = L.kids[s];
        const uint32_t a = __hip_atomic_fetch_add(&L.arrive[s], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
        const bool left = k.x == cur;
        const uint32_t sib = left ? k.y : k.x;
        const bool leaf = sib >= I;
        const uint32_t at = sib - (leaf ? I + lo : lo);  // the sibling arrived here, so it is in the tile
        if (a != 1 || at >= kUpTile) {
            climbing = false;  // first arrival: the sibling continues (or a malformed tree)
            break;
        }
        const Pay o = leaf ? L.leaf[at] : L.node[at];
        pay = left ? op.merge(p, cur, sib, pay, o) : op.merge(p, sib, cur, o, pay);
        L.node[s] = pay;
        cur = p;
        p = L.parent[s];
    }
    __syncthreads();
    if (t < nin && L.arrive[t] == 2u) op.store(lo + t, L.node[t]);

    // Two arrivals of this lane may be left: its own climb's next parent lies
    // outside the tile, and the tile node lo + t was reached by one child.
#pragma unroll 1
    for (int round = 0; round < 2; ++round) {
        bool go = round == 0 && climbing && p < I;
        if (round == 1 && t < nin && L.arrive[t] == 1u) {
            p = lo + t;
            const uint2 k = L.kids[t];
#pragma unroll
            for (int j = 0; j < 2; ++j) {  // the child that arrived
                const uint32_t c = j == 0 ? k.x : k.y;
                const uint32_t at = c >= I ? c - I - lo : c - lo;
                if (at < kUpTile && c < total && (c >= I || L.arrive[at] == 2u)) {
                    cur = c;
                    pay = c >= I ? L.leaf[at] : L.node[at];
                    go = true;
                }
            }
        }
        if (!go) continue;
        // children, parent and arrivals of the next two nodes
        UpTopo A = up_topo(p, I, visit, op), B = up_topo(A.parent, I, visit, op);
        Pay o{};  // the sibling's payload, if its arrival was seen
        bool have = false;
        auto look = [&](const UpTopo& T, uint32_t child) {
            const uint32_t sib = T.kids.x == child ? T.kids.y : T.kids.x;
            have = T.seen == 1 && sib < total;
            asm volatile("" ::: "memory");
            if (have) o = op.fetch(sib);
        };
        look(A, cur);
        for (uint32_t step = 0; step < nf; ++step) {
            const bool left = A.kids.x == cur;
            const uint32_t sib = left ? A.kids.y : A.kids.x;
            const UpTopo C = up_topo(B.parent, I, visit, op);
            if (have) {
                op.store(cur, pay);
                __hip_atomic_fetch_add(&visit[p], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                op.publish(cur, pay);
                drain();
                const uint32_t a = __hip_atomic_fetch_add(&visit[p], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (a != 1 || sib >= total) break;  // first arrival: the sibling continues
                asm volatile("" ::: "memory");
                o = op.fetch(sib);
            }
            pay = left ? op.merge(p, cur, sib, pay, o) : op.merge(p, sib, cur, o, pay);
            look(B, p);
            cur = p;
            p = A.parent;
            A = B;
            B = C;
            if (p >= I) {  // the root
                op.store(cur, pay);
                break;
            }
        }
    }
}

inline dim3 up_grid(uint32_t nf) { return dim3((nf + kUpTile - 1) / kUpTile); }

// Bounds, primitive count and SAH cost (ct = 1.0, ci = 1.2) of a tree's nodes,
// from the leaves' bounds (lbvh.cu:399-457, atrbvh.cu:124-179).
struct BoundsPay {
    f3 mn, mx;
    uint32_t count;
    float cost;
};
struct BoundsUp {
    kr_bvh_node* nodes;
    const uint32_t* parents;
    uint32_t* counts;
    float* costs;

    static __device__ __forceinline__ float area(f3 mn, f3 mx) {
        const f3 d = sub3(mx, mn);
        return 2.0f * (d.x * d.y + d.x * d.z + d.y * d.z);
    }
    __device__ __forceinline__ uint2 kids(uint32_t p) const {
        return make_uint2(nodes[p].u.children.left, nodes[p].u.children.right);
    }
    __device__ __forceinline__ uint32_t parent(uint32_t n) const { return parents[n]; }
    __device__ __forceinline__ BoundsPay leaf(uint32_t n) const {
        const kr_aabb3 b = nodes[n].bounds;
        BoundsPay r{f3{b.min.x, b.min.y, b.min.z}, f3{b.max.x, b.max.y, b.max.z}, 1u, 0.0f};
        r.cost = 1.0f * area(r.mn, r.mx);
        counts[n] = 1u;
        costs[n] = r.cost;
        return r;
    }
    __device__ __forceinline__ BoundsPay merge(uint32_t, uint32_t, uint32_t, const BoundsPay& a,
                                               const BoundsPay& b) const {
        BoundsPay r;  // kr_aabb_expand by both corners of the right child
        r.mn = vm::vmin3(vm::vmin3(a.mn, b.mn), b.mx);
        r.mx = vm::vmax3(vm::vmax3(a.mx, b.mn), b.mx);
        r.count = a.count + b.count;
        r.cost = (float)1.2 * area(r.mn, r.mx) + b.cost + a.cost;
        return r;
    }
    __device__ __forceinline__ void store(uint32_t n, const BoundsPay& r) const {
        nodes[n].bounds.min = kr_vec3{r.mn.x, r.mn.y, r.mn.z};
        nodes[n].bounds.max = kr_vec3{r.mx.x, r.mx.y, r.mx.z};
        counts[n] = r.count;
        costs[n] = r.cost;
    }
    __device__ __forceinline__ void publish(uint32_t n, const BoundsPay& r) const {
        float* b = &nodes[n].bounds.min.x;
        st_agent(b, r.mn.x);
        st_agent(b + 1, r.mn.y);
        st_agent(b + 2, r.mn.z);
        st_agent(b + 3, r.mx.x);
        st_agent(b + 4, r.mx.y);
        st_agent(b + 5, r.mx.z);
        st_agent(&counts[n], r.count);
        st_agent(&costs[n], r.cost);
    }
    __device__ __forceinline__ BoundsPay fetch(uint32_t n) const {
        const float* b = &nodes[n].bounds.min.x;
        return BoundsPay{f3{ld_agent(b), ld_agent(b + 1), ld_agent(b + 2)},
                         f3{ld_agent(b + 3), ld_agent(b + 4), ld_agent(b + 5)}, ld_agent(&counts[n]),
                         ld_agent(&costs[n])};
    }
};

}  // namespace obvh
