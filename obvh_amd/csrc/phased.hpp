// phased.hpp -- state of the phased bottom-up protocol (the ATRBVH optimiser).
//
// A pass visits every internal node after both of its children.  Phase k runs
// workgroups that own leaf positions [w*chunk_k, (w+1)*chunk_k); the last one,
// the top pass, is one group for everything.  Phase 0 starts one lane per leaf;
// later phases start from the nodes the previous phase deferred.  Each deferred
// node is listed with a key, a leaf position of its subtree known to the lane
// that deferred it, and is taken by the workgroup whose chunk holds the key;
// that workgroup runs it when the node's whole leaf span lies in its chunk and
// defers it again otherwise.  Other workgroups decide from the key alone and
// never read the node: a pass that restructures the tree (ATRBVH treelets) may
// rewire a deferred node's children as soon as its owner has completed it and
// an ancestor.  A lane that completes a child adds (tag << 32) | 1 to the
// parent's 64-bit arrival word (tag = (phase << 24) | (workgroup + 1), one tag
// for the whole top pass); the first arrival stops, the second continues if the
// first came from an earlier kernel (visible after the kernel boundary) or from
// its own group, and otherwise defers the parent to the next phase.  Inside a
// kernel a group orders its data by workgroup-scope acq_rel, the top pass by
// waiting for its stores and invalidating its L1; no device-scope release is
// issued.  The top pass owns every leaf and never defers.
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "obvh/obvh.h"

namespace obvh {

constexpr int kPhases = 2;  // phases that defer, at most

struct PhaseWs {
    uint64_t* visit;   // per internal node: arrivals (low word) + sum of tags (high word)
    uint32_t* nlist;   // per phase: number of deferred nodes
    uint2* list;       // per phase: deferred nodes and their keys (I + 1 entries each)
};

inline void phase_carve(PhaseWs* ws, Carver& c, uint32_t nf) {
    ws->visit = c.take<uint64_t>((size_t)nf + 1);
    ws->nlist = c.take<uint32_t>(4);
    ws->list = c.take<uint2>((size_t)kPhases * ((size_t)nf + 1));
}

// Zero the arrival words and the deferred-list counters (grid-stride).
__device__ __forceinline__ void phase_clear(const PhaseWs& ws, uint32_t nf) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0)
        for (int k = 0; k < 4; ++k) ws.nlist[k] = 0;
    for (uint32_t i = t; i < nf; i += gridDim.x * blockDim.x) ws.visit[i] = 0;
}

}  // namespace obvh
