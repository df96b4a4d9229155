// lbvh.hpp -- internal interface of the LBVH builder (lbvh.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "obvh/obvh.h"
#include "radix.hpp"

namespace obvh {

struct LbvhWs {
    int32_t* cbox;       // centroid box as order-preserving keys (min xyz, max xyz)
    uint32_t* visit;     // per internal node: children done (bottom-up pass)
    uint32_t* keys;      // Morton codes by face, then sorted
    uint32_t* vals;      // face ids in sorted order
    uint32_t* keys_tmp;  // the sort's other buffers
    uint32_t* vals_tmp;
    RadixWs radix;
};

// The tree's search probes up to 2^30 positions past its node in an int (more
// faces gave a wrong tree), and the sort holds as many pairs.
constexpr uint32_t kLbvhMaxFaces = 1u << 30;
static_assert(kLbvhMaxFaces <= kRadixMax, "the sort's limit");

size_t lbvh_carve(LbvhWs* ws, void* base, size_t cap, uint32_t nf);
kr_error lbvh_launch(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, kr_bvh_node* nodes, uint32_t* parents,
                     uint32_t* counts, float* costs, uint32_t* mortons, void* workspace, size_t ws_bytes,
                     hipStream_t stream, uint32_t polls = kRadixPolls);

}  // namespace obvh
