// transform.hip -- AABB-BVH -> OBB-tree transform on gfx950.
//
// Method of the reference GPU transform (src/ads/common/cuda/transforms.cu
// :213-964), restructured for CDNA4:
//
//  climb_leaves  one lane per leaf, 512-leaf workgroups: the leaf's 7-slab
//                k-DOP (3 vertices, first vertex wins ties), then a bottom-up climb
//                in which the second child to arrive at a parent merges the
//                two k-DOPs.  Arrivals at parents inside the workgroup's range
//                are counted in LDS; the rest use a 64-bit global arrival
//                word tagged with the workgroup, and parents whose children
//                finished in different workgroups are deferred.  Then the
//                leaf OBBs and matrices (transforms.cu:803-834).
//  climb_upper   the deferred parents and everything above them, eight lanes a
//                path, k-DOPs handed over past the L2 caches.  The merge
//                takes the right child's extreme only if strictly better, so
//                ties go to the left child and the selected vertex ids do
//                not depend on scheduling.  k-DOPs carry vertex ids, not
//                positions (7 x {min, id, max, id} = 112 B per node); spans
//                carry an exact gap flag from leaf counts.
//  candidates    one lane per internal node: gather the 14 extremal vertices
//                and run the base-triangle + ditetrahedron search in
//                registers (transforms.cu:413-756), together with each refit
//                tile's ancestor chain.  Large trees search the nodes the tile
//                climb completed on a second stream beside climb_upper and
//                the others after it.
//  cand_redo     the search in reference mode for nodes with non-finite or
//                huge extremal points.
//  refit         exact projection range of every subtree vertex on each
//                node's candidate axes (transforms.cu:836-900): per-lane walks
//                below each wave's common ancestor, DPP wave reductions above
//                it (both reading the tile's own nodes from an LDS copy), a
//                tile-wide pass over the tile's distinct vertices for the
//                tile's ancestor chain, LDS keys per workgroup, global
//                atomics.
//  finalize      one lane per internal node: OBB vs AABB by half area, extent
//                floor, inverse(T * R * S) (transforms.cu:905-964).
//
// Tie rule, degenerate nodes and floating point follow the reference with
// the decisions documented in the oracle (oracle/transform.c).
#include <float.h>

#include <mutex>

#include "common.hpp"
#include "transform.hpp"

namespace obvh {

constexpr uint32_t kInvalid = 0xFFFFFFFFu;

struct Mat4 {
    float v[16];
};

__device__ __forceinline__ f3 ldv(const kr_vec3* V, uint32_t i) {
    kr_vec3 a = V[i];
    return f3{a.x, a.y, a.z};
}

// kr_minverse4, vecmath.h:946-1075.
__device__ __forceinline__ void minverse4(const float* m, float* out) {
    float r[16];
    r[0] = m[5] * m[10] * m[15] - m[5] * m[11] * m[14] - m[9] * m[6] * m[15] +
           m[9] * m[7] * m[14] + m[13] * m[6] * m[11] - m[13] * m[7] * m[10];
    r[4] = -m[4] * m[10] * m[15] + m[4] * m[11] * m[14] + m[8] * m[6] * m[15] -
           m[8] * m[7] * m[14] - m[12] * m[6] * m[11] + m[12] * m[7] * m[10];
    r[8] = m[4] * m[9] * m[15] - m[4] * m[11] * m[13] - m[8] * m[5] * m[15] +
           m[8] * m[7] * m[13] + m[12] * m[5] * m[11] - m[12] * m[7] * m[9];
    r[12] = -m[4] * m[9] * m[14] + m[4] * m[10] * m[13] + m[8] * m[5] * m[14] -
            m[8] * m[6] * m[13] - m[12] * m[5] * m[10] + m[12] * m[6] * m[9];
    r[1] = -m[1] * m[10] * m[15] + m[1] * m[11] * m[14] + m[9] * m[2] * m[15] -
           m[9] * m[3] * m[14] - m[13] * m[2] * m[11] + m[13] * m[3] * m[10];
    r[5] = m[0] * m[10] * m[15] - m[0] * m[11] * m[14] - m[8] * m[2] * m[15] +
           m[8] * m[3] * m[14] + m[12] * m[2] * m[11] - m[12] * m[3] * m[10];
    r[9] = -m[0] * m[9] * m[15] + m[0] * m[11] * m[13] + m[8] * m[1] * m[15] -
           m[8] * m[3] * m[13] - m[12] * m[1] * m[11] + m[12] * m[3] * m[9];
    r[13] = m[0] * m[9] * m[14] - m[0] * m[10] * m[13] - m[8] * m[1] * m[14] +
            m[8] * m[2] * m[13] + m[12] * m[1] * m[10] - m[12] * m[2] * m[9];
    r[2] = m[1] * m[6] * m[15] - m[1] * m[7] * m[14] - m[5] * m[2] * m[15] +
           m[5] * m[3] * m[14] + m[13] * m[2] * m[7] - m[13] * m[3] * m[6];
    r[6] = -m[0] * m[6] * m[15] + m[0] * m[7] * m[14] + m[4] * m[2] * m[15] -
           m[4] * m[3] * m[14] - m[12] * m[2] * m[7] + m[12] * m[3] * m[6];
    r[10] = m[0] * m[5] * m[15] - m[0] * m[7] * m[13] - m[4] * m[1] * m[15] +
            m[4] * m[3] * m[13] + m[12] * m[1] * m[7] - m[12] * m[3] * m[5];
    r[14] = -m[0] * m[5] * m[14] + m[0] * m[6] * m[13] + m[4] * m[1] * m[14] -
            m[4] * m[2] * m[13] - m[12] * m[1] * m[6] + m[12] * m[2] * m[5];
    r[3] = -m[1] * m[6] * m[11] + m[1] * m[7] * m[10] + m[5] * m[2] * m[11] -
           m[5] * m[3] * m[10] - m[9] * m[2] * m[7] + m[9] * m[3] * m[6];
    r[7] = m[0] * m[6] * m[11] - m[0] * m[7] * m[10] - m[4] * m[2] * m[11] +
           m[4] * m[3] * m[10] + m[8] * m[2] * m[7] - m[8] * m[3] * m[6];
    r[11] = -m[0] * m[5] * m[11] + m[0] * m[7] * m[9] + m[4] * m[1] * m[11] -
            m[4] * m[3] * m[9] - m[8] * m[1] * m[7] + m[8] * m[3] * m[5];
    r[15] = m[0] * m[5] * m[10] - m[0] * m[6] * m[9] - m[4] * m[1] * m[10] +
            m[4] * m[2] * m[9] + m[8] * m[1] * m[6] - m[8] * m[2] * m[5];
    float det = m[0] * r[0] + m[1] * r[4] + m[2] * r[8] + m[3] * r[12];
    if (det == 0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) out[i] = (i % 5 == 0) ? 1.0f : 0.0f;
        return;
    }
    det = 1.0f / det;
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i] = r[i] * det;
}

// kr_mmul4, vecmath.h:1214-1234.
__device__ __forceinline__ void mmul4(const float* l, const float* r, float* o) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            o[4 * c + i] = l[i] * r[4 * c] + l[4 + i] * r[4 * c + 1] + l[8 + i] * r[4 * c + 2] +
                           l[12 + i] * r[4 * c + 3];
}

// inverse(T(mid) * (R(v0,v1,v2) * S(2 ext))), transforms.cu:832-834,939-942.
__device__ __forceinline__ void obb_matrix(f3 v0, f3 v1, f3 v2, f3 mid, f3 ext, float* out) {
    float R[16] = {v0.x, v0.y, v0.z, 0, v1.x, v1.y, v1.z, 0, v2.x, v2.y, v2.z, 0, 0, 0, 0, 1};
    float S[16] = {ext.x * 2.0f, 0, 0, 0, 0, ext.y * 2.0f, 0, 0, 0, 0, ext.z * 2.0f, 0, 0, 0, 0, 1};
    float T[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, mid.x, mid.y, mid.z, 1};
    float RS[16], TRS[16];
    mmul4(R, S, RS);
    mmul4(T, RS, TRS);
    minverse4(TRS, out);
}

// One box (15 floats, kr_obb3 order) and one matrix (16 floats) into
// staging rows.
__device__ __forceinline__ void obb_row(float* d, f3 mid, f3 v0, f3 v1, f3 v2, f3 ext) {
    d[0] = mid.x; d[1] = mid.y; d[2] = mid.z;
    d[3] = v0.x; d[4] = v0.y; d[5] = v0.z;
    d[6] = v1.x; d[7] = v1.y; d[8] = v1.z;
    d[9] = v2.x; d[10] = v2.y; d[11] = v2.z;
    d[12] = ext.x; d[13] = ext.y; d[14] = ext.z;
}

// ------------------------------------------------------ batch map --
//
// Numbering of a batch of trees joined into one combined tree (see the batch
// section below).

struct BatchMap {
    const uint32_t* prim_off;  // K + 1 leaf offsets L_t
    uint32_t K;
    uint32_t Nsum;             // sum of N_t
};

// Tree of input node g: the last t with 2 L_t - t <= g.
__device__ __forceinline__ uint32_t batch_tree_of_node(const BatchMap& m, uint32_t g) {
    uint32_t lo = 0, hi = m.K;  // nb(lo) <= g < nb(hi)
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (2u * m.prim_off[mid] - mid <= g) lo = mid; else hi = mid;
    }
    return lo;
}
__device__ __forceinline__ uint32_t batch_tree_of_leaf(const BatchMap& m, uint32_t f) {
    uint32_t lo = 0, hi = m.K;  // L(lo) <= f < L(hi)
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (m.prim_off[mid] <= f) lo = mid; else hi = mid;
    }
    return lo;
}
// Combined index of local node j of tree t (N leaves, first leaf Lt); j must be < 2N - 1.
__device__ __forceinline__ uint32_t batch_map(const BatchMap& m, uint32_t t, uint32_t Lt, uint32_t N, uint32_t j) {
    if (j + 1 < N) return Lt + j + (t + 1 < m.K ? 1u : 0u);
    return (m.Nsum - 1) + Lt + (j - (N - 1));
}
// Output index of combined node c (a box the caller receives), or kInvalid
// for an unused slot.  K == 0: no batch, the identity.
__device__ __forceinline__ uint32_t batch_out_index(const BatchMap& m, uint32_t c) {
    if (m.K == 0) return c;
    const uint32_t Ic = m.Nsum - 1;
    if (c >= Ic) {  // leaf position c - Ic
        const uint32_t pos = c - Ic;
        const uint32_t t = batch_tree_of_leaf(m, pos);
        const uint32_t Lt = m.prim_off[t], N = m.prim_off[t + 1] - Lt;
        return 2 * Lt - t + (N - 1) + (pos - Lt);
    }
    const uint32_t t = batch_tree_of_leaf(m, c);
    const uint32_t Lt = m.prim_off[t];
    if (t + 1 < m.K) {
        if (c == Lt) return kInvalid;  // unused slot
        return 2 * Lt - t + (c - Lt - 1);
    }
    return 2 * Lt - t + (c - Lt);
}

// Output staging for R consecutive nodes (R = the workgroup size): boxes at
// row stride 15 floats, matrices at row stride 17 (odd strides: no LDS bank
// conflicts), written back to HBM as contiguous dwords.
constexpr int kStage = 256;
template <int R>
struct StageT {
    float ob[R * 15];
    float mt[R * 17];
    uint32_t orow[R];  // output node of each row (batches)
};
using Stage = StageT<kStage>;

template <int R>
__device__ __forceinline__ void stage_nan(StageT<R>& st, uint32_t r) {
    const float nan = __builtin_nanf("");
#pragma unroll
    for (int q = 0; q < 15; ++q) st.ob[r * 15 + q] = nan;
#pragma unroll
    for (int q = 0; q < 16; ++q) st.mt[r * 17 + q] = nan;
}

// Dwords g[0 .. n) = at(j), written by a workgroup of R threads as 16-byte
// stores from the first 16-byte boundary of g on, the dwords before it and
// after the last full vector one by one.
template <int R, class At>
__device__ __forceinline__ void flush_dwords(float* g, uint32_t n, At at) {
    const uint32_t h = min((uint32_t)(((16u - ((uint32_t)(uintptr_t)g & 15u)) & 15u) >> 2), n);
    const uint32_t body = (n - h) >> 2;
    for (uint32_t j = threadIdx.x; j < h; j += R) g[j] = at(j);
    float4* gv = reinterpret_cast<float4*>(g + h);
    for (uint32_t v = threadIdx.x; v < body; v += R) {
        const uint32_t j = h + 4 * v;
        gv[v] = make_float4(at(j), at(j + 1), at(j + 2), at(j + 3));
    }
    for (uint32_t j = h + 4 * body + threadIdx.x; j < n; j += R) g[j] = at(j);
}

// Rows first .. first + cnt - 1 (combined indices) to their output nodes: the
// same node indices, or for a batch each tree's own layout (runs of
// consecutive rows stay consecutive; top nodes are dropped).
template <int R>
__device__ __forceinline__ void stage_flush(StageT<R>& st, kr_obb3* obbs, kr_mat4* mats, size_t first, uint32_t cnt,
                                            const BatchMap& m) {
    if (m.K == 0) {
        flush_dwords<R>(reinterpret_cast<float*>(obbs) + first * 15, cnt * 15, [&](uint32_t j) { return st.ob[j]; });
        flush_dwords<R>(reinterpret_cast<float*>(mats) + first * 16, cnt * 16,
                        [&](uint32_t j) { return st.mt[(j >> 4) * 17 + (j & 15)]; });
        return;
    }
    // Rows of one tree (nearly always) are consecutive there too.  An index
    // map's offset never decreases and a hole starts its tree, so the two ends
    // tell.
    const uint32_t o0 = batch_out_index(m, (uint32_t)first), o1 = batch_out_index(m, (uint32_t)first + cnt - 1);
    if (o0 != kInvalid && o1 != kInvalid && o1 - o0 == cnt - 1) {
        flush_dwords<R>(reinterpret_cast<float*>(obbs) + (size_t)o0 * 15, cnt * 15, [&](uint32_t j) { return st.ob[j]; });
        flush_dwords<R>(reinterpret_cast<float*>(mats) + (size_t)o0 * 16, cnt * 16,
                        [&](uint32_t j) { return st.mt[(j >> 4) * 17 + (j & 15)]; });
        return;
    }
    if (threadIdx.x < cnt) st.orow[threadIdx.x] = batch_out_index(m, (uint32_t)first + threadIdx.x);
    __syncthreads();
    float* go = reinterpret_cast<float*>(obbs);
    for (uint32_t j = threadIdx.x; j < cnt * 15; j += R) {
        const uint32_t r = j / 15, o = st.orow[r];
        if (o != kInvalid) go[(size_t)o * 15 + (j - r * 15)] = st.ob[j];
    }
    float* gm = reinterpret_cast<float*>(mats);
    for (uint32_t j = threadIdx.x; j < cnt * 16; j += R) {
        const uint32_t o = st.orow[j >> 4];
        if (o != kInvalid) gm[(size_t)o * 16 + (j & 15)] = st.mt[(j >> 4) * 17 + (j & 15)];
    }
}

// ------------------------------------------------------------ k-DOP --

// The tree's topology: the children of an internal node, the face of a leaf,
// read from the caller's nodes (36 bytes each) or from a batch's combined
// ones (8 bytes each: no kernel reads a node's bounds).
struct TreeNodes {
    const uint32_t* w;  // of node 0
    uint32_t stride;    // words per node

    __device__ __forceinline__ uint2 kids(uint32_t i) const {
        const uint32_t* p = w + (size_t)i * stride;
        return make_uint2(p[0], p[1]);
    }
    __device__ __forceinline__ uint32_t face(uint32_t i) const { return w[(size_t)i * stride]; }
};
static TreeNodes tree_nodes(const kr_bvh_node* nodes) {
    static_assert(sizeof(kr_bvh_node) == 36 && offsetof(kr_bvh_node, u) == 24, "children follow the bounds");
    return TreeNodes{reinterpret_cast<const uint32_t*>(nodes) + 6, 9};
}

struct Kdop {
    float mn[7], mx[7];
    uint32_t imn[7], imx[7];
};

__device__ __forceinline__ void kdop_store(float4* kd, uint32_t node, const Kdop& k) {
#pragma unroll
    for (int s = 0; s < 7; ++s)
        kd[(size_t)node * 7 + s] = make_float4(k.mn[s], __uint_as_float(k.imn[s]), k.mx[s], __uint_as_float(k.imx[s]));
}
__device__ __forceinline__ void kdop_load(const float4* kd, uint32_t node, Kdop& k) {
#pragma unroll
    for (int s = 0; s < 7; ++s) {
        float4 a = kd[(size_t)node * 7 + s];
        k.mn[s] = a.x; k.imn[s] = __float_as_uint(a.y);
        k.mx[s] = a.z; k.imx[s] = __float_as_uint(a.w);
    }
}

// Leaf OBB from the triangle frame, transforms.cu:803-834.
__device__ __forceinline__ void leaf_obb(f3 v0, f3 v1, f3 v2, float* ob, float* mt) {
    f3 e0 = sub3(v1, v0);
    f3 e1 = sub3(v2, v0);
    f3 a2 = vm::cross(e0, e1);
    f3 a0 = vm::normalize(e0);
    f3 a1 = vm::normalize(vm::cross(a0, a2));
    float R[16] = {a0.x, a0.y, a0.z, 0, a1.x, a1.y, a1.z, 0, a2.x, a2.y, a2.z, 0, 0, 0, 0, 1};
    float Ri[16];
    minverse4(R, Ri);
    auto xf = [&](f3 r) {  // kr_vtransform3
        return f3{Ri[0] * r.x + Ri[4] * r.y + Ri[8] * r.z + Ri[12],
                  Ri[1] * r.x + Ri[5] * r.y + Ri[9] * r.z + Ri[13],
                  Ri[2] * r.x + Ri[6] * r.y + Ri[10] * r.z + Ri[14]};
    };
    f3 l0 = xf(v0), l1 = xf(v1), l2 = xf(v2);
    f3 mx = vm::vmax3(l0, vm::vmax3(l1, l2));
    f3 mn = vm::vmin3(l0, vm::vmin3(l1, l2));
    f3 mid = vm::mul1(add3(mx, mn), 0.5f);
    f3 ext = vm::vmax3(vm::mul1(sub3(mx, mn), 0.5f), f3{0.001f, 0.001f, 0.001f});
    f3 m = vm::mul1(a0, mid.x);
    m = add3(m, vm::mul1(a1, mid.y));
    m = add3(m, vm::mul1(a2, mid.z));
    obb_row(ob, m, a0, a1, a2, ext);
    float M[16];
    obb_matrix(a0, a1, a2, m, ext, M);
#pragma unroll
    for (int q = 0; q < 16; ++q) mt[q] = M[q];
}

// Arrival word of an unused internal slot of a batch: complete, tagged so
// that the per-node kernels skip it (arrival tags never sum to this).
constexpr uint32_t kHoleTag = 0xFFFFFFFFu;
__device__ __forceinline__ bool hole(uint64_t v) { return (uint32_t)(v >> 32) == kHoleTag; }

__global__ void batch_holes(TreeWs ws, BatchMap m) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k + 1 < m.K; k += gridDim.x * blockDim.x) {
        const uint32_t idx = m.prim_off[k];
        ws.visit[idx] = ((uint64_t)kHoleTag << 32) | 2ull;
        ws.span[idx] = make_uint2(1u, 0u);  // empty: holds no refit tile
    }
}

__global__ void tree_clear(uint64_t* visit, uint32_t n, TreeWs ws) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) {
        *ws.error = 0;
        for (int k = 0; k < kNodeLists; ++k) ws.nlist[k] = 0;
    }
    for (uint32_t i = t; i < n; i += gridDim.x * blockDim.x) visit[i] = 0;
}

// Arrival word of an internal node: low 32 bits count the children that
// finished, high 32 bits sum their tags.  tag = (phase << 24) | (owner + 1)
// identifies the kernel (0 climb_leaves, 1 climb_upper) and the workgroup that
// completed the child.
__device__ __forceinline__ bool complete(uint64_t v) { return (uint32_t)v == 2u; }
__device__ __forceinline__ uint32_t make_tag(uint32_t phase, uint32_t owner) { return (phase << 24) | (owner + 1u); }

__device__ __forceinline__ void merge_left_first(const Kdop& L, const Kdop& R, Kdop& m) {
    m = L;
#pragma unroll
    for (int s = 0; s < 7; ++s) {
        if (R.mn[s] < m.mn[s]) { m.mn[s] = R.mn[s]; m.imn[s] = R.imn[s]; }
        if (R.mx[s] > m.mx[s]) { m.mx[s] = R.mx[s]; m.imx[s] = R.imx[s]; }
    }
}

// Leaf k-DOP of one triangle: 7 slabs, first vertex wins ties.
__device__ __forceinline__ void leaf_kdop(f3 v0, f3 v1, f3 v2, const uint32_t vid[3], Kdop& k) {
    const f3 vs[3] = {v0, v1, v2};
    float pr[7];
    slab7(vs[0], pr);
#pragma unroll
    for (int s = 0; s < 7; ++s) { k.mn[s] = k.mx[s] = pr[s]; k.imn[s] = k.imx[s] = vid[0]; }
#pragma unroll
    for (int j = 1; j < 3; ++j) {
        slab7(vs[j], pr);
#pragma unroll
        for (int s = 0; s < 7; ++s) {
            if (pr[s] < k.mn[s]) { k.mn[s] = pr[s]; k.imn[s] = vid[j]; }
            if (pr[s] > k.mx[s]) { k.mx[s] = pr[s]; k.imx[s] = vid[j]; }
        }
    }
}

// Leaf span of a subtree: first and last leaf position below it.  Bit 31 of
// .y is set when the subtree does not hold every position from first to
// last (its leaf count is below the width; the count of such a node is kept
// beside the span); leaf positions are < 2^31.
constexpr uint32_t kGap = 0x80000000u;
__device__ __forceinline__ uint32_t span_hi(uint2 s) { return s.y & ~kGap; }
__device__ __forceinline__ bool span_gap(uint2 s) { return (s.y & kGap) != 0; }
__device__ __forceinline__ uint2 leaf_span(uint32_t pos) { return make_uint2(pos, pos); }
// Leaves below a node: the span's width, or the kept count if it has a gap.
__device__ __forceinline__ uint32_t span_count(uint2 s, uint32_t kept) {
    return span_gap(s) ? kept : span_hi(s) - s.x + 1u;
}
__device__ __forceinline__ uint2 span_join(uint2 a, uint32_t ca, uint2 b, uint32_t cb, uint32_t& c) {
    const uint32_t lo = min(a.x, b.x), hi = max(span_hi(a), span_hi(b));
    c = ca + cb;
    return make_uint2(lo, hi | (hi - lo + 1u != c ? kGap : 0u));
}
// Span and leaf count of node c from global memory (the count word is read
// unconditionally, beside the span, and used only for a gapped span).
__device__ __forceinline__ uint2 span_load(const TreeWs& ws, uint32_t c, uint32_t I, uint32_t& cnt) {
    if (c >= I) {
        cnt = 1;
        return leaf_span(c - I);
    }
    const uint2 s = ws.span[c];
    const uint32_t kept = ws.count[c];
    cnt = span_count(s, kept);
    return s;
}
__device__ __forceinline__ void span_store(TreeWs& ws, uint32_t c, uint2 s, uint32_t cnt) {
    ws.span[c] = s;
    if (span_gap(s)) ws.count[c] = cnt;
}

// Node lists (ws.list, counts in ws.nlist): the nodes the tile climb defers, the
// nodes completed after it, and those the candidate search hands to reference
// mode.
constexpr int kDeferList = 0;
constexpr int kUpperList = 1;
constexpr int kRedoList = 2;
static_assert(kRedoList < kNodeLists, "one list per slot");

// A deferred node is marked in bit 63 of its arrival word: its count already
// reads 2 (both children arrived), but its k-DOP is made by climb_upper, so
// the candidate launch that runs beside it must skip it.
constexpr uint64_t kDeferred = 1ull << 63;
__device__ __forceinline__ void defer(TreeWs& ws, uint32_t node, uint32_t I) {
    atomicOr(reinterpret_cast<unsigned long long*>(&ws.visit[node]), (unsigned long long)kDeferred);
    const uint32_t slot = atomicAdd(&ws.nlist[kDeferList], 1u);
    if (slot < I) ws.list[(size_t)kDeferList * (I + 1) + slot] = node;
}

// k-DOP of leaf node `leaf` from the mesh.
__device__ __forceinline__ bool leaf_kdop_global(const kr_bvh_node* nodes, const kr_vec3* V, const kr_uvec4* F,
                                                 uint32_t leaf, uint32_t N, Kdop& k) {
    const uint32_t f = nodes[leaf].u.primitivesOffset;
    if (f >= N) return false;
    const kr_uvec4 face = F[f];
    const uint32_t vid[3] = {face.x, face.y, face.z};
    leaf_kdop(ldv(V, face.x), ldv(V, face.y), ldv(V, face.z), vid, k);
    return true;
}

// The tiles' part of the bottom-up k-DOP pass.  Workgroup w owns leaf positions
// [w*kTile, (w+1)*kTile) and the internal nodes with the same indices (for a
// Karras-ordered tree these are the internal nodes whose leaves lie in the
// range).  The workgroup first loads the tile's topology into LDS (children
// and parents of its internal nodes, vertex ids of its leaves) and checks that every child of its internal nodes points back to it.
// Then one lane per leaf climbs: at a parent in the tile the arrival is
// counted in LDS, the first child stops and the second merges, reading the
// sibling's k-DOP from LDS (internal node of the tile, or a leaf's k-DOP
// left in the parent's slot), recomputing it (a leaf that left none) or
// loading it (node completed outside the tile's index range).  At the
// first level two leaf siblings in one wave merge without an arrival count:
// the left one takes the right one's k-DOP by lane shuffles.  Parents outside
// the tile use the global arrival word with the workgroup's tag; such a parent is deferred to climb_upper when its
// children finished in different workgroups.  Finally tile nodes reached by
// one child only are folded into the global arrival words, and the k-DOPs,
// spans and arrival words of tile nodes completed here are written back
// contiguously.  The merge keeps the left child's extreme on ties.  Last,
// the tile's leaf boxes (transforms.cu:803-834) from the triangles each lane
// loaded, staged in the same LDS and written back contiguously.
//
// Bound by latency at two workgroups of 78 KB per CU: of a workgroup's 46 us on
// a 1M-leaf tree the loads take 7, the climb 16 (about 13 levels), the k-DOPs'
// write-back 8, the leaf boxes 13.  1M leaves 130 us (2.6 TB/s written), 2M 255.
// A half-reached node's count is looked at after the write-back and its leaf
// child's k-DOP comes from LDS (before, from the vertices again): transforms of
// 2M leaves 853 -> 839 us, 3.8M 1625 -> 1611.  Eight lanes per node above the
// first level, as in climb_upper, took 186 us for 1M.
constexpr uint32_t kTile = 512;  // leaves per workgroup

struct ClimbTile {
    float4 kd[kTile][7];        // k-DOP of internal node lo + s, once completed here
    uint2 span[kTile];
    uint32_t cnt[kTile];        // leaves below internal node lo + s
    uint32_t lid[kTile][3];     // vertex ids of leaf position lo + s
    uint32_t arrive[kTile];     // arrivals at internal node lo + s from this workgroup
    uint2 kids[kTile];          // children of internal node lo + s
    uint32_t par_int[kTile];    // parent of internal node lo + s
    uint32_t par_leaf[kTile];   // parent of the leaf at position lo + s
};
union ClimbLds {
    ClimbTile L;
    StageT<kTile> st;           // after the climb: the leaf boxes
};

__device__ __forceinline__ void tile_leaf_kdop(const ClimbTile& L, const kr_vec3* V, uint32_t s, Kdop& k) {
    const uint32_t vid[3] = {L.lid[s][0], L.lid[s][1], L.lid[s][2]};
    leaf_kdop(ldv(V, vid[0]), ldv(V, vid[1]), ldv(V, vid[2]), vid, k);
}

__global__ __launch_bounds__(kTile) void climb_leaves(TreeNodes nodes,
                                                      const uint32_t* __restrict__ parents,
                                                      const kr_vec3* __restrict__ V,
                                                      const kr_uvec4* __restrict__ F, TreeWs ws, uint32_t N,
                                                      kr_obb3* obbs, kr_mat4* mats, BatchMap bm) {
    __shared__ ClimbLds U;
    ClimbTile& L = U.L;
    const uint32_t I = N - 1, total = 2 * N - 1;
    const uint32_t t = threadIdx.x;
    const uint32_t lo = blockIdx.x * kTile;
    const uint32_t tag = make_tag(0, blockIdx.x);
    const uint32_t pos = lo + t;

    // tile topology and the lane's leaf
    Kdop k = {};
    bool climbing = false;
    f3 v0 = f3{0, 0, 0}, v1 = v0, v2 = v0;  // the lane's triangle, for its leaf box
    // the tile's internal nodes' loads go out before the chain leaf -> face ->
    // vertices waits
    uint32_t l = 0, r = 0, par = kInvalid, f = kInvalid, leaf_parent = kInvalid;
    uint64_t slot = 0;
    if (pos < I) {
        const uint2 lr = nodes.kids(pos);
        l = lr.x;
        r = lr.y;
        par = parents[pos];
        slot = ws.visit[pos];
    }
    if (pos < N) {
        leaf_parent = parents[I + pos];
        f = nodes.face(I + pos);
    }
    kr_uvec4 face = {};
    if (f < N) face = F[f];
    if (pos < I) {
        L.kids[t] = make_uint2(l, r);
        L.par_int[t] = par;
    }
    L.par_leaf[t] = leaf_parent;
    if (pos < N) {
        if (f < N) {
            const uint32_t vid[3] = {face.x, face.y, face.z};
            L.lid[t][0] = vid[0];
            L.lid[t][1] = vid[1];
            L.lid[t][2] = vid[2];
            v0 = ldv(V, vid[0]);
            v1 = ldv(V, vid[1]);
            v2 = ldv(V, vid[2]);
            leaf_kdop(v0, v1, v2, vid, k);
            climbing = true;
        } else {
            L.lid[t][0] = kInvalid;  // never climbs, never read as a sibling
            atomicOr(ws.error, 4u);  // faces has one entry per leaf
        }
    }
    L.arrive[t] = 0;
    __syncthreads();

    // every child points back (an unused slot of a batch has none)
    if (pos < I && !hole(slot)) {
        const auto points_back = [&](uint32_t c) {
            if (c >= total) return false;
            const uint32_t s = (c < I ? c : c - I) - lo;
            return (s < kTile ? (c < I ? L.par_int[s] : L.par_leaf[s]) : parents[c]) == pos;
        };
        if (!points_back(l) || !points_back(r)) atomicOr(ws.error, 2u);
    }

    // First level, all lanes together: two leaf siblings in one wave are
    // merged by the left one (the right one's k-DOP comes by a lane shuffle)
    // without an arrival count.  Any other leaf with a parent in the tile
    // leaves its k-DOP in the parent's LDS slot before it arrives (unless it is
    // the right one of two leaves of the tile), so that a sibling arriving
    // second reads it from LDS instead of recomputing it.
    uint32_t cur = I + pos;
    uint2 span = leaf_span(pos);
    uint32_t count = 1;
    uint32_t p = leaf_parent;
    bool climb = climbing;  // the lane climbs on past the first level
    {
        const uint64_t climbers = __ballot(climbing);
        uint32_t src = (uint32_t)lane_id(), ps = p - lo, sib = kInvalid;
        bool pair_left = false, pair_right = false, stash = false;
        if (climbing && p < I && ps < kTile) {
            const uint2 kc = L.kids[ps];
            const bool am_left = kc.x == cur;
            if (am_left || kc.y == cur) {  // otherwise the climb below reports it
                sib = am_left ? kc.y : kc.x;
                const uint32_t sl = sib - I - (pos - (uint32_t)lane_id());  // the sibling leaf's lane
                if (sib >= I && sib < total && sl < (uint32_t)kWave && ((climbers >> sl) & 1ull)) {
                    pair_left = am_left;
                    pair_right = !am_left;
                    src = sl;
                } else {
                    stash = sib < I || am_left || sib - I - lo >= kTile;
                }
            }
        }
        Kdop o;
#pragma unroll
        for (int q = 0; q < 7; ++q) {  // every lane of the wave takes part
            o.mn[q] = __shfl(k.mn[q], (int)src, kWave);
            o.mx[q] = __shfl(k.mx[q], (int)src, kWave);
            o.imn[q] = (uint32_t)__shfl((int)k.imn[q], (int)src, kWave);
            o.imx[q] = (uint32_t)__shfl((int)k.imx[q], (int)src, kWave);
        }
        if (pair_right) climb = false;  // the left sibling merges
        if (pair_left) {
            Kdop m;
            merge_left_first(k, o, m);
            k = m;
            span = span_join(span, count, leaf_span(sib - I), 1u, count);
#pragma unroll
            for (int q = 0; q < 7; ++q)
                L.kd[ps][q] = make_float4(k.mn[q], __uint_as_float(k.imn[q]), k.mx[q], __uint_as_float(k.imx[q]));
            L.span[ps] = span;
            L.cnt[ps] = count;
            L.arrive[ps] = 2u;  // both children: no other lane arrives here
            cur = p;
            p = L.par_int[ps];
        }
        if (stash) {
#pragma unroll
            for (int q = 0; q < 7; ++q)
                L.kd[ps][q] = make_float4(k.mn[q], __uint_as_float(k.imn[q]), k.mx[q], __uint_as_float(k.imx[q]));
        }
    }

    if (climb) {
        for (uint32_t step = 0; p != kInvalid; ++step) {
            if (p >= I || step >= N) { atomicOr(ws.error, 1u); break; }
            const uint32_t s = p - lo;
            uint32_t sib, pp;
            bool am_left;
            if (s < kTile) {  // parent in the tile: LDS arrival
                const uint2 kc = L.kids[s];  // topology: read before the arrival
                pp = L.par_int[s];
                const uint32_t cnt =
                    __hip_atomic_fetch_add(&L.arrive[s], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (cnt == 0) break;  // first arrival: the sibling continues
                if (cnt != 1) { atomicOr(ws.error, 2u); break; }
                am_left = kc.x == cur;
                if (!am_left && kc.y != cur) { atomicOr(ws.error, 2u); break; }
                sib = am_left ? kc.y : kc.x;
            } else {  // parent outside the tile: publish, then global arrival
                kdop_store(ws.kdop, cur, k);
                span_store(ws, cur, span, count);
                const uint2 lr = nodes.kids(p);
                const uint32_t l = lr.x, rr = lr.y;
                pp = parents[p];
                const uint64_t old = __hip_atomic_fetch_add(&ws.visit[p], ((uint64_t)tag << 32) | 1ull,
                                                            __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
                const uint32_t cnt = (uint32_t)old;
                if (cnt == 0) break;
                if (cnt != 1) { atomicOr(ws.error, 2u); break; }
                if ((uint32_t)(old >> 32) != tag) { defer(ws, p, I); break; }  // other workgroup
                am_left = l == cur;
                if (!am_left && rr != cur) { atomicOr(ws.error, 2u); break; }
                sib = am_left ? rr : l;
            }
            // the sibling finished in this workgroup
            Kdop o;
            uint2 so;
            uint32_t co;
            if (sib >= I) {
                const uint32_t ss = sib - I - lo;
                if (sib >= total || ss >= kTile) { atomicOr(ws.error, 2u); break; }
                // a leaf left its k-DOP in the parent's slot unless this lane
                // is its left leaf sibling (from another wave)
                const uint32_t from = s < kTile && (cur < I || !am_left) ? s : kInvalid;
                if (from != kInvalid) {
#pragma unroll
                    for (int q = 0; q < 7; ++q) {
                        const float4 a = L.kd[from][q];
                        o.mn[q] = a.x; o.imn[q] = __float_as_uint(a.y);
                        o.mx[q] = a.z; o.imx[q] = __float_as_uint(a.w);
                    }
                } else {
                    tile_leaf_kdop(L, V, ss, o);
                }
                so = leaf_span(sib - I);
                co = 1;
            } else if (sib - lo < kTile) {  // completed in this tile: k-DOP in LDS
                const uint32_t ss = sib - lo;
#pragma unroll
                for (int q = 0; q < 7; ++q) {
                    const float4 a = L.kd[ss][q];
                    o.mn[q] = a.x; o.imn[q] = __float_as_uint(a.y);
                    o.mx[q] = a.z; o.imx[q] = __float_as_uint(a.w);
                }
                so = L.span[ss];
                co = L.cnt[ss];
            } else {
                kdop_load(ws.kdop, sib, o);
                so = span_load(ws, sib, I, co);
            }
            Kdop m;
            if (am_left) merge_left_first(k, o, m); else merge_left_first(o, k, m);
            k = m;
            span = span_join(span, count, so, co, count);
            if (s < kTile) {
#pragma unroll
                for (int q = 0; q < 7; ++q)
                    L.kd[s][q] = make_float4(k.mn[q], __uint_as_float(k.imn[q]), k.mx[q], __uint_as_float(k.imx[q]));
                L.span[s] = span;
                L.cnt[s] = count;
            } else {
                kdop_store(ws.kdop, p, k);
                span_store(ws, p, span, count);
            }
            cur = p;
            p = pp;
        }
    }
    __syncthreads();

    // Tile nodes reached by one child: publish a tile-leaf child (its k-DOP
    // is in the node's slot), then the global arrival: the other child
    // finishes in another workgroup.  What the count held is looked at last.
    uint64_t old = 0;
    const bool half = pos < I && L.arrive[t] == 1u;
    if (half) {
        const uint2 kc = L.kids[t];
        const uint32_t c2[2] = {kc.x, kc.y};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t ss = c2[j] - I - lo;
            if (c2[j] >= I && c2[j] < total && ss < kTile && L.lid[ss][0] != kInvalid) {
                float4* d = ws.kdop + (size_t)c2[j] * 7;
#pragma unroll
                for (int q = 0; q < 7; ++q) d[q] = L.kd[t][q];
                ws.span[c2[j]] = leaf_span(c2[j] - I);
            }
        }
        old = __hip_atomic_fetch_add(&ws.visit[pos], ((uint64_t)tag << 32) | 1ull, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    // write back the tile nodes completed here
    const uint32_t nin = lo < I ? min(kTile, I - lo) : 0u;
    float4* kd = ws.kdop + (size_t)lo * 7;
    float4 row[7];
    bool done[7];
#pragma unroll
    for (int u = 0; u < 7; ++u) {  // all LDS reads, then the stores (row by row 1M took 430 us, now 426)
        const uint32_t j = t + u * kTile, ss = j / 7;
        row[u] = L.kd[ss][j - ss * 7];
        done[u] = j < nin * 7 && L.arrive[ss] == 2u;
    }
#pragma unroll
    for (int u = 0; u < 7; ++u)
        if (done[u]) kd[t + u * kTile] = row[u];
    if (t < nin && L.arrive[t] == 2u) {
        span_store(ws, pos, L.span[t], L.cnt[t]);
        ws.visit[pos] = ((uint64_t)tag << 33) | 2ull;
    }
    // the leaf boxes (a bad face id gives a NaN row; the climb reported it)
    __syncthreads();
    if (pos < N) {
        if (climbing) leaf_obb(v0, v1, v2, &U.st.ob[t * 15], &U.st.mt[t * 17]);
        else stage_nan(U.st, t);
    }
    __syncthreads();
    stage_flush(U.st, obbs, mats, (size_t)I + lo, min(kTile, N - lo), bm);
    if (half) {
        if ((uint32_t)old == 1u) defer(ws, pos, I);
        else if ((uint32_t)old != 0u) atomicOr(ws.error, 2u);
    }
}

// The rest of the bottom-up k-DOP pass: the nodes the tile climb deferred (both
// children complete) and everything above them, in one launch.  Eight lanes
// take a deferred node and follow its path to the root: lanes 0..6 hold a slab
// each of the k-DOP, lane 7 the span and leaf count, so a level's loads and
// stores are one or two instructions over a few cache lines.  Children,
// parents and arrival words are loaded two levels ahead (arrival words past the
// L2 caches).  At a parent p
//   - whose other child was seen to have arrived (in the tile climb or here):
//     its data was loaded one level ahead; the path goes on at once;
//   - otherwise the node is stored with agent-scope accesses (past the L2
//     caches), then its arrival counted; the first path to arrive ends, the
//     second loads the sibling past the caches and goes on.
// Nobody waits, and a node is stored before its arrival is counted, so no order
// of the workgroups matters.  Completed nodes are collected in LDS (one
// counter for all of them would take an atomic of the chip per node) and
// appended to a list for the candidate search.
//
// Bound by latency: a level takes 1.5 us on an idle chip (5120 triangles: 15
// levels, 23 us) and 3 us beside the candidate search, which hides it (26 levels
// of a 1M icosphere 91 us, a 2M one 128, a 2M hairball's ATRBVH 215).  Timed
// against each other on 1M and 2M triangles: 77 and 117 us; without the loads
// ahead 114 and 334; with eight paths in a wave from the start 107, 226, and 31
// for 5120 triangles (a wave is as slow as its slowest path); 32768-leaf
// workgroups with hand-overs in LDS and one last workgroup, which it replaced,
// 106, 190 and 30.  Random topology (nearly every node is up here), whole transform:
// 100000 leaves 14.1 ms then, 8.6 now.  The waves run at raised priority: they
// are few, and issue little between their waits.
struct Topo {  // children, parent and arrival word of a node (zero / kInvalid past the internal nodes)
    uint32_t l, r, parent;
    uint64_t v;
};
__device__ __forceinline__ Topo topo_load(TreeNodes nodes, const uint32_t* __restrict__ parents,
                                          const TreeWs& ws, uint32_t p, uint32_t I) {
    Topo T = {0u, 0u, kInvalid, 0ull};
    if (p < I) {
        const uint2 lr = nodes.kids(p);
        T.l = lr.x;
        T.r = lr.y;
        T.parent = parents[p];
        T.v = ld_agent(&ws.visit[p]);
    }
    return T;
}

constexpr int kPathLanes = 8;
constexpr uint32_t kUpperThreads = kWave;  // one wave per workgroup: paths spread over the chip
constexpr uint32_t kUpperDone = 512;       // completed nodes a workgroup collects before it appends them

// Lane q of a path's share of a node: slab q (lanes 0..6), or the span and
// leaf count (lane 7).
template <bool kAgent>
__device__ __forceinline__ uint4 path_load(const TreeWs& ws, uint32_t node, uint32_t I, int q) {
    auto ld64 = [](const void* p) {
        const uint64_t* w = static_cast<const uint64_t*>(p);
        const uint64_t v = kAgent ? ld_agent(w) : *w;
        return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
    };
    if (q < 7) {
        const float4* k = &ws.kdop[(size_t)node * 7 + q];
        const uint2 a = ld64(k), b = ld64(reinterpret_cast<const uint2*>(k) + 1);
        return make_uint4(a.x, a.y, b.x, b.y);
    }
    if (node >= I) {
        const uint2 sp = leaf_span(node - I);
        return make_uint4(sp.x, sp.y, 1u, 0u);
    }
    const uint2 sp = ld64(&ws.span[node]);
    const uint32_t kept = kAgent ? ld_agent(&ws.count[node]) : ws.count[node];
    return make_uint4(sp.x, sp.y, span_count(sp, kept), 0u);
}
template <bool kAgent>
__device__ __forceinline__ void path_store(const TreeWs& ws, uint32_t node, int q, uint4 k) {
    auto st64 = [](void* p, uint32_t x, uint32_t y) {
        uint64_t* w = static_cast<uint64_t*>(p);
        const uint64_t v = (uint64_t)y << 32 | x;
        if (kAgent) st_agent(w, v);
        else *w = v;
    };
    if (q < 7) {
        float4* d = &ws.kdop[(size_t)node * 7 + q];
        st64(d, k.x, k.y);
        st64(reinterpret_cast<uint2*>(d) + 1, k.z, k.w);
        return;
    }
    st64(&ws.span[node], k.x, k.y);
    if (kAgent) st_agent(&ws.count[node], k.z);
    else ws.count[node] = k.z;
}
__device__ __forceinline__ uint4 path_merge(uint4 l, uint4 r, int q) {
    if (q < 7) {  // merge_left_first of one slab
        if (__uint_as_float(r.x) < __uint_as_float(l.x)) { l.x = r.x; l.y = r.y; }
        if (__uint_as_float(r.z) > __uint_as_float(l.z)) { l.z = r.z; l.w = r.w; }
        return l;
    }
    uint32_t c;
    const uint2 sp = span_join(make_uint2(l.x, l.y), l.z, make_uint2(r.x, r.y), r.z, c);
    return make_uint4(sp.x, sp.y, c, 0u);
}

__global__ __launch_bounds__(kUpperThreads) void climb_upper(TreeNodes nodes,
                                                             const uint32_t* __restrict__ parents, TreeWs ws,
                                                             uint32_t N) {
    __builtin_amdgcn_s_setprio(3);  // wave priority
    const uint32_t I = N - 1, total = 2 * N - 1;
    const int q = (int)(threadIdx.x % kPathLanes), lead = lane_id() - q;
    const uint32_t nin = min(ws.nlist[kDeferList], I);
    const uint32_t* in = ws.list + (size_t)kDeferList * (I + 1);
    const uint64_t mine = (uint64_t)make_tag(1, 0) << 32 | 1ull;
    __shared__ uint32_t done[kUpperDone], ndone;
    if (threadIdx.x == 0) ndone = 0;
    __syncthreads();
    auto append = [&](uint32_t slot, uint32_t node) {
        if (slot < I) ws.list[(size_t)kUpperList * (I + 1) + slot] = node;
    };
    auto completed = [&](uint32_t node) {
        if (q != 0) return;
        const uint32_t s = __hip_atomic_fetch_add(&ndone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (s < kUpperDone) done[s] = node;
        else append(atomicAdd(&ws.nlist[kUpperList], 1u), node);
    };
    // one path per wave as far as the waves go, then a second, ...
    for (uint32_t r = blockIdx.x + threadIdx.x / kPathLanes * gridDim.x; r < nin;
         r += gridDim.x * (kUpperThreads / kPathLanes)) {
        uint32_t cur = in[r];
        if (cur >= I) { atomicOr(ws.error, 1u); continue; }
        uint32_t p = parents[cur];
        Topo A = topo_load(nodes, parents, ws, p, I);
        const uint2 lr = nodes.kids(cur);
        const uint32_t l0 = lr.x, r0 = lr.y;
        if (l0 >= total || r0 >= total) { atomicOr(ws.error, 2u); continue; }
        uint4 k = path_merge(path_load<false>(ws, l0, I, q), path_load<false>(ws, r0, I, q), q);
        Topo B = topo_load(nodes, parents, ws, A.parent, I);
        completed(cur);
        uint4 o = make_uint4(0, 0, 0, 0);  // the sibling, if its arrival was seen
        bool have = false;
        auto fetch = [&](const Topo& T, uint32_t child) {
            const uint32_t sib = T.l == child ? T.r : T.l;
            have = (uint32_t)T.v == 1u && sib < total;
            asm volatile("" ::: "memory");
            if (have) o = path_load<true>(ws, sib, I, q);
        };
        fetch(A, cur);
        for (uint32_t step = 0;; ++step) {  // the same for the eight lanes
            const bool am_left = A.l == cur;
            const uint32_t sib = am_left ? A.r : A.l;
            if (p >= I || step >= N || sib >= total || (!am_left && A.r != cur)) {
                path_store<false>(ws, cur, q, k);
                if (p != kInvalid) atomicOr(ws.error, p >= I || step >= N ? 1u : 2u);
                break;
            }
            const Topo C = topo_load(nodes, parents, ws, B.parent, I);
            if (have) {
                path_store<false>(ws, cur, q, k);
                if (q == 0) ws.visit[p] = A.v + mine;
            } else {
                path_store<true>(ws, cur, q, k);
                drain();
                uint64_t old = 0;
                if (q == 0)
                    old = __hip_atomic_fetch_add(&ws.visit[p], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint32_t c = (uint32_t)__shfl((int)(uint32_t)old, lead);
                if (c == 0) break;  // first arrival: the sibling's path goes on
                if (c != 1) { atomicOr(ws.error, 2u); break; }
                asm volatile("" ::: "memory");
                o = path_load<true>(ws, sib, I, q);
            }
            k = am_left ? path_merge(k, o, q) : path_merge(o, k, q);
            fetch(B, p);
            completed(p);
            cur = p;
            p = A.parent;
            A = B;
            B = C;
        }
    }
    __syncthreads();
    const uint32_t nd = min(ndone, kUpperDone);
    uint32_t base = 0;
    if (threadIdx.x == 0 && nd) base = atomicAdd(&ws.nlist[kUpperList], nd);
    base = (uint32_t)__shfl((int)base, 0);
    for (uint32_t s = threadIdx.x; s < nd; s += kUpperThreads) append(base + s, done[s]);
}

// ------------------------------------------------------- candidates --

struct Best {
    float q;
    f3 b0, b1, b2;
    f3 dmin, dmax;
};

// (min, max) of 14 projections (transforms.cu:418-434).  v_min / v_max give the same value as the
// reference's compare-and-select rule (kmin / kmax) except for the sign of a
// zero result and for NaN inputs; a zero result, or a node whose points are
// not all finite and bounded (`sane`), takes the compare-and-select chain.
__device__ __forceinline__ void minmax14(const float (&p)[14], bool sane, float& mn, float& mx) {
    float a = fminf(p[0], p[1]), b = fmaxf(p[0], p[1]);
#pragma unroll
    for (int i = 2; i < 14; ++i) {
        a = fminf(a, p[i]);
        b = fmaxf(b, p[i]);
    }
    if (!sane || a == 0.0f || b == 0.0f) {
        a = p[0];
        b = p[0];
#pragma unroll
        for (int i = 1; i < 14; ++i) {
            a = kmin(a, p[i]);
            b = kmax(b, p[i]);
        }
    }
    mn = a;
    mx = b;
}

__device__ __forceinline__ void proj14(const f3* P, f3 d, bool sane, float& mn, float& mx) {
    float a = dot3(P[0], d), b = a;
#pragma unroll
    for (int i = 1; i < 14; ++i) {
        const float p = dot3(P[i], d);
        a = fminf(a, p);
        b = fmaxf(b, p);
    }
    if (!sane || a == 0.0f || b == 0.0f) {  // same projections, reference rule
        a = dot3(P[0], d);
        b = a;
#pragma unroll
        for (int i = 1; i < 14; ++i) {
            const float p = dot3(P[i], d);
            a = kmin(a, p);
            b = kmax(b, p);
        }
    }
    mn = a;
    mx = b;
}

// The candidate search over a point list P of NP points (NP a compile-time
// count).  Reference mode (kRef, NP = 14): the node's 14 extremal points in
// the reference's interleaved order, each projection range with the
// compare-and-select fallback above.  Distinct mode: the node's distinct
// extremal points, first occurrences in the interleaved order, padded to NP
// with copies of the first point.  Every search over the list is a
// first-index strict compare (a later copy of a point never wins) and every
// range a min / max (the same value for a multiset and its set), so both
// modes choose the same candidate with the same axes and lengths.  They can
// differ only in the sign of a zero range end, which no decision uses
// (lengths, qualities and their compares treat -0 as +0) and which the refit
// replaces: the refit's range is the key minimum / maximum over every
// subtree vertex, the extremal points included.  Distinct mode needs finite,
// bounded points (v_min / v_max); other nodes take reference mode.
template <int NP, bool kRef>
struct Pts {
    const f3* P;
    bool sane;  // reference mode: the points are finite and bounded

    __device__ __forceinline__ void proj(f3 d, float& mn, float& mx) const {
        if (kRef) {
            proj14(P, d, sane, mn, mx);
            return;
        }
        float a = dot3(P[0], d), b = a;
#pragma unroll
        for (int i = 1; i < NP; ++i) {
            const float p = dot3(P[i], d);
            a = fminf(a, p);
            b = fmaxf(b, p);
        }
        mn = a;
        mx = b;
    }
    __device__ __forceinline__ float2 projv(f3 d) const {
        float mn, mx;
        proj(d, mn, mx);
        return make_float2(mn, mx);
    }
};

__device__ __forceinline__ f3 pick(bool c, f3 a, f3 b) { return f3{c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z}; }
__device__ __forceinline__ float2 pick2(bool c, float2 a, float2 b) {
    return make_float2(c ? a.x : b.x, c ? a.y : b.y);
}

// One face of the ditetrahedron, transforms.cu:484-544: the normal's
// projection range, then for each edge e[k] (its range pe[k] computed by
// the caller: an edge is shared by up to three faces, its range is computed
// once with identical arithmetic) the third axis m = e x n; a candidate
// replaces the best one when its quality is strictly lower.
template <int NP, bool kRef>
__device__ __forceinline__ void face(const Pts<NP, kRef>& P, f3 n, float nmn, float nmx, f3 e0, f3 e1, f3 e2,
                                     float2 pe0, float2 pe1, float2 pe2, Best& b) {
    const float leny = nmx - nmn;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f3 e = k == 0 ? e0 : (k == 1 ? e1 : e2);
        const float2 pe = k == 0 ? pe0 : (k == 1 ? pe1 : pe2);
        const f3 m = vm::cross(e, n);
        float mmn, mmx;
        P.proj(m, mmn, mmx);
        const float lenx = pe.y - pe.x;
        const float lenz = mmx - mmn;
        const float q = quality(f3{lenx, leny, lenz});
        if (q < b.q) {
            b.q = q;
            b.dmax = f3{pe.y, nmx, mmx};
            b.dmin = f3{pe.x, nmn, mmn};
            b.b0 = e;
            b.b1 = n;
            b.b2 = m;
        }
    }
}

// Farthest slab pair (transforms.cu:437-456) over the interleaved list,
// first pair wins ties: its index s.
__device__ __forceinline__ int farthest_pair(const f3 (&P)[14]) {
    int at = 0;
    float d2b = vm::dist2(P[0], P[1]);
#pragma unroll
    for (int s = 1; s < 7; ++s) {
        const float d2 = vm::dist2(P[2 * s], P[2 * s + 1]);
        const bool c = d2 > d2b;
        d2b = c ? d2 : d2b;
        at = c ? s : at;
    }
    return at;
}

// Base triangle on the farthest pair (p0, p1), then the ditetrahedron
// (transforms.cu:546-674), over the list P.  The apex faces run as loops
// (two apexes, three faces each, in the reference's candidate order), so
// that the code per point count stays small.
template <int NP, bool kRef>
__device__ __forceinline__ void cand_search(const Pts<NP, kRef>& L, f3 p0, f3 p1, Best& b, int& degen) {
    const float eps = 0.000001f;
    const f3* P = L.P;
    degen = 0;
    if (vm::dist2(p0, p1) < eps) {
        degen = 1;
        return;
    }
    const f3 e0 = vm::normalize(sub3(p0, p1));
    float dm = vm::dist_inf_edge(P[0], p0, e0);
    f3 p2 = P[0];
#pragma unroll
    for (int i = 1; i < NP; ++i) {
        const float d = vm::dist_inf_edge(P[i], p0, e0);
        const bool c = d > dm;
        dm = c ? d : dm;
        p2 = pick(c, P[i], p2);
    }
    if (dm < eps) {
        degen = 1;
        return;
    }
    const f3 e1 = vm::normalize(sub3(p1, p2));
    const f3 e2 = vm::normalize(sub3(p2, p0));
    const f3 nn = vm::normalize(vm::cross(e1, e0));
    const float2 pe0 = L.projv(e0), pe1 = L.projv(e1), pe2 = L.projv(e2);
    // the normal's projections: its range, then the apexes (extreme points
    // along n, first index wins, transforms.cu:609-628)
    float pn[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) pn[i] = dot3(P[i], nn);
    float nmn, nmx;
    if (kRef) {
        minmax14(*reinterpret_cast<const float(*)[14]>(pn), L.sane, nmn, nmx);
    } else {
        nmn = pn[0];
        nmx = pn[0];
#pragma unroll
        for (int i = 1; i < NP; ++i) {
            nmn = fminf(nmn, pn[i]);
            nmx = fmaxf(nmx, pn[i]);
        }
    }
    // the apexes' validity first: a node without one is degenerate and
    // keeps b at the AABB (its range then holds the AABB for finalize)
    float lo = pn[0], hi = pn[0];
#pragma unroll
    for (int i = 1; i < NP; ++i) {
        lo = pn[i] < lo ? pn[i] : lo;
        hi = pn[i] > hi ? pn[i] : hi;
    }
    const float tri = dot3(p0, nn);
    const bool q0v = hi - eps > tri;
    const bool q1v = lo + eps < tri;
    if (!q0v && !q1v) {
        degen = 1;
        return;
    }
    face(L, nn, nmn, nmx, e0, e1, e2, pe0, pe1, pe2, b);
    lo = pn[0];
    hi = pn[0];
    f3 q1 = P[0], q0 = P[0];
#pragma unroll
    for (int i = 1; i < NP; ++i) {
        const bool cl = pn[i] < lo, ch = pn[i] > hi;
        lo = cl ? pn[i] : lo;
        q1 = pick(cl, P[i], q1);
        hi = ch ? pn[i] : hi;
        q0 = pick(ch, P[i], q0);
    }
    // the node's first valid apex (q0, candidates 3..11, or else q1), then q1
    // (12..20) if both are; on apex q the faces j = 0, 1, 2 have edges
    // (e_j, f_{j+1}, f_j) with f_i = q - p_i normalised and normal
    // cross(f_{j+1}, e_j) normalised (transforms.cu:641-700).  A node of four
    // distinct points has one apex: its wave runs the loop once, whichever
    // side each lane's apex is on.
#pragma unroll 1
    for (int a = 0; a < 2; ++a) {
        if (a == 1 && !(q0v && q1v)) continue;
        const f3 q = pick(a == 0 && q0v, q0, q1);
        const f3 f0 = vm::normalize(sub3(q, p0));
        const f3 f1 = vm::normalize(sub3(q, p1));
        const f3 f2 = vm::normalize(sub3(q, p2));
        const float2 pf0 = L.projv(f0), pf1 = L.projv(f1), pf2 = L.projv(f2);
#pragma unroll 1
        for (int j = 0; j < 3; ++j) {
            const f3 ej = pick(j == 0, e0, pick(j == 1, e1, e2));
            const float2 pej = pick2(j == 0, pe0, pick2(j == 1, pe1, pe2));
            const f3 fa = pick(j == 0, f1, pick(j == 1, f2, f0));
            const float2 pfa = pick2(j == 0, pf1, pick2(j == 1, pf2, pf0));
            const f3 fb = pick(j == 0, f0, pick(j == 1, f1, f2));
            const float2 pfb = pick2(j == 0, pf0, pick2(j == 1, pf1, pf2));
            const f3 nf = vm::normalize(vm::cross(fa, ej));
            float fmn, fmx;
            L.proj(nf, fmn, fmx);
            face(L, nf, fmn, fmx, ej, fa, fb, pej, pfa, pfb, b);
        }
    }
}

// Per internal node the candidate search (transforms.cu:677-756).  The
// search's loops run over the node's distinct extremal points: on average
// 5.4 of the 14 on a mesh LBVH (two triangles sharing an edge have four).  A
// wave runs the loops for the largest distinct count among its lanes, so the
// workgroup first sorts its 512 nodes by that count (LDS counting sort), lane
// t takes the t-th node in that order, and the wave runs the search compiled
// for 4, 6, 8 or 14 points.
constexpr int kCandBlock = 256;

struct CandTile {
    uint32_t cid[kCandBlock][15];   // distinct extremal vertex ids in list order (odd stride)
    uint32_t pair[kCandBlock][2];   // vertex ids of the farthest slab pair
    uint8_t cnt[kCandBlock];        // number of distinct ids; 0 = nothing to search; 15 = reference mode
    uint16_t order[kCandBlock];
    uint32_t node[kCandBlock];
    uint32_t hist[16];
};

__device__ __forceinline__ void kdop_ids(const Kdop& k, uint32_t (&id)[14]) {
#pragma unroll
    for (int s = 0; s < 7; ++s) {
        id[2 * s] = k.imn[s];
        id[2 * s + 1] = k.imx[s];
    }
}

// Finite and below 2^61 in magnitude: no projection can be NaN or overflow.
__device__ __forceinline__ bool sane_points(const f3* P, int n) {
    uint32_t ex = 0;
    for (int i = 0; i < n; ++i) {
        ex = max(ex, __float_as_uint(P[i].x) & 0x7F800000u);
        ex = max(ex, __float_as_uint(P[i].y) & 0x7F800000u);
        ex = max(ex, __float_as_uint(P[i].z) & 0x7F800000u);
    }
    return ex <= ((127u + 60u) << 23);
}

// aq: half area of the node's AABB (the k-DOP's first three slabs), kept
// so that finalize reads the k-DOP only where the AABB wins.  The range
// starts as the result's projection range: for a degenerate node (which
// the refit skips and finalize boxes by its AABB) the search leaves b at
// the AABB, so finalize reads that from the range, not from the k-DOP.
__device__ __forceinline__ void store_cand(TreeWs& ws, uint32_t node, const Best& b, int degen, float aq) {
    Cand c;
    c.b[0] = b.b0.x; c.b[1] = b.b0.y; c.b[2] = b.b0.z;
    c.b[3] = b.b1.x; c.b[4] = b.b1.y; c.b[5] = b.b1.z;
    c.b[6] = b.b2.x; c.b[7] = b.b2.y; c.b[8] = b.b2.z;
    c.degen = degen;
    c.aq = aq;
    c.pad = 0;
    ws.cand[node] = c;
    int32_t* rk = &ws.range[(size_t)node * 6];
    rk[0] = f2ord(b.dmin.x); rk[1] = f2ord(b.dmin.y); rk[2] = f2ord(b.dmin.z);
    rk[3] = f2ord(b.dmax.x); rk[4] = f2ord(b.dmax.y); rk[5] = f2ord(b.dmax.z);
}

__device__ __forceinline__ Best aabb_best(const Kdop& k) {
    const f3 alen = f3{k.mx[0] - k.mn[0], k.mx[1] - k.mn[1], k.mx[2] - k.mn[2]};
    return Best{quality(alen), f3{1, 0, 0}, f3{0, 1, 0}, f3{0, 0, 1}, f3{k.mn[0], k.mn[1], k.mn[2]},
                f3{k.mx[0], k.mx[1], k.mx[2]}};
}

// Reference mode over the node's 14 points in list order, for the rare
// nodes with non-finite or huge extremal points (list kRedoList), run by
// cand_redo.

__device__ __forceinline__ void cand_ref(const kr_vec3* __restrict__ V, TreeWs& ws, uint32_t node) {
    Kdop k;
    kdop_load(ws.kdop, node, k);
    uint32_t id[14];
    kdop_ids(k, id);
    f3 Q[14];
#pragma unroll
    for (int i = 0; i < 14; ++i) Q[i] = ldv(V, id[i]);
    const int at = farthest_pair(Q);
    f3 p0 = Q[0], p1 = Q[1];
#pragma unroll
    for (int s = 1; s < 7; ++s)
        if (at == s) { p0 = Q[2 * s]; p1 = Q[2 * s + 1]; }
    Best b = aabb_best(k);
    const float aq = b.q;
    int degen = 0;
    const Pts<14, true> L{Q, sane_points(Q, 14)};
    cand_search(L, p0, p1, b, degen);
    store_cand(ws, node, b, degen, aq);
}

// Distinct-mode search of one node with the list padded to NP points.
template <int NP>
__device__ __forceinline__ void cand_distinct(const kr_vec3* __restrict__ V, TreeWs& ws, const CandTile& T,
                                              uint32_t s, uint32_t node, int cnt) {
    f3 P[NP];
    P[0] = ldv(V, T.cid[s][0]);
#pragma unroll
    for (int i = 1; i < NP; ++i) P[i] = i < cnt ? ldv(V, T.cid[s][i]) : P[0];  // copies of the first point pad the list
    const float4* kd = &ws.kdop[(size_t)node * 7];
    const float4 s0 = kd[0], s1 = kd[1], s2 = kd[2];
    const f3 alen = f3{s0.z - s0.x, s1.z - s1.x, s2.z - s2.x};
    const float aq = quality(alen);
    Best b = {aq, f3{1, 0, 0}, f3{0, 1, 0}, f3{0, 0, 1}, f3{s0.x, s1.x, s2.x}, f3{s0.z, s1.z, s2.z}};
    const f3 p0 = ldv(V, T.pair[s][0]), p1 = ldv(V, T.pair[s][1]);
    int degen = 0;
    const Pts<NP, false> L{P, true};
    cand_search(L, p0, p1, b, degen);
    store_cand(ws, node, b, degen, aq);
}

__device__ __forceinline__ bool holds(uint2 sp, uint32_t first, uint32_t last) {
    return sp.x <= first && sp.y >= last && !(sp.y & kGap);
}

// The ancestors of refit tile `tile` that hold all of its leaves: from the
// tile's first leaf up to the lowest node whose span covers the tile without
// a gap, then that node and its ancestors (at most kTChain; the next one is
// kept for a walk).
__device__ void tile_chain(const uint32_t* __restrict__ parents, TreeWs& ws, uint32_t N, uint32_t tile) {
    const uint32_t I = N - 1, lo = tile * kRTile, thi = min(lo + kRTile, N) - 1;
    uint32_t p = parents[I + lo];
    for (uint32_t step = 0; p < I && step < N && !holds(ws.span[p], lo, thi); ++step) p = parents[p];
    uint32_t n = 0;
    while (p < I && n < kTChain) {
        ws.tchain[(size_t)tile * kTChain + n] = p;
        ++n;
        p = parents[p];
    }
    ws.tmeta[tile] = make_uint2(n, p < I ? p : kInvalid);
}

// Arrival word of a node completed by the tile climb: both tags are phase 0
// (tag = owner + 1 < 2^23), so their sum stays below 2^24; climb_upper adds
// a tag of at least 2^24, a deferred node carries bit 63 (kDeferred) and a
// hole's word is all ones.
__device__ __forceinline__ bool tile_complete(uint64_t v) { return complete(v) && (uint32_t)(v >> 32) < (1u << 24); }

// One workgroup's nodes (node[t] for lane t, kInvalid for none).
__device__ __forceinline__ void cand_block(const kr_vec3* __restrict__ V, TreeWs& ws, uint32_t I, CandTile& T,
                                           uint32_t node, bool bad) {
    const uint32_t t = threadIdx.x;
    if (t < 16) T.hist[t] = 0;
    T.node[t] = node;
    __syncthreads();
    // 1. the lane's own node: distinct ids and the farthest slab pair
    {
        uint32_t cnt = 0;
        if (node < I) {
            if (hole(ws.visit[node]) || bad) {
                Cand c = {};
                c.degen = 1;
                ws.cand[node] = c;
            } else {
                Kdop k;
                kdop_load(ws.kdop, node, k);
                uint32_t id[14];
                kdop_ids(k, id);
                f3 P[14];
#pragma unroll
                for (int i = 0; i < 14; ++i) P[i] = ldv(V, id[i]);
                if (!sane_points(P, 14)) {  // reference mode, after this kernel
                    const uint32_t slot = atomicAdd(&ws.nlist[kRedoList], 1u);
                    if (slot < I) ws.list[(size_t)kRedoList * (I + 1) + slot] = node;
                } else {
                    const int at = farthest_pair(P);
                    uint32_t a = id[0], b = id[1];
#pragma unroll
                    for (int s = 1; s < 7; ++s)
                        if (at == s) { a = id[2 * s]; b = id[2 * s + 1]; }
                    T.pair[t][0] = a;
                    T.pair[t][1] = b;
#pragma unroll
                    for (int i = 0; i < 14; ++i) {
                        bool dup = false;
#pragma unroll
                        for (int j = 0; j < i; ++j) dup |= id[j] == id[i];
                        if (!dup) T.cid[t][cnt++] = id[i];
                    }
                }
            }
        }
        T.cnt[t] = (uint8_t)cnt;
        // counting sort by distinct count (rank within a count from an LDS
        // atomic: the order among equal counts does not matter)
        const uint32_t r = atomicAdd(&T.hist[cnt], 1u);
        __syncthreads();
        if (t == 0) {
            uint32_t acc = 0;
            for (int c = 0; c < 16; ++c) {
                const uint32_t h = T.hist[c];
                T.hist[c] = acc;
                acc += h;
            }
        }
        __syncthreads();
        T.order[T.hist[cnt] + r] = (uint16_t)t;
        __syncthreads();
    }
    // 2. the t-th node in count order, searched over the wave's point count
    const uint32_t s = T.order[t];
    const int cnt = T.cnt[s];
    const int n = wave_max_i32(cnt);  // every lane is active here
    if (cnt != 0) {
        const uint32_t nd = T.node[s];
        if (n <= 4) cand_distinct<4>(V, ws, T, s, nd, cnt);
        else if (n <= 6) cand_distinct<6>(V, ws, T, s, nd, cnt);
        else if (n <= 8) cand_distinct<8>(V, ws, T, s, nd, cnt);
        else cand_distinct<14>(V, ws, T, s, nd, cnt);
    }
    __syncthreads();  // T is reused by the workgroup's next round
}

// The candidate search.  Large trees take two launches.  kTileNodes: the nodes
// the tile climb completed (index order, one round per workgroup), beside
// climb_upper, which leaves most of the chip idle; holes get an AABB record.
// kUpperNodes: the nodes climb_upper completed (their list).  Small trees take
// one, kAllNodes, after climb_upper.  In the last two workgroups below
// `cblocks` find the refit tiles' ancestor chains.
enum CandNodes { kTileNodes, kUpperNodes, kAllNodes };
template <int kNodes>
__global__ __launch_bounds__(kCandBlock, 4) void candidates(const kr_vec3* __restrict__ V,
                                                            const uint32_t* __restrict__ parents, TreeWs ws,
                                                            uint32_t N, uint32_t cblocks) {
    __shared__ CandTile T;
    const uint32_t t = threadIdx.x, I = N - 1;
    if (kNodes != kTileNodes && blockIdx.x < cblocks) {
        const uint32_t tile = blockIdx.x * kCandBlock + t;
        if (tile < (N + kRTile - 1) / kRTile) {
            if (*ws.error != 0) ws.tmeta[tile] = make_uint2(0u, kInvalid);
            else tile_chain(parents, ws, N, tile);
        }
        return;
    }
    const bool bad = *ws.error != 0;
    if (kNodes != kUpperNodes) {
        const uint32_t node = (blockIdx.x - cblocks) * kCandBlock + t;
        bool mine = false;
        if (node < I) {
            const uint64_t vw = ws.visit[node];
            mine = hole(vw) || (kNodes == kAllNodes ? complete(vw) : tile_complete(vw));
        }
        cand_block(V, ws, I, T, mine ? node : kInvalid, bad);
        return;
    }
    const uint32_t nb = gridDim.x - cblocks, nup = min(ws.nlist[kUpperList], I);
    const uint32_t* up = ws.list + (size_t)kUpperList * (I + 1);
    for (uint32_t base = (blockIdx.x - cblocks) * kCandBlock; base < nup; base += nb * kCandBlock)  // uniform
        cand_block(V, ws, I, T, base + t < nup ? up[base + t] : kInvalid, bad);
}

// The candidate search in reference mode on the nodes the distinct-mode
// search handed back (a separate launch after candidates: its registers do
// not add to the distinct-mode search's).
constexpr uint32_t kRedoBlocks = 8;
__global__ __launch_bounds__(1024) void cand_redo(const kr_vec3* __restrict__ V, TreeWs ws, uint32_t I) {
    const uint32_t nredo = min(ws.nlist[kRedoList], I);
    const uint32_t* redo = ws.list + (size_t)kRedoList * (I + 1);
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < nredo; r += gridDim.x * blockDim.x)
        cand_ref(V, ws, redo[r]);
}

// ------------------------------------------------------------ refit --
//
// Exact projection range of every subtree vertex on each internal node's
// candidate axes (transforms.cu:836-900), as order-preserving int32 keys
// (-0 orders below +0), min/max over the subtree's vertices.  A workgroup
// takes a tile of 512 consecutive leaves and splits each leaf's ancestors
// in three tiers:
//   A  below the lowest ancestor holding all 64 leaves of the lane's wave:
//      each group of four lanes folds its triangles' keys into LDS (a slot
//      per internal node of the tile's index range, a small hash for other
//      nodes);
//   B  from that node up to the lowest ancestor holding the whole tile: the
//      wave walks together, reduces the 64 lanes' keys with DPP and one lane
//      folds them into LDS;
//   C  the tile's common ancestor and everything above it: the tile's
//      distinct vertices are collected once (LDS hash set on vertex ids) and
//      each wave takes some of those ancestors, looping over the distinct
//      vertices instead of 3 per triangle.
// "Holds all leaves of a range" is read from the span: its first and last
// leaf cover the range and the leaves below are contiguous.  LDS results are
// folded into global memory at the end.  Without the
// tile-wide pass (too many distinct vertices, or no tile-common node) tier B
// continues to the root.
// The walks of tiers A and B read the parent, span and axes of nodes in the
// tile's own index range [lo, lo + 512) from an LDS copy made at the start
// (a Karras tree numbers every node below the tile-common node inside that
// range; other nodes are read from global memory).  The ancestors for tier C
// (the tile-common node and up to kTChain - 1 of its ancestors) were listed
// per tile by the candidate kernel's leading workgroups, so no workgroup
// walks the ~10-30 dependent parent loads itself; ancestors beyond the list
// (very deep trees) are walked by every wave with its lanes' triangles.
//
// Bound by latency and LDS throughput at three workgroups of 52 KB per CU: of a
// workgroup's 67 us on a 1M-leaf tree the loads and the vertex set take 18,
// tier A 20, tier B 8, tier C 10, the write-back 7.  1M leaves 118 us, 129
// before the leaf's loads started ahead of the set-up, the vertices' positions
// came from their lanes' registers instead of a second gather, an axis read
// became three 16-byte words read a level ahead, and the keys of a node inside
// the tile replaced its range instead of being merged into it; 3.8M leaves 331,
// from 374.

constexpr int kRHash = 256;      // LDS hash for ancestors outside the tile's index range
constexpr int kVSet = 2048;      // distinct vertex ids per tile (hash set)
constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr int32_t kKeyHi = 0x7FFFFFFF, kKeyLo = (int32_t)0x80000000;

// An internal node for tiers A and B: three 16-byte words, the candidate axes
// (9 floats), the parent and the span; bit 31 of the span's first leaf marks a
// degenerate node.
struct RefitNode {
    float4 w[3];

    __device__ __forceinline__ void set(const float b[9], uint32_t parent, uint2 span, bool degen) {
        w[0] = make_float4(b[0], b[1], b[2], b[3]);
        w[1] = make_float4(b[4], b[5], b[6], b[7]);
        w[2] = make_float4(b[8], __uint_as_float(parent), __uint_as_float(span.x | (degen ? kGap : 0u)),
                           __uint_as_float(span.y));
    }
    __device__ __forceinline__ f3 axis(int a) const {
        return a == 0 ? f3{w[0].x, w[0].y, w[0].z} : a == 1 ? f3{w[0].w, w[1].x, w[1].y} : f3{w[1].z, w[1].w, w[2].x};
    }
    __device__ __forceinline__ uint32_t parent() const { return __float_as_uint(w[2].y); }
    __device__ __forceinline__ uint2 span() const {
        return make_uint2(__float_as_uint(w[2].z) & ~kGap, __float_as_uint(w[2].w));
    }
    __device__ __forceinline__ bool degen() const { return (__float_as_uint(w[2].z) & kGap) != 0; }
};

struct RefitTile {
    int32_t tk[kRTile][6];        // keys of internal node lo + s: min b0..b2, max b0..b2
    uint32_t hkey[kRHash];
    int32_t hval[kRHash][6];
    uint32_t vkey[kVSet];        // distinct vertex ids of the tile's triangles
    union {
        RefitNode nd[kRTile];    // internal nodes lo .. lo + 511, until tiers A and B end
        float upos[3 * kRTile][3];  // then: the distinct vertices' positions, compacted
    };
    uint32_t chain[kTChain];     // tile-common node and its ancestors
    uint32_t nchain, nuniq, overflow, rest, unsafe;
};

// Lanes below this one in a ballot.
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ RefitNode refit_node(const RefitTile& R, const TreeWs& ws, const uint32_t* parents,
                                                uint32_t lo, uint32_t p) {
    if (p - lo < kRTile) return R.nd[p - lo];
    RefitNode n;
    const Cand c = ws.cand[p];
    n.set(c.b, parents[p], ws.span[p], c.degen != 0);
    return n;
}

// Order-preserving key of a float (same map as f2ord, without a branch).
__device__ __forceinline__ int32_t okey(float f) {
    const int32_t i = __float_as_int(f);
    return i ^ ((i >> 31) & 0x7FFFFFFF);
}

// Unconditional: reading the current keys first to skip atomics made every
// fold wait for a load of a line other workgroups update (about a fifth of
// the refit's time on a 2M-leaf tree).
__device__ __forceinline__ void fold_global(int32_t* rk, const int32_t v[6]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        atomicMin(&rk[a], v[a]);
        atomicMax(&rk[3 + a], v[3 + a]);
    }
}

__device__ __forceinline__ void fold_lds(int32_t* slot, const int32_t v[6]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        atomicMin(&slot[a], v[a]);
        atomicMax(&slot[3 + a], v[3 + a]);
    }
}

// One step of fold_quads: lanes i and i ^ kBit with the same tag combine their
// keys, and the upper one drops out (a tag of its own).
template <int kBit, int kPerm>
__device__ __forceinline__ void fold_quad_step(uint32_t& tag, int32_t k[6]) {
    const bool same = (uint32_t)dpp_mov<kPerm>((int32_t)tag) == tag;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int32_t mn = min(k[a], dpp_mov<kPerm>(k[a])), mx = max(k[3 + a], dpp_mov<kPerm>(k[3 + a]));
        k[a] = same ? mn : k[a];
        k[3 + a] = same ? mx : k[3 + a];
    }
    if (same && (lane_id() & kBit)) tag = 0x80000000u | (uint32_t)lane_id();
}
// Keys of the lanes that hold the same node p, combined within each group of
// four lanes.  Called by the whole wave, lanes without keys with on = false.
// True for the lanes left to fold: where a node's leaves are consecutive lanes,
// one or two of a group.  The LDS atomics of one wave on one node are made one
// lane after the other and bound the tier; a lane's key reads before them, to
// skip some, took as long (both on 1M triangles, with the reads 437 us the
// transform, all lanes' atomics 434, groups of four 429, of sixteen 433).
__device__ __forceinline__ bool fold_quads(bool on, uint32_t p, int32_t k[6]) {
    const uint32_t mine = on ? p : 0x80000000u | (uint32_t)lane_id();
    uint32_t tag = mine;
    fold_quad_step<1, 0xB1>(tag, k);  // quad_perm [1,0,3,2]
    fold_quad_step<2, 0x4E>(tag, k);  // quad_perm [2,3,0,1]
    return on && tag == mine;
}

__device__ __forceinline__ void fold_tile(RefitTile& R, int32_t* range, uint32_t lo, uint32_t p, const int32_t k[6]) {
    if (p - lo < kRTile) {
        fold_lds(R.tk[p - lo], k);
        return;
    }
    uint32_t h = (p * 2654435761u) >> 24;
    for (int probe = 0; probe < 16; ++probe) {  // linear probing
        uint32_t key = R.hkey[h];
        if (key == kEmpty) key = atomicCAS(&R.hkey[h], kEmpty, p);
        if (key == kEmpty || key == p) {
            fold_lds(R.hval[h], k);
            return;
        }
        h = (h + 1) & (kRHash - 1);
    }
    fold_global(&range[(size_t)p * 6], k);
}

// Keys of one triangle's projection range on the node's axes.  The
// reference reduces the three projections with kr_min / kr_max from vertex 0
// and lets the result enter the node's range only when strictly beyond it
// (transforms.cu:855-897).  For finite vertices (fin) the dot products are
// never NaN and that is the integer min / max of the keys (up to the sign of
// a zero).  Otherwise the compare-and-select chain is evaluated as written,
// and a NaN result gives the neutral key, i.e. never enters the range.
__device__ __forceinline__ void tri_keys(const f3 axes[3], f3 v0, f3 v1, f3 v2, bool fin, int32_t k[6]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const f3 b = axes[a];
        const float d0 = dot3(v0, b), d1 = dot3(v1, b), d2 = dot3(v2, b);
        if (fin) {
            const int32_t k0 = okey(d0), k1 = okey(d1), k2 = okey(d2);
            k[a] = min(min(k0, k1), k2);
            k[3 + a] = max(max(k0, k1), k2);
        } else {
            const float lo = kmin(kmin(d0, d1), d2), hi = kmax(kmax(d0, d1), d2);
            k[a] = lo == lo ? okey(lo) : kKeyHi;
            k[3 + a] = hi == hi ? okey(hi) : kKeyLo;
        }
    }
}

// All coordinates finite (exponent field not all ones).
__device__ __forceinline__ bool finite3(f3 v) {
    const uint32_t m = 0x7F800000u;
    return (__float_as_uint(v.x) & m) != m && (__float_as_uint(v.y) & m) != m && (__float_as_uint(v.z) & m) != m;
}

__device__ __forceinline__ void wave_keys(int32_t k[6]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        k[a] = wave_min_i32(k[a]);
        k[3 + a] = wave_max_i32(k[3 + a]);
    }
}

__global__ __launch_bounds__(kRTile) void refit(TreeNodes nodes,
                                               const uint32_t* __restrict__ parents,
                                               const kr_vec3* __restrict__ V,
                                               const kr_uvec4* __restrict__ F, TreeWs ws, uint32_t N) {
    __shared__ RefitTile R;
    __shared__ uint32_t bad;
    const uint32_t I = N - 1, t = threadIdx.x;
    const uint32_t lo = blockIdx.x * kRTile;
    const uint32_t thi = min(lo + kRTile, N) - 1;  // last leaf position of the tile
    const uint32_t pos = lo + t;
    const bool valid = pos < N;
    // the chain leaf -> face -> vertices starts first: the tile's set-up runs under its latency
    const uint32_t f = valid ? nodes.face(I + pos) : kInvalid;
    const uint32_t leaf_parent = valid ? parents[I + pos] : kInvalid;
#pragma unroll
    for (int a = 0; a < 3; ++a) { R.tk[t][a] = kKeyHi; R.tk[t][3 + a] = kKeyLo; }
    if (t < kRHash) {
        R.hkey[t] = kEmpty;
#pragma unroll
        for (int a = 0; a < 3; ++a) { R.hval[t][a] = kKeyHi; R.hval[t][3 + a] = kKeyLo; }
    }
    for (uint32_t h = t; h < kVSet; h += kRTile) R.vkey[h] = kEmpty;
    if (pos < I) {  // the tile's own index range, for tiers A and B
        const Cand c = ws.cand[pos];
        R.nd[t].set(c.b, parents[pos], ws.span[pos], c.degen != 0);
    }
    if (t == 0) {
        bad = *ws.error;  // one read per workgroup: the exit is uniform
        const uint2 m = ws.tmeta[blockIdx.x];
        R.nchain = min(m.x, (uint32_t)kTChain);
        R.rest = m.y;
        R.nuniq = 0;
        R.overflow = 0;
        R.unsafe = 0;
    }
    if (t < kTChain) R.chain[t] = ws.tchain[(size_t)blockIdx.x * kTChain + t];  // entries past the count unused
    kr_uvec4 face = {};
    if (f < N) face = F[f];  // (a face id out of range set the error, and the workgroup ends below)
    __syncthreads();
    if (bad != 0) return;

    const uint32_t wlo = pos - (uint32_t)lane_id();
    const uint32_t whi = min(wlo + kWave - 1, N - 1);
    f3 v[3] = {f3{0, 0, 0}, f3{0, 0, 0}, f3{0, 0, 0}};
    bool fin = true;
    uint32_t own = 0;  // bit j: the tile's distinct vertices list vertex j from this lane
    if (valid) {
        const uint32_t vid[3] = {face.x, face.y, face.z};
#pragma unroll
        for (int j = 0; j < 3; ++j) v[j] = ldv(V, vid[j]);
        uint32_t h[3], key[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            h[j] = (vid[j] * 2654435761u) >> 21;
            key[j] = R.vkey[h[j]];
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {  // distinct vertex ids of the tile
            bool placed = false;
            for (int probe = 0; probe < 32 && !placed; ++probe) {
                if (probe != 0) {
                    h[j] = (h[j] + 1) & (kVSet - 1);
                    key[j] = R.vkey[h[j]];
                }
                if (key[j] == kEmpty) {
                    key[j] = atomicCAS(&R.vkey[h[j]], kEmpty, vid[j]);
                    if (key[j] == kEmpty) own |= 1u << j;
                }
                placed = key[j] == kEmpty || key[j] == vid[j];
            }
            if (!placed) R.overflow = 1;
        }
        fin = finite3(v[0]) && finite3(v[1]) && finite3(v[2]);
        // the tile-wide pass projects vertices, not triangles: a tile with a
        // non-finite vertex keeps the per-triangle rule up to the root
        if (!fin) R.overflow = 1;
        if (!sane_points(v, 3)) R.unsafe = 1;
    }
    // places of the lane's own vertices in the list: one count per wave
    const uint64_t o0 = __ballot(own & 1u), o1 = __ballot(own & 2u), o2 = __ballot(own & 4u);
    uint32_t u0 = 0;
    if (lane_id() == 0) u0 = atomicAdd(&R.nuniq, (uint32_t)(__popcll(o0) + __popcll(o1) + __popcll(o2)));
    u0 = __builtin_amdgcn_readfirstlane(u0) + lanes_below(o0) + lanes_below(o1) + lanes_below(o2);
    __syncthreads();
    // tier C needs the tile-common node (chain[0]) and a vertex set that fit
    const bool tile_pass = R.overflow == 0 && R.nchain != 0;
    const uint32_t q0 = tile_pass ? R.chain[0] : kInvalid;

    if (wlo < N) {  // wave-uniform
        // tier A: the next node is read while this one's keys are made
        uint32_t common = kInvalid, p = leaf_parent;
        bool on = valid && p < I;
        RefitNode c = {};
        if (on) c = refit_node(R, ws, parents, lo, p);
        for (uint32_t step = 0; step < N && __ballot(on) != 0; ++step) {  // uniform
            if (on && holds(c.span(), wlo, whi)) {
                common = p;
                on = false;
            }
            const uint32_t pp = on ? c.parent() : kInvalid;
            RefitNode n = c;
            if (pp < I) n = refit_node(R, ws, parents, lo, pp);
            const f3 axes[3] = {c.axis(0), c.axis(1), c.axis(2)};
            int32_t k[6];
            tri_keys(axes, v[0], v[1], v[2], fin, k);
            if (fold_quads(on && !c.degen(), p, k)) fold_tile(R, ws.range, lo, p, k);
            on = pp < I;
            c = n;
            p = pp;
        }
        // tier B; lane 0 is valid (wlo < N) and a well-formed tree gives
        // every valid lane the same node
        const uint32_t c0 = __builtin_amdgcn_readfirstlane(common);
        if (__ballot(valid && common != c0) != 0) {
            if (lane_id() == 0) atomicOr(ws.error, 2u);
        } else if (c0 < I && c0 != q0) {  // tier C takes q0 and above
            uint32_t q = c0;
            RefitNode c = refit_node(R, ws, parents, lo, q);
            for (uint32_t step = 0; step < N; ++step) {  // uniform
                const uint32_t qp = __builtin_amdgcn_readfirstlane(c.parent());
                const bool last = qp >= I || qp == q0;
                RefitNode n = c;
                if (!last) n = refit_node(R, ws, parents, lo, qp);
                if (!c.degen()) {
                    const f3 axes[3] = {c.axis(0), c.axis(1), c.axis(2)};
                    int32_t k[6];
                    if (valid) {
                        tri_keys(axes, v[0], v[1], v[2], fin, k);
                    } else {
#pragma unroll
                        for (int a = 0; a < 3; ++a) { k[a] = kKeyHi; k[3 + a] = kKeyLo; }
                    }
                    wave_keys(k);
                    if (lane_id() == 0) fold_tile(R, ws.range, lo, q, k);
                }
                if (last) break;
                q = qp;
                c = n;
            }
        }
    }
    __syncthreads();

    if (tile_pass) {
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (own & (1u << j)) {
                R.upos[u0][0] = v[j].x;
                R.upos[u0][1] = v[j].y;
                R.upos[u0][2] = v[j].z;
                ++u0;
            }
        __syncthreads();
        // tier C over the distinct vertices; each wave reads the axes and
        // current keys of its next ancestor while it works on this one (the
        // keys only filter the atomics: they only move outwards, so an early
        // read never skips a needed update)
        const uint32_t nu = R.nuniq, nc = R.nchain;
        const uint32_t step_c = kRTile / kWave;
        uint32_t j = (uint32_t)wave_id();
        uint32_t qc = 0;
        Cand c = {};
        int32_t cur[6] = {0, 0, 0, 0, 0, 0};
        if (j < nc) {
            qc = __builtin_amdgcn_readfirstlane(R.chain[j]);
            c = ws.cand[qc];
#pragma unroll
            for (int a = 0; a < 6; ++a) cur[a] = ws.range[(size_t)qc * 6 + a];
        }
        for (; j < nc; j += step_c) {
            uint32_t qn = 0;
            Cand cn = {};
            int32_t curn[6] = {0, 0, 0, 0, 0, 0};
            if (j + step_c < nc) {
                qn = __builtin_amdgcn_readfirstlane(R.chain[j + step_c]);
                cn = ws.cand[qn];
#pragma unroll
                for (int a = 0; a < 6; ++a) curn[a] = ws.range[(size_t)qn * 6 + a];
            }
            if (!c.degen) {
                int32_t k[6];
#pragma unroll
                for (int a = 0; a < 3; ++a) { k[a] = kKeyHi; k[3 + a] = kKeyLo; }
                for (uint32_t u = (uint32_t)lane_id(); u < nu; u += kWave) {
                    const f3 p = f3{R.upos[u][0], R.upos[u][1], R.upos[u][2]};
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const int32_t kk = okey(dot3(p, f3{c.b[3 * a], c.b[3 * a + 1], c.b[3 * a + 2]}));
                        k[a] = min(k[a], kk);
                        k[3 + a] = max(k[3 + a], kk);
                    }
                }
                wave_keys(k);
                if (lane_id() == 0) {
                    int32_t* rk = &ws.range[(size_t)qc * 6];
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        if (k[a] < cur[a]) atomicMin(&rk[a], k[a]);
                        if (k[3 + a] > cur[3 + a]) atomicMax(&rk[3 + a], k[3 + a]);
                    }
                }
            }
            qc = qn;
            c = cn;
#pragma unroll
            for (int a = 0; a < 6; ++a) cur[a] = curn[a];
        }
        // ancestors beyond the recorded batch (very deep trees): every wave
        // walks them with its lanes' triangles
        uint32_t q = R.rest;
        if (wlo < N) {
            for (uint32_t step = 0; q != kInvalid && q < I && step < N; ++step) {  // uniform
                const Cand c = ws.cand[q];
                if (!c.degen) {
                    int32_t k[6];
                    if (valid) {
                        const f3 axes[3] = {f3{c.b[0], c.b[1], c.b[2]}, f3{c.b[3], c.b[4], c.b[5]},
                                            f3{c.b[6], c.b[7], c.b[8]}};
                        tri_keys(axes, v[0], v[1], v[2], fin, k);
                    } else {
#pragma unroll
                        for (int a = 0; a < 3; ++a) { k[a] = kKeyHi; k[3 + a] = kKeyLo; }
                    }
                    wave_keys(k);
                    if (lane_id() == 0) fold_global(&ws.range[(size_t)q * 6], k);
                }
                q = __builtin_amdgcn_readfirstlane(parents[q]);
            }
        }
    }
    __syncthreads();
    // Write the tile's LDS keys to global memory.  A node whose leaves all lie
    // in this tile has no contributor outside this workgroup, and within it
    // only the LDS slot (tier C, which folds with atomics, never takes such a
    // node except the tile-common node, whose span is the tile): its keys
    // replace the candidate search's range, which came from some of the same
    // vertices by the same dot products.  Where the tile has a non-finite or
    // huge vertex that range may hold more (the search's reference mode), and
    // the keys are merged into it; the other nodes' are merged with atomics.
    if (lo + t < I && (R.tk[t][0] != kKeyHi || R.tk[t][3] != kKeyLo)) {
        const uint32_t node = lo + t;
        const uint2 sp = ws.span[node];
        int32_t* rk = &ws.range[(size_t)node * 6];
        const bool chain_node = node == q0;
        if (sp.x >= lo && span_hi(sp) <= thi && !chain_node) {
            int32_t k[6];
#pragma unroll
            for (int a = 0; a < 6; ++a) k[a] = R.tk[t][a];
            if (R.unsafe) {
#pragma unroll
                for (int a = 0; a < 3; ++a) { k[a] = min(rk[a], k[a]); k[3 + a] = max(rk[3 + a], k[3 + a]); }
            }
#pragma unroll
            for (int a = 0; a < 6; ++a) rk[a] = k[a];
        } else {
            fold_global(rk, R.tk[t]);
        }
    }
    if (t < kRHash && R.hkey[t] != kEmpty) fold_global(&ws.range[(size_t)R.hkey[t] * 6], R.hval[t]);
}

// --------------------------------------------------------- finalize --
//
// One lane per internal node (transforms.cu:905-964): OBB vs AABB by half
// area, extent floor, inverse(T * R * S).  Boxes and matrices are staged in
// LDS (odd row strides, no bank conflicts) and written back as contiguous
// dwords.

__global__ __launch_bounds__(kStage) void finalize(TreeWs ws, kr_obb3* obbs, kr_mat4* mats, uint32_t I,
                                                   BatchMap bm) {
    __shared__ Stage st;
    const uint32_t base = blockIdx.x * kStage;
    const uint32_t node = base + threadIdx.x;
    float* ob = &st.ob[threadIdx.x * 15];
    float* mt = &st.mt[threadIdx.x * 17];
    if (node < I) {
        const uint64_t vw = ws.visit[node];
        if (!complete(vw)) atomicOr(ws.error, 8u);  // a malformed tree: the node never completed
        if (*ws.error != 0 || !complete(vw) || hole(vw)) {
            stage_nan(st, threadIdx.x);
        } else {
            const Cand c = ws.cand[node];
            const int32_t* rk = &ws.range[(size_t)node * 6];
            const f3 rmn = f3{ord2f(rk[0]), ord2f(rk[1]), ord2f(rk[2])};
            const f3 rmx = f3{ord2f(rk[3]), ord2f(rk[4]), ord2f(rk[5])};
            f3 v0, v1, v2, mn, mx;
            if (!c.degen && quality(sub3(rmx, rmn)) < c.aq) {
                v0 = f3{c.b[0], c.b[1], c.b[2]};
                v1 = f3{c.b[3], c.b[4], c.b[5]};
                v2 = f3{c.b[6], c.b[7], c.b[8]};
                mn = rmn;
                mx = rmx;
            } else {  // the AABB: the k-DOP's first three slabs
                v0 = f3{1, 0, 0};
                v1 = f3{0, 1, 0};
                v2 = f3{0, 0, 1};
                if (c.degen) {  // the candidate step kept them in the range, which the refit skips
                    mn = rmn;
                    mx = rmx;
                } else {
                    const float4* kd = &ws.kdop[(size_t)node * 7];
                    const float4 s0 = kd[0], s1 = kd[1], s2 = kd[2];
                    mn = f3{s0.x, s1.x, s2.x};
                    mx = f3{s0.z, s1.z, s2.z};
                }
            }
            const f3 mid = vm::mul1(add3(mn, mx), 0.5f);
            const f3 ext = vm::vmax3(vm::mul1(sub3(mx, mn), 0.5f), f3{0.001f, 0.001f, 0.001f});
            f3 m = vm::mul1(v0, mid.x);
            m = add3(m, vm::mul1(v1, mid.y));
            m = add3(m, vm::mul1(v2, mid.z));
            obb_row(ob, m, v0, v1, v2, ext);
            float M[16];
            obb_matrix(v0, v1, v2, m, ext, M);
#pragma unroll
            for (int q = 0; q < 16; ++q) mt[q] = M[q];
        }
    }
    __syncthreads();
    stage_flush(st, obbs, mats, base, min((uint32_t)kStage, I - min(base, I)), bm);
}

__global__ void copy_ids(const kr_bvh_node* __restrict__ nodes, const kr_vec3* __restrict__ V,
                         const kr_uvec4* __restrict__ F, TreeWs ws, uint32_t* ids, uint32_t total) {
    const uint32_t node = blockIdx.x * blockDim.x + threadIdx.x;
    if (node >= total) return;
    const uint32_t I = (total - 1) / 2, N = I + 1;
    Kdop k;
    bool ok = *ws.error == 0;
    if (ok) {
        if (node < I) {
            ok = complete(ws.visit[node]);
            if (ok) kdop_load(ws.kdop, node, k);
        } else {
            ok = leaf_kdop_global(nodes, V, F, node, N, k);
        }
    }
#pragma unroll
    for (int s = 0; s < 7; ++s) {
        ids[(size_t)node * 14 + s] = ok ? k.imn[s] : 0xFFFFFFFFu;
        ids[(size_t)node * 14 + 7 + s] = ok ? k.imx[s] : 0xFFFFFFFFu;
    }
}

__global__ void copy_status(const uint32_t* error, uint32_t* status) { *status = *error; }

// ------------------------------------------------------------- host --

size_t tree_carve(TreeWs* ws, void* base, size_t cap, uint32_t N) {
    Carver c{(char*)base, 0, cap};
    const size_t I = N ? N - 1 : 0, total = N ? 2 * (size_t)N - 1 : 0;
    ws->visit = c.take<uint64_t>(I + 1);
    ws->error = c.take<uint32_t>(8);
    ws->nlist = ws->error ? ws->error + 2 : nullptr;  // error[2 .. 2 + kNodeLists)
    ws->list = c.take<uint32_t>((size_t)kNodeLists * (I + 1));
    ws->span = c.take<uint2>(total);
    ws->count = c.take<uint32_t>(I + 1);
    ws->kdop = c.take<float4>(total * 7);
    ws->cand = c.take<Cand>(I + 1);
    ws->range = c.take<int32_t>((I + 1) * 6);
    const size_t tiles = ((size_t)N + kRTile - 1) / kRTile;
    ws->tchain = c.take<uint32_t>(tiles * kTChain);
    ws->tmeta = c.take<uint2>(tiles);
    return c.used;
}

// Per device: a second stream (default priority) and the events that fork the
// first candidate launch onto it and join it back.  One lock covers a call's enqueue
// sequence between them, so calls from several host threads cannot interleave
// their record / wait pairs.
namespace {
struct SideStream {
    hipStream_t s = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};
// Up to this many leaves all kernels run on the caller's stream: the hand-offs
// between streams cost 10-15 us, more than the top of the tree takes from the
// candidate search beside it.  Measured, one stream / two (icospheres, us):
// 100820 leaves 127 / 142, 200000 165 / 170, 264500 202 / 201, 338000 221 / 213,
// 499280 267 / 254, 1003520 454 / 424.
constexpr uint32_t kOneStream = 1u << 18;
constexpr int kMaxDevices = 64;
std::mutex g_side_mu;
SideStream g_side[kMaxDevices];

kr_error side_stream(SideStream** out) {
    int dev = 0;
    OBVH_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return "obvh_obb_tree: device ordinal out of range";
    SideStream& ss = g_side[dev];
    if (ss.s == nullptr) {
        OBVH_HIP_TRY(hipStreamCreateWithFlags(&ss.s, hipStreamNonBlocking));
        OBVH_HIP_TRY(hipEventCreateWithFlags(&ss.fork, hipEventDisableTiming));
        OBVH_HIP_TRY(hipEventCreateWithFlags(&ss.join, hipEventDisableTiming));
    }
    *out = &ss;
    return nullptr;
}
}  // namespace

static kr_error tree_run(TreeNodes nodes, const uint32_t* parents, const kr_vec3* V, const kr_uvec4* F, kr_obb3* obbs,
                         kr_mat4* mats, uint32_t N, void* workspace, size_t ws_bytes, hipStream_t stream,
                         const BatchMap& bm) {
    TreeWs ws;
    size_t need = tree_carve(&ws, workspace, ws_bytes, N);
    if (workspace == nullptr || ws_bytes < need) return "obvh_obb_tree: workspace too small";
    const uint32_t I = N - 1;
    auto blocks = [](uint32_t n, uint32_t b) { return dim3((n + b - 1) / b); };
    hipLaunchKernelGGL(tree_clear, dim3(1024), dim3(256), 0, stream, ws.visit, I + 1, ws);
    if (bm.K > 1)
        hipLaunchKernelGGL(batch_holes, dim3(min((bm.K + 255) / 256, 1024u)), dim3(256), 0, stream, ws, bm);
    hipLaunchKernelGGL(climb_leaves, blocks(N, kTile), dim3(kTile), 0, stream, nodes, parents, V, F, ws, N, obbs, mats,
                       bm);
    if (I > 0) {
        // About one deferred node per tile, if the leaves lie in tree order;
        // at most an eighth of the chip's waves, so that the candidate search
        // beside it fills the rest (64 trees of 3.8M triangles: 1696 us with up
        // to 1024, 1773 with up to 8192).
        const dim3 upper_grid(min(N / kTile + 1, 1024u));
        const uint32_t cb = (((N + kRTile - 1) / kRTile) + kCandBlock - 1) / kCandBlock;  // the refit tiles' chains
        if (N <= kOneStream) {
            if (N > kTile)
                hipLaunchKernelGGL(climb_upper, upper_grid, dim3(kUpperThreads), 0, stream, nodes, parents, ws, N);
            hipLaunchKernelGGL(candidates<kAllNodes>, dim3(cb + (I + kCandBlock - 1) / kCandBlock), dim3(kCandBlock), 0,
                               stream, V, parents, ws, N, cb);
        } else {
            // The candidate search of the nodes the tile climb completed
            // (nearly all of them; VALU-bound) runs on the side stream beside
            // the top of the tree (latency-bound on a few waves) and its
            // search on the caller's stream, joined before the refit.  The
            // other way round the top's waves come last onto a full chip: 2M
            // triangles 890 us against 876.
            std::lock_guard<std::mutex> lock(g_side_mu);
            SideStream* side = nullptr;
            if (kr_error e = side_stream(&side)) return e;
            const uint32_t ub = min((I + kCandBlock - 1) / kCandBlock, 1024u);
            OBVH_HIP_TRY(hipEventRecord(side->fork, stream));
            hipLaunchKernelGGL(climb_upper, upper_grid, dim3(kUpperThreads), 0, stream, nodes, parents, ws, N);
            OBVH_HIP_TRY(hipStreamWaitEvent(side->s, side->fork, 0));
            hipLaunchKernelGGL(candidates<kTileNodes>, blocks(I, kCandBlock), dim3(kCandBlock), 0, side->s, V, parents,
                               ws, N, 0u);
            hipLaunchKernelGGL(candidates<kUpperNodes>, dim3(cb + ub), dim3(kCandBlock), 0, stream, V, parents, ws, N,
                               cb);
            OBVH_HIP_TRY(hipEventRecord(side->join, side->s));
            OBVH_HIP_TRY(hipStreamWaitEvent(stream, side->join, 0));
        }
        hipLaunchKernelGGL(cand_redo, dim3(kRedoBlocks), dim3(1024), 0, stream, V, ws, I);
        hipLaunchKernelGGL(refit, blocks(N, kRTile), dim3(kRTile), 0, stream, nodes, parents, V, F, ws, N);
        hipLaunchKernelGGL(finalize, blocks(I, kStage), dim3(kStage), 0, stream, ws, obbs, mats, I, bm);
    }
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

kr_error tree_launch(const kr_bvh_node* nodes, const uint32_t* parents, const kr_vec3* V,
                     const kr_uvec4* F, kr_obb3* obbs, kr_mat4* mats, uint32_t* ids, uint32_t N,
                     void* workspace, size_t ws_bytes, hipStream_t stream) {
    if (N == 0) return nullptr;
    if (kr_error e = tree_run(tree_nodes(nodes), parents, V, F, obbs, mats, N, workspace, ws_bytes, stream,
                              BatchMap{nullptr, 0, 0}))
        return e;
    if (ids) {
        TreeWs ws;
        tree_carve(&ws, workspace, ws_bytes, N);
        const uint32_t total = 2 * N - 1;
        hipLaunchKernelGGL(copy_ids, dim3((total + 255) / 256), dim3(256), 0, stream, nodes, V, F, ws, ids, total);
        OBVH_HIP_TRY(hipGetLastError());
    }
    return nullptr;
}

// ------------------------------------------------------------ batch --
//
// Many trees in one transform.  The batch's trees (tree t: N_t >= 1 leaves,
// nodes, parents, faces and vertices back to back, indices local to the
// tree) become one forest in the single-tree numbering, so that every
// kernel runs once for the whole batch.  Each node's k-DOP, candidate axes,
// refit range and box depend only on its own subtree, so the forest gives
// every tree's nodes exactly the per-tree results.  The numbering keeps each
// tree Karras-aligned: with L_t the first leaf position of tree t (prefix
// sum of N_s), its internal node j goes to L_t + j + 1 (t < K - 1) or
// L_t + j (the last tree) and its leaf i to (sum N - 1) + L_t + i; the
// internal slots L_k (k < K - 1) stay unused (holes: marked complete with
// tag kHoleTag, skipped by the per-node kernels).  Every tree root has no
// parent.  Tree t's nodes start at 2 L_t - t in the input layout.
//
// The combined nodes keep the children alone (8 bytes of 36), and boxes and
// matrices of rows that lie in one tree go out as in a single transform: 64
// trees of 3.8M triangles 1611 us with whole nodes and a row map, now 1554
// (gathers 191 -> 151, leaf boxes and finalize 40 less; the nodes' gather moves
// 395 MB in 110 us).

// The tree of element i, found once for a workgroup whose 256 elements lie in one
// tree (nearly all of them), per lane otherwise.
template <class Of, class Begin>
__device__ __forceinline__ uint32_t of_group(Of of, Begin begin, uint32_t i, uint32_t n) {
    const uint32_t first = i - threadIdx.x;
    const uint32_t t = of(__builtin_amdgcn_readfirstlane(first));
    return first + 256u <= begin(t + 1) || n <= begin(t + 1) ? t : of(i);
}

// One lane per input node: write the combined node and parent.  Bad local
// indices (children, parents, face ids outside the tree, an empty tree) set
// the batch error word and are mapped out of range, where the transform's
// own checks report them.
__global__ void batch_gather_nodes(BatchMap m, const kr_bvh_node* __restrict__ nodes,
                                   const uint32_t* __restrict__ parents, uint2* cn, uint32_t* cp,
                                   uint32_t* berr, uint32_t total_in) {
    const uint32_t total = 2 * m.Nsum - 1;
    for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < total_in; g += gridDim.x * blockDim.x) {
        const uint32_t t = of_group([&](uint32_t i) { return batch_tree_of_node(m, i); },
                                    [&](uint32_t k) { return 2u * m.prim_off[k] - k; }, g, total_in);
        const uint32_t Lt = m.prim_off[t], N = m.prim_off[t + 1] - Lt;
        if (N == 0) { atomicOr(berr, 1u); continue; }
        const uint32_t nb = 2 * Lt - t, j = g - nb, nn = 2 * N - 1;
        if (j >= nn) { atomicOr(berr, 1u); continue; }
        const uint32_t c = batch_map(m, t, Lt, N, j);
        uint2 o = make_uint2(nodes[g].u.children.left, nodes[g].u.children.right);
        if (j + 1 < N) {
            const uint32_t l = o.x, r = o.y;
            if (l >= nn || r >= nn) atomicOr(berr, 2u);
            o.x = l < nn ? batch_map(m, t, Lt, N, l) : total;
            o.y = r < nn ? batch_map(m, t, Lt, N, r) : total;
        } else {
            if (o.x >= N) atomicOr(berr, 4u);
            o.x = o.x < N ? Lt + o.x : 0xFFFFFFFFu;  // its face
        }
        cn[c] = o;
        const uint32_t p = parents[g];
        uint32_t cpar;
        if (p == kInvalid) cpar = j == 0 ? kInvalid : total;  // only the root has none
        else cpar = p < nn ? batch_map(m, t, Lt, N, p) : total;
        if ((p == kInvalid) != (j == 0) || (p != kInvalid && p >= nn)) atomicOr(berr, 2u);
        cp[c] = cpar;
    }
    // the unused internal slots L_k (k < K - 1) between the trees
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k + 1 < m.K; k += gridDim.x * blockDim.x) {
        const uint32_t idx = m.prim_off[k];
        cn[idx] = make_uint2(0u, 0u);
        cp[idx] = kInvalid;
    }
}

// One lane per face: vertex ids rebased to the batch's vertex array.
__global__ void batch_gather_faces(BatchMap m, const uint32_t* __restrict__ vert_off,
                                   const kr_uvec4* __restrict__ faces, kr_uvec4* cf, uint32_t* berr) {
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < m.Nsum; f += gridDim.x * blockDim.x) {
        const uint32_t t = of_group([&](uint32_t i) { return batch_tree_of_leaf(m, i); },
                                    [&](uint32_t k) { return m.prim_off[k]; }, f, m.Nsum);
        const uint32_t vb = vert_off[t], nv = vert_off[t + 1] - vb;
        kr_uvec4 a = faces[f];
        if (a.x >= nv || a.y >= nv || a.z >= nv) {
            atomicOr(berr, 8u);  // rebased to vertex 0 of the batch: never read outside the array
            a.x = a.x < nv ? vb + a.x : 0u;
            a.y = a.y < nv ? vb + a.y : 0u;
            a.z = a.z < nv ? vb + a.z : 0u;
        } else {
            a.x += vb;
            a.y += vb;
            a.z += vb;
        }
        cf[f] = a;
    }
}

struct BatchWs {
    uint2* nodes;  // children, or a leaf's face and 0
    uint32_t* parents;
    kr_uvec4* faces;
    uint32_t* berr;
    void* tree_ws;
    size_t tree_ws_bytes;
};

size_t batch_carve(BatchWs* w, void* base, size_t cap, uint32_t Nsum) {
    Carver c{(char*)base, 0, cap};
    const size_t total = 2 * (size_t)Nsum - 1;
    w->berr = c.take<uint32_t>(4);
    w->nodes = c.take<uint2>(total);
    w->parents = c.take<uint32_t>(total);
    w->faces = c.take<kr_uvec4>(Nsum);
    TreeWs tw;
    w->tree_ws_bytes = tree_carve(&tw, nullptr, 0, Nsum);
    w->tree_ws = c.take<char>(w->tree_ws_bytes);
    return c.used;
}

size_t batch_workspace_size(uint32_t Nsum) {
    BatchWs w;
    return batch_carve(&w, nullptr, 0, Nsum);
}

__global__ void batch_clear(uint32_t* berr) {
    if (threadIdx.x == 0) *berr = 0;
}

kr_error tree_batch_launch(const kr_bvh_node* nodes, const uint32_t* parents, const kr_vec3* V, const kr_uvec4* F,
                           const uint32_t* prim_off, const uint32_t* vert_off, uint32_t K, uint32_t Nsum,
                           kr_obb3* obbs, kr_mat4* mats, void* workspace, size_t ws_bytes, hipStream_t stream) {
    if (K == 0 || Nsum == 0) return nullptr;
    if (Nsum < K) return "obvh_obb_tree_batch: every tree needs at least one primitive";
    BatchWs w;
    const size_t need = batch_carve(&w, workspace, ws_bytes, Nsum);
    if (workspace == nullptr || ws_bytes < need) return "obvh_obb_tree_batch: workspace too small";
    const BatchMap m{prim_off, K, Nsum};
    const uint32_t total_in = 2 * Nsum - K;
    auto grid = [](uint32_t n) { return dim3(min((n + 255) / 256, 65536u)); };
    hipLaunchKernelGGL(batch_clear, dim3(1), dim3(64), 0, stream, w.berr);
    hipLaunchKernelGGL(batch_gather_nodes, grid(max(total_in, K)), dim3(256), 0, stream, m, nodes, parents, w.nodes,
                       w.parents, w.berr, total_in);
    hipLaunchKernelGGL(batch_gather_faces, grid(Nsum), dim3(256), 0, stream, m, vert_off, F, w.faces, w.berr);
    OBVH_HIP_TRY(hipGetLastError());
    // climb_leaves and finalize write every node's box and matrix straight
    // to its place in the caller's per-tree layout
    return tree_run(TreeNodes{reinterpret_cast<const uint32_t*>(w.nodes), 2}, w.parents, V, w.faces, obbs, mats, Nsum,
                    w.tree_ws, w.tree_ws_bytes, stream, m);
}

__global__ void copy_batch_status(const uint32_t* berr, const uint32_t* error, uint32_t* status) {
    const uint32_t b = *berr;
    uint32_t s = *error;
    if (b & 1u) s |= 16u;  // an empty tree or a node outside its tree
    if (b & 2u) s |= 2u;
    if (b & 4u) s |= 4u;
    if (b & 8u) s |= 32u;
    *status = s;
}

kr_error tree_batch_status_launch(const void* workspace, size_t ws_bytes, uint32_t Nsum, uint32_t* status,
                                  hipStream_t stream) {
    BatchWs w;
    const size_t need = batch_carve(&w, const_cast<void*>(workspace), ws_bytes, Nsum);
    if (workspace == nullptr || ws_bytes < need) return "obvh_obb_tree_batch_status: workspace too small";
    TreeWs tw;
    tree_carve(&tw, w.tree_ws, w.tree_ws_bytes, Nsum);
    hipLaunchKernelGGL(copy_batch_status, dim3(1), dim3(1), 0, stream, w.berr, tw.error, status);
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

kr_error tree_status_launch(const void* workspace, size_t ws_bytes, uint32_t N, uint32_t* status,
                            hipStream_t stream) {
    TreeWs ws;
    const size_t need = tree_carve(&ws, const_cast<void*>(workspace), ws_bytes, N);
    if (workspace == nullptr || ws_bytes < need) return "obvh_obb_tree_status: workspace too small";
    hipLaunchKernelGGL(copy_status, dim3(1), dim3(1), 0, stream, ws.error, status);
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

const char* tree_status_string(uint32_t err) {
    if (err & 2u) return "obvh_obb_tree: parent/child links disagree";
    if (err & 1u) return "obvh_obb_tree: parent index out of range or cycle";
    if (err & 4u) return "obvh_obb_tree: leaf face id out of range";
    if (err & 8u) return "obvh_obb_tree: internal node never completed (malformed tree)";
    if (err & 16u) return "obvh_obb_tree_batch: empty tree in the batch or node outside its tree";
    if (err & 32u) return "obvh_obb_tree_batch: face vertex id outside its tree's vertices";
    if (err != 0u) return "obvh_obb_tree: unknown device error";
    return nullptr;
}

}  // namespace obvh
