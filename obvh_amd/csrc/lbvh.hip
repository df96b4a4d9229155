// lbvh.hip -- LBVH builder on gfx950 (the input side of the transform).
//
// Follows the reference build (src/ads/lbvh_gpu/lbvh.cu:252-457 and the
// sequence at :1640-1692):
//  1. centroid box of the triangle-box centres.  The reference reduction
//     (src/ads/common/cuda/transforms.cu:1127-1190) seeds every LDS slot of a
//     256-thread block with vertices[0] and lets out-of-range threads leave
//     before reducing, so for face counts that are not a multiple of 256 the
//     box also covers vertices[0]; that is reproduced because the Morton codes
//     (and so the tree) depend on it.  Exact min/max via integer atomics on
//     order-preserving float keys.
//  2. 30-bit Morton code of the offset triangle-box centre, safe divide by
//     the centroid extent (lbvh.cu:252-282, vecmath.h:698-716,760).
//  3. stable LSD radix sort of (code, face) pairs over 30 bits (radix.hpp),
//     the equivalent of thrust::stable_sort_by_key (lbvh.cu:1670).
//  4. Karras radix tree, duplicate codes split by 32 + clz(i ^ j)
//     (lbvh.cu:284-396); leaves written in sorted order.
//  5. bottom-up bounds, primitive counts, SAH costs (ct = 1.0, ci = 1.2),
//     lbvh.cu:399-457, in one launch (bottomup.hpp).
#include <float.h>

#include "bottomup.hpp"
#include "common.hpp"
#include "lbvh.hpp"

namespace obvh {

constexpr uint32_t kInv = 0xFFFFFFFFu;

__device__ __forceinline__ f3 ldv3(const kr_vec3* V, uint32_t i) {
    kr_vec3 a = V[i];
    return f3{a.x, a.y, a.z};
}

struct Box {
    f3 mn, mx;
};
__device__ __forceinline__ Box expand3(Box b, f3 a) { return Box{vm::vmin3(b.mn, a), vm::vmax3(b.mx, a)}; }
__device__ __forceinline__ Box tri_box(const kr_vec3* V, kr_uvec4 f) {
    f3 a = ldv3(V, f.x);
    Box b{a, a};
    b = expand3(b, ldv3(V, f.y));
    b = expand3(b, ldv3(V, f.z));
    return b;
}
__device__ __forceinline__ f3 box_center(Box b) {
    return f3{(b.mn.x + b.mx.x) * 0.5f, (b.mn.y + b.mx.y) * 0.5f, (b.mn.z + b.mx.z) * 0.5f};
}
__global__ void lbvh_init(const kr_vec3* V, uint32_t nf, LbvhWs ws) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) {
        if (nf % 256u != 0) {  // vertices[0] joins the centroid box (see header)
            f3 v = ldv3(V, 0);
            ws.cbox[0] = f2ord(v.x); ws.cbox[1] = f2ord(v.y); ws.cbox[2] = f2ord(v.z);
            ws.cbox[3] = f2ord(v.x); ws.cbox[4] = f2ord(v.y); ws.cbox[5] = f2ord(v.z);
        } else {
            for (int k = 0; k < 3; ++k) { ws.cbox[k] = 0x7FFFFFFF; ws.cbox[3 + k] = (int32_t)0x80000000; }
        }
    }
    for (uint32_t i = t; i < nf; i += gridDim.x * blockDim.x) ws.visit[i] = 0;
    for (uint32_t i = t; i < ws.radix.words; i += gridDim.x * blockDim.x) ws.radix.hist[i] = 0;
}

constexpr int kBoxThreads = 1024;
constexpr int kBoxGroups = 2 * kBoxThreads / 256, kBoxGroupWaves = 256 / kWave;

__global__ __launch_bounds__(kBoxThreads) void lbvh_centroid_box(const kr_vec3* V, const kr_uvec4* F, uint32_t nf,
                                                         LbvhWs ws) {
    __shared__ float sh[6][2 * kBoxThreads / kWave], group[6][kBoxGroups];
    const float INF = FLT_MAX * 2.0f;
    float mn[2][3] = {{INF, INF, INF}, {INF, INF, INF}}, mx[2][3] = {{-INF, -INF, -INF}, {-INF, -INF, -INF}};
    const uint32_t stride = gridDim.x * kBoxThreads;
    for (uint32_t f0 = blockIdx.x * kBoxThreads + threadIdx.x; f0 < nf; f0 += 2 * stride) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t f = f0 + h * stride;
            if (f >= nf) continue;
            const f3 c = box_center(tri_box(V, F[f]));
            mn[h][0] = fminf(mn[h][0], c.x); mn[h][1] = fminf(mn[h][1], c.y); mn[h][2] = fminf(mn[h][2], c.z);
            mx[h][0] = fmaxf(mx[h][0], c.x); mx[h][1] = fmaxf(mx[h][1], c.y); mx[h][2] = fmaxf(mx[h][2], c.z);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
        for (int k = 0; k < 3; ++k) {
            const float a = wave_min(mn[h][k]), b = wave_max(mx[h][k]);
            if (lane_id() == 0) {
                sh[k][h * (kBoxThreads / kWave) + wave_id()] = a;
                sh[3 + k][h * (kBoxThreads / kWave) + wave_id()] = b;
            }
        }
    __syncthreads();
    // The bounds of each 256 threads, of a thread's first, third, ... and of its
    // second, fourth, ... face: a bound that is not finite is left out (no
    // faces, or one of infinite extent among them, whose fellows' bound is then
    // left out too).  Up to 2^19 faces these are 256 consecutive faces.
    if (threadIdx.x < 6 * kBoxGroups) {
        const int k = threadIdx.x % 6, g = threadIdx.x / 6;
        const float* w = &sh[k][g * kBoxGroupWaves];
        float a = w[0];
        for (int i = 1; i < kBoxGroupWaves; ++i) a = k < 3 ? fminf(a, w[i]) : fmaxf(a, w[i]);
        if (!(a != INF && a != -INF)) a = k < 3 ? INF : -INF;
        group[k][g] = a;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int k = threadIdx.x;
        float a = group[k][0];
        for (int g = 1; g < kBoxGroups; ++g) a = k < 3 ? fminf(a, group[k][g]) : fmaxf(a, group[k][g]);
        if (a != INF && a != -INF) {
            // filtered: only a workgroup that improves the current bound
            // issues the atomic (thousands of same-address atomics serialise:
            // 2048 workgroups took 27 us, 256 take 10)
            const int32_t key = f2ord(a);
            const int32_t cur = __hip_atomic_load(&ws.cbox[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (k < 3 ? key < cur : key > cur) {
                if (k < 3) atomicMin(&ws.cbox[k], key);
                else atomicMax(&ws.cbox[k], key);
            }
        }
    }
}

__device__ __forceinline__ uint32_t stretch3(uint32_t x) {
    x &= 0x3ffu;
    x = (x | (x << 16)) & 0x30000ffu;
    x = (x | (x << 8)) & 0x300f00fu;
    x = (x | (x << 4)) & 0x30c30c3u;
    x = (x | (x << 2)) & 0x9249249u;
    return x;
}
__device__ __forceinline__ uint32_t quant10(float v) { return (uint32_t)kmin(kmax(v * 1024.0f, 0.0f), 1023.0f); }
__device__ __forceinline__ float safe_div(float a, float b) { return (b != 0.0f) ? a / b : 0.0f; }

constexpr int kPasses = 4;  // 8-bit digits of a 30-bit code

// Morton codes, and how often each digit value occurs for the sort (one set
// of global atomics per workgroup, hence at most 256 of them).
__global__ __launch_bounds__(1024) void lbvh_codes(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, LbvhWs ws) {
    __shared__ uint32_t h[kPasses * kRadixBins];
    for (uint32_t i = threadIdx.x; i < kPasses * kRadixBins; i += blockDim.x) h[i] = 0;
    __syncthreads();
    const f3 cmn = f3{ord2f(ws.cbox[0]), ord2f(ws.cbox[1]), ord2f(ws.cbox[2])};
    const f3 cmx = f3{ord2f(ws.cbox[3]), ord2f(ws.cbox[4]), ord2f(ws.cbox[5])};
    const f3 neg = f3{-cmn.x, -cmn.y, -cmn.z};
    const f3 ext = sub3(cmx, cmn);
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < nf; f += gridDim.x * blockDim.x) {
        Box b = tri_box(V, F[f]);
        Box o{add3(b.mn, neg), add3(b.mx, neg)};  // kr_aabb_offset3(bbox, -cell.min)
        f3 c = box_center(o);
        c = f3{safe_div(c.x, ext.x), safe_div(c.y, ext.y), safe_div(c.z, ext.z)};
        const uint32_t key = stretch3(quant10(c.x)) << 2 | stretch3(quant10(c.y)) << 1 | stretch3(quant10(c.z));
        ws.keys[f] = key;
        radix_count<kPasses>(key, h);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kPasses * kRadixBins; i += blockDim.x)
        if (h[i]) atomicAdd(&ws.radix.hist[i], h[i]);
}

// The sorted codes around a workgroup's nodes in LDS (most nodes span a few
// leaves, so nearly every probe of their searches lands there).
constexpr int kTreeThreads = 256;
constexpr int kWindow = 3 * kTreeThreads;  // from kTreeThreads before the first node on
struct Codes {
    const uint32_t* c;
    const uint32_t* window;
    int first, n;  // first: index of window[0]
    __device__ __forceinline__ uint32_t at(int j) const {
        const uint32_t w = (uint32_t)(j - first);
        return w < (uint32_t)kWindow ? window[w] : c[j];
    }
    __device__ __forceinline__ int delta(int i, int j) const {
        if (j > n - 1 || j < 0) return -1;
        const uint32_t a = at(i), b = at(j);
        if (a == b) return 32 + __clz((uint32_t)i ^ (uint32_t)j);
        return __clz(a ^ b);
    }
};
__device__ __forceinline__ int lid(int num) {
    if (num == 1) return 0;
    if (num % 2 == 1) return num / 2 + 1;
    return num / 2;
}

// Children and parents of the radix tree (Karras).  The nodes' bounds and the
// leaves follow in lbvh_aabbs.
__global__ __launch_bounds__(kTreeThreads) void lbvh_tree(uint32_t nf, LbvhWs ws, kr_bvh_node* nodes,
                                                          uint32_t* parents, uint32_t* mortons) {
    __shared__ uint32_t window[kWindow];
    const uint32_t t = blockIdx.x * kTreeThreads + threadIdx.x;
    const int n = (int)nf, i = (int)t;
    const int first = (int)(blockIdx.x * kTreeThreads) - kTreeThreads;
    for (int w = (int)threadIdx.x; w < kWindow; w += kTreeThreads) {
        const int j = first + w;
        window[w] = j >= 0 && j < n ? ws.keys[j] : 0u;
    }
    __syncthreads();
    if (t >= nf) return;
    const uint32_t I = nf - 1;
    if (mortons) mortons[t] = window[kTreeThreads + threadIdx.x];
    if (t == 0) parents[0] = kInv;
    if (t >= I) return;
    const Codes c{ws.keys, window, first, n};
    const int da = c.delta(i, i + 1), db = c.delta(i, i - 1);
    const int d = (da - db > 0) - (da - db < 0);
    const int dmin = c.delta(i, i - d);
    int lmax = 2;
    while (c.delta(i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int s = lmax / 2; s >= 1; s /= 2)
        if (c.delta(i, i + (l + s) * d) > dmin) l += s;
    const int j = i + l * d;
    const int dnode = c.delta(i, j);
    int s = 0;
    for (int q = lid(l); q >= 1; q = lid(q))
        if (c.delta(i, i + (s + q) * d) > dnode) s += q;
    const int split = i + s * d + (d < 0 ? d : 0);
    const bool lleaf = ((i < j ? i : j) == split);
    const bool rleaf = ((i > j ? i : j) == split + 1);
    const uint32_t li = (uint32_t)split + (lleaf ? I : 0);
    const uint32_t ri = (uint32_t)split + 1 + (rleaf ? I : 0);
    parents[li] = t;
    parents[ri] = t;
    kr_bvh_node& N = nodes[t];
    N.u.children.left = li;
    N.u.children.right = ri;
    N.nPrimitives = 0;
    N.axis = 0;
    N.pad_ = 0;
}

// The bottom-up pass over the bounds; a leaf's come from its triangle, and its
// node is written here.
struct LbvhUp : BoundsUp {
    const kr_vec3* V;
    const kr_uvec4* F;
    const uint32_t* vals;
    uint32_t I;
    __device__ __forceinline__ BoundsPay leaf(uint32_t n) const {
        const uint32_t prim = vals[n - I];
        const Box b = tri_box(V, F[prim]);
        kr_bvh_node L;
        L.bounds.min = kr_vec3{b.mn.x, b.mn.y, b.mn.z};
        L.bounds.max = kr_vec3{b.mx.x, b.mx.y, b.mx.z};
        L.u.children.left = prim;
        L.u.children.right = 0;
        L.nPrimitives = 1;
        L.axis = 0;
        L.pad_ = 0;
        nodes[n] = L;
        BoundsPay r{b.mn, b.mx, 1u, 0.0f};
        r.cost = 1.0f * area(r.mn, r.mx);
        counts[n] = 1u;
        costs[n] = r.cost;
        return r;
    }
};

__global__ __launch_bounds__(kUpTile) void lbvh_aabbs(LbvhUp op, uint32_t nf, uint32_t* visit) {
    __shared__ UpTile<BoundsPay> L;
    bottom_up(nf, visit, L, op);
}

size_t lbvh_carve(LbvhWs* ws, void* base, size_t cap, uint32_t nf) {
    Carver c{(char*)base, 0, cap};
    ws->cbox = c.take<int32_t>(8);
    ws->visit = c.take<uint32_t>(nf);
    ws->keys = c.take<uint32_t>(nf);
    ws->vals = c.take<uint32_t>(nf);
    ws->keys_tmp = c.take<uint32_t>(nf);
    ws->vals_tmp = c.take<uint32_t>(nf);
    radix_carve(&ws->radix, c, nf, kPasses);
    return c.used;
}

kr_error lbvh_launch(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, kr_bvh_node* nodes, uint32_t* parents,
                     uint32_t* counts, float* costs, uint32_t* mortons, void* workspace, size_t ws_bytes,
                     hipStream_t stream, uint32_t polls) {
    if (nf == 0) return "obvh_lbvh_build: no faces";
    if (nf > kLbvhMaxFaces) return "obvh_lbvh_build: too many faces";
    LbvhWs ws;
    size_t need = lbvh_carve(&ws, workspace, ws_bytes, nf);
    if (!workspace || ws_bytes < need) return "obvh_lbvh_build: workspace too small";
    auto blocks = [](uint32_t n, uint32_t b) { return dim3((n + b - 1) / b); };
    uint32_t gb = (nf + 255) / 256;
    if (gb > 2048) gb = 2048;
    hipLaunchKernelGGL(lbvh_init, dim3(gb), dim3(256), 0, stream, V, nf, ws);
    hipLaunchKernelGGL(lbvh_centroid_box, dim3(min((nf + kBoxThreads - 1) / kBoxThreads, 256u)), dim3(kBoxThreads), 0,
                       stream, V, F, nf, ws);
    hipLaunchKernelGGL(lbvh_codes, dim3(min((nf + 1023) / 1024, 256u)), dim3(1024), 0, stream, V, F, nf, ws);
    radix_sort<kPasses>(ws.keys, ws.vals, ws.keys_tmp, ws.vals_tmp, nf, ws.radix, polls, stream);
    hipLaunchKernelGGL(lbvh_tree, blocks(nf, kTreeThreads), dim3(kTreeThreads), 0, stream, nf, ws, nodes, parents,
                       mortons);
    hipLaunchKernelGGL(lbvh_aabbs, up_grid(nf), dim3(kUpTile), 0, stream,
                       LbvhUp{{nodes, parents, counts, costs}, V, F, ws.vals, nf - 1}, nf, ws.visit);
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

}  // namespace obvh
