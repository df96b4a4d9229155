// atrbvh.hip -- ATRBVH builder on gfx950: 64-bit Morton LBVH followed by the
// agglomerative treelet optimiser (src/ads/atrbvh_gpu; the flow of
// atrbvh.cu:258-470).
//
//  atr_scene      scene box over the triangle boxes (atrbvh.cu:262-290)
//  atr_codes      63-bit Morton code of each triangle-box centre normalised
//                 by the scene box (LBVH.cu:9-93, Commons.cuh:422-430,602-645)
//  (sort)         stable radix sort of (code, face) over 63 bits (rocPRIM),
//                 the equivalent of cub::DeviceRadixSort (CubWrapper.cu:8-46)
//  atr_tree       Karras radix tree, duplicates split by 64 + clz(i ^ j)
//                 (LBVH.cu:156-302), and the leaves, as 64-byte working records
//  atr_treelets   one optimiser pass: bottom-up over the current tree; a node
//                 holding at least gamma triangles is optimised as a treelet
//                 root right after its subtree (AgglomerativeTreelet.cu:
//                 405-561, Treelet.cuh:55-127).  A half-wave (32 lanes) forms
//                 the treelet (largest-area expansion), takes the distances
//                 (union box areas), merges the closest pair ts-1 times and
//                 writes the new topology when its SAH is lower, choosing as
//                 the reference's 32-lane __shfl_down tournaments do, ties
//                 included; then it goes on with the parent.  The first pass
//                 also makes the working boxes and areas (LBVH.cu:551-665).
//  atr_export     nodes, parents and leaf bounds from the records
//  (final)        bounds / counts / costs bottom-up with kr_aabb_expand
//                 (atrbvh.cu:95-179).
// The optimiser passes use the phased arrival protocol of phased.hpp, the last
// pass that of bottomup.hpp.
// Working-box min/max order -0 below +0 (as fminf/fmaxf on the reference
// GPU); the final bounds use kr_min/kr_max like kr_aabb_expand.
#include <float.h>

#include <rocprim/device/device_radix_sort.hpp>

#include "atrbvh.hpp"
#include "bottomup.hpp"
#include "common.hpp"

namespace obvh {

constexpr uint32_t kNoNode = 0xFFFFFFFFu;

__device__ __forceinline__ float zmin(float a, float b) {
    return a < b ? a : (b < a ? b : (__builtin_signbit(a) ? a : b));
}
__device__ __forceinline__ float zmax(float a, float b) {
    return a > b ? a : (b > a ? b : (__builtin_signbit(a) ? b : a));
}
__device__ __forceinline__ f3 ldv3a(const kr_vec3* V, uint32_t i) {
    const kr_vec3 a = V[i];
    return f3{a.x, a.y, a.z};
}

// calculateBoundingBoxSurfaceArea (Commons.cuh:96-103)
__device__ __forceinline__ float box_area3(float x, float y, float z) { return 2 * (x * y + x * z + y * z); }
__device__ __forceinline__ float box_area(float4 mn, float4 mx) {
    return box_area3(mx.x - mn.x, mx.y - mn.y, mx.z - mn.z);
}
// calculateLeafBoundingBox (LBVH.cu:414-430)
__device__ __forceinline__ void tri_box(const kr_vec3* V, const kr_uvec4 f, float4& mn, float4& mx) {
    const f3 a = ldv3a(V, f.x), b = ldv3a(V, f.y), c = ldv3a(V, f.z);
    mn = make_float4(zmin(zmin(a.x, b.x), c.x), zmin(zmin(a.y, b.y), c.y), zmin(zmin(a.z, b.z), c.z), 0.0f);
    mx = make_float4(zmax(zmax(a.x, b.x), c.x), zmax(zmax(a.y, b.y), c.y), zmax(zmax(a.z, b.z), c.z), 0.0f);
}

// expandBits64 (Commons.cuh:602-613)
__device__ __forceinline__ uint64_t expand_bits64(uint64_t v) {
    v &= 0x1fffffu;
    v = (v | v << 32) & 0x1f00000000ffffull;
    v = (v | v << 16) & 0x1f0000ff0000ffull;
    v = (v | v << 8) & 0x100f00f00f00f00full;
    v = (v | v << 4) & 0x10c30c30c30c30c3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}
__device__ __forceinline__ uint64_t discretize21(float x) {
    return (uint64_t)fminf(fmaxf(x * 2097152.0f, 0.0f), 2097151.0f);  // NaN -> 0
}

// ----------------------------------------------------------- build --

__device__ __forceinline__ void pass_clear(const AtrWs& ws, uint32_t nf) {
    phase_clear(ws.ph, nf);
    if (blockIdx.x == 0 && threadIdx.x < 64) ws.top[threadIdx.x] = 0;
}
__global__ void atr_init(AtrWs ws, uint32_t nf) {
    pass_clear(ws, nf);
    if (blockIdx.x == 0 && threadIdx.x < 6) ws.sbox[threadIdx.x] = threadIdx.x < 3 ? 0x7FFFFFFF : (int32_t)0x80000000;
}

constexpr int kBoxThreads = 1024;

__global__ __launch_bounds__(kBoxThreads) void atr_scene(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, AtrWs ws) {
    int32_t mn[3] = {0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF}, mx[3] = {(int32_t)0x80000000, (int32_t)0x80000000,
                                                                   (int32_t)0x80000000};
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < nf; f += gridDim.x * blockDim.x) {
        const kr_uvec4 face = F[f];
        const uint32_t vid[3] = {face.x, face.y, face.z};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const f3 p = ldv3a(V, vid[j]);
            const int32_t k[3] = {f2ord(p.x), f2ord(p.y), f2ord(p.z)};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                mn[a] = min(mn[a], k[a]);
                mx[a] = max(mx[a], k[a]);
            }
        }
    }
    // wave, then workgroup reduction; one filtered atomic per key and
    // workgroup (a few thousand same-address atomics would serialise)
    __shared__ int32_t part[kBoxThreads / kWave][6];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        mn[a] = wave_min_i32(mn[a]);
        mx[a] = wave_max_i32(mx[a]);
    }
    if (lane_id() == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            part[wave_id()][a] = mn[a];
            part[wave_id()][3 + a] = mx[a];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        int32_t v = part[0][a];
        for (int w = 1; w < kBoxThreads / kWave; ++w) v = a < 3 ? min(v, part[w][a]) : max(v, part[w][a]);
        const int32_t cur = __hip_atomic_load(&ws.sbox[a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (a < 3 ? v < cur : v > cur) {
            if (a < 3) atomicMin(&ws.sbox[a], v);
            else atomicMax(&ws.sbox[a], v);
        }
    }
}

__global__ void atr_codes(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, AtrWs ws) {
    const uint32_t f = blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    float4 mn, mx;
    tri_box(V, F[f], mn, mx);
    const float smn[3] = {ord2f(ws.sbox[0]), ord2f(ws.sbox[1]), ord2f(ws.sbox[2])};
    const float smx[3] = {ord2f(ws.sbox[3]), ord2f(ws.sbox[4]), ord2f(ws.sbox[5])};
    const float cmn[3] = {mn.x, mn.y, mn.z}, cmx[3] = {mx.x, mx.y, mx.z};
    uint64_t d[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float c = (cmx[a] + cmn[a]) * 0.5f;
        d[a] = expand_bits64(discretize21((c - smn[a]) / (smx[a] - smn[a])));
    }
    ws.keys_in[f] = (d[0] << 2) | (d[1] << 1) | d[2];
    ws.vals_in[f] = f;
}

// longestCommonPrefix (LBVH.cu:173-187), the sorted codes around a
// workgroup's nodes in LDS (most nodes span a few leaves).
constexpr int kTreeThreads = 256;
constexpr int kWindow = 3 * kTreeThreads;  // from kTreeThreads before the first node on
struct Codes64 {
    const uint64_t* k;
    const uint64_t* window;
    int first, n;  // first: index of window[0]
    __device__ __forceinline__ uint64_t at(int j) const {
        const uint32_t w = (uint32_t)(j - first);
        return w < (uint32_t)kWindow ? window[w] : k[j];
    }
    __device__ __forceinline__ int lcp(int i, int j, uint64_t ki) const {
        if (j < 0 || j >= n) return -1;
        const uint64_t kj = at(j);
        if (ki == kj) return 64 + __clz(i ^ j);
        return __clzll((long long)(ki ^ kj));
    }
};

// Working record of a node, four float4 (64 B, half a cache line, so that one
// trip to memory brings everything a treelet reads of a node):
//   [0] box min, surface area        [1] box max, SAH cost of the subtree
//   [2] left, right, parent, 0       (a leaf: face id, 0, parent, 0)
//   [3] first and last leaf position, triangles below, 0
// The box has fminf/fmaxf semantics with -0 below +0.  `nodes` and `parents`
// are written from the records once, after the optimiser (atr_export).
struct AtrRec {
    float4* r;
    __device__ __forceinline__ explicit AtrRec(const AtrWs& ws, uint32_t node) : r(ws.rec + 4 * (size_t)node) {}
    __device__ __forceinline__ uint4 topo() const { return *reinterpret_cast<const uint4*>(r + 2); }
    __device__ __forceinline__ uint4 span() const { return *reinterpret_cast<const uint4*>(r + 3); }
    __device__ __forceinline__ void set_sah(float v) const { reinterpret_cast<float*>(r + 1)[3] = v; }
    __device__ __forceinline__ void set_kids(uint32_t l, uint32_t rr) const {
        *reinterpret_cast<uint2*>(r + 2) = make_uint2(l, rr);
    }
    __device__ __forceinline__ void set_parent(uint32_t p) const { reinterpret_cast<uint32_t*>(r + 2)[2] = p; }
    __device__ __forceinline__ void set_span(uint32_t lo, uint32_t hi, uint32_t tri) const {
        *reinterpret_cast<uint4*>(r + 3) = make_uint4(lo, hi, tri, 0u);
    }
};

__global__ __launch_bounds__(kTreeThreads) void atr_tree(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, float ct,
                                                         AtrWs ws) {
    __shared__ uint64_t window[kWindow];
    const int i = (int)(blockIdx.x * kTreeThreads + threadIdx.x);
    const int n = (int)nf;
    const uint32_t I = nf - 1;
    const int first = (int)(blockIdx.x * kTreeThreads) - kTreeThreads;
    for (int w = (int)threadIdx.x; w < kWindow; w += kTreeThreads) {
        const int j = first + w;
        window[w] = j >= 0 && j < n ? ws.keys_out[j] : 0ull;
    }
    __syncthreads();
    if (i >= n) return;
    {  // leaf i in code order
        const uint32_t face = ws.vals_out[i];
        const AtrRec L(ws, I + (uint32_t)i);
        float4 mn, mx;
        tri_box(V, F[face], mn, mx);
        mn.w = box_area(mn, mx);
        mx.w = ct * mn.w;
        L.r[0] = mn;
        L.r[1] = mx;
        L.set_kids(face, 0u);
        L.set_span((uint32_t)i, (uint32_t)i, 1u);
    }
    if (i == 0) AtrRec(ws, 0u).set_parent(kNoNode);  // the root (or the only leaf)
    if (i >= n - 1) return;
    const Codes64 k{ws.keys_out, window, first, n};
    const uint64_t ki = window[kTreeThreads + threadIdx.x];
    const int l1 = k.lcp(i, i + 1, ki), l2 = k.lcp(i, i - 1, ki);
    const int dir = (0 < l1 - l2) - (l1 - l2 < 0);
    const int min_lcp = k.lcp(i, i - dir, ki);
    int lmax = 2;
    while (k.lcp(i, i + lmax * dir, ki) > min_lcp) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (k.lcp(i, i + (l + t) * dir, ki) > min_lcp) l += t;
    const int j = i + l * dir;
    const int node_lcp = k.lcp(i, j, ki);
    int s = 0, divisor = 2;
    const int max_div = 1 << (32 - __clz(l));
    while (divisor <= max_div) {
        const int t = (l + divisor - 1) / divisor;
        if (k.lcp(i, i + (s + t) * dir, ki) > node_lcp) s += t;
        divisor <<= 1;
    }
    const int split = i + s * dir + min(dir, 0);
    const uint32_t li = (uint32_t)split + (min(i, j) == split ? I : 0u);
    const uint32_t ri = (uint32_t)split + 1 + (max(i, j) == split + 1 ? I : 0u);
    AtrRec(ws, (uint32_t)i).set_kids(li, ri);
    AtrRec(ws, li).set_parent((uint32_t)i);
    AtrRec(ws, ri).set_parent((uint32_t)i);
}

__global__ void atr_clear(AtrWs ws, uint32_t nf) { pass_clear(ws, nf); }

// ------------------------------------------------------- optimiser --
//
// A treelet is a chain of dependent steps (find the largest leaf, read its
// children, again; find the closest pair, merge, again), so a pass is bound
// by latency: tree levels x time per treelet (a 200 K-triangle hairball has
// 24 levels of treelet roots).  Hence
//  - one half-wave (32 lanes, as the reference's warps) per treelet and per
//    path to the root: the lanes climb alone below the first treelet roots,
//    which go to a ready list; the half-waves of the workgroup then take
//    roots from it and each follows its path upwards.  (Running the treelets
//    on the wave whose lane completed the node put a phase's few roots,
//    neighbours in the deferred list, on one wave, two at a time.  A whole
//    wave per treelet makes one 10 % faster but halves their number in
//    flight: 1.75 against 1.65 ms for the build and transform below);
//  - one 64-byte record per node and the top four levels of a treelet's
//    subtree read level by level: four trips to memory instead of two per
//    expansion;
//  - tournaments as integer DPP minima and a ballot instead of shuffle
//    rounds, boxes in LDS, distances in registers.
// 200 K-triangle hairball, treelet size 9, 2 passes: 5529 -> 790 us (930 with
// the top in two launches of 8192-leaf workgroups and one workgroup); a treelet
// takes about 20 K cycles (5 K reading, 4 K forming, 10 K merging).

// The top pass (everything above the chunks) runs on one XCD, whose L2 all its
// CUs share: a half-wave that completes a node waits until its records are in
// the L2, counts its arrival, and the one that arrives second drops its CU's L1
// and goes on with the parent.  So what were two launches' longest paths one
// after the other is one path (300 and 340 us a pass of a 200 K hairball with
// 8192-leaf workgroups and one for the rest, 255 and 260 now), and reads stay L2 hits (past the L2, for all XCDs, a trip takes twice as
// long, four of them a treelet).  The grid covers every CU of the chip; the
// first workgroup to arrive names the XCD, those of the others end.  Any one
// workgroup would do all the work.  Builds at the same time tend to share an
// XCD: one 200 K hairball takes 945 us, 2 and 4 on as many streams 1105 and 1458
// (5674, 5765 and 6032 us in phases of single workgroups).
constexpr int kXccId = 20 | (4 - 1) << 11;  // s_getreg: XCC_ID, 4 bits
constexpr int kTopNext = 32;  // of ws.top: entries taken ([0]: the XCD, plus one); a cache line of its own
constexpr int kTopThreads = 512;      // 16 half-waves per CU (8 take the same time)
constexpr uint32_t kTopBlocks = 256;  // a workgroup per CU of every XCD
// From this many leaves on, 8192-leaf workgroups on all XCDs come between: the
// roots are then more than one XCD's 512 half-waves are quick with.  Builds of
// icospheres and hairballs, 2 passes, without / with them, treelet size 7: 68 K
// 611-637 / 780-803 us, 180 K 834-843 / 900-919, 220 K 923-930 / 945-978, 260 K
// 991-997 / 974-996, 300 K 1231-1241 / 1119-1156, 340 K 1304 / 1152-1207; size 9:
// 220 K 1019-1045 / 1089-1138, 260 K 1077 / 1104-1148, 300 K 1322-1345 /
// 1259-1316, 340 K 1406-1417 / 1282-1357.  400 K hairball 1442 / 1255, 1 M 2848 /
// 1850, 2 M 5290 / 2950 (with 4096 leaves 2 M 3295 and 338 K 1125, with 16384
// 2922 and 1194).
constexpr uint32_t kTopLeaves = 1u << 18;

constexpr int kDistStride = kMaxTreelet + 1;  // odd: the lanes of a row update touch different banks

struct TreeletLds {
    float4 box[kMaxTreelet][2];  // treelet leaf: min, SAH; max, node id
    uint2 kids[kMaxTreelet];     // its children; after its merge step, those of the node the step made
    float area[kMaxTreelet];
    float dist[kMaxTreelet * kDistStride];  // union areas, [row][column], row > column
};

constexpr int kHalf = 32;
constexpr int kHeapLevels = 4;  // levels below a treelet root loaded at once
constexpr int kHeapNodes = (2 << kHeapLevels) - 2;
constexpr int kPairSteps = (kMaxTreelet * (kMaxTreelet - 1) / 2 + kHalf - 1) / kHalf;  // distance entries per lane

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// LOWER_TRM_ROW / LOWER_TRM_COL (TriangularMatrix.cuh:37-52)
__device__ __forceinline__ int trm_row(int index) { return (int)((-1 + sqrtf(8.0f * index + 1)) / 2) + 1; }
__device__ __forceinline__ int trm_index(int row, int col) { return ((row - 1) * row) / 2 + col; }

// Lane a of the lower half's value in the lower half, lane b of the upper
// half's in the upper half (a, b uniform, within the half).
__device__ __forceinline__ uint32_t half_pick(uint32_t v, int a, int b, bool upper) {
    const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)v, a);
    const uint32_t y = (uint32_t)__builtin_amdgcn_readlane((int)v, kHalf + b);
    return upper ? y : x;
}
__device__ __forceinline__ float half_pickf(float v, int a, int b, bool upper) {
    return __uint_as_float(half_pick(__float_as_uint(v), a, b, upper));
}
// Integer min / max over each half (every lane active).
template <bool MIN>
__device__ __forceinline__ int32_t half_reduce(int32_t v, bool upper) {
    auto f = [](int32_t a, int32_t b) { return MIN ? min(a, b) : max(a, b); };
    v = f(v, dpp_mov<0xB1>(v));
    v = f(v, dpp_mov<0x4E>(v));
    v = f(v, dpp_mov<0x141>(v));
    v = f(v, dpp_mov<0x140>(v));
    const int32_t a = f(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16));
    const int32_t b = f(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48));
    return upper ? b : a;
}
// The other lane of a pair (lane ^ 1).
__device__ __forceinline__ float dpp_xor1(float v) {
    const int i = __float_as_int(v);
    return __int_as_float(dpp_mov<0xB1>(i));
}
__device__ __forceinline__ uint32_t dpp_xor1(uint32_t v) {
    return (uint32_t)dpp_mov<0xB1>((int)v);
}

// Box min / max.  v_min_f32 and v_max_f32 order -0 below +0 and so equal zmin
// and zmax on values that are not NaN; kSane says that they are not.
template <bool kSane>
__device__ __forceinline__ float bmin(float a, float b) {
    if (!kSane) return zmin(a, b);
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
template <bool kSane>
__device__ __forceinline__ float bmax(float a, float b) {
    if (!kSane) return zmax(a, b);
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// calculateBoundingBoxAndSurfaceArea (Commons.cuh:173-181)
template <bool kSane>
__device__ __forceinline__ float join_area(float4 amn, float4 amx, float4 bmn, float4 bmx) {
    return box_area3(bmax<kSane>(amx.x, bmx.x) - bmin<kSane>(amn.x, bmn.x),
                     bmax<kSane>(amx.y, bmx.y) - bmin<kSane>(amn.y, bmn.y),
                     bmax<kSane>(amx.z, bmx.z) - bmin<kSane>(amn.z, bmn.z));
}

// The ts - 1 merges of the closest pair (AgglomerativeTreelet.cu:80-222) over
// the treelet leaves in S, one treelet per half of the wave.  The step at
// `last` leaves in slot `last` the node it makes: box, SAH and children (its
// id is tin[last - 1]).  Returns the SAH of the whole treelet.
//
// The closest-pair search of a half is the reference's 32-lane strided scan
// and __shfl_down tournament: among equal distances the lane (entry mod 32)
// whose bit-reversed number is lowest wins, and within a lane the lowest
// entry.  Lane hl plays the reference's lane rev(hl) (`logical`), so the winner
// is the lowest set bit of a ballot.
//
// kSane: every box coordinate is below 2^61 in magnitude, so distances are
// finite and not negative (their bits order as integers) and the union is
// symmetric: each lane keeps its entries' distances in registers and makes
// those that a merge touches again from the boxes.  A wave alone on its SIMD
// issues this chain at about 5 cycles an instruction, so its length is its
// time (1400 cycles per merge while the matrix was moved through LDS, as the
// general form still does).
template <bool kSane>
__device__ __forceinline__ float treelet_merge(TreeletLds& S, int ts, float ci, int hl, int logical, bool upper,
                                               uint32_t tin, const uint32_t (&pair_rc)[kPairSteps]) {
    const int npairs = ts * (ts - 1) / 2;
    float dist[kPairSteps];
    auto entry = [&](int k) { return (int)(pair_rc[k] >> 8) * kDistStride + (int)(pair_rc[k] & 255u); };
    auto measure = [&](int k) {
        const int r = (int)(pair_rc[k] >> 8), c = (int)(pair_rc[k] & 255u);
        return join_area<kSane>(S.box[r][0], S.box[r][1], S.box[c][0], S.box[c][1]);
    };
#pragma unroll
    for (int k = 0; k < kPairSteps; ++k) {
        if (kHalf * k >= npairs) break;
        dist[k] = measure(k);
        if (!kSane && logical + kHalf * k < npairs) S.dist[entry(k)] = dist[k];
    }
    wave_sync();
    float total = 0.0f;
    for (int last = ts - 1; last > 0; --last) {
        const int size = last * (1 + last) / 2;
        // findMinimumDistance
        float moved = 0.0f;
        if (!kSane) moved = S.dist[last * kDistStride + min(hl, kMaxTreelet)];
        int32_t key = 0x7F7FFFFF;  // FLT_MAX
        uint32_t rc = 1u << 8;     // entry 0
#pragma unroll
        for (int k = 0; k < kPairSteps; ++k) {
            if (kHalf * k >= size) break;
            const float d = kSane ? dist[k] : S.dist[entry(k)];
            const int32_t kk = kSane ? __float_as_int(d) : f2ord(d + 0.0f);
            if (logical + kHalf * k < size && (kSane || d < FLT_MAX) && kk < key) { key = kk; rc = pair_rc[k]; }
        }
        const int32_t best = half_reduce<true>(key, upper);
        const uint64_t eq = __ballot(key == best);
        rc = half_pick(rc, __builtin_ctz((uint32_t)eq), __builtin_ctz((uint32_t)(eq >> 32)), upper);
        const int row = (int)(rc >> 8), col = (int)(rc & 255u);
        // updateState
        const float4 r0 = S.box[row][0], r1 = S.box[row][1], c0 = S.box[col][0], c1 = S.box[col][1];
        const float4 l0 = S.box[last][0], l1 = S.box[last][1];
        const float4 nmn = make_float4(bmin<kSane>(c0.x, r0.x), bmin<kSane>(c0.y, r0.y), bmin<kSane>(c0.z, r0.z), 0.0f);
        const float4 nmx = make_float4(bmax<kSane>(c1.x, r1.x), bmax<kSane>(c1.y, r1.y), bmax<kSane>(c1.z, r1.z), 0.0f);
        total = (r0.w + c0.w) + ci * box_area(nmn, nmx);
        const uint32_t made = half_pick(tin, last - 1, last - 1, upper);
        wave_sync();
        if (hl == row) {  // the last slot moves to the pair's free slot
            S.box[row][0] = l0;
            S.box[row][1] = l1;
        }
        if (hl == col || hl == last) {
            S.box[hl][0] = make_float4(nmn.x, nmn.y, nmn.z, total);
            S.box[hl][1] = make_float4(nmx.x, nmx.y, nmx.z, __uint_as_float(made));
        }
        if (hl == last) S.kids[last] = make_uint2(__float_as_uint(r1.w), __float_as_uint(c1.w));
        wave_sync();
        // updateDistancesMatrix
        if (kSane) {
#pragma unroll
            for (int k = 0; k < kPairSteps; ++k) {
                if (kHalf * k >= size - last) break;  // the entries of the next step
                const int r = (int)(pair_rc[k] >> 8), c = (int)(pair_rc[k] & 255u);
                const float d = measure(k);
                if (r == row || r == col || c == row || c == col) dist[k] = d;
            }
        } else if (hl < last) {
            if (hl != row) S.dist[max(row, hl) * kDistStride + min(row, hl)] = moved;
            wave_sync();
            const int a = max(col, hl), b = min(col, hl);
            if (hl != col)
                S.dist[a * kDistStride + b] = join_area<false>(S.box[a][0], S.box[a][1], S.box[b][0], S.box[b][1]);
        }
        wave_sync();
    }
    return total;
}

// One optimiser pass, one phase of the bottom-up protocol (phased.hpp).
// kFirst: the pass also makes the internal nodes' working boxes.  kTop: the top
// pass (chunk is nf), with small nodes on the same paths as the treelet roots.
template <bool kFirst, int kThreads, bool kTop>
__global__ __launch_bounds__(kThreads) void atr_treelets(AtrWs ws, uint32_t nf, int ts, int gamma, float ci,
                                                     uint32_t phase, uint32_t chunk) {
    __shared__ TreeletLds lds[kThreads / kHalf];
    __shared__ uint32_t nready, nextready;
    const uint32_t I = nf - 1;
    if (kTop) {  // the first workgroup's XCD takes all; the others' end here
        __shared__ bool join;
        if (threadIdx.x == 0) {
            const uint32_t xcd = __builtin_amdgcn_s_getreg(kXccId) + 1u;
            const uint32_t old = atomicCAS(&ws.top[0], 0u, xcd);
            join = old == 0u || old == xcd;
        }
        __syncthreads();
        if (!join) return;
    }
    const uint32_t tag = (phase << 24) | (kTop ? 1u : blockIdx.x + 1u);
    const uint64_t lo = (uint64_t)blockIdx.x * chunk, hi = lo + chunk;
    const uint32_t nin = phase == 0 ? 0 : min(ws.ph.nlist[phase - 1], I);
    const uint2* in = phase == 0 ? nullptr : ws.ph.list + (size_t)(phase - 1) * (I + 1);
    uint2* out = ws.ph.list + (size_t)phase * (I + 1);
    // The roots this workgroup takes have disjoint leaf spans inside its
    // chunk, so there are at most `chunk` of them.
    uint32_t* ready = ws.ready + lo;
    if (threadIdx.x == 0) nready = nextready = 0;
    if (!kTop) __syncthreads();
    auto defer = [&](uint32_t node, uint32_t key) {
        const uint32_t slot = atomicAdd(&ws.ph.nlist[phase], 1u);
        if (slot < I) out[slot] = make_uint2(node, key);
    };

    // Below the treelet roots: one lane per leaf (or deferred node).
    const uint32_t nstart = kTop ? 0 : phase == 0 ? chunk : nin;
    for (uint32_t r0 = threadIdx.x; r0 < nstart; r0 += blockDim.x) {
        uint32_t p;          // the node to complete next
        bool both = false;   // its children are known to be complete
        uint32_t key;        // a leaf position below it
        if (phase == 0) {
            const uint64_t pos = lo + r0;
            if (pos >= nf) break;
            key = (uint32_t)pos;
            p = AtrRec(ws, I + key).topo().z;
        } else {
            // Ownership comes from the listed key only: once its owner has
            // completed the node and an ancestor, a treelet there may rewire
            // the node's children while other workgroups still scan this
            // list.
            const uint2 e = in[r0];
            p = e.x;
            key = e.y;
            if (p >= I || key < lo || key >= hi) continue;
            const uint4 t = AtrRec(ws, p).topo();
            const uint4 sl = AtrRec(ws, t.x).span(), sr = AtrRec(ws, t.y).span();
            if (min(sl.x, sr.x) < lo || max(sl.y, sr.y) >= hi) {  // wider than this workgroup: next phase
                defer(p, min(sl.x, sr.x));
                continue;
            }
            both = true;
        }
        for (uint32_t step = 0; p < I && step < nf; ++step) {
            const AtrRec P(ws, p);
            const uint4 t = P.topo();
            if (!both) {
                const uint64_t old = __hip_atomic_fetch_add(&ws.ph.visit[p], ((uint64_t)tag << 32) | 1ull,
                                                            __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
                const uint32_t t1 = (uint32_t)(old >> 32);
                if ((uint32_t)old == 0) break;  // first arrival: the sibling continues
                if (t1 != tag && (t1 >> 24) >= phase) {
                    defer(p, key);
                    break;
                }
            }
            both = false;
            const AtrRec L(ws, t.x), R(ws, t.y);
            const uint4 sl = L.span(), sr = R.span();
            const uint32_t tri = sl.z + sr.z;
            if ((int32_t)tri >= gamma) {
                const uint32_t slot = atomicAdd(&nready, 1u);
                if (slot < chunk && lo + slot < nf) ready[slot] = p;  // always (the roots' spans are disjoint)
                break;
            }
            const float4 lb = L.r[1], rb = R.r[1];
            float area;
            if (kFirst) {
                const float4 la = L.r[0], ra = R.r[0];
                float4 mn = make_float4(zmin(la.x, ra.x), zmin(la.y, ra.y), zmin(la.z, ra.z), 0.0f);
                float4 mx = make_float4(zmax(lb.x, rb.x), zmax(lb.y, rb.y), zmax(lb.z, rb.z), 0.0f);
                area = box_area(mn, mx);
                mn.w = area;
                mx.w = ci * area + lb.w + rb.w;
                P.r[0] = mn;
                P.r[1] = mx;
            } else {
                area = P.r[0].w;
                P.set_sah(ci * area + lb.w + rb.w);
            }
            P.set_span(min(sl.x, sr.x), max(sl.y, sr.y), tri);
            p = t.z;
        }
    }
    __syncthreads();

    // The treelets: each half-wave takes a ready root and follows its path
    // up to the first arrival at a node, a deferred node or the tree's root.
    const bool upper = lane_id() >= kHalf;
    const int hl = lane_id() & (kHalf - 1);
    TreeletLds& S = lds[2 * wave_id() + (upper ? 1 : 0)];
    const int logical = (int)(__brev((uint32_t)hl) >> 27);
    uint32_t pair_rc[kPairSteps];  // row << 8 | column of distance entry logical + 32 k
#pragma unroll
    for (int k = 0; k < kPairSteps; ++k) {
        const int e = min(logical + kHalf * k, kMaxTreelet * (kMaxTreelet - 1) / 2 - 1), r = trm_row(e);
        pair_rc[k] = (uint32_t)(r << 8 | (e - trm_index(r, 0)));
    }
    const uint32_t nroots = kTop ? nin : (uint32_t)min((uint64_t)min(nready, chunk), (uint64_t)nf - lo);
    bool have = false;
    uint32_t root = 0, steps = 0;
    uint4 rt = make_uint4(0u, 0u, kNoNode, 0u);  // the root's left, right, parent
    for (;;) {
        {  // idle halves take the next ready root
            const uint64_t idle = __ballot(!have && hl == 0);
            if (idle) {
                uint32_t slot = 0;
                if (!have && hl == 0)
                    slot = kTop ? __hip_atomic_fetch_add(&ws.top[kTopNext], 1u, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP)
                                : atomicAdd(&nextready, 1u);
                slot = half_pick(slot, 0, 0, upper);
                if (!have && slot < nroots) {
                    root = kTop ? in[slot].x : ready[slot];
                    have = root < I;
                    if (have) rt = AtrRec(ws, root).topo();
                    steps = 0;
                }
            }
            if (__ballot(have) == 0) break;
            if (kTop) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // what the XCD's other CUs wrote
        }
        const AtrRec X(ws, root);
        const uint32_t parent = rt.z;
        uint4 pt = make_uint4(0u, 0u, kNoNode, 0u);  // the parent's topology, needed after the treelet
        if (have && parent < I) pt = AtrRec(ws, parent).topo();

        // The top four levels of the subtree, one node per lane (the children
        // of lane x's node on lanes 2x + 2 and 2x + 3): four trips to memory
        // instead of one per expansion.
        uint32_t id = hl == 0 ? rt.x : rt.y, lkid = 0, rkid = 0, tin = root;
        float4 mn = make_float4(0, 0, 0, 0), mx = mn;
        uint4 sp = make_uint4(0u, 0u, 0u, 0u);
        float4 xmn = mn, xmx = mn;
        bool loaded = have && hl < 2;
        if (loaded) {
            const AtrRec C(ws, id);
            mn = C.r[0];
            mx = C.r[1];
            const uint4 t = C.topo();
            lkid = t.x;
            rkid = t.y;
            sp = C.span();
            if (!kFirst && hl == 0) {
                xmn = X.r[0];
                xmx = X.r[1];
            }
        }
#pragma unroll
        for (int level = 1; level < kHeapLevels; ++level) {
            const int first = (2 << level) - 2;  // lanes [first, 2 first + 2)
            const int up = (hl - 2) >> 1;
            const uint32_t pid = (uint32_t)__shfl((int)id, up, kHalf);
            const uint32_t pl = (uint32_t)__shfl((int)lkid, up, kHalf), pr = (uint32_t)__shfl((int)rkid, up, kHalf);
            const bool pok = __shfl((int)loaded, up, kHalf) != 0;
            if (hl >= first && hl < 2 * first + 2 && pok && pid < I) {
                id = (hl & 1) ? pr : pl;
                loaded = true;
                const AtrRec C(ws, id);
                mn = C.r[0];
                mx = C.r[1];
                const uint4 t = C.topo();
                lkid = t.x;
                rkid = t.y;
            }
        }
        // the root's own box, SAH, triangles and span (lane 0 of the half)
        const uint32_t tri = sp.z + dpp_xor1(sp.z);
        const uint32_t slo = min(sp.x, dpp_xor1(sp.x)), shi = max(sp.y, dpp_xor1(sp.y));
        if (kFirst) {
            xmn = make_float4(zmin(mn.x, dpp_xor1(mn.x)), zmin(mn.y, dpp_xor1(mn.y)), zmin(mn.z, dpp_xor1(mn.z)), 0.0f);
            xmx = make_float4(zmax(mx.x, dpp_xor1(mx.x)), zmax(mx.y, dpp_xor1(mx.y)), zmax(mx.z, dpp_xor1(mx.z)), 0.0f);
            xmn.w = box_area(xmn, xmx);
        }
        xmx.w = ci * xmn.w + mx.w + dpp_xor1(mx.w);

        // (the top pass also gets nodes below gamma: no treelet)
        const bool work = have && (!kTop || (int32_t)half_pick(tri, 0, 0, upper) >= gamma);
        bool keep = false;
        if (!kTop || __ballot(work) != 0) {
            // formTreelet (Treelet.cuh:55-127): expand the treelet leaf with the
            // largest area ts - 2 times.  A single largest area among values that
            // compare is the reference's winner whatever its tournament order.
            // The loop stops early (for both halves) at a tie, an area that does
            // not compare, or a node whose children are below the loaded levels.
            int slot = hl < 2 ? hl : -1;  // treelet leaf index of this lane's node
            int it = 0;
            for (; it < ts - 2; ++it) {
                const bool inner = work && slot >= 0 && id < I;
                const int32_t key = inner && mn.w >= 0.0f ? __float_as_int(mn.w + 0.0f) + 1 : 0;
                const int32_t best = half_reduce<false>(key, upper);
                const uint64_t eq = __ballot(key == best && work);
                const uint32_t ea = (uint32_t)eq, eb = (uint32_t)(eq >> 32);
                constexpr uint32_t kLoaded = (1u << (kHeapNodes / 2 - 1)) - 1;  // lanes whose children are loaded
                if ((ea & (ea - 1)) != 0 || (eb & (eb - 1)) != 0 || ((ea | eb) & ~kLoaded) != 0 ||
                    __ballot(inner && !(mn.w >= 0.0f)) != 0)
                    break;  // wave-uniform
                const int ia = ea ? __builtin_ctz(ea) : 0, ib = eb ? __builtin_ctz(eb) : 0;
                const uint32_t rep = half_pick(id, ia, ib, upper);
                const int from = (int)half_pick((uint32_t)slot, ia, ib, upper);
                const int idx = upper ? ib : ia;
                if (hl == it + 1) tin = rep;
                if (hl == idx) slot = -1;
                if (hl == 2 * idx + 2) slot = from;
                if (hl == 2 * idx + 3) slot = it + 2;
            }
            // to leaf order: lane hl takes treelet leaf hl
            if (work && slot >= 0) {
                S.box[slot][0] = make_float4(mn.x, mn.y, mn.z, mx.w);
                S.box[slot][1] = make_float4(mx.x, mx.y, mx.z, __uint_as_float(id));
                S.kids[slot] = make_uint2(lkid, rkid);
                S.area[slot] = mn.w;
            }
            wave_sync();
            const int sl = min(hl, kMaxTreelet - 1);
            {
                const float4 b0 = S.box[sl][0], b1 = S.box[sl][1];
                mn = make_float4(b0.x, b0.y, b0.z, S.area[sl]);
                mx = make_float4(b1.x, b1.y, b1.z, b0.w);
                id = __float_as_uint(b1.w);
            }
            // the remaining expansions, by the reference's tournament where the
            // largest area is tied or does not compare
            if (it < ts - 2) {
                const uint2 kk = S.kids[sl];
                lkid = kk.x;
                rkid = kk.y;
                for (; it < ts - 2; ++it) {
                    int idx = -1;
                    float w = -FLT_MAX;
                    if (work && hl < 2 + it) {
                        idx = hl;
                        w = id >= I ? -FLT_MAX : mn.w;
                    }
                    for (int n = 2 + it, amount = n / 2; n > 1; n = (n + 1) / 2, amount = n / 2) {
                        const int oi = __shfl_down(idx, amount, kHalf);
                        const float ow = __shfl_down(w, amount, kHalf);
                        if (ow > w) { w = ow; idx = oi; }
                    }
                    const int ia = __builtin_amdgcn_readlane(idx, 0) & (kHalf - 1);
                    const int ib = __builtin_amdgcn_readlane(idx, kHalf) & (kHalf - 1);
                    const uint32_t rep = half_pick(id, ia, ib, upper);
                    const uint32_t l2 = half_pick(lkid, ia, ib, upper), r2 = half_pick(rkid, ia, ib, upper);
                    idx = upper ? ib : ia;
                    if (hl == it + 1) tin = rep;
                    if (work && (hl == idx || hl == it + 2)) {
                        id = hl == idx ? l2 : r2;
                        const AtrRec C(ws, id);
                        mn = C.r[0];
                        mx = C.r[1];
                        const uint4 t = C.topo();
                        lkid = t.x;
                        rkid = t.y;
                    }
                }
                wave_sync();
                if (hl < ts) {
                    S.box[hl][0] = make_float4(mn.x, mn.y, mn.z, mx.w);
                    S.box[hl][1] = make_float4(mx.x, mx.y, mx.z, __uint_as_float(id));
                }
                wave_sync();
            }

            const float big = fmaxf(fmaxf(fmaxf(fabsf(mn.x), fabsf(mn.y)), fmaxf(fabsf(mn.z), fabsf(mx.x))),
                                    fmaxf(fabsf(mx.y), fabsf(mx.z)));
            const bool sane = big < 0x1p61f && mn.x == mn.x && mn.y == mn.y && mn.z == mn.z && mx.x == mx.x &&
                              mx.y == mx.y && mx.z == mx.z;
            float total;
            if (__ballot(work && hl < ts && !sane) == 0)
                total = treelet_merge<true>(S, ts, ci, hl, logical, upper, tin, pair_rc);
            else
                total = treelet_merge<false>(S, ts, ci, hl, logical, upper, tin, pair_rc);

            // updateTreelet: keep the new topology when its SAH is lower
            const uint64_t better = __ballot(work && hl == 0 && total < xmx.w);
            keep = ((better >> (upper ? kHalf : 0)) & 1ull) != 0;
        }
        const uint32_t v = (uint32_t)__shfl_up((int)tin, 1, kHalf);  // tin[hl - 1]
        if (have && hl == 0) {
            X.set_span(slo, shi, tri);
            if (!keep) {
                if (kFirst) X.r[0] = xmn;
                if (kFirst) X.r[1] = xmx;
                else X.set_sah(xmx.w);
            }
        }
        if (keep && hl >= 1 && hl < ts) {
            const float4 b0 = S.box[hl][0], b1 = S.box[hl][1];
            const uint2 kk = S.kids[hl];
            float4 nmn = make_float4(b0.x, b0.y, b0.z, 0.0f), nmx = make_float4(b1.x, b1.y, b1.z, b0.w);
            nmn.w = box_area(nmn, nmx);
            const AtrRec N(ws, v);
            N.r[0] = nmn;
            N.r[1] = nmx;
            N.set_kids(kk.x, kk.y);
            AtrRec(ws, kk.x).set_parent(v);
            AtrRec(ws, kk.y).set_parent(v);
        }

        // up to the parent
        if (kTop) drain();  // this half's records are in the XCD's L2
        bool arrive = have && parent < I && ++steps <= nf;
        uint64_t old = 0;
        if (arrive && hl == 0)
            old = __hip_atomic_fetch_add(&ws.ph.visit[parent], ((uint64_t)tag << 32) | 1ull, __ATOMIC_ACQ_REL,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
        const uint32_t count = half_pick((uint32_t)old, 0, 0, upper);
        const uint32_t t1 = half_pick((uint32_t)(old >> 32), 0, 0, upper);
        have = arrive && count != 0;  // else the sibling continues
        if (have && t1 != tag && (t1 >> 24) >= phase) {
            if (hl == 0) defer(parent, slo);
            have = false;
        }
        root = parent;
        rt = pt;
    }
}

// The tree from the records: topology, leaf bounds and faces (internal bounds
// follow bottom-up).
__global__ __launch_bounds__(256) void atr_export(AtrWs ws, uint32_t nf, kr_bvh_node* nodes, uint32_t* parents) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= 2 * nf - 1) return;
    const AtrRec R(ws, v);
    const uint4 t = R.topo();
    kr_bvh_node n = {};
    n.u.children.left = t.x;  // a leaf: the face id (primitivesOffset)
    n.u.children.right = t.y;
    if (v >= nf - 1) {
        const float4 mn = R.r[0], mx = R.r[1];
        n.bounds.min = kr_vec3{mn.x, mn.y, mn.z};
        n.bounds.max = kr_vec3{mx.x, mx.y, mx.z};
        n.nPrimitives = 1;
    }
    nodes[v] = n;
    parents[v] = t.z;
}

// Bounds / counts / costs of the final tree (atrbvh.cu:124-179: ct = 1.0,
// ci = 1.2, kr_aabb_expand), the same pass as the LBVH builder's.
__global__ __launch_bounds__(kUpTile) void atr_final(BoundsUp op, uint32_t nf, uint32_t* visit) {
    __shared__ UpTile<BoundsPay> L;
    bottom_up(nf, visit, L, op);
}

// ------------------------------------------------------------- host --

static size_t atr_sort_bytes(uint32_t nf) {
    size_t bytes = 0;
    rocprim::radix_sort_pairs((void*)nullptr, bytes, (uint64_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr,
                              (uint32_t*)nullptr, nf, 0, 63);
    return bytes;
}

size_t atr_carve(AtrWs* ws, void* base, size_t cap, uint32_t nf) {
    Carver c{(char*)base, 0, cap};
    const size_t total = nf ? 2 * (size_t)nf - 1 : 0;
    phase_carve(&ws->ph, c, nf);
    ws->sbox = c.take<int32_t>(8);
    ws->keys_in = c.take<uint64_t>(nf);
    ws->keys_out = c.take<uint64_t>(nf);
    ws->vals_in = c.take<uint32_t>(nf);
    ws->vals_out = c.take<uint32_t>(nf);
    ws->rec = c.take<float4>(4 * total);
    ws->ready = c.take<uint32_t>(nf);
    ws->top = c.take<uint32_t>(64);
    ws->sort_bytes = atr_sort_bytes(nf);
    ws->sort_tmp = c.take<char>(ws->sort_bytes);
    return c.used;
}

kr_error atr_launch(const kr_vec3* V, const kr_uvec4* F, uint32_t nf, int treelet_size, int iterations, float ci,
                    float ct, kr_bvh_node* nodes, uint32_t* parents, uint32_t* counts, float* costs, void* workspace,
                    size_t ws_bytes, hipStream_t stream) {
    if (nf == 0) return "obvh_atrbvh_build: no faces";
    if (treelet_size < 3 || treelet_size > kMaxTreelet) return "obvh_atrbvh_build: treelet size must be 3..20";
    if (iterations < 0) return "obvh_atrbvh_build: negative iteration count";
    AtrWs ws;
    const size_t need = atr_carve(&ws, workspace, ws_bytes, nf);
    if (!workspace || ws_bytes < need) return "obvh_atrbvh_build: workspace too small";
    auto blocks = [](uint32_t n, uint32_t b) { return dim3((n + b - 1) / b); };
    uint32_t gb = (nf + 255) / 256;
    if (gb > 2048) gb = 2048;
    hipLaunchKernelGGL(atr_init, dim3(gb), dim3(256), 0, stream, ws, nf);
    hipLaunchKernelGGL(atr_scene, dim3(min((nf + kBoxThreads - 1) / kBoxThreads, 256u)), dim3(kBoxThreads), 0, stream, V, F,
                       nf, ws);
    hipLaunchKernelGGL(atr_codes, blocks(nf, 256), dim3(256), 0, stream, V, F, nf, ws);
    size_t sb = ws.sort_bytes;
    OBVH_HIP_TRY(rocprim::radix_sort_pairs(ws.sort_tmp, sb, ws.keys_in, ws.keys_out, ws.vals_in, ws.vals_out, nf, 0,
                                           63, stream));
    hipLaunchKernelGGL(atr_tree, blocks(nf, kTreeThreads), dim3(kTreeThreads), 0, stream, V, F, nf, ct, ws);
    int gamma = treelet_size;
    for (int it = 0; it < iterations && nf > 1; ++it) {
        if (it > 0) hipLaunchKernelGGL(atr_clear, dim3(gb), dim3(256), 0, stream, ws, nf);
        // Phases of 512 leaves, 8192 (large meshes) and all.  Each costs its own
        // path of treelets.
        auto tile = it == 0 ? atr_treelets<true, 512, false> : atr_treelets<false, 512, false>;
        hipLaunchKernelGGL(tile, dim3((nf + 511) / 512), dim3(512), 0, stream, ws, nf, treelet_size, gamma, ci, 0u,
                           min(512u, nf));
        uint32_t phase = 1;
        if (nf > kTopLeaves) {
            auto mid = it == 0 ? atr_treelets<true, 1024, false> : atr_treelets<false, 1024, false>;
            hipLaunchKernelGGL(mid, dim3((nf + 8191) / 8192), dim3(1024), 0, stream, ws, nf, treelet_size, gamma, ci,
                               phase, 8192u);
            ++phase;
        }
        if (nf > 512) {
            auto top = it == 0 ? atr_treelets<true, kTopThreads, true> : atr_treelets<false, kTopThreads, true>;
            hipLaunchKernelGGL(top, dim3(kTopBlocks), dim3(kTopThreads), 0, stream, ws, nf, treelet_size, gamma, ci,
                               phase, nf);
        }
        gamma *= 2;
    }
    hipLaunchKernelGGL(atr_export, blocks(2 * nf - 1, 256), dim3(256), 0, stream, ws, nf, nodes, parents);
    hipLaunchKernelGGL(atr_clear, dim3(gb), dim3(256), 0, stream, ws, nf);
    hipLaunchKernelGGL(atr_final, up_grid(nf), dim3(kUpTile), 0, stream, BoundsUp{nodes, parents, counts, costs}, nf,
                       reinterpret_cast<uint32_t*>(ws.ph.visit));
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

}  // namespace obvh
