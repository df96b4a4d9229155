// dito.hip -- DiTO-14 oriented bounding boxes of point sets on gfx950.
//
// Method: Larsson & Kallberg DiTO-14 exactly as the reference CPU code
// computes it (src/common/algorithm/dito/dito.cpp:478-538), plus the 0.001
// extent floor of kr_points_obb (src/common/geometry.cpp:249).  The GPU
// driver of the reference (dito.cu:614-744: four synchronised launches,
// float CAS atomics per point, last-writer index selection) is replaced by:
//
//  setup     one workgroup scans the set sizes into a tile table (a set is
//            cut into tiles of `tile` points) and writes the result of empty
//            sets; a grid kernel fills tile -> set.
//  pass 1    workgroups (4 x wave64) take tiles in grid-stride order (one
//            tile per workgroup by default), form the 7 slab projections of
//            every point and keep per slab side the extreme and the point that
//            reached it first; equal to the reference's sequential
//            strict-compare scan.  Output: 14 (value, index) pairs per tile.
//  cand      one wave per set reduces its tile partials, then runs the
//            candidate search (base triangle + ditetrahedron, up to 21 axis
//            triples) over a 14-entry point array held in registers: every
//            lane computes the common prefix, 21 lanes evaluate one axis
//            triple each, and a (quality, id) minimum picks the winner.
//  pass 2    the same tiles project every point on the 3 chosen axes (fused
//            min/max of 3 dot products), 6 floats per tile.
//  final     one wave per set reduces and finalises the box.
//
// No atomics or cross-workgroup fences: kernel boundaries order the phases.
// Each pass reads 12 B per point, 24 B per point per fit, at 6.0-6.2 TB/s of the
// 6.3-6.5 that plain streaming reads reach here, from HBM or from the Infinity
// Cache alike: an axis pass arranged to follow its slab pass through that cache
// (one launch, tiles in an order with a lag) was no faster than two passes.
// A single set takes one launch, or two of more than 262144 points (see
// "one-launch fits" and "two-launch fits" below).
#include <float.h>
#include <stddef.h>

#include <atomic>

#include "common.hpp"
#include "dito.hpp"

namespace obvh {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kRows = 8;     // points per lane in one unrolled step
constexpr int kChunk = 512;  // tiles are multiples of it
constexpr uint32_t kNoIdx = 0xFFFFFFFFu;

struct PtsSoA {
    const float* x;
    const float* y;
    const float* z;
    __device__ __forceinline__ f3 load(uint64_t i) const { return f3{x[i], y[i], z[i]}; }
};
struct PtsAoS {
    const float* xyz;
    __device__ __forceinline__ f3 load(uint64_t i) const {
        return f3{xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]};
    }
};

__device__ __forceinline__ uint64_t set_off(const uint64_t* offs, uint64_t single, uint32_t s) {
    return offs ? offs[s] : (s ? single : 0);
}

// ---------------------------------------------------------------- setup --

// A set whose offsets decrease or run past `total` is invalid: it gets no
// tiles, a NaN box and degenerate = 4, so no later pass reads or writes
// outside the point arrays or the carved tile arrays (`cap_tiles` entries).
__device__ __forceinline__ bool set_valid(uint64_t b, uint64_t e, uint64_t total) { return b <= e && e <= total; }

__device__ __forceinline__ kr_obb3 nan_box() {
    const float nan = __builtin_nanf("");
    kr_obb3 o;
    o.mid = o.v0 = o.v1 = o.v2 = o.ext = kr_vec3{nan, nan, nan};
    return o;
}
__device__ __forceinline__ obvh_dito_trace plain_trace(int degenerate) {
    obvh_dito_trace t = {};
    t.pair_k = t.p2_sel = t.q0_sel = t.q1_sel = -1;
    t.best = -1;
    t.degenerate = degenerate;
    t.result_aabb = degenerate == 3;
    return t;
}

// Batches up to this size get their tile table from the set-up's one workgroup
// (four searches of a lane at a time, in LDS), which saves a launch: 8 sets of
// 20 points 34.0 -> 31.0 us, 1000 of 10 36.3 -> 33.6, 290 of 30000 66.5 -> 65.9.
// A wave writing set after set took 4 us more than the launch at 1000 sets.
constexpr uint32_t kFillSets = 1024;
constexpr size_t kFillTiles = 16384;

__global__ __launch_bounds__(1024) void dito_setup(const uint64_t* offs, uint64_t single_count,
                                                   uint32_t nsets, uint32_t tile, uint64_t total,
                                                   uint32_t cap_tiles, bool fill, DitoWs ws,
                                                   kr_obb3* out, obvh_dito_trace* trace) {
    // (sums of tiles in 64 bits: sets that overlap may need any number of them)
    __shared__ uint64_t carry, wsum[1024 / kWave];
    __shared__ uint32_t limit, firsts[kFillSets];
    if (threadIdx.x == 0) {
        carry = 0;
        limit = 0xFFFFFFFFu;
    }
    if (threadIdx.x == 0 && offs == nullptr) {
        ws.offsets_single[0] = 0;
        ws.offsets_single[1] = single_count;
    }
    __syncthreads();
    for (uint32_t base = 0; base < nsets; base += blockDim.x) {
        const uint32_t s = base + threadIdx.x;
        uint32_t nt = 0;
        if (s < nsets) {
            const uint64_t b = set_off(offs, single_count, s), e = set_off(offs, single_count, s + 1);
            const uint64_t n = e - b;
            if (!set_valid(b, e, total)) {
                out[s] = nan_box();
                if (trace) trace[s] = plain_trace(4);
            } else if (n != 0) {
                nt = (uint32_t)((n + tile - 1) / tile);
            } else {
                // DiTO_14 of an empty set (dito.cpp:498-502) + extent floor.
                kr_obb3 o;
                o.mid = kr_vec3{0, 0, 0};
                o.v0 = kr_vec3{1, 0, 0};
                o.v1 = kr_vec3{0, 1, 0};
                o.v2 = kr_vec3{0, 0, 1};
                o.ext = kr_vec3{0.001f, 0.001f, 0.001f};
                out[s] = o;
                if (trace) trace[s] = plain_trace(3);
            }
        }
        uint64_t v = nt;
        const int lane = lane_id();
#pragma unroll
        for (int m = 1; m < kWave; m <<= 1) {
            const uint64_t o = __shfl_up((unsigned long long)v, m, kWave);
            if (lane >= m) v += o;
        }
        if (lane == kWave - 1) wsum[wave_id()] = v;
        __syncthreads();
        uint64_t wpre = 0;
        for (int w = 0; w < wave_id(); ++w) wpre += wsum[w];
        const uint64_t incl = carry + wpre + v;
        // Offsets that never decrease need at most cap_tiles - 1 tiles.  Where
        // others (sets that overlap) need more than the arrays hold, the sets
        // from the first that does not fit on are invalid: no tiles, a NaN box.
        if (nt != 0 && incl > cap_tiles) {
            if (incl - nt <= cap_tiles) atomicMin(&limit, (uint32_t)(incl - nt));  // the first of them
            out[s] = nan_box();
            if (trace) trace[s] = plain_trace(4);
        }
        __syncthreads();
        const uint32_t first = (uint32_t)min(incl - nt, (uint64_t)limit);
        if (s < nsets) ws.first_tile[s] = first;
        if (fill && s < nsets) firsts[s] = first;
        if (threadIdx.x == blockDim.x - 1) carry = incl;
        __syncthreads();
    }
    const uint32_t T = (uint32_t)min(carry, (uint64_t)limit);
    if (threadIdx.x == 0) ws.first_tile[nsets] = T;
    if (!fill) return;
    // the tile table, as dito_tile_table makes it: four searches of a lane at a time
    for (uint32_t t0 = threadIdx.x; t0 < T; t0 += 4 * blockDim.x) {
        uint32_t at[4] = {0, 0, 0, 0};
        for (uint32_t step = kFillSets / 2; step != 0; step >>= 1) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (at[k] + step < nsets && firsts[at[k] + step] <= t0 + k * blockDim.x) at[k] += step;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (t0 + k * blockDim.x < T) ws.tile_set[t0 + k * blockDim.x] = at[k];
    }
}

__global__ __launch_bounds__(256) void dito_tile_table(uint32_t nsets, DitoWs ws) {
    const uint32_t T = ws.first_tile[nsets];
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < T; t += gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = nsets;  // first_tile[lo] <= t < first_tile[hi]
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (ws.first_tile[mid] <= t) lo = mid; else hi = mid;
        }
        ws.tile_set[t] = lo;  // last set starting at or before t: skips empty sets
    }
}

// --------------------------------------------------------------- pass 1 --

// The lower half of the wave keeps a over its own and the upper half's lane,
// the upper half b.
__device__ __forceinline__ float min_swap32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return fminf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// The same between the even and odd rows of 16 lanes.
__device__ __forceinline__ float min_swap16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return fminf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <int kCtrl>
__device__ __forceinline__ float dpp_movf(float v) {
    return __int_as_float(dpp_mov<kCtrl>(__float_as_int(v)));
}
// Minima of 14 values over the wave by recursive halving (each step halves the
// values a lane carries: 16 minima instead of 84): lanes 4q .. 4q + 3 get that
// of value 7 (q / 8) + q % 8 (q % 8 < 7).
__device__ __forceinline__ float wave_min14(const float (&v)[14]) {
    const float INF = FLT_MAX * 2.0f;
    float w[8], u[4];
#pragma unroll
    for (int k = 0; k < 7; ++k) w[k] = min_swap32(v[k], v[7 + k]);
    w[7] = INF;
#pragma unroll
    for (int k = 0; k < 4; ++k) u[k] = min_swap16(w[k], w[k + 4]);
    const bool b3 = (lane_id() & 8) != 0, b2 = (lane_id() & 4) != 0;
    const float x0 = fminf(b3 ? u[2] : u[0], dpp_movf<0x128>(b3 ? u[0] : u[2]));  // row_ror:8
    const float x1 = fminf(b3 ? u[3] : u[1], dpp_movf<0x128>(b3 ? u[1] : u[3]));
    float y = fminf(b2 ? x1 : x0, dpp_movf<0x141>(b2 ? x0 : x1));  // row_half_mirror
    y = fminf(y, dpp_movf<0x4E>(y));
    return fminf(y, dpp_movf<0xB1>(y));
}
// Minima of 6 values: lanes 8q .. 8q + 7 get that of value 3 (q / 4) + q % 4
// (q % 4 < 3).
__device__ __forceinline__ float wave_min6(const float (&v)[6]) {
    const float INF = FLT_MAX * 2.0f;
    float w[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) w[k] = min_swap32(v[k], v[3 + k]);
    const float u0 = min_swap16(w[0], w[2]), u1 = min_swap16(w[1], INF);
    const bool b3 = (lane_id() & 8) != 0;
    float y = fminf(b3 ? u1 : u0, dpp_movf<0x128>(b3 ? u0 : u1));
    y = fminf(y, dpp_movf<0x141>(y));
    y = fminf(y, dpp_movf<0x4E>(y));
    return fminf(y, dpp_movf<0xB1>(y));
}

template <int kThreads>
struct FitLds {
    float wext[kThreads / kWave][16];  // per wave: slab minima (slots 0..6) and negated maxima (8..14)
    float ext[16];                     // of the tile
    uint32_t idx[16];                  // where they are first reached (point or chunk), within the tile
    float wrng[kThreads / kWave][8];   // per wave: minima (0..2) and negated maxima (4..6) on the axes
    float rng[8];
    SetState st;
    uint32_t last, given;
};
__device__ __forceinline__ int side_slot(int side) { return side < 7 ? side : side + 1; }

// Ranges of two more points on the three axes.
__device__ __forceinline__ void axes_step(f3 p, f3 q, const f3 (&b)[3], float (&r)[6]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float d = dot3(p, b[k]), e = dot3(q, b[k]);
        r[k] = fminf(fminf(r[k], d), e);
        r[3 + k] = fmaxf(fmaxf(r[3 + k], d), e);
    }
}
// Slab extremes of two more points (a three-operand min / max each).
__device__ __forceinline__ void slabs_step(f3 p, f3 q, float (&e)[14]) {
    float u[7], v[7];
    slab7(p, u);
    slab7(q, v);
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        e[k] = fminf(fminf(e[k], u[k]), v[k]);
        e[7 + k] = fmaxf(fmaxf(e[7 + k], u[k]), v[k]);
    }
}
__device__ __forceinline__ void state_axes(const SetState& st, f3 (&b)[3]) {  // uniform
    float ax[9];
#pragma unroll
    for (int k = 0; k < 9; ++k)
        ax[k] = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(st.ax[k])));
#pragma unroll
    for (int k = 0; k < 3; ++k) b[k] = f3{ax[3 * k], ax[3 * k + 1], ax[3 * k + 2]};
}

// The tile's slab extremes into L.ext (maxima negated), L.idx cleared; e: each
// lane's, maxima negated.
template <int kThreads>
__device__ __forceinline__ void tile_extremes(const float (&e)[14], FitLds<kThreads>& L) {
    const float y = wave_min14(e);
    if ((lane_id() & 3) == 0) L.wext[wave_id()][lane_id() >> 2] = y;
    __syncthreads();
    if (threadIdx.x < 16) {
        float a = L.wext[0][threadIdx.x];
        for (int w = 1; w < kThreads / kWave; ++w) a = fminf(a, L.wext[w][threadIdx.x]);
        L.ext[threadIdx.x] = a;
        L.idx[threadIdx.x] = kNoIdx;
    }
    __syncthreads();
}


// A tile's points: uniform pointers and 32-bit byte offsets, so that a load is
// one instruction (a 64-bit address per lane costs two more).  load4: four
// consecutive points, at any alignment of the arrays.
__device__ __forceinline__ float load_at(const float* p, uint32_t byte) {
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + byte);
}
__device__ __forceinline__ float4 load4_at(const float* p, uint32_t byte) {
    float4 v;
    __builtin_memcpy(&v, reinterpret_cast<const char*>(p) + byte, sizeof(v));
    return v;
}
struct TileSoA {
    const float *x, *y, *z;
    __device__ __forceinline__ TileSoA(const PtsSoA& p, uint64_t base) : x(p.x + base), y(p.y + base), z(p.z + base) {}
    __device__ __forceinline__ f3 load(uint32_t i) const {
        return f3{load_at(x, 4 * i), load_at(y, 4 * i), load_at(z, 4 * i)};
    }
    __device__ __forceinline__ void load4(uint32_t i, f3* p) const {
        const float4 a = load4_at(x, 4 * i), b = load4_at(y, 4 * i), c = load4_at(z, 4 * i);
        p[0] = f3{a.x, b.x, c.x};
        p[1] = f3{a.y, b.y, c.y};
        p[2] = f3{a.z, b.z, c.z};
        p[3] = f3{a.w, b.w, c.w};
    }
};
struct TileAoS {
    const float* xyz;
    __device__ __forceinline__ TileAoS(const PtsAoS& p, uint64_t base) : xyz(p.xyz + 3 * base) {}
    __device__ __forceinline__ f3 load(uint32_t i) const {
        return f3{load_at(xyz, 12 * i), load_at(xyz, 12 * i + 4), load_at(xyz, 12 * i + 8)};
    }
    __device__ __forceinline__ void load4(uint32_t i, f3* p) const {
        const float4 a = load4_at(xyz, 12 * i), b = load4_at(xyz, 12 * i + 16), c = load4_at(xyz, 12 * i + 32);
        p[0] = f3{a.x, a.y, a.z};
        p[1] = f3{a.w, b.x, b.y};
        p[2] = f3{b.z, b.w, c.x};
        p[3] = f3{c.y, c.z, c.w};
    }
};
__device__ __forceinline__ TileSoA tile_of(const PtsSoA& p, uint64_t base) { return TileSoA(p, base); }
__device__ __forceinline__ TileAoS tile_of(const PtsAoS& p, uint64_t base) { return TileAoS(p, base); }

// A tile is read in steps of 2048 points, 512 consecutive ones per wave: lane l
// takes points 4 l .. 4 l + 3 of each half.  Row r = 8 c + j of a lane (step c)
// is point tile_point(r) of the tile; a lane's rows ascend.
constexpr uint32_t kStepPts = kBlock * kRows;
static_assert(kRows == 8, "two halves of four points");
__device__ __forceinline__ uint32_t tile_point(uint32_t r) {
    return (r >> 3) * kStepPts + (threadIdx.x >> 6) * (kStepPts / kWaves) + ((r >> 2) & 1u) * (4 * kWave) +
           (threadIdx.x & (kWave - 1)) * 4 + (r & 3u);
}

// f(c, points) for every step c of a tile's cnt points.  Past the end a lane
// gets copies of the last point, which no strict rule takes.
template <class T, class F>
__device__ __forceinline__ void stream_tile(const T& pts, uint32_t cnt, F f) {
    uint32_t c = 0;
    for (; (c + 1) * kStepPts <= cnt; ++c) {
        f3 p[kRows];
        pts.load4(tile_point(8 * c), p);
        pts.load4(tile_point(8 * c + 4), p + 4);
        f(c, p);
    }
    if (c * kStepPts + (threadIdx.x >> 6) * (kStepPts / kWaves) < cnt) {  // wave-uniform
        f3 p[kRows];
#pragma unroll
        for (int j = 0; j < kRows; ++j) p[j] = pts.load(min(tile_point(8 * c + j), cnt - 1));
        f(c, p);
    }
}

// Slab pass over a tile of cnt points: its 14 extremes (L.ext, maxima negated)
// and the points where they are first reached (L.idx; kNoIdx: nowhere, all NaN
// or beyond infinity).  Streaming, bound by memory (6.0 TB/s): per point and
// side one strict compare and two selects keep the first point that reaches
// the extreme, as the sequential scan does; NaN values are never taken.  What
// a small tile cost was the reduction: shuffling 14 (value, index) pairs
// through the wave was 700 instructions; now the values halve (45) and only
// the lanes that hold an extreme look at indices.  Ends with a barrier.
template <class T>
__device__ __forceinline__ void tile_pass1(const T& pts, uint32_t cnt, FitLds<kBlock>& L) {
    const float INF = FLT_MAX * 2.0f;
    float run[14];     // extremes, maxima negated
    uint32_t row[14];  // where they were first reached
#pragma unroll
    for (int k = 0; k < 14; ++k) { run[k] = INF; row[k] = 0xFFFFFFFFu; }
    stream_tile(pts, cnt, [&](uint32_t c, const f3 (&p)[kRows]) {
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            float pr[7];
            slab7(p[j], pr);
#pragma unroll
            for (int k = 0; k < 14; ++k) {
                const float v = k < 7 ? pr[k] : -pr[k - 7];
                if (v < run[k]) { run[k] = v; row[k] = 8 * c + j; }
            }
        }
    });
    tile_extremes(run, L);
#pragma unroll
    for (int k = 0; k < 14; ++k) {
        const bool hit = run[k] == L.ext[side_slot(k)] && row[k] != 0xFFFFFFFFu;
        if (__ballot(hit) == 0) continue;  // (one atomic per wave: of equal points every lane is here)
        const int32_t first = wave_min_i32(hit ? (int32_t)tile_point(row[k]) : 0x7FFFFFFF);
        if (lane_id() == 0) atomicMin(&L.idx[side_slot(k)], (uint32_t)first);
    }
    __syncthreads();
}

// The tile's pairs (value, index within the set; `first`: of the tile's first
// point) by threads 0..13.
__device__ __forceinline__ void store_pairs(const FitLds<kBlock>& L, uint32_t first, float* v_out, uint32_t* i_out) {
    if (threadIdx.x >= 14) return;
    const int side = threadIdx.x, slot = side_slot(side);
    const uint32_t i = L.idx[slot];
    v_out[side] = side < 7 ? L.ext[slot] : -L.ext[slot];
    i_out[side] = i == kNoIdx ? kNoIdx : first + i;
}

__global__ __launch_bounds__(kBlock) void dito_pass1(PtsSoA pts, const uint64_t* offs, uint32_t nsets, uint32_t tile,
                                                     DitoWs ws) {
    __shared__ FitLds<kBlock> L;
    const uint32_t T = ws.first_tile[nsets];
    for (uint32_t t = blockIdx.x; t < T; t += gridDim.x) {
        const uint32_t s = ws.tile_set[t];
        const uint64_t sbeg = offs[s], send = offs[s + 1];
        const uint64_t first = (uint64_t)(t - ws.first_tile[s]) * tile;
        tile_pass1(tile_of(pts, sbeg + first), (uint32_t)min((uint64_t)tile, send - sbeg - first), L);
        store_pairs(L, (uint32_t)first, &ws.part1_v[(size_t)t * 14], &ws.part1_i[(size_t)t * 14]);
    }
}

// ----------------------------------------- candidate search (one wave) --
//
// dito.cpp:347-418 over a 14-entry point list `sel`.  Sets of n <= 14 points
// use their n points followed by copies of sel[0]: a copy never wins a strict
// comparison against the first occurrence, so every result equals the
// n-point search.  Candidate ids: 0..2 base triangle, 3..11 upper tetra,
// 12..20 lower tetra.  Every lane computes the common prefix (extreme pair,
// base triangle, normal, apexes); lane c < 21 evaluates candidate c with the
// same operations as the sequential scan.  The scan keeps the first candidate
// whose quality is strictly below the best so far, starting from the AABB's:
// that is the lexicographic minimum of (quality, id) over the candidates,
// kept when it is strictly below the AABB's quality; a NaN quality or an
// absent candidate (apex not valid) never wins.

__device__ __forceinline__ void ext_projs(const f3* sel, f3 d, float& mn, float& mx) {
    float p = dot3(sel[0], d);
    mn = p;
    mx = p;
#pragma unroll
    for (int i = 1; i < 14; ++i) {
        p = dot3(sel[i], d);
        if (p < mn) mn = p;  // dito.cpp:198-202
        if (p > mx) mx = p;
    }
}

// Quality of candidate c (dito.cpp:309-345 for one edge of one triangle), its
// axes in b0..b2; +inf when the candidate does not exist.
__device__ __forceinline__ float eval_candidate(const f3* sel, int c, f3 n, f3 e0, f3 e1, f3 e2, f3 p0, f3 p1,
                                                f3 p2, f3 q0, f3 q1, bool q0v, bool q1v, f3& b0, f3& b1, f3& b2) {
    const int face = c / 3, k = c - 3 * face;
    f3 nf = n, ea = e0, eb = e1, ec = e2;
    if (face > 0) {
        const bool up = face <= 3;
        if (up ? !q0v : !q1v) return FLT_MAX * 2.0f;
        const f3 q = up ? q0 : q1;
        const f3 f0 = dm::normalize(sub3(q, p0));
        const f3 f1 = dm::normalize(sub3(q, p1));
        const f3 f2 = dm::normalize(sub3(q, p2));
        const int fi = (face - 1) % 3;  // dito.cpp:394-417
        if (fi == 0) {
            nf = dm::normalize(dm::cross(f1, e0)); ea = e0; eb = f1; ec = f0;
        } else if (fi == 1) {
            nf = dm::normalize(dm::cross(f2, e1)); ea = e1; eb = f2; ec = f1;
        } else {
            nf = dm::normalize(dm::cross(f0, e2)); ea = e2; eb = f0; ec = f2;
        }
    }
    const f3 e = k == 0 ? ea : (k == 1 ? eb : ec);
    float nmin, nmax, emin, emax, mmin, mmax;
    ext_projs(sel, nf, nmin, nmax);
    const f3 m = dm::cross(e, nf);
    ext_projs(sel, e, emin, emax);
    ext_projs(sel, m, mmin, mmax);
    b0 = e;
    b1 = nf;
    b2 = m;
    return quality(f3{emax - emin, nmax - nmin, mmax - mmin});
}

// Run by every lane of a wave; the results are uniform.
__device__ void dito_candidate_search(const float mn[7], const float mx[7], const f3 minv[7], const f3 maxv[7],
                                      const f3 sel[14], SetState& st, obvh_dito_trace& tr) {
    const float eps = 0.000001f;
    const f3 almid = f3{(mn[0] + mx[0]) * 0.5f, (mn[1] + mx[1]) * 0.5f, (mn[2] + mx[2]) * 0.5f};
    const f3 allen = f3{mx[0] - mn[0], mx[1] - mn[1], mx[2] - mn[2]};
    st.almid[0] = almid.x; st.almid[1] = almid.y; st.almid[2] = almid.z;
    st.allen[0] = allen.x; st.allen[1] = allen.y; st.allen[2] = allen.z;
    st.alval = quality(allen);

    int kstar = 0;
    float dbest = dm::sqdist(maxv[0], minv[0]);
#pragma unroll
    for (int k = 1; k < 7; ++k) {
        const float d = dm::sqdist(maxv[k], minv[k]);
        if (d > dbest) { dbest = d; kstar = k; }
    }
    f3 p0 = minv[0], p1 = maxv[0];
#pragma unroll
    for (int k = 1; k < 7; ++k)
        if (kstar == k) { p0 = minv[k]; p1 = maxv[k]; }
    tr.pair_k = kstar;
    if (dm::sqdist(p0, p1) < eps) {  // degenerate case 1 -> AABB
        st.mode = 1;
        tr.degenerate = 1;
        return;
    }
    const f3 e0 = dm::normalize(sub3(p0, p1));
    int ip2 = 0;
    f3 p2 = sel[0];
    float dmax;
    {
        f3 u0 = sub3(sel[0], p0);
        float t = dot3(e0, u0);
        dmax = len2(u0) - t * t / len2(e0);
#pragma unroll
        for (int i = 1; i < 14; ++i) {
            u0 = sub3(sel[i], p0);
            t = dot3(e0, u0);
            const float d = len2(u0) - t * t / len2(e0);
            if (d > dmax) { dmax = d; ip2 = i; p2 = sel[i]; }
        }
    }
    tr.p2_sel = ip2;
    if (dmax < eps) {  // degenerate case 2 -> line-aligned box (dito.cpp:451-476)
        const f3 u = e0;
        f3 r = u;
        if (fabsf(u.x) > fabsf(u.y) && fabsf(u.x) > fabsf(u.z)) r.x = 0;
        else if (fabsf(u.y) > fabsf(u.z)) r.y = 0;
        else r.z = 0;
        if (len2(r) < eps) r = f3{1, 1, 1};
        const f3 v = dm::normalize(dm::cross(u, r));
        const f3 w = dm::normalize(dm::cross(u, v));
        st.ax[0] = u.x; st.ax[1] = u.y; st.ax[2] = u.z;
        st.ax[3] = v.x; st.ax[4] = v.y; st.ax[5] = v.z;
        st.ax[6] = w.x; st.ax[7] = w.y; st.ax[8] = w.z;
        st.mode = 2;
        tr.degenerate = 2;
        return;
    }
    const f3 e1 = dm::normalize(sub3(p1, p2));
    const f3 e2 = dm::normalize(sub3(p2, p0));
    const f3 n = dm::normalize(dm::cross(e1, e0));

    float pr = dot3(sel[0], n);
    float lo = pr, hi = pr;
    int ilo = 0, ihi = 0;
    f3 q1 = sel[0], q0 = sel[0];
#pragma unroll
    for (int i = 1; i < 14; ++i) {
        pr = dot3(sel[i], n);
        if (pr < lo) { lo = pr; ilo = i; q1 = sel[i]; }
        if (pr > hi) { hi = pr; ihi = i; q0 = sel[i]; }
    }
    const float tri = dot3(p0, n);
    const int q0v = (hi - eps > tri) ? 1 : 0;
    const int q1v = (lo + eps < tri) ? 1 : 0;
    tr.q0_sel = ihi;
    tr.q1_sel = ilo;
    tr.q0_valid = q0v;
    tr.q1_valid = q1v;

    const int lane = lane_id();
    const float INF = FLT_MAX * 2.0f;
    f3 b0 = f3{1, 0, 0}, b1 = f3{0, 1, 0}, b2 = f3{0, 0, 1};
    float q = INF;
    if (lane < 21) q = eval_candidate(sel, lane, n, e0, e1, e2, p0, p1, p2, q0, q1, q0v != 0, q1v != 0, b0, b1, b2);
    if (!(q == q)) q = INF;  // NaN never compares below anything
    int id = lane;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
        const float oq = __shfl_xor(q, m, kWave);
        const int oid = __shfl_xor(id, m, kWave);
        if (oq < q || (oq == q && oid < id)) { q = oq; id = oid; }
    }
    int best_id = -1;
    if (q < st.alval) {  // strictly better than the AABB (and than every earlier candidate)
        best_id = id;
        b0 = f3{__shfl(b0.x, id), __shfl(b0.y, id), __shfl(b0.z, id)};
        b1 = f3{__shfl(b1.x, id), __shfl(b1.y, id), __shfl(b1.z, id)};
        b2 = f3{__shfl(b2.x, id), __shfl(b2.y, id), __shfl(b2.z, id)};
    } else {
        b0 = f3{1, 0, 0};
        b1 = f3{0, 1, 0};
        b2 = f3{0, 0, 1};
    }
    st.ax[0] = b0.x; st.ax[1] = b0.y; st.ax[2] = b0.z;
    st.ax[3] = b1.x; st.ax[4] = b1.y; st.ax[5] = b1.z;
    st.ax[6] = b2.x; st.ax[7] = b2.y; st.ax[8] = b2.z;
    st.mode = 0;
    tr.degenerate = 0;
    tr.best = best_id;
}

// One wave: the set's slab extremes (indices within the set, 14 sides) from
// the partials of its nt tiles (first tile ft).  kAgent: the partials were
// written by other workgroups of this launch.
template <bool kAgent>
__device__ __forceinline__ void reduce_partials(uint32_t ft, uint32_t nt, const float* part1_v,
                                                const uint32_t* part1_i, uint32_t (&ix)[14]) {
    const int lane = lane_id();
    // Lane l reduces side l % 16 (sides 0..13) over the tiles j = l / 16
    // (mod 4); two shuffle steps join the four groups.  (value, index) pairs
    // order lexicographically (no NaN values: pass 1 never takes one), so
    // the order of the reduction does not matter.
    const int side = lane & 15;
    const bool mn = side < 7;
    float a = mn ? FLT_MAX * 2.0f : -FLT_MAX * 2.0f;
    uint32_t ai = kNoIdx;
    if (side < 14) {
        // sixteen tiles' pairs are read before any is compared: one
        // memory round trip per 64 tiles instead of one per 4
        constexpr int kB = 16;
        for (uint32_t j0 = (uint32_t)(lane >> 4); j0 < nt; j0 += 4 * kB) {
            float ov[kB];
            uint32_t oi[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                const uint32_t j = j0 + 4u * u;
                const size_t at = (size_t)(ft + j) * 14 + side;
                ov[u] = j < nt ? (kAgent ? ld_agent(&part1_v[at]) : part1_v[at]) : 0.0f;
                oi[u] = j < nt ? (kAgent ? ld_agent(&part1_i[at]) : part1_i[at]) : kNoIdx;
            }
#pragma unroll
            for (int u = 0; u < kB; ++u) {
                if (j0 + 4u * u >= nt) continue;
                const bool better = (ai == kNoIdx) || (mn ? pair_better<true>(a, ai, ov[u], oi[u])
                                                          : pair_better<false>(a, ai, ov[u], oi[u]));
                if (better) { a = ov[u]; ai = oi[u]; }
            }
        }
    }
#pragma unroll
    for (int m = 16; m < kWave; m <<= 1) {
        const float ov = __shfl_xor(a, m, kWave);
        const uint32_t oi = (uint32_t)__shfl_xor((int)ai, m, kWave);
        if (mn ? pair_better<true>(a, ai, ov, oi) : pair_better<false>(a, ai, ov, oi)) { a = ov; ai = oi; }
    }
#pragma unroll
    for (int k = 0; k < 14; ++k) ix[k] = (uint32_t)__builtin_amdgcn_readlane((int)ai, k);
}

// One wave: the candidate search of a set (n points from sbeg) from its slab
// extremes' indices; st and tr in every lane.
template <class P>
__device__ __forceinline__ void set_search(P pts, uint64_t sbeg, uint64_t n, uint32_t (&ix)[14], SetState& st,
                                           obvh_dito_trace& tr) {
    // The reference scan starts from point 0 and compares strictly
    // (dito.cpp:116-173): a slab whose value at point 0 is NaN stays (NaN, 0),
    // since no later compare against NaN succeeds; otherwise NaN values are
    // never taken and the result is the (value, first index) minimum over
    // the other points, which is what the reductions above computed.  A side
    // without an index has no value beyond infinity: point 0 holds it.
    {
        const f3 pt0 = pts.load(sbeg);
        float pr0[7];
        slab7(pt0, pr0);
#pragma unroll
        for (int k = 0; k < 7; ++k)
            if (pr0[k] != pr0[k]) ix[k] = ix[7 + k] = 0;
    }
#pragma unroll
    for (int side = 0; side < 14; ++side)
        if ((uint64_t)ix[side] >= n) ix[side] = 0;
    tr = {};
    tr.pair_k = tr.p2_sel = tr.q0_sel = tr.q1_sel = -1;
    tr.best = -1;
    float mn[7], mx[7];
    f3 minv[7], maxv[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        tr.slab_min_idx[k] = ix[k];
        tr.slab_max_idx[k] = ix[7 + k];
        minv[k] = pts.load(sbeg + ix[k]);
        maxv[k] = pts.load(sbeg + ix[7 + k]);
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        float pr[7];
        slab7(minv[k], pr);
        mn[k] = pr[k];
        slab7(maxv[k], pr);
        mx[k] = pr[k];
    }
    f3 sel[14];
    if (n > 14) {
#pragma unroll
        for (int k = 0; k < 7; ++k) { sel[k] = minv[k]; sel[7 + k] = maxv[k]; }
    } else {
        sel[0] = pts.load(sbeg);
#pragma unroll
        for (int i = 1; i < 14; ++i) sel[i] = (uint64_t)i < n ? pts.load(sbeg + i) : sel[0];
    }
    st = {};
    dito_candidate_search(mn, mx, minv, maxv, sel, st, tr);
}

// One wave: reduce the nt tile partials of a set (points [sbeg, send),
// first tile ft), then search; state and trace written by lane 0.
template <class P>
__device__ __forceinline__ void set_cand(P pts, uint64_t sbeg, uint64_t send, uint32_t ft, uint32_t nt,
                                         const float* part1_v, const uint32_t* part1_i, SetState* state,
                                         obvh_dito_trace* trace) {
    uint32_t ix[14];
    reduce_partials<false>(ft, nt, part1_v, part1_i, ix);
    SetState st;
    obvh_dito_trace tr;
    set_search(pts, sbeg, send - sbeg, ix, st, tr);
    if (lane_id() == 0) {
        *state = st;
        *trace = tr;
    }
}

// One wave per set: reduce the tile partials, then the wave searches.
__global__ __launch_bounds__(kBlock) void dito_cand(PtsSoA pts, const uint64_t* offs, uint32_t nsets, uint64_t total,
                                                    DitoWs ws, obvh_dito_trace* trace) {
    const uint32_t s = blockIdx.x * kWaves + wave_id();
    if (s >= nsets) return;
    const uint64_t sbeg = offs[s], send = offs[s + 1];
    if (send == sbeg || !set_valid(sbeg, send, total)) return;
    const uint32_t ft = ws.first_tile[s], nt = ws.first_tile[s + 1] - ft;
    if (nt == 0) return;
    set_cand(pts, sbeg, send, ft, nt, ws.part1_v, ws.part1_i, &ws.state[s], &trace[s]);
}

// --------------------------------------------------------------- pass 2 --

// Each lane's ranges of a tile's cnt points on the set's three axes (min b0..b2,
// max b0..b2).
template <class T>
__device__ __forceinline__ void tile_ranges(const T& pts, uint32_t cnt, const SetState* st, float (&r)[6]) {
    const float INF = FLT_MAX * 2.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) { r[k] = INF; r[3 + k] = -INF; }
    if (st->mode == 1) return;
    f3 b[3];
    state_axes(*st, b);
    stream_tile(pts, cnt, [&](uint32_t, const f3 (&p)[kRows]) {
#pragma unroll
        for (int j = 0; j < kRows; j += 2) axes_step(p[j], p[j + 1], b, r);
    });
}

// Ranges of a tile's cnt points on the set's three axes: 6 floats (min b0..b2,
// max b0..b2) written to out6 by threads 0..7.  Ends with a barrier.
template <class T>
__device__ __forceinline__ void tile_pass2(const T& pts, uint32_t cnt, const SetState* st, FitLds<kBlock>& L,
                                           float* out6) {
    float r[6];
    tile_ranges(pts, cnt, st, r);
#pragma unroll
    for (int k = 3; k < 6; ++k) r[k] = -r[k];
    const float y = wave_min6(r);
    if ((lane_id() & 7) == 0) L.wrng[wave_id()][lane_id() >> 3] = y;
    __syncthreads();
    const int q = threadIdx.x;
    if (q < 8 && (q & 3) < 3) {
        float a = L.wrng[0][q];
        for (int w = 1; w < kWaves; ++w) a = fminf(a, L.wrng[w][q]);
        out6[q < 4 ? q : q - 1] = q < 4 ? a : -a;
    }
    __syncthreads();
}

__global__ __launch_bounds__(kBlock) void dito_pass2(PtsSoA pts, const uint64_t* offs, uint32_t nsets, uint32_t tile,
                                                     DitoWs ws) {
    __shared__ FitLds<kBlock> L;
    const uint32_t T = ws.first_tile[nsets];
    for (uint32_t t = blockIdx.x; t < T; t += gridDim.x) {
        const uint32_t s = ws.tile_set[t];
        const uint64_t sbeg = offs[s], send = offs[s + 1];
        const uint64_t first = (uint64_t)(t - ws.first_tile[s]) * tile;
        tile_pass2(tile_of(pts, sbeg + first), (uint32_t)min((uint64_t)tile, send - sbeg - first), &ws.state[s], L,
                   &ws.part2[(size_t)t * 6]);
    }
}

// ---------------------------------------------------------------- final --

// The box of a set from its ranges on the axes (min b0..b2, max b0..b2); one
// lane.  Returns whether it is the AABB.
template <class P>
__device__ __forceinline__ int set_box(P pts, uint64_t sbeg, float (&a)[6], const SetState& st, kr_obb3* out) {
    const f3 b0 = f3{st.ax[0], st.ax[1], st.ax[2]};
    const f3 b1 = f3{st.ax[3], st.ax[4], st.ax[5]};
    const f3 b2 = f3{st.ax[6], st.ax[7], st.ax[8]};
    // computeObbDimensions (dito.cpp:421-426) starts from point 0 with strict
    // compares: a NaN projection of point 0 stays, later NaNs are skipped
    // (fminf / fmaxf above skip them too).
    if (st.mode != 1) {
        const f3 p0 = pts.load(sbeg);
        const float d[3] = {dot3(p0, b0), dot3(p0, b1), dot3(p0, b2)};
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (d[k] != d[k]) a[k] = a[3 + k] = d[k];
    }
    const f3 bmn = f3{a[0], a[1], a[2]}, bmx = f3{a[3], a[4], a[5]};
    const f3 blen = sub3(bmx, bmn);
    kr_obb3 o;
    int result_aabb;
    if (st.mode == 2 || (st.mode == 0 && quality(blen) < st.alval)) {
        // finalizeOBB, dito.cpp:428-440
        const f3 ext = dm::scale(0.5f, blen);
        const f3 q = dm::scale(0.5f, add3(bmn, bmx));
        f3 mid = dm::scale(q.x, b0);
        mid = add3(mid, dm::scale(q.y, b1));
        mid = add3(mid, dm::scale(q.z, b2));
        o.mid = kr_vec3{mid.x, mid.y, mid.z};
        o.v0 = kr_vec3{b0.x, b0.y, b0.z};
        o.v1 = kr_vec3{b1.x, b1.y, b1.z};
        o.v2 = kr_vec3{b2.x, b2.y, b2.z};
        o.ext = kr_vec3{ext.x, ext.y, ext.z};
        result_aabb = 0;
    } else {  // finalizeAxisAlignedOBB, dito.cpp:442-449
        const f3 e = dm::scale(0.5f, f3{st.allen[0], st.allen[1], st.allen[2]});
        o.mid = kr_vec3{st.almid[0], st.almid[1], st.almid[2]};
        o.v0 = kr_vec3{1, 0, 0};
        o.v1 = kr_vec3{0, 1, 0};
        o.v2 = kr_vec3{0, 0, 1};
        o.ext = kr_vec3{e.x, e.y, e.z};
        result_aabb = 1;
    }
    // kr_points_obb extent floor (geometry.cpp:249)
    o.ext.x = kmax(o.ext.x, 0.001f);
    o.ext.y = kmax(o.ext.y, 0.001f);
    o.ext.z = kmax(o.ext.z, 0.001f);
    *out = o;
    return result_aabb;
}

// One wave: reduce the nt tile ranges of a set (first tile ft) and write
// its box (lane 0).
template <class P>
__device__ __forceinline__ void set_final(P pts, uint64_t sbeg, uint32_t ft, uint32_t nt, const float* part2,
                                          const SetState* state, kr_obb3* out, obvh_dito_trace* trace) {
    const float INF = FLT_MAX * 2.0f;
    float a[6] = {INF, INF, INF, -INF, -INF, -INF};
    for (uint32_t j = lane_id(); j < nt; j += kWave) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const float o = part2[(size_t)(ft + j) * 6 + k];
            a[k] = k < 3 ? fminf(a[k], o) : fmaxf(a[k], o);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) { a[k] = wave_min(a[k]); a[3 + k] = wave_max(a[3 + k]); }
    if (lane_id() == 0) trace->result_aabb = set_box(pts, sbeg, a, *state, out);
}

__global__ __launch_bounds__(kBlock) void dito_final(PtsSoA pts, const uint64_t* offs, uint32_t nsets, uint64_t total,
                                                     DitoWs ws, kr_obb3* out, obvh_dito_trace* trace) {
    const uint32_t s = blockIdx.x * kWaves + wave_id();
    if (s >= nsets) return;
    const uint64_t sbeg = offs[s], send = offs[s + 1];
    if (send == sbeg || !set_valid(sbeg, send, total)) return;
    const uint32_t ft = ws.first_tile[s], nt = ws.first_tile[s + 1] - ft;
    if (nt == 0) return;
    set_final(pts, sbeg, ft, nt, ws.part2, &ws.state[s], &out[s], &trace[s]);
}

// ------------------------------------------------------- one-launch fits --
//
// A single set in one launch: its tiles hand their partial results over inside
// the launch with the agent-scope accesses above.
//
// No tile depends on another one being scheduled: a tile that has polled for the
// set's state long enough gives up and ends, and the searching tile takes its
// axis pass over.  At most `cap` tiles wait, an eighth of the workgroups the
// device holds, so that this does not happen unless the chip is held by others
// for milliseconds (larger sets take two launches).  A tile gives up by writing
// kGaveUp to its axis partial and then counting itself in sync->flag; it still
// does its own pass if the count shows that the state is there and the mark was
// not taken yet.  The searching tile sees in the count, as it publishes the
// state, whether to look for marks.  (A count that comes after the last tile's
// reset only makes the next call look: every tile clears its mark before it
// counts its slab pass.)

constexpr uint32_t kStateUp = 1u << 31;       // sync->flag: the state is there; below: tiles that gave up
constexpr uint32_t kGaveUp = 0x7FC00001u;     // NaN, as no axis partial is
constexpr uint32_t kTakenOver = 0x7FC00002u;

constexpr int kStateWords = sizeof(SetState) / 4;
constexpr int kTraceWords = sizeof(obvh_dito_trace) / 4;
constexpr int kTraceResult = offsetof(obvh_dito_trace, result_aabb) / 4;
static_assert(kStateWords <= kWave && kTraceWords <= kWave, "copied by one wave");

// Points [first, first + cnt) of tile rows j (index j * kThreads + thread);
// past the end a copy of the last one, which no strict rule takes.
template <class P, int J, int kThreads>
__device__ __forceinline__ void load_tile(P pts, uint64_t first, uint32_t cnt, f3 (&p)[J]) {
    const uint32_t t = threadIdx.x;
    if (cnt == (uint32_t)(J * kThreads)) {  // uniform
#pragma unroll
        for (int j = 0; j < J; ++j) p[j] = pts.load(first + (uint32_t)j * kThreads + t);
        return;
    }
#pragma unroll
    for (int c = 0; c < J; c += kRows) {
        if ((uint32_t)(c * kThreads) < cnt) {
#pragma unroll
            for (int j = c; j < c + kRows; ++j) p[j] = pts.load(first + min((uint32_t)j * kThreads + t, cnt - 1));
        } else {
#pragma unroll
            for (int j = c; j < c + kRows; ++j) p[j] = p[0];
        }
    }
}

template <int kSide>
__device__ __forceinline__ float slab_side(f3 p) {  // the side's projection, negated for a maximum
    float pr[7];
    slab7(p, pr);
    return kSide < 7 ? pr[kSide % 7] : -pr[kSide % 7];
}

// Where the tile reaches its extreme on one side: the lanes whose own extreme
// equals it (usually one lane of one wave) look for the first of their points.
template <int kSide, int J, int kThreads>
__device__ __forceinline__ void find_side(const f3 (&p)[J], uint32_t cnt, float own, FitLds<kThreads>& L) {
    const float target = L.ext[side_slot(kSide)];
    if (__ballot(own == target) == 0) return;
    uint32_t at = kNoIdx;
#pragma unroll
    for (int c = J - kRows; c >= 0; c -= kRows) {
        if ((uint32_t)(c * kThreads) >= cnt) continue;
#pragma unroll
        for (int j = c + kRows - 1; j >= c; --j)
            if (slab_side<kSide>(p[j]) == target) at = (uint32_t)j;
    }
    // (one atomic per wave: in a set of equal points every lane is here)
    const int32_t first = wave_min_i32(at == kNoIdx ? 0x7FFFFFFF : (int32_t)(at * kThreads + threadIdx.x));
    if (lane_id() == 0 && first != 0x7FFFFFFF) atomicMin(&L.idx[side_slot(kSide)], (uint32_t)first);
}

__device__ __forceinline__ uint32_t* axis_mark(const DitoWs& ws, uint32_t tile) {
    return reinterpret_cast<uint32_t*>(&ws.part2[(size_t)tile * 6]);
}
// The mark of a tile that gave up goes to one side: back to the tile, or to the
// searching tile.
__device__ __forceinline__ bool claim_mark(uint32_t* mark, uint32_t to) {
    uint32_t expected = kGaveUp;
    return __hip_atomic_compare_exchange_strong(mark, &expected, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
}

// Wave 0: the set's state for the axis pass, after the flag shows it.  False
// when it is not there after `polls` polls: the tile's axis pass is the
// searching tile's.
__device__ __forceinline__ bool wait_state(FitSync* sync, const SetState* state, uint32_t* mark, uint32_t polls,
                                           SetState* lds) {
    uint32_t up = 0;
    for (uint32_t i = 0; i < polls && up < kStateUp; ++i) {
        if (i > 0) __builtin_amdgcn_s_sleep(8);
        up = __builtin_amdgcn_readfirstlane((int)ld_agent(&sync->flag));
    }
    if (up < kStateUp) {
        bool mine = false;
        if (lane_id() == 0) {
            st_agent(mark, kGaveUp);
            drain();
            up = __hip_atomic_fetch_add(&sync->flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            mine = up >= kStateUp && claim_mark(mark, 0u);
        }
        if (__ballot(mine) == 0) return false;
    }
    asm volatile("" ::: "memory");
    if (lane_id() < kStateWords)
        reinterpret_cast<uint32_t*>(lds)[lane_id()] = ld_agent(reinterpret_cast<const uint32_t*>(state) + lane_id());
    return true;
}

// After the slab pass of tile `part` of nt (partials from tile ft), L.ext and
// L.idx (indices from the tile's first point, `first` of the set): publish
// them; the last tile searches.  Returns whether this workgroup did (L.st then
// holds the state, `gave` of thread 0 how many tiles had given up waiting for
// it).  Ends with a barrier.
template <class P, int kThreads>
__device__ __forceinline__ bool tile_search(P pts, uint64_t sbeg, uint64_t n, uint32_t first, uint32_t part,
                                            uint32_t ft, uint32_t nt, const DitoWs& ws, SetState* state,
                                            FitSync* sync, obvh_dito_trace* trace, FitLds<kThreads>& L,
                                            uint32_t& gave) {
    const int lane = lane_id(), wave = wave_id();
    gave = 0;
    if (nt > 1) {
        if (wave == 0) {
            if (lane < 14) {
                const size_t at = (size_t)(ft + part) * 14 + lane;
                const int slot = side_slot(lane);
                const uint32_t i = L.idx[slot];
                st_agent(&ws.part1_v[at], lane < 7 ? L.ext[slot] : -L.ext[slot]);
                st_agent(&ws.part1_i[at], i == kNoIdx ? kNoIdx : first + i);
            }
            if (lane == 14) st_agent(axis_mark(ws, ft + part), 0u);
            drain();
            if (lane == 0)
                L.last = __hip_atomic_fetch_add(&sync->done1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == nt - 1;
        }
        __syncthreads();
        if (L.last == 0) return false;
    }
    if (wave == 0) {
        uint32_t ix[14];
        if (nt == 1) {
#pragma unroll
            for (int k = 0; k < 14; ++k) ix[k] = (uint32_t)__builtin_amdgcn_readfirstlane((int)L.idx[side_slot(k)]);
        } else {
            asm volatile("" ::: "memory");
            reduce_partials<true>(ft, nt, ws.part1_v, ws.part1_i, ix);
        }
        SetState st;
        obvh_dito_trace tr;
        set_search(pts, sbeg, n, ix, st, tr);
        if (lane == 0) L.st = st;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (nt > 1) {
            if (lane < kStateWords)
                st_agent(reinterpret_cast<uint32_t*>(state) + lane, reinterpret_cast<const uint32_t*>(&L.st)[lane]);
            drain();
            if (lane == 0)
                gave = __hip_atomic_fetch_or(&sync->flag, kStateUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (trace && lane == 0) {  // the box's workgroup writes result_aabb
#pragma unroll
            for (int k = 0; k < kTraceWords; ++k)
                if (k != kTraceResult) reinterpret_cast<uint32_t*>(trace)[k] = reinterpret_cast<const uint32_t*>(&tr)[k];
        }
    }
    __syncthreads();
    return true;
}

// After the axis pass: r, each lane's ranges (maxima not negated).  The last
// tile of the set writes the box.
template <class P, int kThreads>
__device__ __forceinline__ void tile_box(P pts, uint64_t sbeg, float (&r)[6], uint32_t part, uint32_t ft, uint32_t nt,
                                         const DitoWs& ws, FitSync* sync, kr_obb3* out, obvh_dito_trace* trace,
                                         FitLds<kThreads>& L) {
    const float INF = FLT_MAX * 2.0f;
    const int lane = lane_id(), wave = wave_id();
#pragma unroll
    for (int k = 3; k < 6; ++k) r[k] = -r[k];
    const float y = wave_min6(r);
    if ((lane & 7) == 0) L.wrng[wave][lane >> 3] = y;
    __syncthreads();
    if (wave != 0) return;
    if (lane < 8) {
        float a = L.wrng[0][lane];
        for (int w = 1; w < kThreads / kWave; ++w) a = fminf(a, L.wrng[w][lane]);
        L.rng[lane] = a;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float a[6];
    if (nt == 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            a[k] = L.rng[k];
            a[3 + k] = -L.rng[4 + k];
        }
    } else {
        if (lane < 6) st_agent(&ws.part2[(size_t)(ft + part) * 6 + lane], lane < 3 ? L.rng[lane] : -L.rng[lane + 1]);
        drain();
        uint32_t old = 0;
        if (lane == 0) old = __hip_atomic_fetch_add(&sync->done2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((uint32_t)__builtin_amdgcn_readfirstlane((int)old) != nt - 1) return;
        asm volatile("" ::: "memory");
        float q[6] = {INF, INF, INF, -INF, -INF, -INF};
        for (uint32_t j0 = lane; j0 < nt; j0 += 4 * kWave) {  // four tiles of a lane a trip to memory
            float o[4][6];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int k = 0; k < 6; ++k)
                    o[u][k] = ld_agent(&ws.part2[(size_t)(ft + min(j0 + u * kWave, nt - 1)) * 6 + k]);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int k = 0; k < 3; ++k) { q[k] = fminf(q[k], o[u][k]); q[3 + k] = fmaxf(q[3 + k], o[u][3 + k]); }
        }
#pragma unroll
        for (int k = 3; k < 6; ++k) q[k] = -q[k];
        const float z = wave_min6(q);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            a[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), 8 * k));
            a[3 + k] = -__int_as_float(__builtin_amdgcn_readlane(__float_as_int(z), 32 + 8 * k));
        }
        if (lane == 0) {  // nobody reads them any more: zero for the next call on this workspace
            st_agent(&sync->done1, 0u);
            st_agent(&sync->done2, 0u);
            st_agent(&sync->flag, 0u);
        }
    }
    if (lane == 0) {
        const int aabb = set_box(pts, sbeg, a, L.st, out);
        if (trace) st_agent(&trace->result_aabb, aabb);
    }
}

// A workgroup keeps its tile's points in registers between the passes; the
// last tile to finish the slab pass searches, the others wait for its state.
// Up to 8192 points one workgroup does it all (no hand-over: 23 -> 12.4 us);
// 131 072 points take 64 tiles (26.7 -> 20.9 us).  Batches read their points
// again instead: tiles that wait in registers for their set's search held
// 75 MB for 68 us each, three times the time of two readings.
template <class P, int J, int kThreads>
__device__ __forceinline__ void one_tile(P pts, uint64_t n, uint32_t part, uint32_t nt, const DitoWs& ws,
                                         uint32_t polls, kr_obb3* out, obvh_dito_trace* trace, FitLds<kThreads>& L) {
    constexpr uint32_t kTilePts = J * kThreads;
    const float INF = FLT_MAX * 2.0f;
    FitSync* sync = reinterpret_cast<FitSync*>(ws.done);
    const uint64_t first = (uint64_t)part * kTilePts;
    const uint32_t cnt = (uint32_t)min((uint64_t)kTilePts, n - first);
    f3 p[J];
    load_tile<P, J, kThreads>(pts, first, cnt, p);
    float e[14];
#pragma unroll
    for (int k = 0; k < 7; ++k) { e[k] = INF; e[7 + k] = -INF; }
#pragma unroll
    for (int j = 0; j < J; j += 2) slabs_step(p[j], p[j + 1], e);
#pragma unroll
    for (int k = 7; k < 14; ++k) e[k] = -e[k];
    tile_extremes(e, L);
    find_side<0>(p, cnt, e[0], L); find_side<1>(p, cnt, e[1], L); find_side<2>(p, cnt, e[2], L);
    find_side<3>(p, cnt, e[3], L); find_side<4>(p, cnt, e[4], L); find_side<5>(p, cnt, e[5], L);
    find_side<6>(p, cnt, e[6], L); find_side<7>(p, cnt, e[7], L); find_side<8>(p, cnt, e[8], L);
    find_side<9>(p, cnt, e[9], L); find_side<10>(p, cnt, e[10], L); find_side<11>(p, cnt, e[11], L);
    find_side<12>(p, cnt, e[12], L); find_side<13>(p, cnt, e[13], L);
    __syncthreads();
    uint32_t gave;
    const bool searched = tile_search(pts, 0, n, (uint32_t)first, part, 0, nt, ws, ws.state, sync, trace, L, gave);
    if (searched) {
        load_tile<P, J, kThreads>(pts, first, cnt, p);  // the search used the registers
    } else {
        if (wave_id() == 0) {
            const bool ok = wait_state(sync, ws.state, axis_mark(ws, part), polls, &L.st);
            if (lane_id() == 0) L.given = ok ? 0u : 1u;
        }
        __syncthreads();
        if (L.given != 0) return;
    }
    f3 b[3];
    state_axes(L.st, b);
    auto axis_pass = [&](uint32_t tile) {
        float r[6] = {INF, INF, INF, -INF, -INF, -INF};
#pragma unroll
        for (int j = 0; j < J; j += 2) axes_step(p[j], p[j + 1], b, r);
        tile_box(pts, 0, r, tile, 0, nt, ws, sync, out, trace, L);
    };
    axis_pass(part);
    if (!searched || nt == 1) return;
    if (threadIdx.x == 0) L.given = gave & ~kStateUp;
    __syncthreads();
    if (L.given == 0) return;
    for (uint32_t t = 0; t < nt; ++t) {  // the tiles that gave up
        __syncthreads();
        if (threadIdx.x == 0) L.last = t != part && claim_mark(axis_mark(ws, t), kTakenOver);
        __syncthreads();
        if (L.last == 0) continue;
        const uint64_t at = (uint64_t)t * kTilePts;
        load_tile<P, J, kThreads>(pts, at, (uint32_t)min((uint64_t)kTilePts, n - at), p);
        axis_pass(t);
    }
}

// A set of n > 0 points, gridDim.x tiles.
template <class P, int J, int kThreads>
__global__ __launch_bounds__(kThreads) void dito_one(P pts, uint64_t n, DitoWs ws, uint32_t polls, kr_obb3* out,
                                                     obvh_dito_trace* trace) {
    __shared__ FitLds<kThreads> L;
    one_tile<P, J, kThreads>(pts, n, blockIdx.x, gridDim.x, ws, polls, out, trace, L);
}

__global__ void dito_one_clear(DitoWs ws) {
    if (threadIdx.x < 4) ws.done[threadIdx.x] = 0;
}

// ------------------------------------------------------- two-launch fits --
//
// Sets of more tiles than may wait: the same hand-overs, the slab pass with the
// search and the axis pass with the box in a launch each.  Bound by the passes'
// latency and by the last tile's reduction of up to 1024 partials by one wave.
// With an agent-scope release and acquire a workgroup (an L2 written back each
// time) 1 M points took 57 us, 4 M 122, 6 M 133, 32 M 283; now 49, 89, 94 and 198.

template <class P>
__global__ __launch_bounds__(kBlock) void dito_one_a(P pts, uint64_t n, uint32_t tile, DitoWs ws,
                                                     obvh_dito_trace* trace) {
    __shared__ FitLds<kBlock> L;
    const uint64_t base = (uint64_t)blockIdx.x * tile;
    tile_pass1(tile_of(pts, base), (uint32_t)min((uint64_t)tile, n - base), L);
    uint32_t gave;
    tile_search(pts, 0, n, (uint32_t)base, blockIdx.x, 0, gridDim.x, ws, ws.state, reinterpret_cast<FitSync*>(ws.done),
                trace, L, gave);
}

template <class P>
__global__ __launch_bounds__(kBlock) void dito_one_b(P pts, uint64_t n, uint32_t tile, DitoWs ws, kr_obb3* out,
                                                     obvh_dito_trace* trace) {
    __shared__ FitLds<kBlock> L;
    if (threadIdx.x == 0) L.st = *ws.state;
    const uint64_t base = (uint64_t)blockIdx.x * tile;
    float r[6];
    tile_ranges(tile_of(pts, base), (uint32_t)min((uint64_t)tile, n - base), ws.state, r);
    tile_box(pts, 0, r, blockIdx.x, 0, gridDim.x, ws, reinterpret_cast<FitSync*>(ws.done), out, trace, L);
}

// ----------------------------------------------------------------- host --

size_t dito_max_tiles(uint32_t nsets, uint64_t total, uint32_t tile) {
    return (size_t)(total / tile) + nsets + 1;
}

size_t dito_carve(DitoWs* ws, void* base, size_t cap, uint32_t nsets, uint64_t total, uint32_t tile) {
    tile = min(tile, kDitoMaxTile);
    Carver c{(char*)base, 0, cap};
    const size_t T = dito_max_tiles(nsets, total, tile);
    ws->offsets_single = c.take<uint64_t>(2);
    ws->done = c.take<uint32_t>(4);
    ws->first_tile = c.take<uint32_t>(nsets + 1);
    ws->tile_set = c.take<uint32_t>(T);
    ws->part1_v = c.take<float>(T * 14);
    ws->part1_i = c.take<uint32_t>(T * 14);
    ws->part2 = c.take<float>(T * 6);
    ws->state = c.take<SetState>(nsets);
    ws->trace_tmp = c.take<obvh_dito_trace>(nsets);
    return c.used;
}

uint32_t dito_auto_tile(uint32_t nsets, uint64_t total) {
    // about 4096 tiles for the whole job, between 512 and 32768 points each
    // (8192 sets, 897 M points: 3.52 ms with 32768, 3.54 with 16384, 3.59 with
    // 65536); up to 65536 for a single set, whose workspace for 2^28 points
    // must fit the static array of the no-allocation entry
    uint64_t want = total / 4096;
    uint64_t t = (want + kChunk - 1) / kChunk * kChunk;
    if (t < (uint64_t)kChunk) t = kChunk;
    const uint64_t most = nsets == 1 ? 65536 : 32768;
    if (t > most) t = most;
    return (uint32_t)t;
}

// Tiles of one set that may wait for each other: an eighth of the workgroups
// the device holds at four per CU.
static kr_error one_cap(uint32_t* cap) {
    static std::atomic<uint32_t> cached[64];
    int dev = 0;
    OBVH_HIP_TRY(hipGetDevice(&dev));
    uint32_t v = dev >= 0 && dev < 64 ? cached[dev].load(std::memory_order_relaxed) : 0;
    if (v == 0) {
        int cus = 0;
        OBVH_HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        v = (uint32_t)max(cus / 2, 1);
        if (dev >= 0 && dev < 64) cached[dev].store(v, std::memory_order_relaxed);
    }
    *cap = v;
    return nullptr;
}

constexpr int kOneRows = 8;  // points per lane of the single fit's workgroups

template <class P>
static void launch_one(P p, uint64_t n, uint32_t tile, uint32_t T, uint32_t cap, DitoWs ws, uint32_t polls,
                       kr_obb3* out, obvh_dito_trace* trace, bool& clear, hipStream_t stream) {
    if (n <= 1024 * kOneRows) {
        hipLaunchKernelGGL((dito_one<P, kOneRows, 1024>), dim3(1), dim3(1024), 0, stream, p, n, ws, polls, out,
                           trace);
        return;
    }
    if (clear) hipLaunchKernelGGL(dito_one_clear, dim3(1), dim3(64), 0, stream, ws);
    clear = false;
    constexpr uint32_t kOneTile = kBlock * kOneRows;
    const uint64_t F = (n + kOneTile - 1) / kOneTile;
    if (F <= cap) {
        hipLaunchKernelGGL((dito_one<P, kOneRows, kBlock>), dim3((uint32_t)F), dim3(kBlock), 0, stream, p, n, ws,
                           polls, out, trace);
        return;
    }
    hipLaunchKernelGGL(dito_one_a<P>, dim3(T), dim3(kBlock), 0, stream, p, n, tile, ws, trace);
    hipLaunchKernelGGL(dito_one_b<P>, dim3(T), dim3(kBlock), 0, stream, p, n, tile, ws, out, trace);
}

kr_error dito_one_launch(const float* x, const float* y, const float* z, const float* xyz, uint64_t n,
                         kr_obb3* out, obvh_dito_trace* trace, void* workspace, size_t ws_bytes, bool& clear,
                         hipStream_t stream, uint32_t polls) {
    if (n == 0) return "obvh_dito: the single-set fit needs at least one point";
    // The two-launch form's tiles: at most 1024, since each workgroup pays one
    // agent-scope release and the last one reduces every tile.  At least the
    // batched path's tile, so the workspace size of obvh_dito_workspace_size
    // always suffices.
    uint64_t tl = (n + 1023) / 1024;
    tl = (tl + kChunk - 1) / kChunk * kChunk;
    const uint32_t tile = (uint32_t)max(max(tl, (uint64_t)4 * kChunk), (uint64_t)dito_auto_tile(1, n));
    DitoWs ws;
    const size_t need = dito_carve(&ws, workspace, ws_bytes, 1, n, tile);
    if (workspace == nullptr || ws_bytes < need) return "obvh_dito: workspace too small";
    const uint64_t T = (n + tile - 1) / tile;
    if (T > dito_max_tiles(1, n, tile)) return "obvh_dito: tile count";
    uint32_t cap = 0;
    if (kr_error e = one_cap(&cap)) return e;
    cap = (uint32_t)min((uint64_t)cap, (uint64_t)dito_max_tiles(1, n, tile));
    if (xyz) launch_one(PtsAoS{xyz}, n, tile, (uint32_t)T, cap, ws, polls, out, trace, clear, stream);
    else launch_one(PtsSoA{x, y, z}, n, tile, (uint32_t)T, cap, ws, polls, out, trace, clear, stream);
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

kr_error dito_launch(const float* x, const float* y, const float* z,
                     const uint64_t* offsets, uint64_t single_count, uint32_t nsets, uint64_t total,
                     kr_obb3* out, obvh_dito_trace* trace, uint32_t tile, uint32_t workers,
                     void* workspace, size_t ws_bytes, hipStream_t stream) {
    if (nsets == 0) return nullptr;
    if (tile == 0) tile = dito_auto_tile(nsets, total);
    if (tile % kChunk != 0) return "obvh_dito: tile_points must be a multiple of 512";
    tile = min(tile, kDitoMaxTile);
    DitoWs ws;
    const size_t need = dito_carve(&ws, workspace, ws_bytes, nsets, total, tile);
    if (workspace == nullptr || ws_bytes < need) return "obvh_dito: workspace too small";
    const uint64_t* offs = offsets ? offsets : ws.offsets_single;
    obvh_dito_trace* tr = trace ? trace : ws.trace_tmp;
    const size_t T = dito_max_tiles(nsets, total, tile);
    // default: one workgroup per tile (measured faster than persistent
    // workgroups looping over tiles)
    if (workers == 0) workers = (uint32_t)(T < 65536 ? T : 65536);
    if (workers > T) workers = (uint32_t)T;
    if (T > 0xFFFFFFF0ull) return "obvh_dito: too many tiles";
    const bool fill = nsets <= kFillSets && T <= kFillTiles;
    hipLaunchKernelGGL(dito_setup, dim3(1), dim3(1024), 0, stream, offsets, single_count, nsets, tile, total,
                       (uint32_t)T, fill, ws, out, tr);
    if (!fill) {
        const uint32_t tb = (uint32_t)min((T + 255) / 256, (size_t)4096);
        hipLaunchKernelGGL(dito_tile_table, dim3(tb), dim3(256), 0, stream, nsets, ws);
    }
    const PtsSoA p{x, y, z};
    const dim3 set_grid((nsets + kWaves - 1) / kWaves);
    hipLaunchKernelGGL(dito_pass1, dim3(workers), dim3(kBlock), 0, stream, p, offs, nsets, tile, ws);
    hipLaunchKernelGGL(dito_cand, set_grid, dim3(kBlock), 0, stream, p, offs, nsets, total, ws, tr);
    hipLaunchKernelGGL(dito_pass2, dim3(workers), dim3(kBlock), 0, stream, p, offs, nsets, tile, ws);
    hipLaunchKernelGGL(dito_final, set_grid, dim3(kBlock), 0, stream, p, offs, nsets, total, ws, out, tr);
    OBVH_HIP_TRY(hipGetLastError());
    return nullptr;
}

}  // namespace obvh
