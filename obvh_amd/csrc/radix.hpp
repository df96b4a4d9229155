// radix.hpp -- stable LSD radix sort of (32-bit key, 32-bit value) pairs.
//
// One launch per 8-bit digit.  The digits' histograms of all passes are made
// beforehand, where the keys are made (radix_count).  A workgroup takes the
// next tile of 1024 to 8192 pairs, ranks its keys within each wave (lanes with
// the same digit find each other by eight ballots), publishes its digit counts
// and looks back over the earlier tiles' for its place, 64 tiles a trip to
// memory, then puts its pairs in digit order in LDS and writes them in runs.
// Counts are handed over with agent-scope accesses: one word holds a count and
// whether it is the tile's own or includes all before it.  (Onesweep: Adinets
// and Merrill, 2022; the look-back is Merrill and Garland's, 2016.)  A tile
// waits only for tiles taken before it, which wait for none after, and only so
// long: past the poll limit it counts the earlier tile's keys itself (the pass's
// input does not change), so the result never depends on the wait.
//
// Bound by latency: a pass over 1 M pairs takes 17 us for 16 MB moved (written
// without the LDS order 22 us; with 256 threads and one look-back thread per
// digit 25).  rocPRIM sorts up to 1 M pairs by merging: 22 launches, 152 us for
// 1 M pairs against 68.
#pragma once
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace obvh {

constexpr int kRadixBits = 8;
constexpr int kRadixBins = 1 << kRadixBits;
constexpr int kRadixThreads = 1024;
constexpr int kRadixWaves = kRadixThreads / kWave;
constexpr int kRadixGroups = kRadixThreads / kRadixBins;  // threads per bin in the look-back
constexpr int kRadixBack = 16;                            // earlier tiles a thread reads at once
constexpr uint32_t kRadixOwn = 1u << 30, kRadixAll = 2u << 30, kRadixMask = kRadixOwn - 1;
constexpr uint32_t kRadixMax = kRadixMask + 1;  // pairs, at most (nobody reads the last tile's word)
constexpr uint32_t kRadixPolls = 1u << 12;  // about a microsecond each

// Per pass: bin counts, then per tile and bin the published word, and the next
// tile; all zero before the sort.
struct RadixWs {
    uint32_t* hist;   // passes x 256
    uint32_t* next;   // passes
    uint32_t* state;  // passes x tiles x 256
    uint32_t words;   // of all three, contiguous from hist
};
// Pairs per thread: small inputs want more workgroups, large ones fewer tiles
// to look back over.  LBVH build with 1 / 2 / 4 / 8: 20 K faces 85 / 87 / 93 / 105 us,
// 100 K 150 / 106 / 110 / 121, 200 K 136 / 131 / 127 / 137, 1 M 334 / 273 / 242 / 246,
// 2 M 565 / 450 / 398 / 371.
inline int radix_items(uint32_t n) { return n <= 32768u ? 1 : n <= 131072u ? 2 : n <= 1250000u ? 4 : 8; }
inline uint32_t radix_tiles(uint32_t n) {
    const uint32_t tile = (uint32_t)radix_items(n) * kRadixThreads;
    return (n + tile - 1) / tile;
}
inline void radix_carve(RadixWs* ws, Carver& c, uint32_t n, int passes) {
    const size_t words = (size_t)passes * ((size_t)radix_tiles(n) + 1) * kRadixBins + 64;
    ws->hist = c.take<uint32_t>(words);
    ws->words = (uint32_t)words;
    ws->next = ws->hist ? ws->hist + (size_t)passes * kRadixBins : nullptr;
    ws->state = ws->hist ? ws->next + 64 : nullptr;
}

// One workgroup's counts of its keys' digits: h is passes x 256 in LDS, zeroed
// and summed by the caller's barriers.
template <int kPasses>
__device__ __forceinline__ void radix_count(uint32_t key, uint32_t (&h)[kPasses * kRadixBins]) {
#pragma unroll
    for (int p = 0; p < kPasses; ++p) atomicAdd(&h[p * kRadixBins + ((key >> (p * kRadixBits)) & (kRadixBins - 1))], 1u);
}

__device__ __forceinline__ uint32_t digit(uint32_t key, int pass) {
    return (key >> (pass * kRadixBits)) & (kRadixBins - 1);
}

// Ranks of a wave's keys (row i, this lane: element first + 64 i of n) among
// its earlier keys of the same digit; h: the wave's counts, zero before.
template <int kItems>
__device__ __forceinline__ void wave_rank(const uint32_t (&key)[kItems], uint32_t first, uint32_t n, int pass,
                                          uint32_t* h, uint32_t (&rank)[kItems]) {
    const uint64_t below = (1ull << lane_id()) - 1;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const uint32_t d = digit(key[i], pass);
        const bool valid = first + i * kWave < n;
        uint64_t same = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kRadixBits; ++b) {
            const bool bit = ((d >> b) & 1u) != 0;
            const uint64_t set = __ballot(bit);
            same &= bit ? set : ~set;
        }
        const uint32_t before = h[d];
        rank[i] = before + (uint32_t)__popcll(same & below);
        __builtin_amdgcn_wave_barrier();
        if (valid && (same & below) == 0) h[d] = before + (uint32_t)__popcll(same);
        __builtin_amdgcn_wave_barrier();
    }
}

// Inclusive scan over a wave.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)v, m, kWave);
        if (lane_id() >= m) v += o;
    }
    return v;
}

// Pass `pass`; vals_in == nullptr: the values are the keys' positions.
template <int kItems>
__global__ __launch_bounds__(kRadixThreads) void radix_pass(const uint32_t* __restrict__ keys_in,
                                                            const uint32_t* __restrict__ vals_in,
                                                            uint32_t* __restrict__ keys_out,
                                                            uint32_t* __restrict__ vals_out, uint32_t n, int pass,
                                                            uint32_t polls, RadixWs ws) {
    __shared__ uint32_t wh[kRadixWaves][kRadixBins];
    __shared__ uint32_t base[kRadixBins];
    __shared__ uint32_t part[kRadixGroups][kRadixBins];  // look-back: sums, bit 31: includes everything before
    __shared__ uint32_t wsum[kRadixBins / kWave], lsum[kRadixBins / kWave];
    __shared__ uint32_t skey[kItems * kRadixThreads], sval[kItems * kRadixThreads];  // the tile's pairs in bin order
    __shared__ uint32_t taken;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const uint32_t bin = tid % kRadixBins, group = tid / kRadixBins;
    if (tid == 0) taken = __hip_atomic_fetch_add(&ws.next[pass], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (uint32_t i = tid; i < kRadixWaves * kRadixBins; i += kRadixThreads) (&wh[0][0])[i] = 0;
    const uint32_t count = group == 0 ? ws.hist[pass * kRadixBins + bin] : 0u;
    __syncthreads();
    const uint32_t tile = taken;
    uint32_t* state = ws.state + ((size_t)pass * gridDim.x + tile) * kRadixBins + bin;

    const uint32_t first = tile * (kItems * kRadixThreads) + wave * (kItems * kWave) + lane;
    uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const uint32_t at = first + i * kWave;
        key[i] = at < n ? keys_in[at] : 0u;
        val[i] = vals_in ? (at < n ? vals_in[at] : 0u) : at;
    }
    wave_rank<kItems>(key, first, n, pass, wh[wave], rank);
    // exclusive scan of the whole sort's bin counts (the first 256 threads)
    uint32_t place = 0, own = 0, before = 0;
    bool done = false;
    uint32_t incl = wave_scan(count);
    if (group == 0) {  // whole waves
        if (lane == kWave - 1) wsum[wave] = incl;
    }
    __syncthreads();
    if (group == 0) {
        place = incl - count;
        for (uint32_t w = 0; w < wave; ++w) place += wsum[w];
        // the tile's count of the bin; the waves' places within it
#pragma unroll
        for (int w = 0; w < kRadixWaves; ++w) {
            const uint32_t c = wh[w][bin];
            wh[w][bin] = own;
            own += c;
        }
        st_agent(state, (tile == 0 ? kRadixAll : kRadixOwn) | own);
        // where the bin starts within the tile
        incl = wave_scan(own);
        if (lane == kWave - 1) lsum[wave] = incl;
    }
    __syncthreads();
    uint32_t local = 0;
    if (group == 0) {
        local = incl - own;
        for (uint32_t w = 0; w < wave; ++w) local += lsum[w];
#pragma unroll
        for (int w = 0; w < kRadixWaves; ++w) wh[w][bin] += local;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        if (first + i * kWave >= n) continue;
        const uint32_t j = wh[wave][digit(key[i], pass)] + rank[i];
        skey[j] = key[i];
        sval[j] = val[i];
    }
    // look back: the threads of a bin read kRadixBack earlier tiles each
    for (uint32_t seen = 0; seen < tile; seen += kRadixGroups * kRadixBack) {  // uniform
        const uint32_t from = seen + group * kRadixBack;
        const uint32_t want = from < tile ? min((uint32_t)kRadixBack, tile - from) : 0u;
        uint32_t sum = 0, got = 0;
        for (uint32_t poll = 0; got < want && poll < polls; ++poll) {
            uint32_t s[kRadixBack];
#pragma unroll
            for (int u = 0; u < kRadixBack; ++u)
                s[u] = (uint32_t)u >= got && (uint32_t)u < want ? ld_agent(state - (size_t)(from + u + 1) * kRadixBins)
                                                                : 0u;
#pragma unroll
            for (int u = 0; u < kRadixBack; ++u) {
                if ((uint32_t)u != got || s[u] == 0) continue;  // not yet published: read again from here
                sum += s[u] & kRadixMask;
                got = (s[u] & kRadixAll) ? want + 1 : got + 1;
            }
        }
#pragma unroll 1
        for (; got < want; ++got) {
            const uint32_t lo = (tile - 1 - (from + got)) * (kItems * kRadixThreads);
#pragma unroll 1
            for (uint32_t k = 0; k < kItems * kRadixThreads; ++k) sum += digit(keys_in[lo + k], pass) == bin ? 1u : 0u;
        }
        part[group][bin] = sum | (got > want ? 0x80000000u : 0u);
        __syncthreads();
        if (group == 0) {
            for (int g = 0; g < kRadixGroups && !done; ++g) {
                const uint32_t q = part[g][bin];
                before += q & 0x7FFFFFFFu;
                done = (q >> 31) != 0;
            }
        }
        if (!__syncthreads_or(group == 0 && !done)) break;
    }
    if (group == 0) {
        if (tile > 0) st_agent(state, kRadixAll | (before + own));
        base[bin] = place + before - local;
    }
    __syncthreads();
    // consecutive lanes write runs of a bin
    const uint32_t cnt = min((uint32_t)(kItems * kRadixThreads), n - tile * (kItems * kRadixThreads));
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        const uint32_t j = i * kRadixThreads + tid;
        if (j >= cnt) continue;
        const uint32_t k = skey[j], to = base[digit(k, pass)] + j;
        keys_out[to] = k;
        vals_out[to] = sval[j];
    }
}

// All passes over n <= kItems * 1024 pairs by one workgroup, in LDS; the
// result goes to keys and vals.
template <int kItems, int kPasses>
__global__ __launch_bounds__(kRadixThreads) void radix_small(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                             uint32_t n) {
    __shared__ uint32_t wh[kRadixWaves][kRadixBins];
    __shared__ uint32_t lsum[kRadixBins / kWave];
    __shared__ uint32_t skey[kItems * kRadixThreads], sval[kItems * kRadixThreads];
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const uint32_t first = wave * (kItems * kWave) + lane;
    uint32_t key[kItems], val[kItems], rank[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        val[i] = first + i * kWave;
        key[i] = val[i] < n ? keys[val[i]] : 0u;
    }
#pragma unroll 1
    for (int pass = 0; pass < kPasses; ++pass) {
        for (uint32_t i = tid; i < kRadixWaves * kRadixBins; i += kRadixThreads) (&wh[0][0])[i] = 0;
        __syncthreads();
        wave_rank<kItems>(key, first, n, pass, wh[wave], rank);
        __syncthreads();
        uint32_t own = 0, incl = 0;
        if (tid < kRadixBins) {  // whole waves
#pragma unroll
            for (int w = 0; w < kRadixWaves; ++w) {
                const uint32_t c = wh[w][tid];
                wh[w][tid] = own;
                own += c;
            }
            incl = wave_scan(own);
            if (lane == kWave - 1) lsum[wave] = incl;
        }
        __syncthreads();
        if (tid < kRadixBins) {
            uint32_t local = incl - own;
            for (uint32_t w = 0; w < wave; ++w) local += lsum[w];
#pragma unroll
            for (int w = 0; w < kRadixWaves; ++w) wh[w][tid] += local;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (first + i * kWave >= n) continue;
            const uint32_t j = wh[wave][digit(key[i], pass)] + rank[i];
            skey[j] = key[i];
            sval[j] = val[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kItems; ++i) {
            if (first + i * kWave >= n) continue;
            key[i] = skey[first + i * kWave];
            val[i] = sval[first + i * kWave];
        }
    }
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
        if (first + i * kWave >= n) continue;
        keys[first + i * kWave] = key[i];
        vals[first + i * kWave] = val[i];
    }
}

// kPasses passes (an even number) over n pairs, the values the keys' positions.
// keys: the keys, then the result with vals; keys_tmp, vals_tmp: scratch.
template <int kPasses>
inline void radix_sort(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t n,
                       const RadixWs& ws, uint32_t polls, hipStream_t stream) {
    static_assert(kPasses % 2 == 0, "the result is in the first buffers");
    if (n <= 4 * kRadixThreads) {  // LBVH build of 2000 faces: 57.6 us, with the launches below 69.7; of 5120 no gain
        auto k = n <= kRadixThreads       ? radix_small<1, kPasses>
                 : n <= 2 * kRadixThreads ? radix_small<2, kPasses>
                                          : radix_small<4, kPasses>;
        hipLaunchKernelGGL(k, dim3(1), dim3(kRadixThreads), 0, stream, keys, vals, n);
        return;
    }
    for (int p = 0; p < kPasses; ++p) {
        const bool odd = (p & 1) != 0;
        const int items = radix_items(n);
        auto k = items == 1 ? radix_pass<1> : items == 2 ? radix_pass<2> : items == 4 ? radix_pass<4> : radix_pass<8>;
        hipLaunchKernelGGL(k, dim3(radix_tiles(n)), dim3(kRadixThreads), 0, stream, odd ? keys_tmp : keys,
                           p == 0 ? nullptr : (odd ? vals_tmp : vals), odd ? keys : keys_tmp, odd ? vals : vals_tmp, n,
                           p, polls, ws);
    }
}

}  // namespace obvh
