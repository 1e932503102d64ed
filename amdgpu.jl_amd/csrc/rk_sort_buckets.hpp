// Sorts of up to 2^20 keys of 4 and 8 bytes by splitters (included by rk_sort.hip).
//
//   sort_sample_kernel     fetches a sample of the keys (larger sorts only; smaller ones fetch it where they rank it)
//   sort_splitters_kernel  ranks the sample by counting and keeps every SB_OVER-th of it: k - 1 splitters
//   sort_tile_kernel       sorts every tile of 4096 keys by bucket -- between which splitters a key lies -- and leaves a table
//                          of where the buckets start in every tile
//   sort_bucket_kernel     a workgroup a bucket: collects its keys from all tiles, sorts them in LDS and writes the result
//
// A radix pass over 10^6 keys is bound by latency, and 8-byte keys take eight of them, one after the other; the four kernels
// here are as many as two passes take and do not get more with the width of the key.  No key is moved to its bucket: a bucket
// takes its runs out of the tiles, so nothing has to know the buckets' sizes before it writes.
// Radix passes -> so, us a call: sortperm Int64[1000003] 136.3 -> 42.3 (kernels 2.9, 5.7, 15.9 and 19.1), Float32 66.0 -> 39;
// sort Float32[1000003] 63.9 -> 33.8, Float64 132 -> 38, Int64 of 20 bits 79.7 -> 38; sort Float32[150000] 48.6 -> 26.0.  Each of
// the kernels moves what it moves in a fraction of its time: what is left is their chains of dependent loads and barriers.
//
// Order: keys are compared together with their index -- (key, index) is a strict order -- so equal keys are split between
// buckets like any others, a bucket's size does not depend on how the keys are distributed, and the permutation is the stable
// one although no kernel here keeps the order of what it moves.
//
// Bucket sizes: a bucket holds the keys between two neighbours among k sampled quantiles, SB_OVER samples apart, so its size
// is spread like a Gamma variable of that shape around n / k.  LDS has room for SB_CAP keys, 2.75 times n / k at 2^20 keys
// and more below; one bucket in 2 million is larger (at 2^20 keys; the fewer the keys, the fewer) and is sorted in memory: such
// a call takes 0.4 to 1 ms.  Where samples are taken depends on the number of keys alone, so for an input it always happens or
// never does.  Nothing but the time depends on a bucket's being small.
#pragma once

#include "rk_common.hpp"

namespace rk {

constexpr uint32_t SB_OVER = 16;                 // samples a bucket
constexpr uint32_t SB_MAX_K = 256, SB_MAX_TILES = 256;
constexpr int SB_SPL_BLOCK = 512, SB_SPL_EACH = 16;
constexpr uint32_t SB_DIRECT_SAMPLES = 1024;     // up to so many samples every workgroup that ranks some fetches all of them
constexpr int SB_TILE_BLOCK = 1024, SB_TILE_ITEMS = 4, SB_TILE = SB_TILE_BLOCK * SB_TILE_ITEMS;
constexpr int SB_SORT_BLOCK = 1024, SB_SORT_ITEMS = 11;
constexpr uint32_t SB_CAP = SB_SORT_BLOCK * SB_SORT_ITEMS;   // keys sorted in LDS
constexpr uint32_t SB_BINS = 4096;               // of a bucket, in LDS
constexpr uint32_t SB_MAX_BIN = 32;              // largest bin whose keys are ranked by comparing them with each other
constexpr uint32_t SB_DIVIDE_BIN = 16;           // if there is a larger one: largest that is not divided
constexpr uint32_t SB_TOGETHER = 24;             // lanes of a wave that go to the bin of the first: from here on they add to it once

// Buckets of a sort of n keys: a power of two (the search among the splitters has no remainder), n / k <= 512 while that is a
// workgroup a compute unit at most, n / k <= 4096 at 2^20 keys.
__host__ __device__ inline uint32_t sb_buckets(int64_t n) {
    uint32_t k = 4;
    while ((int64_t)k * 512 < n && k < SB_MAX_K) k *= 2;
    return k;
}

// Where the j-th of s samples is taken: somewhere in the j-th of s equal stretches (a multiplicative hash of j decides where),
// so that samples are in index order and a step that the data repeats is not met in step.
__device__ __forceinline__ uint32_t sb_sample_pos(uint32_t j, uint32_t s, uint32_t n) {
    const uint32_t a = (uint32_t)((uint64_t)j * n / s), b = (uint32_t)((uint64_t)(j + 1u) * n / s);
    uint32_t h = (j + 1u) * 0x9e3779b1u;
    h ^= h >> 15;
    h *= 0x85ebca77u;
    return a + __umulhi(h, b - a);
}

// ---- splitters -------------------------------------------------------------------------------------------------
// s = k * SB_OVER samples, all in every workgroup's LDS; a workgroup ranks SB_SPL_EACH of them against all.  s^2 comparisons
// are 16.8 million at most, 1.3 us of the chip's vector instructions; sorting the samples in one workgroup would leave the
// others idle for longer.  ctl: of sorts that run no radix pass.
// With many samples it is the fetching that counts -- a line of memory for every sample, in every workgroup -- and a kernel in
// front packs them (compact).
template <typename T>
__global__ __launch_bounds__(256) void sort_sample_kernel(const T* __restrict__ keys, uint32_t n, int rev, uint32_t s, typename SortKey<T>::U* __restrict__ compact) {
    typedef typename SortKey<T>::U U;
    const uint32_t j = blockIdx.x * 256u + threadIdx.x;
    if (j < s) compact[j] = enc_bits<T>(__builtin_bit_cast(U, keys[sb_sample_pos(j, s, n)]), rev, (U)0);
}

template <typename T, bool DIRECT>
__global__ __launch_bounds__(SB_SPL_BLOCK) void sort_splitters_kernel(const T* __restrict__ keys, uint32_t n, int rev, SortCtl* ctl, uint32_t k,
                                                                      const typename SortKey<T>::U* __restrict__ compact,
                                                                      typename SortKey<T>::U* __restrict__ spl_key, uint32_t* __restrict__ spl_pos) {
    typedef typename SortKey<T>::U U;
    constexpr uint32_t PARTS = SB_SPL_BLOCK / SB_SPL_EACH, MOST = DIRECT ? SB_DIRECT_SAMPLES : SB_MAX_K * SB_OVER, UNR = MOST / SB_SPL_BLOCK;
    __shared__ U smp[MOST];
    __shared__ uint32_t below[SB_SPL_EACH];
    const uint32_t tid = threadIdx.x, s = k * SB_OVER;
    U v[UNR];
#pragma unroll
    for (uint32_t u = 0; u < UNR; ++u) {
        uint32_t j = tid + u * SB_SPL_BLOCK;
        j = j < s ? j : s - 1u;
        v[u] = DIRECT ? __builtin_bit_cast(U, keys[sb_sample_pos(j, s, n)]) : compact[j];
    }
    if (ctl != nullptr && blockIdx.x == 0 && tid == 0) ctl->nexec = 0u;
    if (tid < SB_SPL_EACH) below[tid] = 0u;
#pragma unroll
    for (uint32_t u = 0; u < UNR; ++u) {
        const uint32_t j = tid + u * SB_SPL_BLOCK;
        if (j < s) smp[j] = DIRECT ? enc_bits<T>(v[u], rev, (U)0) : v[u];
    }
    __syncthreads();
    // of the samples in front an equal one counts as smaller
    const uint32_t j0 = blockIdx.x * SB_SPL_EACH, j = j0 + tid % SB_SPL_EACH, i0 = tid / SB_SPL_EACH;
    const U mine = smp[j];
    uint32_t c = 0, i = i0;
#pragma unroll 8
    for (; i < j0; i += PARTS) c += smp[i] <= mine ? 1u : 0u;
    if (i < j0 + SB_SPL_EACH) {                              // (PARTS >= SB_SPL_EACH: once at most)
        const U x = smp[i];
        c += (x < mine || (x == mine && i < j)) ? 1u : 0u;
        i += PARTS;
    }
#pragma unroll 8
    for (; i < s; i += PARTS) c += smp[i] < mine ? 1u : 0u;
    atomicAdd(&below[tid % SB_SPL_EACH], c);
    __syncthreads();
    if (tid < SB_SPL_EACH) {
        const uint32_t r = below[tid];
        if (r != 0u && r % SB_OVER == 0u) {
            spl_key[r / SB_OVER - 1u] = mine;
            spl_pos[r / SB_OVER - 1u] = sb_sample_pos(j, s, n);
        }
    }
}

// ---- tiles --------------------------------------------------------------------------------------------------------
// Every key searches the splitters in LDS, takes its place among the tile's keys of the bucket with an LDS atomic (their order
// does not matter), and the tile is written in the order of the buckets (sortperm: with the keys' indices in the tile).
// table[tile][bucket] = where the bucket starts in the tile | its size << 16.  Summed down the tiles that is also how many keys
// lie in the buckets in front and how many in the bucket, so no workgroup adds to anything that others add to.
template <typename T, bool PERM>
__global__ __launch_bounds__(SB_TILE_BLOCK) void sort_tile_kernel(const T* __restrict__ keys, uint32_t n, int rev, uint32_t k,
                                                                  const typename SortKey<T>::U* __restrict__ spl_key,
                                                                  const uint32_t* __restrict__ spl_pos, uint32_t* __restrict__ table,
                                                                  typename SortKey<T>::U* __restrict__ tile_key, uint16_t* __restrict__ tile_val) {
    typedef typename SortKey<T>::U U;
    constexpr int BLOCK = SB_TILE_BLOCK, ITEMS = SB_TILE_ITEMS;
    __shared__ U lds_key[SB_TILE];
    __shared__ uint16_t lds_val[PERM ? SB_TILE : 1];
    __shared__ U skey[SB_MAX_K];
    __shared__ uint32_t spos[SB_MAX_K], cnt[SB_MAX_K], wsum[SB_MAX_K / WAVE];
    const uint32_t tid = threadIdx.x, e0 = blockIdx.x * (uint32_t)SB_TILE;
    U key[ITEMS];
    uint32_t bucket[ITEMS], rank[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t e = e0 + tid + i * BLOCK;
        key[i] = __builtin_bit_cast(U, keys[e < n ? e : n - 1u]);
    }
    if (tid < k) {
        skey[tid] = tid < k - 1u ? spl_key[tid] : (U)0;
        spos[tid] = tid < k - 1u ? spl_pos[tid] : 0u;
        cnt[tid] = 0u;
    }
    __syncthreads();
    bool tie = false;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) { key[i] = enc_bits<T>(key[i], rev, (U)0); bucket[i] = 0u; }
    // splitters below the key: the searches of a lane's keys go side by side
    for (uint32_t step = k / 2u; step != 0u; step /= 2u) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) bucket[i] += skey[bucket[i] + step - 1u] < key[i] ? step : 0u;
    }
    // one that equals the key: the index decides
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) tie = tie || (bucket[i] < k - 1u && skey[bucket[i]] == key[i]);
    if (tie) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) bucket[i] = 0u;
        for (uint32_t step = k / 2u; step != 0u; step /= 2u) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const U x = skey[bucket[i] + step - 1u];
                bucket[i] += (x < key[i] || (x == key[i] && spos[bucket[i] + step - 1u] <= e0 + tid + i * BLOCK)) ? step : 0u;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        rank[i] = 0u;
        if (e0 + tid + i * BLOCK < n) rank[i] = atomicAdd(&cnt[bucket[i]], 1u);
    }
    __syncthreads();
    uint32_t c = 0u, inc = 0u;
    if (tid < SB_MAX_K) {
        if (tid < k) c = cnt[tid];
        inc = wave_scan_inclusive(c, OpAdd(), 0u);
        if (tid % WAVE == WAVE - 1) wsum[tid / WAVE] = inc;
    }
    __syncthreads();
    if (tid < k) {
        uint32_t start = inc - c;
        for (uint32_t w = 0; w < tid / WAVE; ++w) start += wsum[w];
        cnt[tid] = start;
        table[blockIdx.x * k + tid] = start | c << 16;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (e0 + tid + i * BLOCK < n) {
            const uint32_t p = cnt[bucket[i]] + rank[i];
            lds_key[p] = key[i];
            if constexpr (PERM) lds_val[p] = (uint16_t)(tid + i * BLOCK);
        }
    }
    __syncthreads();
    const uint32_t m = n - e0 < (uint32_t)SB_TILE ? n - e0 : (uint32_t)SB_TILE;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t p = tid + i * BLOCK;
        if (p < m) {
            tile_key[e0 + p] = lds_key[p];
            if constexpr (PERM) tile_val[e0 + p] = lds_val[p];
        }
    }
}

// ---- radix passes in LDS ------------------------------------------------------------------------------------------
// One stable pass over m keys of a workgroup of 16 waves by an 8-bit digit: item i of lane l of wave w is element
// (w * per + i) * 64 + l, before and after; `per` items a lane are in use.  cnt: 16 x 256 words.
template <bool PERM, int ITEMS, typename U, typename Digit>
__device__ __forceinline__ void sb_radix_pass(U (&key)[ITEMS], uint32_t (&val)[PERM ? ITEMS : 1], uint32_t per, uint32_t m, Digit&& digit, U* lds_key,
                                              uint32_t* lds_val, uint32_t* cnt, uint32_t* wsum) {
    constexpr int BLOCK = 1024, NW = BLOCK / WAVE;
    const uint32_t tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, first = wave * per * WAVE + lane;
    uint32_t* wcnt = cnt + wave * 256u;
    uint32_t rank[ITEMS];
    *(uint4*)&cnt[tid * 4u] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i >= per) continue;
        const bool valid = first + i * WAVE < m;
        const uint32_t d = digit(key[i], val[PERM ? i : 0]);
        uint32_t same_lo, same_hi;
        match_digit_halves(d, same_lo, same_hi);
        const uint64_t vm = __ballot(valid);
        same_lo &= (uint32_t)vm;
        same_hi &= (uint32_t)(vm >> 32);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi, __builtin_amdgcn_mbcnt_lo(same_lo, 0u));
        rank[i] = __hip_atomic_load(&wcnt[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) + below;
        __builtin_amdgcn_wave_barrier();
        if (valid && below == 0u)
            __hip_atomic_fetch_add(&wcnt[d], (uint32_t)__builtin_popcount(same_lo) + (uint32_t)__builtin_popcount(same_hi), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t total = 0u, inc = 0u;
    if (tid < 256u) {
        for (int w = 0; w < NW; ++w) total += cnt[w * 256 + tid];
        inc = wave_scan_inclusive(total, OpAdd(), 0u);
        if (lane == WAVE - 1) wsum[wave] = inc;
    }
    __syncthreads();
    if (tid < 256u) {
        uint32_t at = inc - total;
        for (uint32_t w = 0; w < wave; ++w) at += wsum[w];
        for (int w = 0; w < NW; ++w) {
            const uint32_t c = cnt[w * 256 + tid];
            cnt[w * 256 + tid] = at;
            at += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i < per && first + i * WAVE < m) {
            const uint32_t p = wcnt[digit(key[i], val[PERM ? i : 0])] + rank[i];
            lds_key[p] = key[i];
            if constexpr (PERM) lds_val[p] = val[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)i < per && first + i * WAVE < m) {
            key[i] = lds_key[first + i * WAVE];
            if constexpr (PERM) val[i] = lds_val[first + i * WAVE];
        }
    }
}

// ---- a bucket ------------------------------------------------------------------------------------------------------
// Bitonic sort of x[0, m) (with y) by the whole workgroup, in LDS or in memory.  The variant whose comparisons all put the
// smaller element first: elements from m on would be larger than any and never move, so they need not exist.
template <bool PERM, typename U>
__device__ __forceinline__ void sb_bitonic(U* x, uint32_t* y, uint32_t m) {
    uint32_t half = 1u;
    while (half * 2u < m) half *= 2u;
    auto order = [&](uint32_t a, uint32_t b) {
        if (b >= m) return;
        const U xa = x[a], xb = x[b];
        if constexpr (PERM) {
            const uint32_t ya = y[a], yb = y[b];
            if (xb < xa || (xb == xa && yb < ya)) { x[a] = xb; x[b] = xa; y[a] = yb; y[b] = ya; }
        } else {
            if (xb < xa) { x[a] = xb; x[b] = xa; }
        }
    };
    for (uint32_t h = 1u; h <= half; h *= 2u) {              // runs of h become runs of 2 h
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < half; i += blockDim.x) {
            const uint32_t o = i & (h - 1u), a = (i - o) * 2u;
            order(a + o, a + 2u * h - 1u - o);
        }
        for (uint32_t j = h / 2u; j != 0u; j /= 2u) {
            __syncthreads();
            for (uint32_t i = threadIdx.x; i < half; i += blockDim.x) {
                const uint32_t o = i & (j - 1u), a = (i - o) * 2u + o;
                order(a, a + j);
            }
        }
    }
    __syncthreads();
}

// Inside a bucket the keys are spread over bins by a monotone, nearly linear map of their distance from the smallest, in no order, and a
// key's place in its bin is the number of smaller keys there: a bin holds a key or two, and a wave compares as often as the largest bin
// it meets has keys.
// sortperm: what is spread are the highest 32 bits that vary of the distance and, behind it, the index, so that few values, many times
// over, are spread as well.
// Should a bin exceed SB_MAX_BIN -- a bucket around zero, where the keys of floats are far from linear; values in clusters, or few of
// them, far apart -- every such bin is divided once more, into as many as it has keys (bins of equal keys: by the index; without one they
// need no order), and those again, SB_LEVELS times.  What even that does not spread is sorted by comparisons, still in LDS.
// A division takes 3 to 5 us, most of it fetching code that nothing else runs; comparing 4096 keys 50.  2^20 keys, us a call, four radix passes or
// fewer / comparing what one division by the bucket's range does not spread / so: sort Int32 (id << 16) + small number 45 / 86 / 48, Float64 of
// whole numbers below 16384 86 / 76 / 51, Float32 of them 56 / 70 / 50; sortperm Int64 (id << 32) + small number 68 / 168 / 59, Float32 of 256
// values in order 45 / 100 / 43, at random 45 / 58 / 53, of 16 46 / 62 / 52, Int32 of 256 42 / 46 / 42, of 16 42 / 50 / 46.
constexpr int SB_LEVELS = 6;

// LDS of a workgroup that sorts a bucket of up to ITEMS * BLOCK keys.
template <typename U, bool PERM, int ITEMS, int BLOCK, uint32_t BINS> struct SbLds {
    static constexpr uint32_t CAP = (uint32_t)(ITEMS * BLOCK);
    // keys and indices of the bucket; while bins are divided, the sizes of the new ones and, for a bin that starts at q, smallest and largest
    // key and index at q / SB_DIVIDE_BIN
    static constexpr uint32_t LARGE = CAP / SB_DIVIDE_BIN;
    static constexpr size_t KEYS = (size_t)CAP * sizeof(U), POOL = KEYS + (PERM ? (size_t)CAP * 4 : 0);
    static constexpr size_t DIVIDE = (size_t)CAP * 4 + (size_t)LARGE * (2 * sizeof(U) + (PERM ? 12 : 4));
    alignas(16) char pool[POOL > DIVIDE ? POOL : DIVIDE];
    alignas(16) uint32_t bins[BINS + 4];
    uint32_t part[4][BLOCK / WAVE];
    U key_lo, key_hi;                                        // smallest and largest key of the bucket, and index
    uint32_t val_lo, val_hi;
    // by one thread, before a barrier
    __device__ __forceinline__ void init() { key_lo = (U)~(U)0; key_hi = (U)0; val_lo = ~0u; val_hi = 0u; }
};

template <typename U> __device__ __forceinline__ U sb_uniform(U x) {
    if constexpr (sizeof(U) == 4) return (U)__builtin_amdgcn_readfirstlane((int)x);
    else return (U)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x) | (U)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32)) << 32;
}

// Bits of x.
template <typename U> __device__ __forceinline__ uint32_t sb_bits(U x) {
    if constexpr (sizeof(U) == 4) return x == 0u ? 0u : 32u - (uint32_t)__clz((int)x);
    else return x == 0ull ? 0u : 64u - (uint32_t)__clzll((long long)x);
}

// Words of LDS that other threads write at the same time.
template <typename U> __device__ __forceinline__ void sb_put(U* p, U x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
template <typename U> __device__ __forceinline__ U sb_get(const U* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// The highest 32 bits of d, a distance of up to `bits` bits, with `word` behind it (sortperm).
template <bool PERM, typename U> __device__ __forceinline__ uint32_t sb_code(U d, uint32_t bits, uint32_t word) {
    const uint32_t top = sizeof(U) == 4 || bits <= 32u ? (uint32_t)d : (uint32_t)((uint64_t)d >> (bits - 32u));
    if constexpr (PERM) return bits >= 32u ? top : (uint32_t)__builtin_amdgcn_alignbit(top, word, bits);
    else return bits >= 32u || bits == 0u ? top : top << (32u - bits);
}

// Thread t holds the elements t, t + BLOCK, ... of the m of the bucket, in any order (for those from m on, where others of the
// thread's row exist, one that does); store(place, key, index) gets each of them.  KNOWN: the indices lie in [vlo, vhi]; otherwise
// the smallest and the largest are looked for.
template <bool PERM, bool KNOWN, int ITEMS, int BLOCK, uint32_t BINS, typename U, typename Store>
__device__ __forceinline__ void sb_sort_bucket(U (&key)[ITEMS], uint32_t (&val)[PERM ? ITEMS : 1], uint32_t m, SbLds<U, PERM, ITEMS, BLOCK, BINS>& lds,
                                               uint32_t vlo, uint32_t vhi, Store&& store) {
    typedef SbLds<U, PERM, ITEMS, BLOCK, BINS> Lds;
    constexpr int NW = BLOCK / WAVE, PER = (int)BINS / BLOCK;
    constexpr uint32_t CAP = Lds::CAP;
    constexpr bool RANGE = PERM && !KNOWN;
    static_assert(PER % 4 == 0, "a thread scans PER bins, four at a time");
    static_assert(CAP < 1u << 16, "place and size in 32 bits");
    U* const lds_key = (U*)lds.pool;
    uint32_t* const lds_val = (uint32_t*)(lds.pool + Lds::KEYS);        // (sortperm only)
    auto& bins = lds.bins;
    auto& part = lds.part;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    U lo = (U)~(U)0, hi = (U)0;
    uint32_t rank[ITEMS];
    if constexpr (RANGE) { vlo = ~0u; vhi = 0u; }
    m = sb_uniform(m);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < PER; c += 4) *(uint4*)&bins[tid * PER + c] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)(i * BLOCK) < m) {
            lo = key[i] < lo ? key[i] : lo;
            hi = key[i] > hi ? key[i] : hi;
            if constexpr (RANGE) {
                vlo = val[i] < vlo ? val[i] : vlo;
                vhi = val[i] > vhi ? val[i] : vhi;
            }
        }
    }
    lo = wave_reduce(lo, OpMin());
    hi = wave_reduce(hi, OpMax());
    if (lane == 0) { atomicMin(&lds.key_lo, lo); atomicMax(&lds.key_hi, hi); }
    if constexpr (RANGE) {
        vlo = wave_reduce(vlo, OpMin());
        vhi = wave_reduce(vhi, OpMax());
        if (lane == 0) { atomicMin(&lds.val_lo, vlo); atomicMax(&lds.val_hi, vhi); }
    }
    __syncthreads();
    lo = sb_uniform(lds.key_lo);
    hi = sb_uniform(lds.key_hi);
    const U span = hi - lo;
    const uint32_t bits = sb_bits(span);
    if constexpr (RANGE) {
        vlo = sb_uniform(lds.val_lo);
        vhi = sb_uniform(lds.val_hi);
    }
    const uint32_t vspan = vhi - vlo, vshift = vspan == 0u ? 0u : 32u - sb_bits(vspan);
    const auto word_of = [&](uint32_t v) -> uint32_t { return PERM ? (v - vlo) << vshift : 0u; };
    // a bin is one value; sortperm: of equal keys, one index
    const bool exact = PERM ? bits == 0u && vspan < BINS : span < (U)BINS;
    // code * scale < BINS * 2^32: the last bin is BINS - 1.  (The two roundings and the reciprocal are off by 3 units of 2^-24
    // at most, the last factor is 8 units below 1.)
    const uint32_t most_code = sb_code<PERM>(span, bits, vspan << vshift);
    const uint32_t scale = exact ? 0u : sb_uniform((uint32_t)((float)BINS * 4294967296.f * __builtin_amdgcn_rcpf((float)most_code + 1.f) * (1.f - 0x1p-21f)));
    auto code_of = [&](U x, uint32_t v) -> uint32_t {
        asm volatile("" : "+v"(x));                // computed again at every use: kept, the bins of eleven keys spilled 20 registers
        return sb_code<PERM>((U)(x - lo), bits, word_of(v));
    };
    auto bin_of = [&](U x, uint32_t v) -> uint32_t {
        if (exact) return PERM ? v - vlo : (uint32_t)(x - lo);
        return __umulhi(code_of(x, v), scale);
    };
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        rank[i] = 0u;
        if ((uint32_t)(i * BLOCK) >= m) continue;
        const bool valid = tid + i * BLOCK < m;
        const uint32_t b = bin_of(key[i], val[PERM ? i : 0]), b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
        const uint64_t same = __ballot(valid && b == b0);
        const uint32_t together = (uint32_t)__popcll(same);
        if (together >= SB_TOGETHER) {                          // (lane 0 is one of them)
            if (lane == 0u) rank[i] = atomicAdd(&bins[b0], together);
            rank[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)rank[i]) + __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
            if (valid && b != b0) rank[i] = atomicAdd(&bins[b], 1u);
        } else if (valid) {
            rank[i] = atomicAdd(&bins[b], 1u);
        }
    }
    __syncthreads();
    uint32_t c[PER], sum = 0u, most = 0u;
#pragma unroll
    for (int j = 0; j < PER; j += 4) {
        const uint4 q = *(const uint4*)&bins[tid * PER + j];
        c[j] = q.x; c[j + 1] = q.y; c[j + 2] = q.z; c[j + 3] = q.w;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) { sum += c[j]; most = c[j] > most ? c[j] : most; }
    const uint32_t inc = wave_scan_inclusive(sum, OpAdd(), 0u);
    most = wave_reduce(most, OpMax());
    if (lane == WAVE - 1) { part[0][wave] = inc; part[1][wave] = most; }
    __syncthreads();
    uint32_t first = inc - sum, largest = 0u;
    for (int w = 0; w < NW; ++w) {
        if ((uint32_t)w < wave) first += part[0][w];
        largest = part[1][w] > largest ? part[1][w] : largest;
    }
    largest = sb_uniform(largest);
#pragma unroll
    for (int j = 0; j < PER; ++j) { const uint32_t q = c[j]; c[j] = first; first += q; }
#pragma unroll
    for (int j = 0; j < PER; j += 4) *(uint4*)&bins[tid * PER + j] = make_uint4(c[j], c[j + 1], c[j + 2], c[j + 3]);
    if (tid == 0) bins[BINS] = m;
    __syncthreads();
    // elements [q0, q1) that come before one, which stands at p
    auto smaller = [&](U x, uint32_t v, uint32_t q0, uint32_t q1) -> uint32_t {
        uint32_t r = 0u;
        constexpr uint32_t FLIGHT = PERM ? 4u : 2u;
        for (uint32_t q = q0; q < q1; q += FLIGHT) {
            U o[FLIGHT];
            uint32_t ov[FLIGHT];
#pragma unroll
            for (uint32_t j = 0; j < FLIGHT; ++j) {
                const uint32_t at = q + j < q1 ? q + j : q;
                o[j] = lds_key[at];
                ov[j] = PERM ? lds_val[PERM ? at : 0] : at;
            }
#pragma unroll
            for (uint32_t j = 0; j < FLIGHT; ++j) r += q + j < q1 && (o[j] < x || (o[j] == x && ov[j] < v)) ? 1u : 0u;
        }
        return r;
    };
    if (exact || largest <= SB_MAX_BIN) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (tid + i * BLOCK < m) {
                const uint32_t p = bins[bin_of(key[i], val[PERM ? i : 0])] + rank[i];
                lds_key[p] = key[i];
                if constexpr (PERM) lds_val[p] = val[i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = tid + i * BLOCK;
            if (p >= m) continue;
            const U x = lds_key[p];
            const uint32_t v = PERM ? lds_val[PERM ? p : 0] : p;
            if (exact) {                                                // nothing to compare
                store(p, x, v);
            } else {
                const uint32_t b = bin_of(x, v), q0 = bins[b];
                store(q0 + smaller(x, v, q0, bins[b + 1u]), x, v);
            }
        }
        return;
    }
    // rank: from here on, where the element's bin starts, and of a bin that can be compared its size << 16 and the element's place in
    // it << 24, of others the element's place << 16
    constexpr uint32_t LARGE = 0x80000000u;
    constexpr int ROWS = ITEMS > 8 ? 4 : 2;                             // whose reads are in flight together
    static_assert(SB_MAX_BIN <= 64u && CAP < 1u << 14, "start, size and place in 31 bits");
    uint32_t* const sub = (uint32_t*)lds.pool;
    U* const bin_lo = (U*)(lds.pool + (size_t)CAP * 4);
    U* const bin_hi = bin_lo + Lds::LARGE;
    uint32_t* const bin_size = (uint32_t*)(bin_hi + Lds::LARGE);
    uint32_t* const bin_vlo = bin_size + Lds::LARGE;                    // (sortperm only)
    uint32_t* const bin_vhi = bin_vlo + Lds::LARGE;
    const auto entry = [](uint32_t r) { return (r & 0xffffu) / SB_DIVIDE_BIN % Lds::LARGE; };
    const auto place_in_bin = [](uint32_t r) { return (r & LARGE) != 0u ? (r & ~LARGE) >> 16 : r >> 24; };
    const auto divides = [](uint32_t r) { return (r & LARGE) != 0u || (r >> 16 & 0xffu) > SB_DIVIDE_BIN; };
    // Of the lanes side by side that go to one entry, the first: 64 that write to one word of LDS take 70 cycles.  (All lanes call.)
    const auto first_of_run = [](uint32_t at) { return (uint32_t)__builtin_amdgcn_update_dpp((int)~at, (int)at, 0x138, 0xf, 0xf, false) != at; };
    const auto enter = [&](bool valid, uint32_t q0, uint32_t size, uint32_t place) -> uint32_t {
        const bool writes = valid && size > SB_DIVIDE_BIN;
        if (first_of_run(writes ? q0 : ~0u) && writes) sb_put(&bin_size[q0 / SB_DIVIDE_BIN], size);
        return size <= SB_MAX_BIN ? q0 | size << 16 | place << 24 : LARGE | q0 | place << 16;
    };
#pragma unroll
    for (int i0 = 0; i0 < ITEMS; i0 += ROWS) {
        uint32_t q0[ROWS], q1[ROWS];
#pragma unroll
        for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
            if ((uint32_t)((i0 + j) * BLOCK) >= m) continue;
            const uint32_t b = bin_of(key[i0 + j], val[PERM ? i0 + j : 0]);
            q0[j] = bins[b];
            q1[j] = bins[b + 1u];
        }
#pragma unroll
        for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
            if ((uint32_t)((i0 + j) * BLOCK) >= m) continue;
            rank[i0 + j] = enter(tid + (i0 + j) * BLOCK < m, q0[j], q1[j] - q0[j], rank[i0 + j]);
        }
    }
    // How bins are first divided: as though their keys were spread evenly in them, with less than 2/5 of the bucket in the largest (around
    // zero, floats have up to 1/20 in a bin, Float64 1/4; two values would have half), otherwise from their smallest to their largest key.
    // Evenly, bins of equal keys are told from others first, unless 4-byte keys have less than 1/8 in the largest: the float buckets
    // around zero of sorts up to 2^20 keys are what those sorts wait for (sort Float32[2^20] 35.8 -> 34.7 us; 64 equal keys a bin 44 -> 51).
    constexpr bool UNSEEN = sizeof(U) == 4 && ITEMS > 8;
    bool any_mixed = true;                                              // there is a bin of different keys
    for (int level = 0; level < SB_LEVELS && largest > SB_MAX_BIN; ++level) {
        const bool evenly = level == 0 && largest * 5u <= m * 2u, unseen = UNSEEN && evenly && largest * 8u <= m;
        if (level != 0) __syncthreads();
        for (uint32_t i = tid; i < m; i += BLOCK) sub[i] = 0u;
        // the range of every bin: from any of its elements, then those outside what is known move it, a few of them first: of a few keys
        // many times over, all 64 lanes of a wave would move the same range, one after the other
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (unseen || (uint32_t)(i * BLOCK) >= m) continue;
            const bool writes = tid + i * BLOCK < m && divides(rank[i]);
            const uint32_t at = entry(rank[i]);
            if (first_of_run(writes ? at : ~0u) && writes) {
                sb_put(&bin_lo[at], key[i]);
                sb_put(&bin_hi[at], key[i]);
                if (PERM && !evenly) { sb_put(&bin_vlo[at], val[PERM ? i : 0]); sb_put(&bin_vhi[at], val[PERM ? i : 0]); }
            }
        }
        __syncthreads();
        bool mixed = false;
        if (evenly && !unseen) {
#pragma unroll
            for (int i0 = 0; i0 < ITEMS; i0 += ROWS) {
                if ((uint32_t)(i0 * BLOCK) >= m) continue;
                U from[ROWS], to[ROWS];
#pragma unroll
                for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                    const uint32_t at = entry(rank[i0 + j]);
                    from[j] = sb_get(&bin_lo[at]);
                    to[j] = sb_get(&bin_hi[at]);
                }
#pragma unroll
                for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                    const int i = i0 + j;
                    if (tid + i * BLOCK < m && divides(rank[i]) && key[i] != from[j]) {
                        mixed = true;
                        if (to[j] == from[j]) sb_put(&bin_hi[entry(rank[i])], key[i]);
                    }
                }
            }
        } else if (!unseen) {
            const auto move = [&](int i, U from, U to, uint32_t vfrom, uint32_t vto) {
                if (tid + i * BLOCK < m && divides(rank[i])) {
                    const uint32_t at = entry(rank[i]);
                    mixed = mixed || key[i] != from || key[i] != to;
                    if (key[i] < from) atomicMin(&bin_lo[at], key[i]);
                    if (key[i] > to) atomicMax(&bin_hi[at], key[i]);
                    if constexpr (PERM) {
                        if (val[i] < vfrom) atomicMin(&bin_vlo[at], val[i]);
                        if (val[i] > vto) atomicMax(&bin_vhi[at], val[i]);
                    }
                }
            };
            if (lane % 16u == 0u) {
                const uint32_t at = entry(rank[0]);
                move(0, sb_get(&bin_lo[at]), sb_get(&bin_hi[at]), PERM ? sb_get(&bin_vlo[at]) : 0u, PERM ? sb_get(&bin_vhi[at]) : 0u);
            }
#pragma unroll
            for (int i0 = 0; i0 < ITEMS; i0 += ROWS) {
                if ((uint32_t)(i0 * BLOCK) >= m) continue;
                U from[ROWS], to[ROWS];
                uint32_t vfrom[ROWS], vto[ROWS];
#pragma unroll
                for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                    const uint32_t at = entry(rank[i0 + j]);
                    from[j] = sb_get(&bin_lo[at]);
                    to[j] = sb_get(&bin_hi[at]);
                    vfrom[j] = PERM ? sb_get(&bin_vlo[at]) : 0u;
                    vto[j] = PERM ? sb_get(&bin_vhi[at]) : 0u;
                }
#pragma unroll
                for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) move(i0 + j, from[j], to[j], vfrom[j], vto[j]);
            }
        }
        if (PERM && !unseen) {
            __syncthreads();
        } else if (!unseen) {
            any_mixed = __syncthreads_or(mixed ? 1 : 0) != 0;
            if (!any_mixed) break;                                      // equal keys need no order
        }
#pragma unroll
        for (int i0 = 0; i0 < ITEMS; i0 += ROWS) {
            if ((uint32_t)(i0 * BLOCK) >= m) continue;
            U from[ROWS], wide[ROWS];
            uint32_t size[ROWS], vfrom[PERM ? ROWS : 1], vwide[PERM ? ROWS : 1];
#pragma unroll
            for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                const uint32_t at = entry(rank[i0 + j]);
                from[j] = bin_lo[at];
                wide[j] = (U)(bin_hi[at] - from[j]);
                size[j] = bin_size[at];
                if constexpr (PERM) {
                    vfrom[j] = evenly ? vlo : bin_vlo[at];
                    vwide[j] = evenly ? vspan : bin_vhi[at] - vfrom[j];
                }
            }
#pragma unroll
            for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                const int i = i0 + j;
                if (tid + i * BLOCK < m) {
                    uint32_t id = rank[i] & 0xffffu;
                    const bool large = divides(rank[i]);
                    const uint32_t bw = sb_bits(wide[j]);
                    if (level != 0 && !large) {
                        atomicAdd(&sub[id], 1u);
                        continue;
                    }
                    if (!large || unseen || (evenly && bw != 0u)) {     // by where in its bin the element lies
                        const uint32_t in_bin = code_of(key[i], val[PERM ? i : 0]) * scale;
                        id += __umulhi(in_bin, large ? size[j] : rank[i] >> 16 & 0xffu);
                    } else if (!PERM && bw == 0u) {
                        id += place_in_bin(rank[i]);
                    } else {
                        uint32_t word = 0u, most_word = 0u;
                        if constexpr (PERM) {
                            const int vs = vwide[j] == 0u ? 0 : __clz((int)vwide[j]);
                            word = (val[i] - vfrom[j]) << vs;
                            most_word = vwide[j] << vs;
                        }
                        // as above: below `size` for all of the bin
                        const uint32_t most_of_bin = sb_code<PERM>(wide[j], bw, most_word);
                        const uint32_t per = (uint32_t)((float)size[j] * 4294967296.f * __builtin_amdgcn_rcpf((float)most_of_bin + 1.f) * (1.f - 0x1p-21f));
                        id += __umulhi(sb_code<PERM>((U)(key[i] - from[j]), bw, word), per);
                    }
                    rank[i] = LARGE | id | atomicAdd(&sub[id], 1u) << 16;
                }
            }
        }
        __syncthreads();
        uint32_t s[ITEMS], total = 0u, top = 0u;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) s[i] = sub[tid * ITEMS + i];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (tid * ITEMS + i >= m) s[i] = 0u;
            total += s[i];
            top = s[i] > top ? s[i] : top;
        }
        const uint32_t run = wave_scan_inclusive(total, OpAdd(), 0u);
        top = wave_reduce(top, OpMax());
        if (lane == WAVE - 1) { part[2][wave] = run; part[3][wave] = top; }
        __syncthreads();
        uint32_t at = run - total;
        largest = 0u;
        for (int w = 0; w < NW; ++w) {
            if ((uint32_t)w < wave) at += part[2][w];
            largest = part[3][w] > largest ? part[3][w] : largest;
        }
        largest = sb_uniform(largest);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            if (tid * ITEMS + i < m) sub[tid * ITEMS + i] = at | s[i] << 16;
            at += s[i];
        }
        __syncthreads();
#pragma unroll
        for (int i0 = 0; i0 < ITEMS; i0 += ROWS) {
            if ((uint32_t)(i0 * BLOCK) >= m) continue;
            uint32_t q[ROWS];
#pragma unroll
            for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) q[j] = sub[rank[i0 + j] & 0xffffu];
#pragma unroll
            for (int j = 0; j < ROWS && i0 + j < ITEMS; ++j) {
                const int i = i0 + j;
                const bool valid = tid + i * BLOCK < m && (level == 0 || divides(rank[i]));
                const uint32_t r = enter(valid, q[j] & 0xffffu, q[j] >> 16, place_in_bin(rank[i]));
                if (valid) rank[i] = r;
            }
        }
    }
    __syncthreads();
    if (any_mixed && largest > SB_MAX_BIN) {                            // in any order
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = tid + i * BLOCK;
            if (p < m) {
                lds_key[p] = key[i];
                if constexpr (PERM) lds_val[p] = val[i];
            }
        }
        sb_bitonic<PERM>(lds_key, lds_val, m);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t p = tid + i * BLOCK;
            if (p < m) store(p, lds_key[p], PERM ? lds_val[PERM ? p : 0] : p);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (tid + i * BLOCK < m) {
            const uint32_t p = (rank[i] & 0xffffu) + place_in_bin(rank[i]);
            lds_key[p] = key[i];
            if constexpr (PERM) lds_val[p] = val[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {                                   // the elements of this thread as it holds them
        if (tid + i * BLOCK < m) {
            const uint32_t q0 = rank[i] & 0xffffu, p = q0 + place_in_bin(rank[i]), v = PERM ? val[PERM ? i : 0] : p;
            if (!PERM && (rank[i] & LARGE) != 0u) store(p, key[i], v);
            else store(q0 + smaller(key[i], v, q0, q0 + (rank[i] >> 16 & 0xffu)), key[i], v);
        }
    }
}

template <typename T, bool PERM>
__global__ __launch_bounds__(SB_SORT_BLOCK) void sort_bucket_kernel(uint32_t k, uint32_t ntiles, const uint32_t* __restrict__ table, int rev,
                                                                    const typename SortKey<T>::U* __restrict__ tile_key, const uint16_t* __restrict__ tile_val,
                                                                    typename SortKey<T>::U* big_key, uint32_t* big_val, T* sorted_out, int64_t* perm_out) {
    typedef typename SortKey<T>::U U;
    constexpr int BLOCK = SB_SORT_BLOCK, ITEMS = SB_SORT_ITEMS;
    __shared__ SbLds<U, PERM, ITEMS, BLOCK, SB_BINS> lds;
    auto& bins = lds.bins;
    auto& part = lds.part;
    uint32_t* const run_off = bins;                          // of a tile: keys of the bucket in the tiles in front (read before bins are)
    uint32_t* const run_at = bins + SB_MAX_TILES;            // where the bucket starts in it
    static_assert(2u * SB_MAX_TILES <= SB_BINS && SB_MAX_TILES <= (uint32_t)BLOCK, "a thread a tile");
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, bucket = blockIdx.x;
    uint32_t entry = 0u;
    if (tid == 0u) lds.init();
    if (tid < ntiles) entry = table[tid * k + bucket];
    const uint32_t before = wave_reduce(entry & 0xffffu, OpAdd());
    const uint32_t run = wave_scan_inclusive(entry >> 16, OpAdd(), 0u);
    const uint64_t there = __ballot((entry >> 16) != 0u);     // tiles that hold keys of the bucket
    if (lane == 0) {
        part[0][wave] = before;
        part[2][wave] = there == 0ull ? ~0u : wave * WAVE + (uint32_t)__builtin_ctzll(there);
        part[3][wave] = there == 0ull ? 0u : wave * WAVE + (WAVE - 1) - (uint32_t)__builtin_clzll(there);
    }
    if (lane == WAVE - 1) part[1][wave] = run;
    __syncthreads();
    uint32_t start = 0u, off = run - (entry >> 16), m = 0u, first_tile = ~0u, last_tile = 0u;
#pragma unroll
    for (int w = 0; w < (int)SB_MAX_TILES / WAVE; ++w) {
        start += part[0][w];
        first_tile = part[2][w] < first_tile ? part[2][w] : first_tile;
        last_tile = part[3][w] > last_tile ? part[3][w] : last_tile;
        if ((uint32_t)w < wave) off += part[1][w];
        m += part[1][w];
    }
    if (tid < SB_MAX_TILES) {
        run_off[tid] = tid < ntiles ? off : ~0u;
        run_at[tid] = entry & 0xffffu;
    }
    __syncthreads();
    // the p-th key of the bucket: in the last tile with no more than p keys in front of it
    auto find = [&](uint32_t p, uint32_t& tile) -> uint32_t {
        tile = 0u;
#pragma unroll
        for (uint32_t step = SB_MAX_TILES / 2u; step != 0u; step /= 2u) tile += run_off[tile + step] <= p ? step : 0u;
        return tile * (uint32_t)SB_TILE + run_at[tile] + (p - run_off[tile]);
    };
    if (m > SB_CAP) {                                        // too large for LDS: compared in memory, slowly
        U* x = PERM ? big_key + start : (U*)sorted_out + start;
        uint32_t* y = PERM ? big_val + start : nullptr;
        for (uint32_t p = tid; p < m; p += BLOCK) {
            uint32_t tile;
            const uint32_t at = find(p, tile);
            x[p] = tile_key[at];
            if constexpr (PERM) y[p] = tile * (uint32_t)SB_TILE + tile_val[at];
        }
        sb_bitonic<PERM>(x, y, m);
        for (uint32_t i = tid; i < m; i += BLOCK) {
            if constexpr (PERM) perm_out[start + i] = (int64_t)y[i] + 1;
            else sorted_out[start + i] = dec_bits<T>(x[i], rev, (U)0);
        }
        return;
    }
    U key[ITEMS];
    uint32_t val[PERM ? ITEMS : 1];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)(i * BLOCK) < m) {
            const uint32_t p = tid + i * BLOCK;
            uint32_t tile;
            const uint32_t at = find(p < m ? p : 0u, tile);
            key[i] = tile_key[at];
            if constexpr (PERM) val[i] = tile * (uint32_t)SB_TILE + tile_val[at];
        }
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);             // searches four at a time: eleven take too many registers
    }
    start = sb_uniform(start);
    sb_sort_bucket<PERM, true, ITEMS, BLOCK, SB_BINS>(key, val, m, lds, sb_uniform(first_tile) * (uint32_t)SB_TILE, sb_uniform(last_tile) * (uint32_t)SB_TILE + (SB_TILE - 1), [&](uint32_t to, U x, uint32_t v) {
        if constexpr (PERM) perm_out[start + to] = (int64_t)v + 1;
        else sorted_out[start + to] = dec_bits<T>(x, rev, (U)0);
    });
}

// ---- sorts that fit a workgroup ---------------------------------------------------------------------------------------
// Up to 4096 keys: radix passes with everything in LDS, one kernel instead of ten or eighteen (sort Float64[1000] 63 -> 16.5 us a
// call, Float64[4096] 66 -> 25, Float32[4096] 42 -> 16.5).  A digit in which no
// two keys differ (integers: relative to the smallest) takes no pass.
constexpr int ST_BLOCK = 1024, ST_ITEMS = 4, ST_MAX = ST_BLOCK * ST_ITEMS;

template <typename T, bool PERM>
__global__ __launch_bounds__(ST_BLOCK) void sort_tiny_kernel(const T* orig, T* sorted_out, int64_t* perm_out, uint32_t n, int rev, SortCtl* ctl) {
    typedef typename SortKey<T>::U U;
    constexpr int BLOCK = ST_BLOCK, ITEMS = ST_ITEMS, NW = BLOCK / WAVE;
    constexpr bool RELATIVE = std::is_integral<T>::value;
    __shared__ U lds_key[ST_MAX];
    __shared__ uint32_t lds_val[PERM ? ST_MAX : 1];
    __shared__ alignas(16) uint32_t cnt[NW * 256];
    __shared__ uint32_t wsum[256 / WAVE];
    __shared__ unsigned long long part[2][NW];
    const uint32_t tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE, per = (n + BLOCK - 1) / BLOCK, first = wave * per * WAVE + lane;
    U key[ITEMS];
    uint32_t val[PERM ? ITEMS : 1];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t e = first + i * WAVE;
        key[i] = __builtin_bit_cast(U, orig[e < n ? e : n - 1u]);
        if constexpr (PERM) val[i] = e;
    }
    U base = enc_bits<T>(__builtin_bit_cast(U, orig[0]), rev, (U)0);
    unsigned long long inv = 0ull;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        key[i] = enc_bits<T>(key[i], rev, (U)0);
        const unsigned long long v = (unsigned long long)(U)~key[i];
        inv = v > inv ? v : inv;
    }
    if constexpr (RELATIVE) {
        inv = wave_reduce(inv, OpMax());
        if (lane == 0) part[0][wave] = inv;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NW; ++w) inv = part[0][w] > inv ? part[0][w] : inv;
        base = (U)~(U)inv;
    }
    U mine = (U)0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        mine |= RELATIVE ? (U)(key[i] - base) : (U)(key[i] ^ base);
        if (RELATIVE) key[i] = (U)(key[i] - base);
    }
    unsigned long long bits = wave_reduce((unsigned long long)mine, OpOr());
    if (lane == 0) part[1][wave] = bits;
    __syncthreads();
    bits = 0ull;
#pragma unroll
    for (int w = 0; w < NW; ++w) bits |= part[1][w];
    uint32_t ran = 0u;
    for (int pass = 0; pass < (int)sizeof(T); ++pass) {
        if (((bits >> (8 * pass)) & 0xffull) == 0ull) continue;
        ++ran;
        sb_radix_pass<PERM, ITEMS>(key, val, per, n, [&](U x, uint32_t) { return digit_of(x, pass); }, lds_key, lds_val, cnt, wsum);
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t e = first + i * WAVE;
        if ((uint32_t)i < per && e < n) {
            if constexpr (PERM) perm_out[e] = (int64_t)val[i] + 1;
            else sorted_out[e] = dec_bits<T>(key[i], rev, RELATIVE ? base : (U)0);
        }
    }
    if (tid == 0) ctl->nexec = ran;
}

}  // namespace rk
