// Sorts of more than 2^20 keys by two levels of splitters (included by rk_sort.hip): 8-byte keys up to 2^26, Float32 up to 2^22.
//
//   sort_sample_kernel, sort_splitters_kernel   255 splitters from 4096 samples (rk_sort_buckets.hpp)
//   sort_split_first_kernel   sorts every tile in LDS by part -- between which splitters a key lies -- and leaves a table of where
//                             the parts start in every tile
//   sort_runs_kernel          for every part, where its runs lie: the columns of that table, summed down the tiles
//   sort_parts_kernel         a workgroup a part: samples it, sorts the samples, keeps every LS_OVER-th as splitters of the part, and
//                             lists the tiles of the part and its buckets
//   sort_split_second_kernel  a tile of a part: collects its keys from the runs and sorts the tile by bucket
//   sort_last_kernel          a workgroup a bucket: collects its keys from the part's tiles, sorts them in LDS and writes the result
//
// Every key is read and written three times, whatever its width, where radix passes of 8 bits read it twice and write it once for
// each of its bytes; and since no kernel has to keep the order of what it moves, a key's place is one LDS atomic instead of a match by
// ballots.  Nothing is scattered over memory: a tile is written where it was read, and the next kernel collects its runs.
//
// Radix passes -> so, us a call: sort Float64[2^21] 248 -> 75, [2^24] 718 -> 315, [2^26] 3093 -> 1162; sort Int64 of 64 bits 262 -> 110,
// 760 -> 357; sortperm Int64 288 -> 120, 1026 -> 484; sort Float32[1500000] 113 -> 58, [2^22] 136 -> 92, two values 135 -> 128, 256 values
// 136 -> 109; sortperm Float32[2^22] 148 -> 106, two values 143 -> 145, 256 values 145 -> 130.  For Float32 beyond, sort takes one move into
// buckets (rk_sort_quantiles.hpp), and sortperm radix passes; so does Int32 at once, which needs a read for the digits that vary, and launches for the
// passes that then do not run (2^21 keys of 20 bits).
// The kernels of sort Float64[2^24]: 61 first, 5 runs, 23 parts, 82 second, 129 last; 256 MiB read and written are 41.  They are bound by
// vector instructions (sort Float32[2^22], a key: 58 first, 85 second, 204 last).
//
// Order, and the sizes of buckets: as in rk_sort_buckets.hpp, (key, index) is a strict order.  Within a part the index is a key's place in
// the part (sort) or its index in the array (sortperm).  A part gets as many buckets as its size asks for, with LS_OVER samples a
// bucket, so up to 2^25 keys one bucket in 10^11 does not fit LDS and is sorted in memory, as in rk_sort_buckets.hpp.  LS_BUCKETS are the
// most that a part gets: at 2^26 keys 3 % of the parts are larger than that is meant for, and one bucket in 10^7 does not fit, in one
// sort of 250.
#pragma once

#include "rk_sort_buckets.hpp"

namespace rk {

constexpr uint32_t LS_PARTS = 256, LS_BUCKETS = 256;           // of a sort; of a part, at most
constexpr uint32_t LS_OVER = 32;                               // samples a bucket
constexpr int LS_BLOCK = 1024;
constexpr uint32_t LS_RUNS = 1024;                             // runs of a tile that LDS holds at a time
constexpr uint32_t LS_TILES = 256;                             // tiles of a part up to which its buckets are sorted in LDS

// Keys a bucket that are sorted in LDS, and on the average, by workgroups of which LDS holds two to four a compute unit.
constexpr int LS_LAST_BLOCK = 512, LS_LAST_ITEMS = 8;
constexpr uint32_t LS_CAP = LS_LAST_BLOCK * LS_LAST_ITEMS, LS_MEAN = LS_CAP * 3 / 8, LS_BINS = 2048;

struct LsTile { uint32_t part, buckets, at, count, first_run, last_run, to, unused; };     // `at`: in the part; `to`: in the array
struct LsBucket { uint32_t first_tile, ntiles, bucket, start; };                           // `start`: of the part

// Splitters in LDS: as a search tree (the root is node 1, a level lies side by side, so the lanes of a wave that have come to
// different nodes of it read different banks) and in order, with their indices.
template <typename U> struct LsSplitters {
    U tree[256], ordered[256];
    uint32_t index[256], cnt[256], wsum[4];
};

// `leaves`: a power of two, at least the number of buckets k; missing splitters compare greater than any key.
template <typename U>
__device__ __forceinline__ void ls_load_splitters(LsSplitters<U>& s, uint32_t k, uint32_t leaves, const U* spl_key, const uint32_t* spl_index) {
    const uint32_t tid = threadIdx.x;
    if (tid < 256u) s.cnt[tid] = 0u;
    if (tid + 1u < leaves) {
        const bool there = tid + 1u < k;
        const U x = there ? spl_key[tid] : (U)~(U)0;
        s.ordered[tid] = x;
        s.index[tid] = there ? spl_index[tid] : ~0u;
        const uint32_t m = tid + 1u, z = (uint32_t)__builtin_ctz(m) + 1u;
        s.tree[(leaves >> z) + (m >> z)] = x;
    }
}

// Sorts a tile by bucket: thread t holds its elements t, t + 1024, ... of which the first `count` exist.  row[b] = where bucket b
// starts in the tile | its size << 16.  index(i): of item i, for keys that equal a splitter.
// Lanes that all go to one bucket (input that is sorted already, or few values) add to its counter once.
template <bool PERM, int ITEMS, bool FULL, typename U, typename V, typename Index>
__device__ __forceinline__ void ls_split_tile(U (&key)[ITEMS], const V (&val)[PERM ? ITEMS : 1], uint32_t count, uint32_t k, uint32_t leaves,
                                              LsSplitters<U>& s, U* lds_key, uint32_t* row, U* out_key, V* out_val, Index&& index) {
    const uint32_t tid = threadIdx.x, lane = tid % WAVE;
    uint32_t place[ITEMS];                                   // bucket | rank in it << 8
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) place[i] = 1u;
    for (uint32_t l = leaves; l > 1u; l /= 2u) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) place[i] = place[i] * 2u + (s.tree[place[i]] < key[i] ? 1u : 0u);
    }
    bool tie = false;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        place[i] -= leaves;
        tie = tie || (place[i] + 1u < k && s.ordered[place[i]] == key[i]);
    }
    if (tie) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) place[i] = 0u;
        for (uint32_t step = leaves / 2u; step != 0u; step /= 2u) {
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const U x = s.ordered[place[i] + step - 1u];
                place[i] += (x < key[i] || (x == key[i] && s.index[place[i] + step - 1u] <= index(i))) ? step : 0u;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const bool valid = FULL || tid + i * LS_BLOCK < count;
        const uint32_t b = place[i], b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)b);
        const uint32_t in = FULL ? (uint32_t)WAVE : (uint32_t)__popcll(__ballot(valid));
        uint32_t r = 0u;
        if (__ballot(valid && b != b0) == 0ull) {            // (the lanes that exist are the first ones)
            if (lane == 0u && in != 0u) r = atomicAdd(&s.cnt[b0], in);
            r = (uint32_t)__builtin_amdgcn_readfirstlane((int)r) + lane;
        } else if (valid) {
            r = atomicAdd(&s.cnt[b], 1u);
        }
        place[i] = b | r << 8;
    }
    __syncthreads();
    uint32_t c = 0u, inc = 0u;
    if (tid < 256u) {
        c = s.cnt[tid];
        inc = wave_scan_inclusive(c, OpAdd(), 0u);
        if (lane == WAVE - 1) s.wsum[tid / WAVE] = inc;
    }
    __syncthreads();
    if (tid < 256u) {
        uint32_t start = inc - c;
        for (uint32_t w = 0; w < tid / WAVE; ++w) start += s.wsum[w];
        s.cnt[tid] = start;
        if (tid < k) row[tid] = start | c << 16;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) place[i] = s.cnt[place[i] & 0xffu] + (place[i] >> 8);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if (FULL || tid + i * LS_BLOCK < count) lds_key[place[i]] = key[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t q = tid + i * LS_BLOCK;
        if (FULL || q < count) out_key[q] = lds_key[q];
    }
    if constexpr (PERM) {
        V* const lds_val = (V*)lds_key;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i)
            if (FULL || tid + i * LS_BLOCK < count) lds_val[place[i]] = val[i];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t q = tid + i * LS_BLOCK;
            if (FULL || q < count) out_val[q] = lds_val[q];
        }
    }
}

// Waves per SIMD that the registers have to allow: two workgroups a compute unit where LDS has room for two.
template <typename U, bool PERM> constexpr int ls_split_waves() { return sizeof(U) == 8 && PERM ? 4 : 8; }

// Integers: keys that differ in a few digits only were sorted by radix passes (ctl->nexec: number of digits).
template <typename T> __device__ __forceinline__ bool ls_not_needed(const SortCtl* ctl) { return std::is_integral<T>::value && ctl->nexec <= SORT_FEW_PASSES; }

// `tile_key` may be `keys`: a workgroup has read its tile before it writes it.
template <typename T, bool PERM, int ITEMS>
__global__ __launch_bounds__(LS_BLOCK, (ls_split_waves<typename SortKey<T>::U, PERM>())) void sort_split_first_kernel(
    const T* keys, uint32_t n, int rev, const SortCtl* ctl, const typename SortKey<T>::U* __restrict__ spl_key, const uint32_t* __restrict__ spl_index,
    uint32_t* __restrict__ table, typename SortKey<T>::U* tile_key, uint16_t* tile_val) {
    typedef typename SortKey<T>::U U;
    constexpr uint32_t TILE = (uint32_t)ITEMS * LS_BLOCK;
    __shared__ U lds_key[TILE];
    __shared__ LsSplitters<U> s;
    if (ls_not_needed<T>(ctl)) return;
    const uint32_t tid = threadIdx.x, e0 = blockIdx.x * TILE, count = n - e0 < TILE ? n - e0 : TILE;
    // all tiles but the last are full: no bounds to check (and to keep) for every key and step
    const auto split = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;
        U key[ITEMS];
        uint16_t val[PERM ? ITEMS : 1];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const uint32_t q = tid + i * LS_BLOCK;
            key[i] = __builtin_bit_cast(U, (keys + e0)[FULL || q < count ? q : 0u]);
        }
        ls_load_splitters(s, LS_PARTS, LS_PARTS, spl_key, spl_index);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            key[i] = enc_bits<T>(key[i], rev, (U)0);
            if constexpr (PERM) val[i] = (uint16_t)(tid + i * LS_BLOCK);
        }
        ls_split_tile<PERM, ITEMS, FULL>(key, val, count, LS_PARTS, LS_PARTS, s, lds_key, table + (size_t)blockIdx.x * LS_PARTS, tile_key + e0,
                                         PERM ? tile_val + e0 : nullptr, [&](int i) { return e0 + tid + i * LS_BLOCK; });
    };
    if (count == TILE) split(std::true_type{}); else split(std::false_type{});
}

// runs[part][tile] = keys of the part in the tiles in front, place of the tile's first key of the part in the tile.  An XCD
// takes 32 neighbouring parts, a line of every row of the table.
template <typename T>
__global__ __launch_bounds__(LS_BLOCK) void sort_runs_kernel(const SortCtl* ctl, uint32_t ntiles, const uint32_t* __restrict__ table, uint2* __restrict__ runs, uint32_t* __restrict__ sizes) {
    constexpr uint32_t UNR = 8;
    __shared__ uint32_t wsum[2][LS_BLOCK / WAVE];
    if (ls_not_needed<T>(ctl)) return;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, part = (blockIdx.x % 8u) * (LS_PARTS / 8u) + blockIdx.x / 8u;
    uint32_t carry = 0u;
    for (uint32_t t0 = 0, turn = 0; t0 < ntiles; t0 += LS_BLOCK * UNR, turn ^= 1u) {
        const uint32_t rest = ntiles - t0, each = rest >= LS_BLOCK * UNR ? UNR : (rest + LS_BLOCK - 1u) / LS_BLOCK, first = t0 + tid * each;
        uint32_t v[UNR], sum = 0u;
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) {
            v[u] = 0u;
            if (u < each && first + u < ntiles) v[u] = table[(size_t)(first + u) * LS_PARTS + part];
        }
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) sum += v[u] >> 16;
        const uint32_t inc = wave_scan_inclusive(sum, OpAdd(), 0u);
        if (lane == WAVE - 1) wsum[turn][wave] = inc;
        __syncthreads();
        uint32_t off = carry + inc - sum;
#pragma unroll
        for (uint32_t w = 0; w < LS_BLOCK / WAVE; ++w) {
            if (w < wave) off += wsum[turn][w];
            carry += wsum[turn][w];
        }
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) {
            if (u < each && first + u < ntiles) runs[(size_t)part * ntiles + first + u] = make_uint2(off, v[u] & 0xffffu);
            off += v[u] >> 16;
        }
    }
    if (tid == 0u) sizes[part] = carry;
}

// A workgroup a part.  Samples are taken as from the whole array, one from somewhere in each of equal stretches of the part; whoever
// holds the run that one falls into says where it lies.
template <typename T, bool PERM>
__global__ __launch_bounds__(LS_BLOCK) void sort_parts_kernel(const SortCtl* ctl, uint32_t ntiles, uint32_t shift,
                                                              const uint32_t* __restrict__ sizes, const uint2* __restrict__ runs,
                                                              const typename SortKey<T>::U* __restrict__ tile_key, const uint16_t* __restrict__ tile_val,
                                                              typename SortKey<T>::U* __restrict__ spl_key, uint32_t* __restrict__ spl_index,
                                                              LsTile* __restrict__ tiles, uint32_t max_tiles, LsBucket* __restrict__ buckets, uint32_t max_buckets) {
    typedef typename SortKey<T>::U U;
    constexpr int ITEMS = (int)(LS_BUCKETS * LS_OVER) / LS_BLOCK;
    __shared__ SbLds<U, true, ITEMS, LS_BLOCK, SB_BINS> lds;
    __shared__ uint32_t smp_at[LS_BUCKETS * LS_OVER];
    __shared__ uint32_t wsum[3][LS_PARTS / WAVE], mine[6], all[2];
    if (ls_not_needed<T>(ctl)) return;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE, part = blockIdx.x, tile = 1u << shift;
    if (tid == 0u) lds.init();
    uint32_t size = 0u, nt = 0u, k = 0u, inc[3] = {0u, 0u, 0u};
    if (tid < LS_PARTS) {
        size = sizes[tid];
        nt = (size + tile - 1u) >> shift;
        k = (size + LS_MEAN - 1u) / LS_MEAN;
        k = k < LS_BUCKETS ? k : LS_BUCKETS;
        inc[0] = wave_scan_inclusive(size, OpAdd(), 0u);
        inc[1] = wave_scan_inclusive(nt, OpAdd(), 0u);
        inc[2] = wave_scan_inclusive(k, OpAdd(), 0u);
        if (lane == WAVE - 1) {
#pragma unroll
            for (int j = 0; j < 3; ++j) wsum[j][wave] = inc[j];
        }
    }
    __syncthreads();
    if (tid < LS_PARTS) {
        for (uint32_t w = 0; w < wave; ++w) {
#pragma unroll
            for (int j = 0; j < 3; ++j) inc[j] += wsum[j][w];
        }
        if (tid == part) {
            mine[0] = size; mine[1] = nt; mine[2] = k;
            mine[3] = inc[0] - size; mine[4] = inc[1] - nt; mine[5] = inc[2] - k;
        }
        if (tid == LS_PARTS - 1u) { all[0] = inc[1]; all[1] = inc[2]; }
    }
    __syncthreads();
    size = mine[0]; nt = mine[1]; k = mine[2];
    const uint32_t start = mine[3], first_tile = mine[4], first_bucket = mine[5];
    if (part == 0u) {                                        // what the grids of the next kernels have too many
        for (uint32_t t = all[0] + tid; t < max_tiles; t += LS_BLOCK) tiles[t].count = 0u;
        for (uint32_t b = all[1] + tid; b < max_buckets; b += LS_BLOCK) buckets[b].ntiles = 0u;
    }
    if (tid < k) buckets[first_bucket + tid] = LsBucket{first_tile, nt, tid, start};
    const uint32_t s = k > 1u ? k * LS_OVER : 0u;
    const uint64_t step = s != 0u ? ((uint64_t)size << 12) / s : 0ull;                    // of a stretch, in 4096ths of a key
    const float per_key = s != 0u ? (float)s / (float)size : 0.f;
    const auto stretch = [&](uint32_t j) { return (uint32_t)((j * step) >> 12); };
    const auto sample = [&](uint32_t j) {
        uint32_t h = (j + 1u) * 0x9e3779b1u;
        h ^= h >> 15;
        h *= 0x85ebca77u;
        const uint32_t a = stretch(j);
        return a + __umulhi(h, stretch(j + 1u) - a);
    };
    constexpr uint32_t UNR = 4;
    for (uint32_t i0 = tid; i0 < ntiles; i0 += LS_BLOCK * UNR) {
        uint2 run[UNR];
        uint32_t next[UNR];
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) {
            const uint32_t i = i0 + u * LS_BLOCK;
            run[u] = make_uint2(0u, 0u);
            next[u] = i + 1u == ntiles ? size : 0u;
            if (i < ntiles) run[u] = runs[(size_t)part * ntiles + i];
            if (i + 1u < ntiles) next[u] = runs[(size_t)part * ntiles + i + 1u].x;
        }
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) {
            const uint32_t i = i0 + u * LS_BLOCK, off = run[u].x, end = next[u];
            if (i >= ntiles || off == end) continue;
            // the tiles that begin and end in the run
            for (uint32_t t = off >> shift; (t << shift) < end; ++t) {
                const uint32_t at = t << shift, count = size - at < tile ? size - at : tile;
                LsTile& d = tiles[first_tile + t];
                if (at >= off) { d.part = part; d.buckets = k; d.at = at; d.count = count; d.first_run = i; d.to = start + at; }
                if (at + count <= end) d.last_run = i;
            }
            // the samples in it: where they lie
            const uint32_t guess = (uint32_t)((float)off * per_key);
            for (uint32_t j = guess > 1u ? guess - 2u : 0u; j < s && stretch(j) < end; ++j) {
                const uint32_t p = sample(j);
                if (p >= off && p < end) smp_at[j] = (i << shift) + run[u].y + (p - off);
            }
        }
    }
    if (s == 0u) return;
    __syncthreads();
    U key[ITEMS];
    uint32_t index[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)(i * LS_BLOCK) < s) {
            const uint32_t j = tid + i * LS_BLOCK < s ? tid + i * LS_BLOCK : 0u, from = smp_at[j];
            key[i] = tile_key[from];
            index[i] = PERM ? (from >> shift << shift) + tile_val[from] : sample(j);
        }
    }
    sb_sort_bucket<true, false, ITEMS, LS_BLOCK, SB_BINS>(key, index, s, lds, 0u, 0u, [&](uint32_t to, U x, uint32_t v) {
        if (to == 0u || to % LS_OVER != 0u) return;
        spl_key[part * LS_BUCKETS + to / LS_OVER - 1u] = x;
        spl_index[part * LS_BUCKETS + to / LS_OVER - 1u] = v;
    });
}

// A tile of a part: elements [at, at + count) of its runs, one after the other.
template <typename T, bool PERM, int ITEMS>
__global__ __launch_bounds__(LS_BLOCK, (ls_split_waves<typename SortKey<T>::U, PERM>())) void sort_split_second_kernel(
    const SortCtl* ctl, const LsTile* __restrict__ tiles, const uint2* __restrict__ runs, uint32_t ntiles, uint32_t shift,
    const typename SortKey<T>::U* __restrict__ spl_key, const uint32_t* __restrict__ spl_index, const typename SortKey<T>::U* __restrict__ in_key,
    const uint16_t* __restrict__ in_val, uint32_t* __restrict__ table, typename SortKey<T>::U* __restrict__ out_key, uint32_t* __restrict__ out_val) {
    typedef typename SortKey<T>::U U;
    constexpr uint32_t TILE = (uint32_t)ITEMS * LS_BLOCK;
    __shared__ U lds_key[TILE];
    __shared__ LsSplitters<U> s;
    __shared__ uint32_t run_off[LS_RUNS + 1], run_from[LS_RUNS];       // of a run: its first element in the tile; in_key[run_from + e] is element e
    __shared__ uint16_t group_run[TILE / WAVE];                        // the run of the first of 64 elements
    if (ls_not_needed<T>(ctl)) return;
    const LsTile d = tiles[blockIdx.x];             // (the same for all lanes: scalar loads)
    if (d.count == 0u) return;
    const uint32_t tid = threadIdx.x;
    uint32_t leaves = 1u;
    while (leaves < d.buckets) leaves *= 2u;
    ls_load_splitters(s, d.buckets, leaves, spl_key + d.part * LS_BUCKETS, spl_index + d.part * LS_BUCKETS);
    const auto split = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;
        uint32_t from[ITEMS];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) from[i] = 0u;
        for (uint32_t r0 = d.first_run; r0 <= d.last_run; r0 += LS_RUNS) {
            const uint32_t left = d.last_run - r0 + 1u, nr = left < LS_RUNS ? left : LS_RUNS;
            __syncthreads();
            for (uint32_t r = tid; r <= nr; r += LS_BLOCK) {
                if (r == left) { run_off[r] = d.count; continue; }
                const uint2 run = runs[(size_t)d.part * ntiles + r0 + r];
                run_off[r] = run.x > d.at ? run.x - d.at : 0u;
                if (r < nr) run_from[r] = ((r0 + r) << shift) + run.y - run.x + d.at;
            }
            __syncthreads();
            const uint32_t begin = run_off[0], end = run_off[nr];
            for (uint32_t r = tid; r < nr; r += LS_BLOCK) {
                const uint32_t a = run_off[r], b = run_off[r + 1u];
                for (uint32_t g = (a + WAVE - 1u) / WAVE; g * WAVE < b; ++g) group_run[g] = (uint16_t)r;
            }
            __syncthreads();
            const auto find = [&](uint32_t q, uint32_t r) {
                while (q >= run_off[r + 1u]) ++r;            // (run_off[nr] = end > q)
                return run_from[r] + q;
            };
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const uint32_t q = tid + i * LS_BLOCK;
                if (q >= begin && q < end) from[i] = find(q, q / WAVE * WAVE >= begin ? group_run[q / WAVE] : 0u);
            }
        }
        U key[ITEMS];
        uint32_t val[PERM ? ITEMS : 1];
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            key[i] = (U)0;
            if (FULL || tid + i * LS_BLOCK < d.count) {
                key[i] = in_key[from[i]];
                if constexpr (PERM) val[i] = (from[i] >> shift << shift) + in_val[from[i]];
            }
        }
        ls_split_tile<PERM, ITEMS, FULL>(key, val, d.count, d.buckets, leaves, s, lds_key, table + (size_t)blockIdx.x * LS_BUCKETS, out_key + d.to,
                                         PERM ? out_val + d.to : nullptr, [&](int i) { return PERM ? val[PERM ? i : 0] : d.at + tid + i * LS_BLOCK; });
    };
    if (d.count == TILE) split(std::true_type{}); else split(std::false_type{});
}

template <typename U, bool PERM> constexpr int ls_last_waves() { return PERM && sizeof(U) == 8 ? 4 : PERM || sizeof(U) == 8 ? 6 : 8; }

// A workgroup a bucket.  xcd_chunk: each XCD takes neighbouring buckets (0: as they come), which share the lines where their runs meet.
template <typename T, bool PERM>
__global__ __launch_bounds__(LS_LAST_BLOCK, (ls_last_waves<typename SortKey<T>::U, PERM>())) void sort_last_kernel(const SortCtl* ctl, const LsBucket* __restrict__ buckets, uint32_t nbuckets,
                                                                            uint32_t xcd_chunk, uint32_t tile_shift, const uint32_t* __restrict__ table, int rev,
                                                                            const typename SortKey<T>::U* __restrict__ tile_key, const uint32_t* __restrict__ tile_val,
                                                                            typename SortKey<T>::U* big_key, uint32_t* big_val, T* sorted_out, int64_t* perm_out) {
    typedef typename SortKey<T>::U U;
    constexpr int BLOCK = LS_LAST_BLOCK, ITEMS = LS_LAST_ITEMS;
    __shared__ SbLds<U, PERM, ITEMS, BLOCK, LS_BINS> lds;
    static_assert(2u * LS_TILES <= LS_BINS && LS_TILES <= (uint32_t)BLOCK, "a thread a tile");
    uint32_t* const run_off = lds.bins;                      // of a tile: keys of the bucket in the tiles in front (read before bins are)
    uint32_t* const run_from = lds.bins + LS_TILES;          // tile_key[run_from + p] is the p-th key of the bucket
    if (ls_not_needed<T>(ctl)) return;
    uint32_t at = blockIdx.x;
    if (xcd_chunk != 0u) {
        at = (blockIdx.x & 7u) * xcd_chunk + (blockIdx.x >> 3);
        if (blockIdx.x >> 3 >= xcd_chunk || at >= nbuckets) return;
    }
    const LsBucket d = buckets[at];
    if (d.ntiles == 0u) return;
    const uint32_t* const column = table + (size_t)d.first_tile * LS_BUCKETS + d.bucket;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    uint32_t entry = 0u, before = 0u, mine = 0u;
    if (tid == 0u) lds.init();
    for (uint32_t t = tid; t < d.ntiles; t += BLOCK) {
        entry = column[(size_t)t * LS_BUCKETS];
        before += entry & 0xffffu;
        mine += entry >> 16;
    }
    before = wave_reduce(before, OpAdd());
    const uint32_t run = wave_scan_inclusive(mine, OpAdd(), 0u);
    if (lane == 0) lds.part[0][wave] = before;
    if (lane == WAVE - 1) lds.part[1][wave] = run;
    __syncthreads();
    uint32_t start = d.start, off = run - mine, m = 0u;
#pragma unroll
    for (int w = 0; w < BLOCK / WAVE; ++w) {
        start += lds.part[0][w];
        if ((uint32_t)w < wave) off += lds.part[1][w];
        m += lds.part[1][w];
    }
    m = sb_uniform(m);
    if (m == 0u) return;
    if (m > LS_CAP || d.ntiles > LS_TILES) {                    // too large for LDS: compared in memory, slowly
        U* x = PERM ? big_key + start : (U*)sorted_out + start;
        uint32_t* y = PERM ? big_val + start : nullptr;
        uint32_t to = 0u;
        for (uint32_t t = 0; t < d.ntiles; ++t) {
            const uint32_t e = column[(size_t)t * LS_BUCKETS], from = d.start + (t << tile_shift) + (e & 0xffffu);
            for (uint32_t p = tid; p < e >> 16; p += BLOCK) {
                x[to + p] = tile_key[from + p];
                if constexpr (PERM) y[to + p] = tile_val[from + p];
            }
            to += e >> 16;
        }
        sb_bitonic<PERM>(x, y, m);
        for (uint32_t i = tid; i < m; i += BLOCK) {
            if constexpr (PERM) perm_out[start + i] = (int64_t)y[i] + 1;
            else sorted_out[start + i] = dec_bits<T>(x[i], rev, (U)0);
        }
        return;
    }
    uint32_t top = 1u;                                       // a power of two, at least the number of tiles
    while (top < d.ntiles) top *= 2u;
    if (tid < LS_TILES) {
        run_off[tid] = tid < d.ntiles ? off : ~0u;
        run_from[tid] = d.start + (tid << tile_shift) + (entry & 0xffffu) - off;
    }
    __syncthreads();
    U key[ITEMS];
    uint32_t val[PERM ? ITEMS : 1];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if ((uint32_t)(i * BLOCK) < m) {
            const uint32_t q = tid + i * BLOCK, p = q < m ? q : 0u;
            uint32_t tile = 0u;
            for (uint32_t step = top / 2u; step != 0u; step /= 2u) tile += run_off[tile + step] <= p ? step : 0u;
            const uint32_t from = run_from[tile] + p;
            key[i] = tile_key[from];
            if constexpr (PERM) val[i] = tile_val[from];
        }
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    start = sb_uniform(start);
    sb_sort_bucket<PERM, false, ITEMS, BLOCK, LS_BINS>(key, val, m, lds, 0u, 0u, [&](uint32_t to, U x, uint32_t v) {
        if constexpr (PERM) perm_out[start + to] = (int64_t)v + 1;
        else sorted_out[start + to] = dec_bits<T>(x, rev, (U)0);
    });
}

// ---- host --------------------------------------------------------------------------------------------------------
constexpr int64_t LS_MAX_KEYS = (int64_t)1 << 26;          // LS_BUCKETS buckets of LS_MEAN keys are 1.5 times a part of so many
constexpr int64_t LS_MAX_FLOATS = (int64_t)1 << 22;        // Float32: figures above

// Keys a tile, of both levels: runs as long as two workgroups a compute unit in LDS allow, but hundreds of tiles.
constexpr int64_t LS_SMALL_TILES = ((int64_t)1 << 22) - 1;  // keys up to which the tiles are the smaller ones
static inline uint32_t ls_tile_shift(int64_t n) { return n <= LS_SMALL_TILES ? 12 : 13; }

struct LsLayout {
    size_t compact_off, spl_key_off, spl_index_off, table_off, sizes_off, runs_off, part_key_off, part_index_off, tiles_off, buckets_off, table2_off, total;
    uint32_t shift, ntiles, max_tiles, max_buckets;
};

static LsLayout ls_layout(size_t off, size_t key_size, int64_t n) {
    LsLayout l{};
    l.shift = ls_tile_shift(n);
    l.ntiles = (uint32_t)((n + ((int64_t)1 << l.shift) - 1) >> l.shift);
    l.max_tiles = (uint32_t)(n >> l.shift) + LS_PARTS;                       // at most one that is not full a part
    l.max_buckets = (uint32_t)(n / LS_MEAN) + LS_PARTS;
    const auto take = [&](size_t bytes) { const size_t at = off; off += (bytes + 255) & ~(size_t)255; return at; };
    l.compact_off = take((size_t)LS_PARTS * SB_OVER * key_size);
    l.spl_key_off = take((size_t)LS_PARTS * key_size);
    l.spl_index_off = take((size_t)LS_PARTS * 4);
    l.table_off = take((size_t)l.ntiles * LS_PARTS * 4);
    l.sizes_off = take((size_t)LS_PARTS * 4);
    l.runs_off = take((size_t)l.ntiles * LS_PARTS * sizeof(uint2));
    l.part_key_off = take((size_t)LS_PARTS * LS_BUCKETS * key_size);
    l.part_index_off = take((size_t)LS_PARTS * LS_BUCKETS * 4);
    l.tiles_off = take((size_t)l.max_tiles * sizeof(LsTile));
    l.buckets_off = take((size_t)l.max_buckets * sizeof(LsBucket));
    l.table2_off = take((size_t)l.max_tiles * LS_BUCKETS * 4);
    l.total = off;
    return l;
}

// first_key: where the tiles of the first level lie (sort!, sort: the result's place); second_key: those of the second.
// sortperm's indices: first_val (16 bits, in the tile), second_val; big_val for a bucket that does not fit LDS, whose keys go to first_key.
template <typename T, bool PERM>
static int32_t sort_split(const LsLayout& l, const void* keys, void* sorted_out, int64_t* perm_out, int64_t n, int rev, char* base, SortCtl* ctl,
                          typename SortKey<T>::U* first_key, typename SortKey<T>::U* second_key, uint32_t* first_val, uint32_t* second_val, hipStream_t stream) {
    typedef typename SortKey<T>::U U;
    U* compact = (U*)(base + l.compact_off);
    U* spl_key = (U*)(base + l.spl_key_off);
    uint32_t* spl_index = (uint32_t*)(base + l.spl_index_off);
    uint32_t* table = (uint32_t*)(base + l.table_off);
    uint32_t* sizes = (uint32_t*)(base + l.sizes_off);
    uint2* runs = (uint2*)(base + l.runs_off);
    U* part_key = (U*)(base + l.part_key_off);
    uint32_t* part_index = (uint32_t*)(base + l.part_index_off);
    LsTile* tiles = (LsTile*)(base + l.tiles_off);
    LsBucket* buckets = (LsBucket*)(base + l.buckets_off);
    uint32_t* table2 = (uint32_t*)(base + l.table2_off);
    constexpr uint32_t SAMPLES = LS_PARTS * SB_OVER;
    sort_sample_kernel<T><<<SAMPLES / 256, 256, 0, stream>>>((const T*)keys, (uint32_t)n, rev, SAMPLES, compact);
    RK_LAUNCH_CHECK();
    sort_splitters_kernel<T, false><<<SAMPLES / SB_SPL_EACH, SB_SPL_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, rev, nullptr, LS_PARTS, compact, spl_key, spl_index);
    RK_LAUNCH_CHECK();
    const auto first = [&](auto items) {
        sort_split_first_kernel<T, PERM, decltype(items)::value><<<l.ntiles, LS_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, rev, ctl, spl_key, spl_index, table, first_key, (uint16_t*)first_val);
    };
    if (l.shift == 12) first(std::integral_constant<int, 4>{});
    else first(std::integral_constant<int, 8>{});
    RK_LAUNCH_CHECK();
    sort_runs_kernel<T><<<LS_PARTS, LS_BLOCK, 0, stream>>>(ctl, l.ntiles, table, runs, sizes);
    RK_LAUNCH_CHECK();
    sort_parts_kernel<T, PERM><<<LS_PARTS, LS_BLOCK, 0, stream>>>(ctl, l.ntiles, l.shift, sizes, runs, first_key, (const uint16_t*)first_val, part_key, part_index, tiles, l.max_tiles, buckets, l.max_buckets);
    RK_LAUNCH_CHECK();
    const auto second = [&](auto items) {
        sort_split_second_kernel<T, PERM, decltype(items)::value><<<l.max_tiles, LS_BLOCK, 0, stream>>>(ctl, tiles, runs, l.ntiles, l.shift, part_key, part_index, first_key, (const uint16_t*)first_val, table2, second_key, second_val);
    };
    if (l.shift == 12) second(std::integral_constant<int, 4>{});
    else second(std::integral_constant<int, 8>{});
    RK_LAUNCH_CHECK();
    const uint32_t chunk = n >= ((int64_t)1 << 23) ? (l.max_buckets + 7u) / 8u : 0u;
    sort_last_kernel<T, PERM><<<chunk != 0u ? chunk * 8u : l.max_buckets, LS_LAST_BLOCK, 0, stream>>>(ctl, buckets, l.max_buckets, chunk, l.shift, table2, rev, second_key, second_val, first_key, first_val, (T*)sorted_out, perm_out);
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

}  // namespace rk
