// sort and sort! of keys of 4 bytes, Float32 from 2^22 and Int32 from 2^23 to 2^26 of them (included by rk_sort.hip): one move into
// buckets, which are sorted on the chip.
//
//   sq_sample_kernel    fetches a sample of the keys, and its smallest and largest
//   sq_table_kernel     counts the samples in SQ_CELLS equal cells between these; from there on, a key's bucket is the straight line
//                       that its cell has for the share of smaller samples, in units of a bucket.  Values in large numbers, and keys far from
//                       all the others, get buckets of their own, and the cells cover the rest: a second launch, which else ends at once
//   sq_count_kernel     the sizes of the buckets, by tile; of floats, which bits vary
//   sq_offsets_kernel   where the buckets lie, and where the keys of each chunk of tiles go; decides
//   sq_scatter_kernel   sorts every tile in LDS by bucket and writes its runs where they belong
//   sq_bucket_kernel    a workgroup a bucket: its keys in registers, spread over bins, put in order in LDS, written once
//
// Every key is read three times and written twice, of integers read once more in front (sort_range_kernel, 50 us of 2^26 keys), whatever its bits; four
// radix passes read it eight times and write it four times, and match digits by ballots because they have to keep the order of what they
// move.  Here nothing has to: equal keys of sort are the same bits, so a key's place is one LDS atomic.
//
// Radix passes -> so, us a call: sort Float32[2^23] 172 -> 128, [2^24] 248 -> 171, [2^26] 758 -> 449; Int32 of 32 bits [2^24] 265 -> 196,
// [2^26] 811 -> 489, of 20 bits [2^24] 234 -> 188, [2^26] 740 -> 460.  The kernels of Float32[2^26]: 8 sample, 18 table, 50 count, 8 offsets, 155
// scatter, 190 buckets; 512 MiB read and written are 81.  By counters (profiles/sort_quantiles_sq_counters.txt) the count is bound by its vector
// instructions, 20 a key.  The scatter and the buckets are neither: vector units busy 43 and 60 %, LDS 35 and 41 % of the time (half of that bank
// conflicts), and over two fifths of a wave's time is waiting, in phases that one workgroup a compute unit does not overlap; the scatter also writes 367 MiB
// for 256 (370 in Int32), runs of ten keys on the average (with tiles of 12288 keys and twice as many workgroups 181, 87 if nothing is written).  The fewer bytes a
// key, the shorter the runs' lines: keys of 8 bytes, and sortperm, whose index would travel along, take two levels of splitters (rk_sort_split.hpp).
// Below 2^22 keys the launches count: Float32[2^22] 91 in rk_sort_split.hpp, 95 so.  Int32[2^22] of 8 bits, one radix pass and eight launches
// for nothing more, 69 -> 76, [2^23] 94 -> 96, [2^24] 132 -> 124; of 32 bits [2^22] 147 -> 108, which the others would pay for.
//
// Float32 around a number or with one in large numbers, radix passes / cells over the whole sampled range / so, us a call of 2^24 and of 2^26 keys: N(1000, 1) with
// 0.1 % zeros 239 / 277 / 243 and 727 / 864 / 604; N(1013, 10) with 0.1 % NaN 241 / 282 / 232 and 734 / 878 / 543; N(20, 5) with 0.1 % -9999 239 / 209 / 234 and
// 742 / 948 / 527; half zeros 248 / 289 / 219 and 743 / 885 / 506; nine in ten zeros 245 / 285 / 194 and 723 / 849 / 437.  Int32 ids with 0.01 % typemax
// 265 / 741 / 220 and 777 / 1025 / 522.  (Of 2^23 keys 0.95 to 1.2 times as fast as radix passes.)
//
// If a bucket exceeds what its workgroup holds (SQ_CAP) all the same, that is known before a key is moved, mostly from the sample, and the radix passes run
// instead: their plan is there, or the plan says that none runs, and the kernels of the other way end at once.  So they do where the sample says that a bucket has
// few values.  That costs them sample, table and launches, and above 2^24 keys passes whose workgroups take several tiles: Float32 of N(0, 1) rounded to 0.001
// [2^24] 258 -> 294, [2^26] 776 -> 897; of 256 levels 242 -> 278, 719 -> 837; Int32 of a power law [2^23] 170 -> 211, [2^24] 238 -> 278, of 16 bits [2^23] 120 -> 138,
// [2^24] 164 -> 181, [2^26] 463 -> 494.
#pragma once

#include <cmath>

#include "rk_sort_buckets.hpp"

namespace rk {

constexpr int SQ_BLOCK = 1024;
constexpr int64_t SQ_TILE = 6 * 4 * SQ_BLOCK;        // keys a tile: what LDS holds beside the tables
constexpr uint32_t SQ_CELLS = 4096;              // of the sampled range
constexpr uint32_t SQ_MAX_K = 2560;              // buckets, a multiple of 64
constexpr uint32_t SQ_GROUP = 16;                // neighbouring keys that are sampled together: a line of memory is fetched anyway
// Samples a bucket.  Half as many take 3.5 + 2 us less of Float32[2^26] and 1 + 0.5 of [2^24], and make the buckets less alike: of N(1000, 1), whose buckets are little more
// than a cell, 485 -> 488 us a call of 2^26 keys and 177 -> 188 of 2^24.
inline uint32_t sq_samples(int64_t n) { return n <= (int64_t)1 << 25 ? 512u : 256u; }
constexpr uint32_t SQ_SAMPLES_EACH = 4;          // samples a thread fetches
constexpr uint32_t SQ_TABLE_GRID = 64;
constexpr uint32_t SQ_CHUNKS = 512;              // of tiles, at most
constexpr uint32_t SQ_CHUNK_TILES = 6;
constexpr uint32_t SQ_COLUMNS = 64;              // buckets that a workgroup of sq_offsets_kernel takes
constexpr uint32_t SQ_FREQUENT = 4;              // values in large numbers, at most: zeros, NaNs, a number that stands for a missing one
constexpr uint32_t SQ_HEAVY = SQ_FREQUENT + 2u;  // and the two beyond which keys are few and far

struct SqCtl {
    uint32_t lo, range, up;                      // a key's cell: the highest 12 bits of its distance from lo, at most range, << up
    uint32_t way;                                // SQ_BUCKETS ...
    uint32_t ok;                                 // the buckets fit
    uint32_t ticket[3];
    uint32_t heavies, heavy[SQ_HEAVY], heavy_bucket[SQ_HEAVY], heavy_size[SQ_HEAVY];       // values with a bucket of their own
};
// SQ_PLANNED: the radix passes run as they are planned: over all digits (floats), or over those that a read of all keys in front has found to
// vary (integers); SQ_SOME_DIGITS: one bucket holds far too many of the samples, or buckets hold few values, and floats get a plan after such a read.
constexpr uint32_t SQ_BUCKETS = 0, SQ_PLANNED = 1, SQ_SOME_DIGITS = 2;
constexpr uint32_t SQ_CHECKED = 16384;           // samples that are looked at for that
// Values a bucket, on the average: with fewer the lanes of a wave meet on few counters in LDS (N(0, 1) rounded to 0.001, three values a bucket of 2^24
// keys: the bucket kernel 281 us for 54, the call 404 for 294 by radix passes; five of 2^23: 288 and 212).
constexpr uint32_t SQ_FEW_VALUES = 8;
// Integers that differ in so few digits are sorted by radix passes, and those of fewer values than there are cells.  Two passes / buckets, 16 bits, us a
// call: 2^24 keys 183 / 199, 2^25 285 / 287, 2^26 534 / 498; 1000 values 191 / 366, 296 / 484, 515 / 538.
constexpr int64_t SQ_TWO_PASSES = (int64_t)1 << 25;
inline uint32_t sq_few_passes(int64_t n) { return n <= SQ_TWO_PASSES ? 2u : 1u; }

// What a cell holds: the share of the samples in front of it, in 65535ths, << 16, and its own.  With the place in the cell as a 16-bit
// fraction that is one product, at most where the next cell starts: a key's share of the k buckets, in 2^-32.
// Keys beyond the ends count as these.  A heavy value stands in a bucket of its own, between those of the smaller and of the larger keys
// of its place, which are two apart then; its keys are counted, not moved, and written by sq_bucket_kernel.
struct SqMap { uint32_t lo, range, up, k, heavies, heavy[SQ_HEAVY]; };
__device__ __forceinline__ uint32_t sq_lines(uint32_t k, uint32_t heavies) { return (heavies != 0u ? k - 2u * SQ_HEAVY : k) << 8; }
__device__ __forceinline__ SqMap sq_map(const SqCtl* ctl, uint32_t k) {
    const uint32_t heavies = sb_uniform(ctl->heavies);
    SqMap m{ctl->lo, ctl->range, ctl->up, sq_lines(k, heavies), heavies, {}};
#pragma unroll
    for (uint32_t h = 0; h < SQ_HEAVY; ++h) m.heavy[h] = sb_uniform(ctl->heavy[h]);
    return m;
}

__device__ __forceinline__ uint32_t sq_bucket(const uint32_t* cells, const SqMap& m, uint32_t key) {
    uint32_t t = __builtin_elementwise_sub_sat(key, m.lo);
    t = (t < m.range ? t : m.range) << m.up;
    const uint32_t cell = cells[t >> 20];
    uint32_t share;
    asm("v_mad_u32_u16 %0, %1, %2, %2" : "=v"(share) : "v"(t >> 4), "v"(cell));
    return (uint32_t)((uint64_t)(share >> 8) * (uint64_t)(m.k & 0xffffffu) >> 32);
}

// f(h, value) for every heavy value.
template <typename F> __device__ __forceinline__ void sq_heavies(const SqMap& m, F&& f) {
    static_assert(SQ_HEAVY == 6u, "");
    if (m.heavies == 0u) return;
    f(0, m.heavy[0]);
    if (m.heavies == 1u) return;
    f(1, m.heavy[1]);
    if (m.heavies == 2u) return;
    f(2, m.heavy[2]);
    if (m.heavies == 3u) return;
    f(3, m.heavy[3]);
    if (m.heavies == 4u) return;
    f(4, m.heavy[4]);
    if (m.heavies == 5u) return;
    f(5, m.heavy[5]);
}

// The buckets b[i] of the keys, as sq_bucket gives them, with those of the heavy values among them.
template <int N> __device__ __forceinline__ void sq_around(const SqMap& m, const uint32_t (&key)[N], uint32_t (&b)[N]) {
    sq_heavies(m, [&](int, uint32_t v) {
#pragma unroll
        for (int i = 0; i < N; ++i) b[i] += (key[i] >= v ? 1u : 0u) + (key[i] > v ? 1u : 0u);
    });
}

// enc_bits / dec_bits of sort and sort!, which keep the bit patterns of NaNs, without branches.  flip: all ones for rev=true.
template <typename T> __device__ __forceinline__ uint32_t sq_enc(uint32_t raw, uint32_t flip) {
    if constexpr (std::is_integral<T>::value) return raw ^ (0x80000000u ^ flip);
    else return ((raw ^ ((uint32_t)((int32_t)raw >> 31) | 0x80000000u)) - 0x007fffffu) ^ flip;
}
template <typename T> __device__ __forceinline__ uint32_t sq_dec(uint32_t key, uint32_t flip) {
    if constexpr (std::is_integral<T>::value) return key ^ (0x80000000u ^ flip);
    const uint32_t u = (key ^ flip) + 0x007fffffu;
    return u ^ ((uint32_t)((int32_t)~u >> 31) | 0x80000000u);
}

// A value that the compiler does not know to be the same as before.
template <typename V> __device__ __forceinline__ V sq_again(V v) { asm volatile("" : "+v"(v)); return v; }
template <typename V> __device__ __forceinline__ V sq_again_uniform(V v) { asm volatile("" : "+s"(v)); return v; }

// p[i] of less than 2^32 bytes: a 32-bit offset to a pointer that all lanes share.
template <typename T> __device__ __forceinline__ T& sq_at(T* p, uint32_t i) {
    return *(T*)((char*)const_cast<typename std::remove_const<T>::type*>(p) + (size_t)(uint32_t)(i * (uint32_t)sizeof(T)));
}

// ---- sample -------------------------------------------------------------------------------------------------------
// Groups of neighbouring keys from somewhere in each of equal stretches of the array.
template <typename T>
__global__ __launch_bounds__(SQ_BLOCK) void sq_sample_kernel(const T* __restrict__ keys, uint32_t n, uint32_t flip, SortCtl* ctl, int first_source, uint32_t few_passes, uint32_t* __restrict__ sample,
                                                             uint2* __restrict__ ends, uint32_t* __restrict__ hist, SqCtl* sq) {
    __shared__ uint32_t part[2][SQ_BLOCK / WAVE];
    const uint32_t tid = threadIdx.x, groups = gridDim.x * (SQ_BLOCK * SQ_SAMPLES_EACH / SQ_GROUP);
    const bool few = std::is_integral<T>::value && (ctl->nexec <= few_passes || (uint32_t)ctl->key_max - ~(uint32_t)ctl->inv_min < SQ_CELLS);
    if (blockIdx.x == 0u && tid == 0u) {
        SqCtl c{};
        c.way = few ? SQ_PLANNED : SQ_BUCKETS;
        *sq = c;
    }
    if (few) return;
    uint32_t v[SQ_SAMPLES_EACH], lo = ~0u, hi = 0u;
#pragma unroll
    for (uint32_t i = 0; i < SQ_SAMPLES_EACH; ++i) {
        const uint32_t s = blockIdx.x * (SQ_BLOCK * SQ_SAMPLES_EACH) + i * SQ_BLOCK + tid, g = s / SQ_GROUP;
        const uint32_t a = (uint32_t)((uint64_t)g * n / groups), b = (uint32_t)((uint64_t)(g + 1u) * n / groups);
        uint32_t h = (g + 1u) * 0x9e3779b1u;
        h ^= h >> 15;
        h *= 0x85ebca77u;
        v[i] = __builtin_bit_cast(uint32_t, keys[a + __umulhi(h, b - a - (SQ_GROUP - 1u)) + s % SQ_GROUP]);     // (b - a >= SQ_GROUP)
    }
#pragma unroll
    for (uint32_t i = 0; i < SQ_SAMPLES_EACH; ++i) {
        v[i] = sq_enc<T>(v[i], flip);
        lo = v[i] < lo ? v[i] : lo;
        hi = v[i] > hi ? v[i] : hi;
        sample[blockIdx.x * (SQ_BLOCK * SQ_SAMPLES_EACH) + i * SQ_BLOCK + tid] = v[i];
    }
    lo = wave_reduce(lo, OpMin());
    hi = wave_reduce(hi, OpMax());
    if (tid % WAVE == 0u) { part[0][tid / WAVE] = lo; part[1][tid / WAVE] = hi; }
    for (uint32_t c = blockIdx.x * SQ_BLOCK + tid; c < SQ_CELLS; c += gridDim.x * SQ_BLOCK) hist[c] = 0u;
    __syncthreads();
    if (tid == 0u) {
        for (int w = 1; w < SQ_BLOCK / WAVE; ++w) {
            lo = part[0][w] < lo ? part[0][w] : lo;
            hi = part[1][w] > hi ? part[1][w] : hi;
        }
        ends[blockIdx.x] = make_uint2(lo, hi);
    }
    if (!std::is_integral<T>::value && blockIdx.x == 0u) {               // as sort_init_kernel
        for (uint32_t i = tid; i < SORT_CTL_CLEAR; i += SQ_BLOCK) ctl->skip[i] = 0u;
        __syncthreads();
        if (tid == 0u) {
            ctl->inv_min = ~0ull;
            sort_make_plan(ctl, 4, false, 0ull, ~0ull, first_source);
        }
    }
}

// Adds one to the counter of each lane; lanes that go where the first one goes add together if they are many (values in large numbers).
// (All lanes call.  Float32[2^26], sq_table_kernel: nine in ten keys zero 38.1 -> 19.0 us, two values 33.4 -> 26.2, normal 18.2 -> 18.8.)
__device__ __forceinline__ void sq_add(uint32_t* cnt, uint32_t c) {
    const uint32_t c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
    const uint32_t same = (uint32_t)__popcll(__ballot(c == c0));
    if (same < SB_TOGETHER) {
        atomicAdd(&cnt[c], 1u);
    } else {
        const bool first = threadIdx.x % WAVE == 0u;
        if (first || c != c0) atomicAdd(&cnt[c], first ? same : 1u);
    }
}

// ---- the buckets' bounds ----------------------------------------------------------------------------------------------
// Counts the samples in cells.  If a few values stand for many of the samples, or nearly all lie in few of the cells -- one NaN or zero among a
// thousand values around 1000 leaves them two -- it says so, and the kernel runs again (REFINE) with these values apart and the cells where the keys
// are: of 2^26 keys of N(1000, 1) 0.1 % zeros, or of N(1013, 10) 0.1 % NaN, are sorted by buckets then.
template <bool REFINE>
__global__ __launch_bounds__(SQ_BLOCK) void sq_table_kernel(const uint32_t* __restrict__ sample, uint32_t samples, const uint2* __restrict__ ends,
                                                            uint32_t nends, uint32_t offset, uint32_t k, uint32_t each, uint32_t too_many, int floats, uint32_t* hist, uint32_t* __restrict__ cells, SqCtl* sq) {
    constexpr uint32_t PER = SQ_CELLS / SQ_BLOCK;
    __shared__ uint32_t h[SQ_CELLS], cnt[SQ_MAX_K];
    __shared__ uint32_t part[4][SQ_BLOCK / WAVE], lds_ticket;
    constexpr uint32_t SQ_PICKS = 128;
    __shared__ uint32_t found, end_cell[2], heavy_cell[SQ_FREQUENT], picked[SQ_FREQUENT], pick[SQ_FREQUENT][SQ_PICKS];
    __shared__ uint32_t frequent, value[SQ_FREQUENT], value_cell[SQ_FREQUENT], value_same[SQ_FREQUENT];
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    if (sq->way == SQ_PLANNED || (REFINE && sq->heavies == 0u)) return;
    uint32_t lo = ~0u, hi = 0u, up = 0u;
    SqMap map{};
    if (REFINE) {
        map = sq_map(sq, k);
        lo = map.lo;
        hi = lo + map.range;
        up = map.up;
    } else {
        for (uint32_t i = tid; i < nends; i += SQ_BLOCK) {
            const uint2 e = ends[i];
            lo = e.x < lo ? e.x : lo;
            hi = e.y > hi ? e.y : hi;
        }
        lo = wave_reduce(lo, OpMin());
        hi = wave_reduce(hi, OpMax());
        if (lane == 0u) { part[0][wave] = lo; part[1][wave] = hi; }
    }
#pragma unroll
    for (uint32_t c = 0; c < PER; ++c) h[tid + c * SQ_BLOCK] = 0u;
    __syncthreads();
    // Cells start where binades do: the density of floats halves or doubles there, which a line in the middle of a cell would not follow.
    const auto divide = [&]() {
        const auto bits_up = [](uint32_t range) { return range == 0u ? 31u : (uint32_t)__clz((int)range); };
        for (up = bits_up(hi - lo);; --up) {
            const uint32_t most = up < 20u ? (1u << (20u - up)) - 1u : 0u, down = (lo + offset) & most;
            const uint32_t from = down < lo ? lo - down : 0u;
            if (bits_up(hi - from) >= up) { lo = from; break; }
        }
    };
    if (!REFINE) {
        for (int w = 0; w < SQ_BLOCK / WAVE; ++w) {
            lo = part[0][w] < lo ? part[0][w] : lo;
            hi = part[1][w] > hi ? part[1][w] : hi;
        }
        divide();
    }
    const uint32_t range = hi - lo;
    const auto is_heavy = [&](uint32_t x) {
        bool heavy = false;
        sq_heavies(map, [&](int, uint32_t w) { heavy = heavy || x == w; });
        return heavy;
    };
    // The lanes of a wave are far apart in the array: of keys in order, neighbours would all add to one cell.
    const uint32_t quads = samples / 4u / SQ_TABLE_GRID;                // (a multiple of WAVE)
    const uint4* const mine = (const uint4*)sample + (size_t)blockIdx.x * quads + lane * (quads / WAVE);
    constexpr uint32_t UNR = 4;
    for (uint32_t i = wave; i < quads / WAVE; i += SQ_BLOCK / WAVE * UNR) {
        uint4 v[UNR];
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) v[u] = mine[i + u * (SQ_BLOCK / WAVE) < quads / WAVE ? i + u * (SQ_BLOCK / WAVE) : 0u];
#pragma unroll
        for (uint32_t u = 0; u < UNR; ++u) {
            if (i + u * (SQ_BLOCK / WAVE) >= quads / WAVE) continue;
            if (!REFINE) {
                sq_add(h, (v[u].x - lo) << up >> 20);
                sq_add(h, (v[u].y - lo) << up >> 20);
                sq_add(h, (v[u].z - lo) << up >> 20);
                sq_add(h, (v[u].w - lo) << up >> 20);
            } else {
                const uint32_t x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint32_t d = __builtin_elementwise_sub_sat(x[j], lo);
                    if (!is_heavy(x[j])) atomicAdd(&h[(d < range ? d : range) << up >> 20], 1u);
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < PER; ++c) {
        const uint32_t x = h[tid + c * SQ_BLOCK];
        if (x != 0u) atomicAdd(&hist[tid + c * SQ_BLOCK], x);
    }
    publish_barrier();
    __syncthreads();
    if (tid == 0u) lds_ticket = atomicAdd(&sq->ticket[REFINE ? 2 : 0], 1u);
    __syncthreads();
    if (lds_ticket != SQ_TABLE_GRID - 1u) return;
    // the last one
    const auto scan = [&](const uint32_t (&c)[PER], uint32_t& all) {        // how many are in front of the thread's cells, and all of them
        uint32_t sum = 0u;
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) sum += c[j];
        const uint32_t inc = wave_scan_inclusive(sum, OpAdd(), 0u);
        __syncthreads();
        if (lane == WAVE - 1) part[2][wave] = inc;
        __syncthreads();
        uint32_t before = inc - sum;
        all = 0u;
        for (uint32_t w = 0; w < SQ_BLOCK / WAVE; ++w) {
            before += w < wave ? part[2][w] : 0u;
            all += part[2][w];
        }
        return before;
    };
    uint32_t c[PER], all;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) c[j] = load_agent(&hist[tid * PER + j]);
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) h[tid * PER + j] = c[j];
    uint32_t before = scan(c, all);
    if constexpr (!REFINE) {
        // the cells beyond which half a bucket's share of the samples lies
        const auto find_ends = [&](uint32_t before, uint32_t all) {
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                const uint32_t behind = all - before - c[j];
                if (before <= each / 2u && before + c[j] > each / 2u) end_cell[0] = tid * PER + j;
                if (behind <= each / 2u && behind + c[j] > each / 2u) end_cell[1] = tid * PER + j;
                before += c[j];
            }
        };
        // whether these leave an eighth of the range or less
        const auto few_cells = [&]() { return up < 20u && end_cell[0] <= end_cell[1] && end_cell[1] - end_cell[0] < SQ_CELLS / 8u; };
        if (tid < SQ_FREQUENT) picked[tid] = 0u;
        if (tid == 0u) { found = 0u; frequent = 0u; end_cell[0] = 0u; end_cell[1] = SQ_CELLS - 1u; }
        __syncthreads();
        find_ends(before, all);
        // a cell far above its neighbours may hold such a value
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            const uint32_t at = tid * PER + j, beside = (at != 0u ? h[at - 1u] : 0u) + (at + 1u < SQ_CELLS ? h[at + 1u] : 0u);
            if (c[j] >= beside + beside / 8u + each / 2u) {
                const uint32_t s = atomicAdd(&found, 1u);
                if (s < SQ_FREQUENT) heavy_cell[s] = at;
            }
        }
        __syncthreads();
        const uint32_t heavy_cells = found <= SQ_FREQUENT ? found : 0u;
        if (range != 0u && (heavy_cells != 0u || few_cells())) {
            const auto add_heavy = [&](uint32_t v) {
                if (is_heavy(v)) return;
#pragma unroll
                for (uint32_t q = 0; q < SQ_HEAVY; ++q) map.heavy[q] = q == map.heavies ? v : map.heavy[q];
                ++map.heavies;
            };
            if (heavy_cells != 0u) {
                // up to 128 of the cell's samples: values that half a bucket's share of the samples, by these, are
                constexpr uint32_t FROM = 4u * SQ_CHECKED, EACH = FROM / 4u / SQ_BLOCK;
#pragma unroll 4
                for (uint32_t u = 0; u < EACH; ++u) {
                    const uint4 v = ((const uint4*)sample)[(lane * (FROM / 4u / WAVE) + u * (SQ_BLOCK / WAVE) + wave) * (samples / FROM)];
                    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        for (uint32_t s = 0; s < heavy_cells; ++s)
                            if ((x[i] - lo) << up >> 20 == heavy_cell[s] && picked[s] < SQ_PICKS) {
                                const uint32_t p = atomicAdd(&picked[s], 1u);
                                if (p < SQ_PICKS) pick[s][p] = x[i];
                            }
                }
                __syncthreads();
                if (tid < heavy_cells && picked[tid] > SQ_PICKS) picked[tid] = SQ_PICKS;
                __syncthreads();
                const uint32_t s = tid / SQ_PICKS, p = tid % SQ_PICKS;
                static_assert(SQ_FREQUENT * SQ_PICKS <= SQ_BLOCK, "a thread a pick");
                if (s < heavy_cells && p < picked[s]) {
                    uint32_t same = 0u, in_front = 0u;
                    for (uint32_t q = 0; q < picked[s]; ++q) {
                        const bool is = pick[s][q] == pick[s][p];
                        same += is ? 1u : 0u;
                        in_front += is && q < p ? 1u : 0u;
                    }
                    if (in_front == 0u && same >= (picked[s] < 16u ? 2u : 3u) && (uint64_t)h[heavy_cell[s]] * same >= (uint64_t)(each / 2u) * picked[s]) {
                        const uint32_t f = atomicAdd(&frequent, 1u);
                        if (f < SQ_FREQUENT) { value[f] = pick[s][p]; value_cell[f] = s; value_same[f] = same; }
                    }
                }
                if (tid == 0u) { end_cell[0] = 0u; end_cell[1] = SQ_CELLS - 1u; }
                __syncthreads();
                if (frequent <= SQ_FREQUENT) {
                    for (uint32_t f = 0; f < frequent; ++f) {
                        add_heavy(value[f]);
                        const uint32_t t = value_cell[f];
#pragma unroll
                        for (uint32_t j = 0; j < PER; ++j)       // what remains
                            if (heavy_cell[t] == tid * PER + j) c[j] -= (uint32_t)((uint64_t)h[tid * PER + j] * value_same[f] / picked[t]);
                    }
                    uint32_t all_of = all;
                    const uint32_t before_of = scan(c, all_of);
                    find_ends(before_of, all_of);
                    __syncthreads();
                }
            }
            // (of more such values at one place the buckets would not fit)
            if (frequent <= SQ_FREQUENT && few_cells()) {
                const uint32_t new_lo = lo + (end_cell[0] << (20u - up));
                const uint64_t end = (uint64_t)lo + ((uint64_t)(end_cell[1] + 1u) << (20u - up)) - 1u;
                const uint32_t new_hi = end < (uint64_t)hi ? (uint32_t)end : hi;
                if (new_lo != 0u) add_heavy(new_lo - 1u);       // keys beyond are no neighbours of those in front: a bucket of both would not be spread
                if (new_hi != ~0u) add_heavy(new_hi + 1u);
                lo = new_lo;
                hi = new_hi;
                divide();
            }
            if (map.heavies != 0u) {
#pragma unroll
                for (uint32_t j = 0; j < PER; ++j) hist[tid * PER + j] = 0u;
                if (tid != 0u) return;
                sq->lo = lo;
                sq->range = hi - lo;
                sq->up = up;
                sq->heavies = map.heavies;
                for (uint32_t q = 0; q < SQ_HEAVY; ++q) sq->heavy[q] = map.heavy[q];
                return;
            }
            // (c may be less by now)
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) c[j] = h[tid * PER + j];
        }
        map = SqMap{lo, range, up, sq_lines(k, 0u), 0u, {}};
    }
    const float per_sample = 65535.f / (float)(all != 0u ? all : 1u);
    const auto share = [&](uint32_t x) { const uint32_t s = (uint32_t)((float)x * per_sample); return s < 65535u ? s : 65535u; };
    uint32_t at = share(before);
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        before += c[j];
        const uint32_t next = share(before);
        h[tid * PER + j] = at << 16 | (next - at);
        cells[tid * PER + j] = at << 16 | (next - at);
        at = next;
    }
    for (uint32_t b = tid; b < k; b += SQ_BLOCK) cnt[b] = 0u;
    constexpr uint32_t QUADS = SQ_CHECKED / 4u / SQ_BLOCK;
    const uint32_t stride = samples / 4u / (SQ_CHECKED / 4u), key0 = sample[0];
    uint32_t varying = 0u, most = 0u, others = 0u, first[QUADS], first_bucket[QUADS];
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < QUADS; ++u) {
        const uint4 v = ((const uint4*)sample)[(lane * (SQ_CHECKED / 4u / WAVE) + u * (SQ_BLOCK / WAVE) + wave) * stride];
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            varying |= x[i] ^ key0;
            b[i] = sq_bucket(h, map, x[i]);
        }
        if constexpr (REFINE) sq_around(map, x, b);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!REFINE) sq_add(cnt, b[i]);
            else if (!is_heavy(x[i])) atomicAdd(&cnt[b[i]], 1u);
            else b[i] = ~0u;
        }
        first[u] = x[0];
        first_bucket[u] = b[0];
    }
    __syncthreads();
    for (uint32_t b = tid; b < k; b += SQ_BLOCK) most = cnt[b] > most ? cnt[b] : most;
    // how many samples, of those that are not neighbours, equal one of their bucket; low half: how many are not that one
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < QUADS; ++u)
        if (first_bucket[u] != ~0u) cnt[first_bucket[u]] = first[u];
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < QUADS; ++u) others += first_bucket[u] != ~0u && cnt[first_bucket[u]] == first[u] ? 1u << 16 : 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < QUADS; ++u)
        if (first_bucket[u] != ~0u) cnt[first_bucket[u]] = u * SQ_BLOCK + tid;
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < QUADS; ++u)
        if (first_bucket[u] != ~0u) others += cnt[first_bucket[u]] == u * SQ_BLOCK + tid ? 0u - (1u << 16) : 1u;
    most = wave_reduce(most, OpMax());
    varying = wave_reduce(varying, OpOr());
    others = wave_reduce(others, OpAdd());
    if (lane == 0u) { part[0][wave] = most; part[1][wave] = varying; part[3][wave] = others; }
    __syncthreads();
    if (tid != 0u) return;
    for (int w = 1; w < SQ_BLOCK / WAVE; ++w) {
        most = part[0][w] > most ? part[0][w] : most;
        varying |= part[1][w];
        others += part[3][w];
    }
    const bool all_vary = (varying & 0xffu) != 0u && (varying >> 8 & 0xffu) != 0u && (varying >> 16 & 0xffu) != 0u && varying >> 24 != 0u;
    const bool few_values = (others >> 16) * SQ_FEW_VALUES > (others & 0xffffu);
    sq->lo = map.lo;
    sq->range = map.range;
    sq->up = map.up;
    if constexpr (REFINE) {
        for (uint32_t q = 0; q < SQ_HEAVY; ++q) {
            uint32_t x[1] = {map.heavy[q]}, b[1] = {sq_bucket(h, map, x[0])};
            sq_around(map, x, b);
            sq->heavy_bucket[q] = q < map.heavies ? b[0] : ~0u;
        }
    }
    sq->way = most <= too_many && !few_values ? SQ_BUCKETS : floats != 0 && !all_vary ? SQ_SOME_DIGITS : SQ_PLANNED;
}

// ---- tiles ----------------------------------------------------------------------------------------------------------
// Thread t holds the 4 * NV keys 4 (t + v * 1024) ... of a tile; `count` of the tile's exist.
template <int NV> struct SqTile {
    uint32_t key[4 * NV];
    template <bool FULL> __device__ __forceinline__ void load(const uint32_t* p, uint32_t count) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const uint32_t at = 4u * (threadIdx.x + v * SQ_BLOCK);
            if (FULL || at + 4u <= count) {
                const auto x = load_nt_elems<uint32_t, 4>(p + at);
#pragma unroll
                for (int j = 0; j < 4; ++j) key[4 * v + j] = x[j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) key[4 * v + j] = p[at + j < count ? at + j : 0u];
            }
        }
    }
    template <bool FULL> __device__ __forceinline__ bool has(int i, uint32_t count) const {
        return FULL || 4u * (threadIdx.x + i / 4 * SQ_BLOCK) + i % 4 < count;
    }
};

// Places r[i] among the keys of the bins b[i], in no order.  Lanes of a wave that all go to one bin (input that is sorted already, or few
// values) add to it once; that is asked for every fourth key, and once for all of them: the additions are in flight together.
// has(i): the key exists.  (All lanes call.)
template <int N, typename Has> __device__ __forceinline__ void sq_take(uint32_t* cnt, const uint32_t (&b)[N], uint32_t (&r)[N], Has&& has) {
    bool together = false;
#pragma unroll
    for (int i = 0; i < N; i += 4) together = together || __ballot(b[i] != (uint32_t)__builtin_amdgcn_readfirstlane((int)b[i])) == 0ull;
    if (!together) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            r[i] = 0u;
            if (has(i)) r[i] = atomicAdd(&cnt[b[i]], 1u);
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t b0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)b[i]), lane = threadIdx.x % WAVE;
            r[i] = 0u;
            if (__ballot(!has(i) || b[i] != b0) == 0ull) {
                if (lane == 0u) r[i] = atomicAdd(&cnt[b0], (uint32_t)WAVE);
                r[i] = (uint32_t)__builtin_amdgcn_readfirstlane((int)r[i]) + lane;
            } else if (has(i)) {
                r[i] = atomicAdd(&cnt[b[i]], 1u);
            }
        }
    }
}

// A chunk of up to SQ_CHUNK_TILES neighbouring tiles.  rows[tile][bucket]: keys of the bucket in the chunk's tiles in front (and a row
// behind the last tile, as of one more); totals[chunk][bucket].  (A row's 16 bits overflow only where the bucket does not fit.)
// The rows stay in LDS until the last tile: a store between two tiles would be waited for with the keys asked for behind it.
template <typename T>
__global__ __launch_bounds__(SQ_BLOCK, 8) void sq_count_kernel(const T* __restrict__ keys, uint32_t n, uint32_t flip, uint32_t k, const uint32_t* __restrict__ cells,
                                                               uint32_t ntiles, uint32_t chunk_tiles, uint32_t* __restrict__ rows,
                                                               uint32_t* __restrict__ totals, uint32_t* __restrict__ seen, const SqCtl* sq) {
    constexpr uint32_t TILE = SQ_TILE;
    constexpr bool INTEGERS = std::is_integral<T>::value;
    __shared__ alignas(16) uint32_t table[SQ_CELLS];
    __shared__ alignas(8) uint32_t cnt[SQ_MAX_K];
    __shared__ uint32_t row[SQ_CHUNK_TILES][SQ_MAX_K / 2u];
    __shared__ uint32_t part[SQ_BLOCK / WAVE];
    const uint32_t tid = threadIdx.x;
    const uint32_t t0 = blockIdx.x * chunk_tiles, t1 = t0 + chunk_tiles < ntiles ? t0 + chunk_tiles : ntiles;
    const uint32_t whole = n / TILE < t1 ? n / TILE : t1;     // the last tile may not be
    constexpr uint32_t UNIT = 8u * SQ_BLOCK, UNITS = TILE / UNIT;         // a tile is read two vectors a lane at a time
    const uint32_t units = whole * UNITS;
    SqTile<2> next;
    const uint32_t way = sq->way;
    if (way == SQ_PLANNED) return;
    if (t0 < whole) next.template load<true>((const uint32_t*)keys + (size_t)t0 * TILE, UNIT);
    const SqMap map = sq_map(sq, k);
#pragma unroll
    for (uint32_t c = 0; c < SQ_CELLS / SQ_BLOCK; c += 4) *(uint4*)&table[4u * tid + c * SQ_BLOCK] = *(const uint4*)&cells[4u * tid + c * SQ_BLOCK];
    for (uint32_t b = tid; b < k; b += SQ_BLOCK) cnt[b] = 0u;
    for (uint32_t b = tid; b < k / 2u; b += SQ_BLOCK) row[0][b] = 0u;
    const uint32_t key0 = sq_enc<T>(__builtin_bit_cast(uint32_t, keys[0]), flip);
    uint32_t varying = 0u, heavy_count[SQ_HEAVY] = {};              // (of the wave)
    const auto add = [&](const SqTile<2>& t, auto&& has) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            uint32_t x[4], b[4], r[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = sq_enc<T>(t.key[4 * v + i], flip);                   // (where there is none, the tile's first)
                if (!INTEGERS) varying |= x[i] ^ key0;
            }
            if (way != SQ_BUCKETS) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = sq_bucket(table, map, x[i]);
            if (map.heavies == 0u) {
                sq_take(cnt, b, r, [&](int i) { return has(4 * v + i); });
                continue;
            }
            uint32_t gone = 0u;
            sq_heavies(map, [&](int h, uint32_t w) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool is = x[i] == w && has(4 * v + i);
                    heavy_count[h] += (uint32_t)__popcll(__ballot(is));
                    gone |= is ? 1u << i : 0u;
                    b[i] += (x[i] >= w ? 1u : 0u) + (x[i] > w ? 1u : 0u);
                }
            });
            sq_take(cnt, b, r, [&](int i) { return has(4 * v + i) && (gone >> i & 1u) == 0u; });
        }
    };
    __syncthreads();
    for (uint32_t tile = t0; tile < whole; ++tile) {
        for (uint32_t u = tile * UNITS; u < (tile + 1u) * UNITS; ++u) {
            const SqTile<2> now = next;
            if (u + 1u < units) next.template load<true>((const uint32_t*)keys + (size_t)(u + 1u) * UNIT, UNIT);
            add(now, [](int) { return true; });
        }
        if (tile + 1u < t1) {
            __syncthreads();
            for (uint32_t b = tid; b < k / 2u; b += SQ_BLOCK) {
                const uint2 c = *(const uint2*)&cnt[2u * b];
                row[tile + 1u - t0][b] = (c.x & 0xffffu) | c.y << 16;
            }
            __syncthreads();
        }
    }
    if (whole < t1) {
        for (uint32_t e0 = whole * TILE; e0 < n; e0 += UNIT) {
            const uint32_t count = n - e0 < UNIT ? n - e0 : UNIT;
            next.template load<false>((const uint32_t*)keys + e0, count);
            add(next, [&](int i) { return next.template has<false>(i, count); });
        }
    }
    __syncthreads();
    if (map.heavies != 0u) {
        sq_heavies(map, [&](int h, uint32_t) {
            if (tid % WAVE == 0u) atomicAdd(&cnt[sq->heavy_bucket[h]], heavy_count[h]);
        });
        __syncthreads();
    }
    for (uint32_t b = tid; b < k; b += SQ_BLOCK) totals[(size_t)blockIdx.x * k + b] = cnt[b];
    for (uint32_t b = tid; b < k / 2u; b += SQ_BLOCK) {
        for (uint32_t tile = t0; tile < t1; ++tile) rows[(size_t)tile * (k / 2u) + b] = row[tile - t0][b];
        if (t1 == ntiles) {
            const uint2 c = *(const uint2*)&cnt[2u * b];
            rows[(size_t)ntiles * (k / 2u) + b] = ntiles % chunk_tiles == 0u ? 0u : (c.x & 0xffffu) | c.y << 16;
        }
    }
    // (a store a chunk, for the kernel behind to put together: 16 atomics a workgroup to one word took 100 us)
    if constexpr (!INTEGERS) {
        varying = wave_reduce(varying, OpOr());
        if (tid % WAVE == 0u) part[tid / WAVE] = varying;
        __syncthreads();
        if (tid != 0u) return;
        for (int w = 1; w < SQ_BLOCK / WAVE; ++w) varying |= part[w];
        seen[blockIdx.x] = varying;
    }
}

// totals[chunk][bucket] becomes where the chunk's keys of the bucket go, from the bucket's start (and those of one more chunk); starts[bucket].
__global__ __launch_bounds__(SQ_BLOCK) void sq_offsets_kernel(uint32_t* totals, uint32_t nchunks, uint32_t k, uint32_t cap, uint32_t* sizes,
                                                              uint32_t* __restrict__ starts, const uint32_t* __restrict__ seen, SqCtl* sq, SortCtl* ctl, int floats, int first_source) {
    constexpr uint32_t GROUPS = SQ_BLOCK / SQ_COLUMNS, ROWS = SQ_CHUNKS / GROUPS;
    __shared__ uint32_t sum[GROUPS][SQ_COLUMNS];
    __shared__ uint32_t part[3][SQ_BLOCK / WAVE], lds_ticket;
    const uint32_t tid = threadIdx.x, g = tid / SQ_COLUMNS, col = blockIdx.x * SQ_COLUMNS + tid % SQ_COLUMNS, lane = tid % WAVE, wave = tid / WAVE;
    const uint32_t each = (nchunks + GROUPS - 1u) / GROUPS, first = g * each;
    const uint32_t way = sq->way;
    if (way == SQ_PLANNED || (way != SQ_BUCKETS && blockIdx.x != 0u)) return;
    uint32_t v[ROWS], mine = 0u;
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
        v[r] = 0u;
        if (r < each && first + r < nchunks) v[r] = totals[(size_t)(first + r) * k + col];
    }
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) mine += v[r];
    sum[g][tid % SQ_COLUMNS] = mine;
    __syncthreads();
    uint32_t before = 0u, all = 0u;
#pragma unroll
    for (uint32_t j = 0; j < GROUPS; ++j) {
        const uint32_t s = sum[j][tid % SQ_COLUMNS];
        before += j < g ? s : 0u;
        all += s;
    }
#pragma unroll
    for (uint32_t r = 0; r < ROWS; ++r) {
        if (r < each && first + r < nchunks) totals[(size_t)(first + r) * k + col] = before;
        before += v[r];
    }
    if (g == 0u) { store_agent(&sizes[col], all); totals[(size_t)nchunks * k + col] = all; }
    publish_barrier();
    __syncthreads();
    if (tid == 0u) lds_ticket = atomicAdd(&sq->ticket[1], 1u);
    __syncthreads();
    if (way == SQ_BUCKETS && lds_ticket != gridDim.x - 1u) return;
    // the last one
    constexpr uint32_t PER = (SQ_MAX_K + SQ_BLOCK - 1u) / SQ_BLOCK;
    const uint32_t heavies = sb_uniform(sq->heavies);
    uint32_t c[PER], total = 0u, most = 0u;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) c[j] = tid * PER + j < k ? load_agent(&sizes[tid * PER + j]) : 0u;
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        total += c[j];
        uint32_t size = c[j];
        for (uint32_t h = 0; h < heavies; ++h)
            if (tid * PER + j == sq->heavy_bucket[h]) {
                sq->heavy_size[h] = size;
                size = 0u;
                sizes[tid * PER + j] = 0u;                   // (nothing to sort)
            }
        most = size > most ? size : most;
    }
    uint32_t varying = 0u;
    for (uint32_t i = tid; floats != 0 && i < nchunks; i += SQ_BLOCK) varying |= seen[i];
    const uint32_t inc = wave_scan_inclusive(total, OpAdd(), 0u);
    most = wave_reduce(most, OpMax());
    varying = wave_reduce(varying, OpOr());
    if (lane == WAVE - 1) { part[0][wave] = inc; part[1][wave] = most; part[2][wave] = varying; }
    __syncthreads();
    uint32_t start = inc - total;
    for (uint32_t w = 0; w < wave; ++w) start += part[0][w];
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) {
        if (tid * PER + j < k) starts[tid * PER + j] = start;
        start += c[j];
    }
    if (tid != 0u) return;
    for (uint32_t w = 0; w < SQ_BLOCK / WAVE; ++w) {
        most = part[1][w] > most ? part[1][w] : most;
        varying |= part[2][w];
    }
    if (way == SQ_BUCKETS && most <= cap) {
        sq->ok = 1u;
        for (int p = 0; p < 4; ++p) ctl->skip[p] = 1u;
        ctl->nexec = ~0u;
    } else if (floats != 0) {
        sort_make_plan(ctl, 4, false, 0u, varying, first_source);
    }
}

// The sizes of a tile's buckets are known, so a key's place in the sorted tile is one addition in LDS.
// Every workgroup takes a tile of every round of gridDim.x, neighbours on one XCD, whose runs meet in its L2; the keys of its next tile are
// asked for when those of this one lie in LDS, before it is written.
// HEAVY: there are heavy values.
template <typename T, bool HEAVY>
__device__ __forceinline__ void sq_scatter_tiles(const T* keys, uint32_t n, uint32_t flip, uint32_t k, const uint32_t* __restrict__ cells, uint32_t ntiles, uint32_t chunk_tiles,
                                                 const uint16_t* __restrict__ rows, const uint32_t* __restrict__ totals, const uint32_t* __restrict__ starts,
                                                 const SqCtl* sq, uint32_t* __restrict__ out, uint32_t* lds_key, uint32_t* table, uint32_t* cnt, uint32_t* to) {
    constexpr uint32_t TILE = SQ_TILE, PER = (SQ_MAX_K + SQ_BLOCK - 1u) / SQ_BLOCK;
    constexpr int NV = SQ_TILE / (4 * SQ_BLOCK), ITEMS = 4 * NV;
    const uint32_t tid = sq_again(threadIdx.x), lane = tid % WAVE, wave = tid / WAVE;
    const uint32_t tile0 = (blockIdx.x & 7u) * (gridDim.x / 8u) + (blockIdx.x >> 3), whole = n / TILE;
    if (tile0 >= ntiles) return;
    uint32_t* const part = lds_key;
    SqTile<NV> t;
    const uint32_t per = (k + SQ_BLOCK - 1u) / SQ_BLOCK;                // bucket tid * per + j
    // keys of the thread's buckets in the tiles in front of a tile, and with those of the tile
    uint32_t before[PER], with[PER];
    const auto fetch_counts = [&](uint32_t tile) {
        const uint32_t* const total = totals + (size_t)(tile / chunk_tiles) * k;
        const uint32_t* const total1 = totals + (size_t)((tile + 1u) / chunk_tiles) * k;
        const uint16_t* const row = rows + (size_t)tile * k;
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            const uint32_t b = tid * per + j < k ? tid * per + j : k - 1u;
            before[j] = sq_at(total, b) + sq_at(row, b);
            with[j] = sq_at(total1, b) + sq_at(row, b + k);
        }
        if (HEAVY) {                                         // (none of a heavy value's are moved)
#pragma unroll
            for (uint32_t h = 0; h < SQ_HEAVY; ++h)
#pragma unroll
                for (uint32_t j = 0; j < PER; ++j)
                    if (tid * per + j == sq->heavy_bucket[h]) with[j] = before[j];
        }
    };
    fetch_counts(tile0);
    if (tile0 < whole) t.template load<true>((const uint32_t*)keys + (size_t)tile0 * TILE, TILE);
    const SqMap map = HEAVY ? sq_map(sq, k) : SqMap{sq->lo, sq->range, sq->up, k << 8, 0u, {}};
    for (uint32_t c = 4u * tid; c < SQ_CELLS; c += 4u * SQ_BLOCK) *(uint4*)&table[c] = *(const uint4*)&cells[c];
    uint32_t first[PER];
#pragma unroll
    for (uint32_t j = 0; j < PER; ++j) first[j] = sq_at(starts, tid * per + j < k ? tid * per + j : k - 1u);
    const auto scatter = [&](uint32_t count, uint32_t next, auto full) {
        constexpr bool FULL = decltype(full)::value, ALL = FULL && !HEAVY;
        uint32_t sum = 0u;
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) sum += j < per && tid * per + j < k ? with[j] - before[j] : 0u;
        const uint32_t inc = wave_scan_inclusive(sum, OpAdd(), 0u);
        if (lane == WAVE - 1) part[wave] = inc;
        __syncthreads();
        uint32_t start = inc - sum;
        for (uint32_t w = 0; w < wave; ++w) start += part[w];
        uint32_t moved = count;
        if constexpr (HEAVY) {
            moved = 0u;
            for (uint32_t w = 0; w < SQ_BLOCK / WAVE; ++w) moved += part[w];
        }
#pragma unroll
        for (uint32_t j = 0; j < PER; ++j) {
            const uint32_t b = tid * per + j;
            if (j < per && b < k) { cnt[b] = start; to[b] = first[j] + before[j] - start; }
            start += with[j] - before[j];
        }
        __syncthreads();
#pragma unroll
        for (int i0 = 0; i0 < ITEMS; i0 += 4) {
            uint32_t b[4], place[4];
            [[maybe_unused]] bool gone[4] = {};              // of a heavy value
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                t.key[i0 + i] = sq_enc<T>(t.key[i0 + i], flip);
                b[i] = sq_bucket(table, map, t.key[i0 + i]);
            }
            if constexpr (HEAVY) {
                const uint32_t x[4] = {t.key[i0], t.key[i0 + 1], t.key[i0 + 2], t.key[i0 + 3]};
                sq_around(map, x, b);
                sq_heavies(map, [&](int, uint32_t w) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) gone[i] = gone[i] || x[i] == w;
                });
            }
            const auto moves = [&](int i) { return t.template has<FULL>(i0 + i, count) && (!HEAVY || !gone[i]); };
            sq_take(cnt, b, place, moves);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (moves(i)) lds_key[place[i]] = t.key[i0 + i];
        }
        if (FULL) {
            t.template load<true>((const uint32_t*)keys + (size_t)(next < whole ? next : 0u) * TILE, TILE);
            fetch_counts(next < ntiles ? next : 0u);
        }
        __syncthreads();
        // the keys' buckets once more: neighbours now share them and their cells
#pragma unroll
        for (int i0 = 0; i0 < ITEMS; i0 += 4) {
            uint32_t x[4], at[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = lds_key[ALL || tid + (i0 + i) * SQ_BLOCK < moved ? tid + (i0 + i) * SQ_BLOCK : 0u];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (HEAVY) at[i] = sq_bucket(table, map, x[i]);
                else at[i] = to[sq_bucket(table, map, x[i])] + tid + (i0 + i) * SQ_BLOCK;
            }
            if constexpr (HEAVY) {
                sq_around(map, x, at);
#pragma unroll
                for (int i = 0; i < 4; ++i) at[i] = to[at[i]] + tid + (i0 + i) * SQ_BLOCK;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (ALL || tid + (i0 + i) * SQ_BLOCK < moved) sq_at(out, at[i]) = x[i];
        }
        __syncthreads();
    };
    uint32_t tile = tile0;
    for (; tile < whole; tile += gridDim.x) scatter(TILE, tile + gridDim.x, std::true_type{});
    if (tile < ntiles) {
        t.template load<false>((const uint32_t*)keys + (size_t)tile * TILE, n - tile * TILE);
        scatter(n - tile * TILE, 0u, std::false_type{});
    }
}

template <typename T>
__global__ __launch_bounds__(SQ_BLOCK, 4) void sq_scatter_kernel(const T* keys, uint32_t n, uint32_t flip, uint32_t k, const uint32_t* __restrict__ cells,
                                                                 uint32_t ntiles, uint32_t chunk_tiles, const uint16_t* __restrict__ rows,
                                                                 const uint32_t* __restrict__ totals, const uint32_t* __restrict__ starts, const SqCtl* sq,
                                                                 uint32_t* __restrict__ out) {
    __shared__ uint32_t lds_key[SQ_TILE];
    __shared__ alignas(16) uint32_t table[SQ_CELLS];
    __shared__ uint32_t cnt[SQ_MAX_K];           // of a bucket: where its next key goes in the tile
    __shared__ uint32_t to[SQ_MAX_K];            // where its keys go, less where it starts in the tile
    if (sq->ok == 0u) return;
    if (sq->heavies == 0u) sq_scatter_tiles<T, false>(keys, n, flip, k, cells, ntiles, chunk_tiles, rows, totals, starts, sq, out, lds_key, table, cnt, to);
    else sq_scatter_tiles<T, true>(keys, n, flip, k, cells, ntiles, chunk_tiles, rows, totals, starts, sq, out, lds_key, table, cnt, to);
}

// ---- a bucket ---------------------------------------------------------------------------------------------------------
// Sorting networks on 16 keys of a lane: of any keys, and of two sorted halves.
__device__ __forceinline__ void sq_order(uint32_t& a, uint32_t& b) {
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    a = lo;
    b = hi;
}
// Batcher's odd-even merge sort, from runs of FROM keys on.
template <int FROM> __device__ __forceinline__ void sq_network(uint32_t (&x)[16]) {
#pragma unroll
    for (int p = FROM; p < 16; p *= 2) {
#pragma unroll
        for (int q = p; q > 0; q /= 2) {
#pragma unroll
            for (int j = q % p; j + q < 16; j += 2 * q) {
#pragma unroll
                for (int i = 0; i < q; ++i)
                    if (i + j + q < 16 && (i + j) / (2 * p) == (i + j + q) / (2 * p)) sq_order(x[i + j], x[i + j + q]);
            }
        }
    }
}

// In memory, by one workgroup: radix passes of 8 bits over the distance from the smallest key.  Of a bucket that bins do not spread: a step of
// a wave is four loads that are asked for while the step in front is worked on.
// a: the keys; b: as much room.  Returns whether the sorted keys are in b.
__device__ bool sq_radix(uint32_t* a, uint32_t* b, uint32_t m, uint32_t lo, uint32_t bits, uint32_t* cnt, uint32_t* wsum) {
    constexpr uint32_t NW = SQ_BLOCK / WAVE;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const uint32_t seg = ((m + NW - 1u) / NW + WAVE - 1u) / WAVE * WAVE, first = wave * seg, end = first + seg < m ? first + seg : m;
    uint32_t* const wcnt = cnt + wave * 256u;
    bool in_b = false;
    for (uint32_t shift = 0; shift < bits; shift += 8u) {
        const uint32_t* const src = in_b ? b : a;
        uint32_t* const dst = in_b ? a : b;
        __syncthreads();
        for (uint32_t i = tid; i < NW * 256u; i += SQ_BLOCK) cnt[i] = 0u;
        __syncthreads();
        for (int move = 0; move < 2; ++move) {
            constexpr int U = 4;
            uint32_t next[U];
            const auto fetch = [&](uint32_t e0) {
#pragma unroll
                for (int u = 0; u < U; ++u) next[u] = e0 + u * WAVE + lane < end ? src[e0 + u * WAVE + lane] : 0u;
            };
            fetch(first);
            for (uint32_t e0 = first; e0 < end; e0 += U * WAVE) {
                uint32_t x[U], at[U];
#pragma unroll
                for (int u = 0; u < U; ++u) x[u] = next[u];
                fetch(e0 + U * WAVE);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const bool valid = e0 + u * WAVE + lane < end;
                    const uint32_t d = (x[u] - lo) >> shift & 0xffu;
                    if (move == 0) {
                        if (valid) atomicAdd(&wcnt[d], 1u);
                        continue;
                    }
                    uint32_t same_lo, same_hi;
                    match_digit_halves(d, same_lo, same_hi);
                    const uint64_t vm = __ballot(valid);
                    same_lo &= (uint32_t)vm;
                    same_hi &= (uint32_t)(vm >> 32);
                    const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi, __builtin_amdgcn_mbcnt_lo(same_lo, 0u));
                    at[u] = __hip_atomic_load(&wcnt[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) + below;
                    __builtin_amdgcn_wave_barrier();
                    if (valid && below == 0u)
                        __hip_atomic_fetch_add(&wcnt[d], (uint32_t)__builtin_popcount(same_lo) + (uint32_t)__builtin_popcount(same_hi), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WAVEFRONT);
                    __builtin_amdgcn_wave_barrier();
                }
                if (move == 0) continue;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (e0 + u * WAVE + lane < end) dst[at[u]] = x[u];
            }
            __syncthreads();
            if (move != 0) continue;
            uint32_t total = 0u, inc = 0u;
            if (tid < 256u) {
                for (uint32_t w = 0; w < NW; ++w) total += cnt[w * 256u + tid];
                inc = wave_scan_inclusive(total, OpAdd(), 0u);
                if (lane == WAVE - 1) wsum[wave] = inc;
            }
            __syncthreads();
            if (tid < 256u) {
                uint32_t at = inc - total;
                for (uint32_t w = 0; w < wave; ++w) at += wsum[w];
                for (uint32_t w = 0; w < NW; ++w) {
                    const uint32_t c = cnt[w * 256u + tid];
                    cnt[w * 256u + tid] = at;
                    at += c;
                }
            }
            __syncthreads();
        }
        in_b = !in_b;
    }
    return in_b;
}

constexpr int SQ_VECTORS = 12;
constexpr uint32_t SQ_CAP = 4u * SQ_VECTORS * SQ_BLOCK, SQ_BINS = 8192, SQ_SLOTS = 31936;
constexpr uint32_t SQ_ROUNDS = 64;             // of merges, at most: sq_radix takes about as long

// Where the 4 slots q lie, and slot s: lanes that each read 16 neighbours, 4 at a time, read different banks.  (Slots stay among their 16.)
__device__ __forceinline__ uint32_t sq_quad(uint32_t q) { return q ^ (q >> 4 & 3u); }
__device__ __forceinline__ uint32_t sq_slot(uint32_t s) { return s ^ (s >> 4 & 12u); }

// Buckets of up to 4 * NV * 1024 keys, which the threads hold.  They are spread over BINS bins by their distance from the smallest, in no
// order, and put into LDS, whole bins at a time (nearly always all of them); there a thread sorts 16 neighbours in registers and
// then, in rounds that start at every other 8th key, merges two neighbouring runs of 8: a bin of s keys lies in (s + 14) / 8 of these at
// most, and so many rounds sort it.  The next bucket's keys are asked for when this one's lie in LDS.
template <typename T>
__global__ __launch_bounds__(SQ_BLOCK, 4) void sq_bucket_kernel(uint32_t* in, const uint32_t* __restrict__ starts, const uint32_t* __restrict__ sizes, uint32_t k,
                                                                    uint32_t flip, const SqCtl* sq, T* out) {
    constexpr uint32_t BINS = SQ_BINS, SLOTS = SQ_SLOTS;
    constexpr int NV = SQ_VECTORS, ITEMS = 4 * NV, NW = SQ_BLOCK / WAVE, PER = (int)BINS / SQ_BLOCK;
    constexpr uint32_t WINDOW = SLOTS - 32u;                 // a window's slots start and end at a multiple of 16 of the bucket's
    constexpr uint32_t WINDOWS = ITEMS * SQ_BLOCK / (WINDOW / 2u) + 2u;
    constexpr int GROUP = NV % 2 == 0 ? 2 : 1;
    static_assert(SLOTS % 16u == 0u && NV % GROUP == 0 && PER % 4 == 0 && WINDOWS < SQ_BLOCK, "shapes");
    static_assert(BINS >= NW * 256u, "counters of sq_radix");
    __shared__ alignas(16) uint32_t bins[BINS];
    __shared__ alignas(16) uint32_t slot[SLOTS];
    __shared__ uint32_t part[4][NW], bound[WINDOWS + 1u], bound_bin[WINDOWS + 1u];
    if (sq->ok == 0u) return;
    const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    SqTile<NV> t;
    // Rows of 4 keys a thread, GROUP of them at a time: those that are all there need no bounds.  (Where there is no key, the first one.)
    const auto whole = [](int v, uint32_t m) { return (uint32_t)(v + GROUP) * (4u * SQ_BLOCK) <= m; };
    const auto none = [](int v, uint32_t m) { return (uint32_t)v * (4u * SQ_BLOCK) >= m; };
    const auto fetch = [&](uint32_t start, uint32_t m) {
        const uint32_t tid = sq_again(threadIdx.x);
        const uint32_t* const from = in + start;
        const int32_t left = (int32_t)m - 4 * (int32_t)tid;
#pragma unroll
        for (int g = 0; g < NV; g += GROUP) {
            if (whole(g, m)) {
#pragma unroll
                for (int v = g; v < g + GROUP; ++v) {
                    const auto x = load_nt_elems<uint32_t, 4>(from + 4u * (tid + v * SQ_BLOCK));
#pragma unroll
                    for (int j = 0; j < 4; ++j) t.key[4 * v + j] = x[j];
                }
            } else if (m != 0u) {
#pragma unroll
                for (int i = 4 * g; i < 4 * (g + GROUP); ++i) t.key[i] = from[left > i / 4 * (4 * SQ_BLOCK) + i % 4 ? 4u * (tid + i / 4 * SQ_BLOCK) + i % 4 : 0u];
            }
        }
    };
    const auto clear_bins = [&]() {
#pragma unroll
        for (int c = 0; c < PER; c += 4) *(uint4*)&bins[4u * tid + c * SQ_BLOCK] = make_uint4(0u, 0u, 0u, 0u);
    };
    // One bucket, whose keys are there; `ahead` asks for the next one's, unless this says that it has not.
    // (sq_again: what is cheap to compute and used in several places is not worth a register between them)
    const auto sort_bucket = [&](uint32_t start, uint32_t m, auto&& ahead) {
        const uint32_t tid = sq_again(threadIdx.x);
        int32_t left = (int32_t)m - 4 * (int32_t)tid;
        const uint32_t m_ = m;
        const auto has = [&](int i) { return left > i / 4 * (4 * SQ_BLOCK) + i % 4; };
        uint32_t lo = ~0u, hi = 0u;
#pragma unroll
        for (int g = 0; g < NV; g += GROUP) {
            if (none(g, m)) continue;
#pragma unroll
            for (int i = 4 * g; i < 4 * (g + GROUP); ++i) {
                lo = t.key[i] < lo ? t.key[i] : lo;
                hi = t.key[i] > hi ? t.key[i] : hi;
            }
        }
        lo = wave_reduce(lo, OpMin());
        hi = wave_reduce(hi, OpMax());
        if (lane == 0u) { part[0][wave] = lo; part[1][wave] = hi; }
        // up to three slots in front of the bucket are empty, so that stores are aligned
        const uint32_t skip = (uint32_t)((uintptr_t)(out + start) >> 2) & 3u, all = skip + m;
        const bool one_window = all <= SLOTS - 16u;
        if (tid <= WINDOWS) { bound[tid] = tid == 0u ? skip : all; bound_bin[tid] = tid == 0u ? 0u : BINS; }
        __syncthreads();
#pragma unroll 4
        for (int w = 0; w < NW; ++w) {
            lo = part[0][w] < lo ? part[0][w] : lo;
            hi = part[1][w] > hi ? part[1][w] : hi;
        }
        lo = sb_uniform(lo);
        hi = sb_uniform(hi);
        const uint32_t span = hi - lo;
        // below BINS for every distance: the distance, the factor and the product are rounded by 2^-24 each.  Distances below
        // BINS - BINS / 256 have a bin each.
        const float per_key = (float)BINS * (1.f - 0x1p-20f) / ((float)span + 1.f);
        const bool exact = span < BINS - BINS / 256u;
        // Of floats of more than three binades -- a bucket around zero, or the one below a range that starts there -- nearly all bits may lie at
        // the ends: such keys are spread by their values.  (Without infinities or NaNs at an end there are none.)
        float value_lo = 0.f, per_value = 0.f;
        bool by_value = false;
        if constexpr (!std::is_integral<T>::value) {
            value_lo = __builtin_bit_cast(float, sq_dec<T>(lo, flip));
            const float width = __builtin_bit_cast(float, sq_dec<T>(hi, flip)) - value_lo;
            per_value = (float)BINS * (1.f - 0x1p-20f) / width;
            if (span > 3u << 23 && __builtin_fabsf(width) < __builtin_inff() && __builtin_fabsf(per_value) < __builtin_inff()) {
                // which of the two spreads the first row better, over an eighth of the bins (over 64 of them a few keys at one place do not show: of 2^24
                // keys of N(0, 1) 1 % of which are a million times as large, one bucket made the call 379 us for 176)
                uint32_t* const coarse = slot;
                coarse[tid] = coarse[SQ_BLOCK + tid] = 0u;
                __syncthreads();
                if (has(0)) {
                    atomicAdd(&coarse[(uint32_t)((float)(t.key[0] - lo) * per_key) / (BINS / SQ_BLOCK)], 1u);
                    atomicAdd(&coarse[SQ_BLOCK + (uint32_t)((__builtin_bit_cast(float, sq_dec<T>(t.key[0], flip)) - value_lo) * per_value) / (BINS / SQ_BLOCK)], 1u);
                }
                __syncthreads();
                const uint32_t by_bits = wave_reduce(coarse[tid], OpMax()), by_val = wave_reduce(coarse[SQ_BLOCK + tid], OpMax());
                if (lane == 0u) { part[2][wave] = by_bits; part[3][wave] = by_val; }
                __syncthreads();
                uint32_t most_bits = 0u, most_val = 0u;
#pragma unroll 4
                for (int w = 0; w < NW; ++w) {
                    most_bits = part[2][w] > most_bits ? part[2][w] : most_bits;
                    most_val = part[3][w] > most_val ? part[3][w] : most_val;
                }
                by_value = sb_uniform(most_val) < sb_uniform(most_bits);
            }
        }
        const auto with_bins = [&](auto&& run) {
            if constexpr (!std::is_integral<T>::value) {
                if (by_value) {
                    run([&](uint32_t x) { return (uint32_t)((__builtin_bit_cast(float, sq_dec<T>(x, flip)) - value_lo) * per_value); });
                    return;
                }
            }
            run([&](uint32_t x) { return (uint32_t)((float)(x - lo) * per_key); });
        };
        with_bins([&](auto&& bin_of) {
            const uint32_t m = sq_again_uniform(m_);
            left = sq_again(left);
#pragma unroll
            for (int g = 0; g < NV; g += GROUP) {
                if (whole(g, m)) {
#pragma unroll
                    for (int i = 4 * g; i < 4 * (g + GROUP); ++i) atomicAdd(&bins[bin_of(t.key[i])], 1u);
                } else if (!none(g, m)) {
#pragma unroll
                    for (int i = 4 * g; i < 4 * (g + GROUP); ++i)
                        if (has(i)) atomicAdd(&bins[bin_of(t.key[i])], 1u);
                }
            }
        });
        __syncthreads();
        {
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
            if (lane == WAVE - 1) { part[2][wave] = inc; part[3][wave] = most; }
            __syncthreads();
            uint32_t first = skip + inc - sum;
#pragma unroll 4
            for (int w = 0; w < NW; ++w) {
                if ((uint32_t)w < wave) first += part[2][w];
                most = part[3][w] > most ? part[3][w] : most;
            }
            if (!one_window && most <= WINDOW / 2u) {
                // Window w ends where the first bin starts from w + 1 steps on.  A step is half a window at least, and no bin is longer.
                const uint32_t step = WINDOW - most;
                uint32_t w = first / step + 1u, next = w * step, at = first;
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    at += c[j];
                    if (at >= next) {
                        bound[w] = at;
                        bound_bin[w] = tid * PER + j + 1u;
                        ++w;
                        next += step;
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < PER; ++j) { const uint32_t q = c[j]; c[j] = first; first += q; }
#pragma unroll
            for (int j = 0; j < PER; j += 4) *(uint4*)&bins[tid * PER + j] = make_uint4(c[j], c[j + 1], c[j + 2], c[j + 3]);
        }
        __syncthreads();
        uint32_t most = 0u;
#pragma unroll 4
        for (int w = 0; w < NW; ++w) most = part[3][w] > most ? part[3][w] : most;
        most = sb_uniform(most);
        bool sorted = one_window || most <= WINDOW / 2u;
        const uint32_t rounds = (exact && !by_value) || most <= 1u ? 0u : (most + 14u) / 8u;
        for (uint32_t w = 0; sorted; ++w) {
            // Slots [from, end) of the bucket lie here, `base` in the first of these; the rest of the 16 that each of the two is one of is empty.
            const uint32_t from = one_window ? skip : sb_uniform(bound[w]), end = one_window ? all : sb_uniform(bound[w + 1u]), base = from & ~15u;
            const uint32_t last = ((end + 15u) & ~15u) - base;
            const auto put = [&](uint32_t x, uint32_t p) { slot[sq_slot(p - base)] = x; };
            with_bins([&](auto&& bin_of) {
                const uint32_t m = sq_again_uniform(m_);
                left = sq_again(left);
                uint32_t p[2][4 * GROUP];                    // the additions of a group are in flight while the keys of the one in front are put
                if (one_window) {
#pragma unroll
                    for (int g = 0; g <= NV; g += GROUP) {
                        if (g < NV && whole(g, m)) {
#pragma unroll
                            for (int i = 0; i < 4 * GROUP; ++i) p[g / GROUP & 1][i] = atomicAdd(&bins[bin_of(t.key[4 * g + i])], 1u);
                        } else if (g < NV && !none(g, m)) {
#pragma unroll
                            for (int i = 0; i < 4 * GROUP; ++i)
                                if (has(4 * g + i)) p[g / GROUP & 1][i] = atomicAdd(&bins[bin_of(t.key[4 * g + i])], 1u);
                        }
                        if (g != 0 && whole(g - GROUP, m)) {
#pragma unroll
                            for (int i = 0; i < 4 * GROUP; ++i) put(t.key[4 * (g - GROUP) + i], p[(g / GROUP & 1) ^ 1][i]);
                        } else if (g != 0 && !none(g - GROUP, m)) {
#pragma unroll
                            for (int i = 0; i < 4 * GROUP; ++i)
                                if (has(4 * (g - GROUP) + i)) put(t.key[4 * (g - GROUP) + i], p[(g / GROUP & 1) ^ 1][i]);
                        }
                    }
                } else {
                    const uint32_t bin0 = sb_uniform(bound_bin[w]), bin1 = sb_uniform(bound_bin[w + 1u]);
#pragma unroll
                    for (int g = 0; g < NV; g += GROUP) {
                        if (none(g, m)) continue;
#pragma unroll
                        for (int i = 4 * g; i < 4 * (g + GROUP); ++i) {
                            const uint32_t b = bin_of(t.key[i]);
                            if (has(i) && b - bin0 < bin1 - bin0) put(t.key[i], atomicAdd(&bins[b], 1u));
                        }
                    }
                }
            });
            if (tid < from - base) slot[sq_slot(tid)] = 0u;                    // (no key is smaller, or larger)
            if (tid < last - (end - base)) slot[sq_slot(end - base + tid)] = ~0u;
            if (end >= all) ahead();
            __syncthreads();
            if (end >= all) clear_bins();
            uint4* const quads = (uint4*)slot;
            const uint32_t most_rounds = rounds < SQ_ROUNDS ? rounds : SQ_ROUNDS;
            for (uint32_t r = 0; r < most_rounds; ++r) {
                bool in_order = true;
                for (uint32_t at = 4u * tid + (r & 1u) * 2u; at + 4u <= last / 4u; at += 4u * SQ_BLOCK) {
                    uint32_t x[16];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint4 q = quads[sq_quad(at + j)];
                        x[4 * j] = q.x; x[4 * j + 1] = q.y; x[4 * j + 2] = q.z; x[4 * j + 3] = q.w;
                    }
                    const bool fine = r != 0u && x[7] <= x[8];
                    if (fine) continue;
                    if (r == 0u) {
                        sq_network<1>(x);
                    } else {
                        in_order = false;
                        sq_network<8>(x);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) quads[sq_quad(at + j)] = make_uint4(x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3]);
                }
                // (a round that changes nothing has found the pairs of both kinds in order; few rounds are not worth the question)
                if (r >= 2u && rounds > 4u) {
                    if (__syncthreads_or(in_order ? 0 : 1) == 0) break;
                } else {
                    __syncthreads();
                }
                if (r + 1u == most_rounds && rounds > most_rounds) sorted = false;
            }
            if (!sorted) break;
            T* const to = out + start - skip + base;         // slot s goes to to[s]
            for (uint32_t s = 4u * tid; s < end - base; s += 4u * SQ_BLOCK) {
                const uint4 q = quads[sq_quad(s / 4u)];
                const uint32_t x[4] = {q.x, q.y, q.z, q.w};
                if (s >= from - base && s + 4u <= end - base) {
                    typename VecOf<uint32_t, 4>::type o;
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[j] = sq_dec<T>(x[j], flip);
                    store_nt((typename VecOf<uint32_t, 4>::type*)(to + s), o);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (s + j >= from - base && s + j < end - base) to[s + j] = __builtin_bit_cast(T, sq_dec<T>(x[j], flip));
                }
            }
            if (end >= all) return true;
            __syncthreads();
        }
        uint32_t* const mine = in + start;
        uint32_t* const other = (uint32_t*)out + start;
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) t.key[i] = 0u;      // (needs their registers)
        const bool there = sq_radix(mine, other, m, lo, sb_bits(span), bins, part[0]);
        for (uint32_t i = tid; i < m; i += SQ_BLOCK) out[start + i] = __builtin_bit_cast(T, sq_dec<T>(there ? other[i] : mine[i], flip));
        __syncthreads();
        clear_bins();
        return false;
    };
    const uint32_t heavies = sq->heavies;
    for (uint32_t h = 0; h < heavies; ++h) {
        const uint32_t b = sq->heavy_bucket[h], m = sq->heavy_size[h], v = sq_dec<T>(sq->heavy[h], flip);
        uint32_t* const to = (uint32_t*)out + starts[b];
        const uint32_t to_line = (0u - (uint32_t)((uintptr_t)to >> 2)) & 3u, head = to_line < m ? to_line : m, quads = (m - head) / 4u;
        typename VecOf<uint32_t, 4>::type o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = v;
        for (uint32_t q = blockIdx.x * SQ_BLOCK + tid; q < quads; q += gridDim.x * SQ_BLOCK) store_nt((typename VecOf<uint32_t, 4>::type*)(to + head + 4u * q), o);
        if (blockIdx.x == h && tid < head) to[tid] = v;
        if (blockIdx.x == h && tid < m - head - 4u * quads) to[head + 4u * quads + tid] = v;
    }
    uint32_t bucket = blockIdx.x, start = sb_uniform(starts[bucket]), m = sb_uniform(sizes[bucket]);
    fetch(start, m);
    clear_bins();
    for (;;) {
        const uint32_t next = bucket + gridDim.x;
        const uint32_t next_start = sb_uniform(starts[next < k ? next : bucket]), next_m = next < k ? sb_uniform(sizes[next]) : 0u;
        if (m == 0u || !sort_bucket(start, m, [&]() { fetch(next_start, next_m); })) fetch(next_start, next_m);
        if (next >= k) break;
        bucket = next;
        start = next_start;
        m = next_m;
        __syncthreads();
    }
}

// ---- host --------------------------------------------------------------------------------------------------------
// The most keys: 2560 buckets and a tile are what fits LDS with the cells here (132 of 160 KiB in the scatter; the count keeps the counters of six tiles), and their runs
// are ten keys.  One more takes the radix passes, 758 us for 449; larger tiles or buckets were not tried.
constexpr int64_t SQ_MIN_INTEGERS = (int64_t)1 << 23, SQ_MAX_KEYS = (int64_t)1 << 26;
constexpr int64_t SQ_MEAN = 26624;                         // keys a bucket, at most: 1.2 times as many lie in LDS at a time
constexpr int64_t SQ_ROUND = 256;                          // buckets: a multiple of a workgroup a compute unit

struct SqLayout {
    size_t sq_off, seen_off, ends_off, hist_off, cells_off, rows_off, totals_off, sizes_off, starts_off, total;
    uint32_t k, sample_grid, ntiles, chunk_tiles, nchunks, too_many;
};

static SqLayout sq_layout(size_t off, int64_t n) {
    SqLayout l{};
    const int64_t rounds = (n + SQ_ROUND * SQ_MEAN - 1) / (SQ_ROUND * SQ_MEAN);
    l.k = (uint32_t)(SQ_ROUND * rounds);
    l.ntiles = (uint32_t)((n + SQ_TILE - 1) / SQ_TILE);
    l.chunk_tiles = (l.ntiles + SQ_CHUNKS - 1u) / SQ_CHUNKS;
    l.nchunks = (l.ntiles + l.chunk_tiles - 1u) / l.chunk_tiles;
    const float fit = (float)SQ_CAP * (float)SQ_CHECKED / (float)n;            // of the samples that are looked at, those of a bucket that just fits
    l.too_many = (uint32_t)(fit + 4.f * std::sqrt(fit));
    l.sample_grid = l.k / (SQ_BLOCK * SQ_SAMPLES_EACH / sq_samples(n));
    const uint32_t k = l.k;
    const auto take = [&](size_t bytes) { const size_t at = off; off += (bytes + 255) & ~(size_t)255; return at; };
    l.sq_off = take(sizeof(SqCtl));
    l.seen_off = take((size_t)SQ_CHUNKS * 4);
    l.ends_off = take((size_t)l.sample_grid * sizeof(uint2));
    l.hist_off = take((size_t)SQ_CELLS * 4);
    l.cells_off = take((size_t)SQ_CELLS * 4);
    l.sizes_off = take((size_t)k * 4);
    l.starts_off = take((size_t)k * 4);
    l.totals_off = take((size_t)(SQ_CHUNKS + 1u) * k * 4);
    l.rows_off = take((size_t)(l.ntiles + 1u) * k * 2);
    l.total = off;
    return l;
}

// `moved`: room for the keys, which holds the sample before.
template <typename T>
static int32_t sort_quantiles(const SqLayout& l, const void* keys, void* sorted_out, int64_t n, int rev, char* base, SortCtl* ctl, int first_source,
                              uint32_t* moved, hipStream_t stream) {
    const uint32_t flip = (rev & SORT_REV) != 0 ? ~0u : 0u;
    SqCtl* sq = (SqCtl*)(base + l.sq_off);
    uint32_t* seen = (uint32_t*)(base + l.seen_off);
    uint2* ends = (uint2*)(base + l.ends_off);
    uint32_t* hist = (uint32_t*)(base + l.hist_off);
    uint32_t* cells = (uint32_t*)(base + l.cells_off);
    uint32_t* sizes = (uint32_t*)(base + l.sizes_off);
    uint32_t* starts = (uint32_t*)(base + l.starts_off);
    uint32_t* totals = (uint32_t*)(base + l.totals_off);
    uint16_t* rows = (uint16_t*)(base + l.rows_off);
    const uint32_t k = l.k;
    const uint32_t cus = (uint32_t)device_info().cus, resident = cus / 8u * 8u;
    const int floats = std::is_integral<T>::value ? 0 : 1;
    sq_sample_kernel<T><<<l.sample_grid, SQ_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, flip, ctl, first_source, sq_few_passes(n), moved, ends, hist, sq);
    RK_LAUNCH_CHECK();
    // from a key to the number whose multiples of 2^23 are binades
    const uint32_t offset = std::is_integral<T>::value ? 0u : flip != 0u ? 1u - 0x007fffffu : 0x007fffffu;
    const uint32_t samples = l.sample_grid * SQ_BLOCK * SQ_SAMPLES_EACH;
    sq_table_kernel<false><<<SQ_TABLE_GRID, SQ_BLOCK, 0, stream>>>(moved, samples, ends, l.sample_grid, offset, k, sq_samples(n), l.too_many, floats, hist, cells, sq);
    RK_LAUNCH_CHECK();
    sq_table_kernel<true><<<SQ_TABLE_GRID, SQ_BLOCK, 0, stream>>>(moved, samples, ends, l.sample_grid, offset, k, sq_samples(n), l.too_many, floats, hist, cells, sq);
    RK_LAUNCH_CHECK();
    sq_count_kernel<T><<<l.nchunks, SQ_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, flip, k, cells, l.ntiles, l.chunk_tiles, (uint32_t*)rows, totals, seen, sq);
    RK_LAUNCH_CHECK();
    sq_offsets_kernel<<<k / SQ_COLUMNS, SQ_BLOCK, 0, stream>>>(totals, l.nchunks, k, SQ_CAP, sizes, starts, seen, sq, ctl, floats, first_source);
    RK_LAUNCH_CHECK();
    sq_scatter_kernel<T><<<l.ntiles < resident ? (l.ntiles + 7u) / 8u * 8u : resident, SQ_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, flip, k, cells, l.ntiles, l.chunk_tiles, rows, totals, starts, sq, moved);
    RK_LAUNCH_CHECK();
    sq_bucket_kernel<T><<<k < cus ? k : cus, SQ_BLOCK, 0, stream>>>(moved, starts, sizes, k, flip, sq, (T*)sorted_out);
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

}  // namespace rk
