// sort! / sortperm! of vectors (src/kernels/sorting.jl:1-3, which forwards to AcceleratedKernels' merge sort):
// least-significant-digit radix sort, 8 bits per pass.
//
// Five ways by the number of keys:
//   up to 4096           one workgroup does all of it in LDS (sort_tiny_kernel, rk_sort_buckets.hpp).
//   up to 2^20           keys of 4 and 8 bytes go through splitters into buckets that are sorted in LDS (rk_sort_buckets.hpp):
//                        such sorts are bound by the latency of their kernels, and these are four or five whatever the width.
//   up to 2^26           keys of 8 bytes, and Float32 up to 2^22, go through two levels of splitters (rk_sort_split.hpp), unless they are
//                        integers with three digits at most from the lowest that varies to the top of their range.
//   up to 2^26           sort of more Float32, and of more than 2^23 Int32, moves the keys into buckets once (rk_sort_quantiles.hpp), unless a bucket
//                        gets too large for that or has few values, or integers differ in one digit (two up to 2^25 keys).
//   the others           the radix passes of this file:
//   sort_init_kernel     clears the control block; no memset: graph-safe
//   sort_range_kernel    one read of the keys: smallest and largest key (integers) and the bits that differ between keys;
//                        the workgroup that finishes last decides which passes run (a digit that is the same in every key
//                        needs none) and which buffer each of them reads.  (Integers are taken relative to the smallest key.)
// and for every pass
//   sort_upsweep_kernel  the 256 digit counts of every tile (one more read of the keys, at streaming speed)
//   sort_pass_kernel     a tile of 4096 keys ranks its keys by digit (wave-level match by ballots, counts in LDS), reorders
//                        the tile in LDS and writes runs of equal digits.  The kernel is bound by its vector instructions
//                        (58 a key, 32 of them the match), not by memory.
//
// How a tile learns where its digits go:
//   up to 256 tiles (2^20 keys of 2 bytes)  every workgroup of the pass sums the columns of the table of counts itself (256 rows
//                        of 512 bytes out of L2, one or two rounds of loads): nothing waits for anything.  A tile or less per
//                        compute unit: it is 16 waves with 4 keys a lane, not 4 waves with 16.
//   beyond               sort_tilescan_kernel: exclusive scan of the counts down the tiles in one launch (chunks of tiles; the
//                        workgroup that finishes last scans the chunk totals and the digit totals); the pass kernel gives
//                        each XCD a contiguous eighth of the tiles.
// Large sorts of floats run every pass (their digits are hardly ever constant) and do without the range read.
//   sort_finish_kernel   moves the result of sort! into the caller's array when an odd number of passes ran
//
// Keys are mapped to unsigned integers that sort like Base.isless (-0.0 < 0.0, NaN last; sortperm makes every NaN the
// canonical one so that they are equal keys, sort! keeps their bit patterns), complemented for rev=true; the mapping is
// applied on the first read and undone on the last write.  The sort is stable, so sortperm keeps equal keys in index
// order (also with rev=true, as Base does).
#include <cstddef>
#include <cstdlib>
#include <type_traits>

#include "rk_common.hpp"

namespace rk {

constexpr int SORT_BLOCK = 256;
constexpr int SORT_MAX_PASSES = 8;

struct SortCtl {                                  // head of the caller's temporary buffer
    uint32_t hist[SORT_MAX_PASSES][256];          // large sorts: first output slot of every digit value (sort_tilescan_kernel)
    // everything from here on is cleared by sort_init_kernel
    uint32_t skip[SORT_MAX_PASSES];
    uint32_t src_is_b[SORT_MAX_PASSES];           // the pass reads buffer B (1) or A (0)
    uint32_t scan_ticket[SORT_MAX_PASSES];        // sort_tilescan_kernel: workgroups that have stored their chunk totals
    uint32_t first_pass, last_pass, nexec;
    uint32_t range_ticket;                        // sort_range_kernel: workgroups that have added their part
    unsigned long long inv_min;                   // ~(smallest mapped key), kept as a maximum so that zero is its identity
    unsigned long long key_max;                   // largest mapped key (integers: range = key_max - smallest)
    unsigned long long varying;                   // bits that are not the same in all mapped keys
};
constexpr int SORT_CTL_CLEAR = (int)((sizeof(SortCtl) - offsetof(SortCtl, skip)) / sizeof(uint32_t));

// ---- key <-> ordered unsigned integer -----------------------------------------------------------------
template <typename T> struct SortKey;
template <> struct SortKey<int16_t> {
    typedef uint16_t U;
    static __device__ __forceinline__ U enc(int16_t v, bool) { return (U)((uint16_t)v ^ 0x8000u); }
    static __device__ __forceinline__ int16_t dec(U u, bool) { return (int16_t)(u ^ 0x8000u); }
};
template <> struct SortKey<int32_t> {
    typedef uint32_t U;
    static __device__ __forceinline__ U enc(int32_t v, bool) { return (U)v ^ 0x80000000u; }
    static __device__ __forceinline__ int32_t dec(U u, bool) { return (int32_t)(u ^ 0x80000000u); }
};
template <> struct SortKey<int64_t> {
    typedef uint64_t U;
    static __device__ __forceinline__ U enc(int64_t v, bool) { return (U)v ^ 0x8000000000000000ull; }
    static __device__ __forceinline__ int64_t dec(U u, bool) { return (int64_t)(u ^ 0x8000000000000000ull); }
};
// Floats: sign-magnitude bits -> unsigned integers in isless order (-0.0 < 0.0), NaN after +Inf.
//   keep == false (sortperm: the keys are not part of the result): every NaN becomes the canonical one, so all NaNs
//                 are equal keys and stay in index order, as isless-equal elements must in a stable sort.
//   keep == true  (sort!): a bijection of the bit patterns, so the sorted array is a permutation of the input, NaN signs
//                 and payloads included.  The plain mapping puts the negative NaNs below -Inf: NLOW of them, keys
//                 0 .. NLOW-1; they are moved above the positive NaNs and everything else shifts down by NLOW.  The
//                 order among NaNs is then by bit pattern, not by index (Base's own float sort moves its NaNs to the
//                 end without keeping their order either).
template <typename U, U NLOW> struct FloatKeyMap {
    static __device__ __forceinline__ U fwd(U std_key) { return std_key < NLOW ? (U)(std_key + (U)(0 - NLOW)) : (U)(std_key - NLOW); }
    static __device__ __forceinline__ U inv(U k) { return k >= (U)(0 - NLOW) ? (U)(k - (U)(0 - NLOW)) : (U)(k + NLOW); }
};
struct half_bits { uint16_t b; };                 // Float16 travels as its bit pattern
template <> struct SortKey<half_bits> {
    typedef uint16_t U;
    typedef FloatKeyMap<uint16_t, 0x03ffu> Map;    // 0xfc01 .. 0xffff are the negative NaNs
    static __device__ __forceinline__ U enc(half_bits v, bool keep) {
        uint16_t b = v.b;
        if (!keep && (b & 0x7fffu) > 0x7c00u) b = 0x7e00u;        // NaN -> canonical, sorts after +Inf
        const U u = (U)((b & 0x8000u) ? ~b : (b ^ 0x8000u));
        return keep ? Map::fwd(u) : u;
    }
    static __device__ __forceinline__ half_bits dec(U k, bool keep) {
        const U u = keep ? Map::inv(k) : k;
        return half_bits{(uint16_t)((u & 0x8000u) ? (u ^ 0x8000u) : ~u)};
    }
};
template <> struct SortKey<float> {
    typedef uint32_t U;
    typedef FloatKeyMap<uint32_t, 0x007fffffu> Map;
    static __device__ __forceinline__ U enc(float v, bool keep) {
        uint32_t b = __builtin_bit_cast(uint32_t, v);
        if (!keep && v != v) b = 0x7fc00000u;
        const U u = (b & 0x80000000u) ? ~b : (b ^ 0x80000000u);
        return keep ? Map::fwd(u) : u;
    }
    static __device__ __forceinline__ float dec(U k, bool keep) {
        const U u = keep ? Map::inv(k) : k;
        return __builtin_bit_cast(float, (u & 0x80000000u) ? (u ^ 0x80000000u) : ~u);
    }
};
template <> struct SortKey<double> {
    typedef uint64_t U;
    typedef FloatKeyMap<uint64_t, 0x000fffffffffffffull> Map;
    static __device__ __forceinline__ U enc(double v, bool keep) {
        uint64_t b = __builtin_bit_cast(uint64_t, v);
        if (!keep && v != v) b = 0x7ff8000000000000ull;
        const U u = (b & 0x8000000000000000ull) ? ~b : (b ^ 0x8000000000000000ull);
        return keep ? Map::fwd(u) : u;
    }
    static __device__ __forceinline__ double dec(U k, bool keep) {
        const U u = keep ? Map::inv(k) : k;
        return __builtin_bit_cast(double, (u & 0x8000000000000000ull) ? (u ^ 0x8000000000000000ull) : ~u);
    }
};

// `rev` here is a set of flags: bit 0 = descending order, bit 1 = keep NaN bit patterns (SORT_KEEP_NAN).
constexpr int SORT_REV = 1, SORT_KEEP_NAN = 2;
// the same mapping on the raw bit pattern: one load path serves the first pass (caller's keys) and the later ones
// and, for integers, relative to the smallest mapped key of the array: small-range integers then have constant high digits,
// whose passes are skipped
template <typename T> __device__ __forceinline__ typename SortKey<T>::U enc_bits(typename SortKey<T>::U raw, int rev, typename SortKey<T>::U umin) {
    typedef typename SortKey<T>::U U;
    const U u = SortKey<T>::enc(__builtin_bit_cast(T, raw), (rev & SORT_KEEP_NAN) != 0);
    return (U)(((rev & SORT_REV) ? (U)~u : u) - umin);
}
template <typename T> __device__ __forceinline__ T dec_bits(typename SortKey<T>::U k, int rev, typename SortKey<T>::U umin) {
    typedef typename SortKey<T>::U U;
    const U u = (U)(k + umin);
    return SortKey<T>::dec((rev & SORT_REV) ? (U)~u : u, (rev & SORT_KEEP_NAN) != 0);
}

template <typename U> __device__ __forceinline__ uint32_t digit_of(U u, int pass) { return (uint32_t)(u >> (8 * pass)) & 0xffu; }

// Mask of the lanes whose digit equals this lane's, as two halves.  Per bit of the digit: e = all ones where the bit is
// set, m = ballot of the bit; (m ^ e) has a one exactly for the lanes that differ from this lane in that bit.  Four vector
// instructions a bit (sign-extended bit, compare into a lane mask, and one three-input bit operation same &= ~(m ^ e) for
// each half of the wave) instead of the five the compiler makes of a ballot.  Call with all 64 lanes active.
// A vector instruction may read a scalar register two wait states after a vector instruction wrote it, at the earliest.  The
// compiler keeps that distance behind its own compares but not behind those of an asm statement, so four compares are one
// block that ends in the two wait states (s_nop 1): whatever follows it may read any of the masks.  (All eight in one block:
// sort(Float32[2^26]) 757.8 against 755.4 us.)
__device__ __forceinline__ void match_digit_halves(uint32_t d, uint32_t& same_lo, uint32_t& same_hi) {
    same_lo = ~0u;
    same_hi = ~0u;
#pragma unroll
    for (int b = 0; b < 8; b += 4) {
        uint32_t e[4];
        uint64_t m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k] = (uint32_t)__builtin_amdgcn_sbfe((int)d, b + k, 1);
        asm volatile("v_cmp_ne_u32_e64 %0, 0, %4\n\t"
                     "v_cmp_ne_u32_e64 %1, 0, %5\n\t"
                     "v_cmp_ne_u32_e64 %2, 0, %6\n\t"
                     "v_cmp_ne_u32_e64 %3, 0, %7\n\t"
                     "s_nop 1"
                     : "=s"(m[0]), "=s"(m[1]), "=s"(m[2]), "=s"(m[3])
                     : "v"(e[0]), "v"(e[1]), "v"(e[2]), "v"(e[3]));
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            same_lo = __builtin_amdgcn_bitop3_b32(same_lo, (uint32_t)m[k], e[k], 0x90);             // a & ~(b ^ c)
            same_hi = __builtin_amdgcn_bitop3_b32(same_hi, (uint32_t)(m[k] >> 32), e[k], 0x90);
        }
    }
}

// Wave-uniform test of a digit for the counting kernel: do at least 8 lanes share the first lane's digit?
__device__ __forceinline__ bool digits_skewed(uint32_t d, bool valid) {
    const uint64_t active = __ballot(valid);
    if (active == 0ull) return false;
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, __ffsll((unsigned long long)active) - 1);
    return __popcll(__ballot(valid && d == d0)) >= 8;
}
// ---- plan: which passes run and what they read --------------------------------------------------------------------
// relative: keys are taken relative to the smallest one (integers), so digits above their range are zero in every key, and
// so are low digits in which the keys do not differ.
// Otherwise (floats) a digit in which no two keys differ is skipped: their exponent bytes are constant or not whatever is
// subtracted.
// first: what the first pass says of its source, SORT_A or SORT_B (it reads the caller's keys either way, and writes the other one);
// SORT_ENDS_IN_A: whichever lets the last pass write buffer A.
constexpr int SORT_A = 0, SORT_B = 1, SORT_ENDS_IN_A = 2;
__device__ __forceinline__ void sort_make_plan(SortCtl* ctl, int passes, bool relative, unsigned long long range, unsigned long long varying,
                                               int first_source) {
    uint32_t runs = 0u;                                      // a bit a pass
    for (int p = 0; p < passes; ++p) {
        const unsigned long long upto = p == 7 ? ~0ull : (1ull << (8 * (p + 1))) - 1ull;
        const bool skip = relative ? (range >> (8 * p)) == 0ull || (varying & upto) == 0ull : ((varying >> (8 * p)) & 0xffull) == 0ull;
        runs |= skip ? 0u : 1u << p;
    }
    uint32_t src_b = first_source == SORT_ENDS_IN_A ? (uint32_t)__popc(runs) & 1u : first_source == SORT_B ? 1u : 0u;
    uint32_t nexec = 0, first = 0xffffffffu, last = 0xffffffffu;
    for (int p = 0; p < passes; ++p) {
        const bool skip = (runs >> p & 1u) == 0u;
        ctl->skip[p] = skip ? 1u : 0u;
        if (skip) continue;
        ctl->src_is_b[p] = src_b;
        src_b ^= 1u;
        if (first == 0xffffffffu) first = (uint32_t)p;
        last = (uint32_t)p;
        ++nexec;
    }
    ctl->first_pass = first;
    ctl->last_pass = last;
    ctl->nexec = nexec;
}

// What the plan says about one pass.  All words are asked for together: read where they are used, each waits for the branch
// that the one before decides, round trips to memory in front of the keys (eight passes over 10^6 keys 138.6 against 136.6 us).
struct SortStep {
    uint32_t skip, src_b, first_pass, last_pass;
    unsigned long long inv_min;
};
__device__ __forceinline__ SortStep sort_step(const SortCtl* ctl, int pass) {
    SortStep s{ctl->skip[pass], ctl->src_is_b[pass], ctl->first_pass, ctl->last_pass, ctl->inv_min};
    asm volatile("" : "+s"(s.skip), "+s"(s.src_b), "+s"(s.first_pass), "+s"(s.last_pass), "+s"(s.inv_min));
    return s;
}

// Sorts of 8-byte integers that take another way unless the plan has few passes (rk_sort_split.hpp) launch so many;
// `pass` is then -1, -2, ... for the first of the digits that vary, the second ...  Returns the digit, -1: there is none to do.
// Three: 2^24 keys in three digits, sortperm Int64 432 us so and 522 by splitters, sort 400 and 382; in four, 547 and 502, 427 and 381.
constexpr uint32_t SORT_FEW_PASSES = 3;
__device__ __forceinline__ int sort_pass_index(const SortCtl* ctl, int pass) {
    if (pass >= 0) return pass;
    if (ctl->nexec > SORT_FEW_PASSES || (uint32_t)-pass > ctl->nexec) return -1;
    int p = -1;
    for (int left = -pass; left != 0;) left -= ctl->skip[++p] == 0u ? 1 : 0;
    return p;
}

// ---- init: clear the control block ----------------------------------------------------------------------------------
// all_passes: large sorts of floats, which run every pass on keys that are not taken relative to the smallest one; their
// plan is made here.
__global__ __launch_bounds__(256) void sort_init_kernel(SortCtl* ctl, int all_passes, int first_source) {
    for (int i = threadIdx.x; i < SORT_CTL_CLEAR; i += 256) ctl->skip[i] = 0u;
    if (all_passes == 0) return;
    __syncthreads();
    if (threadIdx.x == 0) {
        ctl->inv_min = ~0ull;
        sort_make_plan(ctl, all_passes, false, 0ull, ~0ull, first_source);
    }
}

// The whole-array read below takes 16-byte vectors from the aligned body [head, head + nvec * VEC) of the keys
// and single elements from the few keys in front of and behind it.
template <typename T, typename F>
__device__ __forceinline__ void for_each_key(const T* __restrict__ keys, int64_t n, int64_t head, int64_t nvec, F&& f) {
    typedef typename SortKey<T>::U U;
    constexpr int VEC = 16 / sizeof(T);
    typedef typename VecOf<U, VEC>::type VU;
    const VU* body = (const VU*)(keys + head);
    constexpr int UNR = 4;                                   // loads in flight per lane
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + (UNR - 1) * stride < nvec; i += UNR * stride) {
        VU v[UNR];
#pragma unroll
        for (int r = 0; r < UNR; ++r) v[r] = load_nt(body + i + r * stride);
#pragma unroll
        for (int r = 0; r < UNR; ++r) {
            U k[VEC];
#pragma unroll
            for (int j = 0; j < VEC; ++j) k[j] = (U)v[r][j];
            f(k, VEC);
        }
    }
    for (; i < nvec; i += stride) {
        const VU v = load_nt(body + i);
        U k[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) k[j] = (U)v[j];
        f(k, VEC);
    }
    if (blockIdx.x == 0) {
        const int64_t tail0 = head + nvec * VEC, extra = head + (n - tail0);     // at most 2 * (VEC - 1) keys
        for (int64_t i = threadIdx.x; i < extra; i += blockDim.x) {
            const int64_t e = i < head ? i : tail0 + (i - head);
            U k[VEC];
            k[0] = __builtin_bit_cast(U, keys[e]);
            f(k, 1);
        }
    }
}

// ---- smallest and largest key, varying bits -----------------------------------------------------------------------------
// One read at streaming speed.  Integers are taken relative to the smallest key: small-range integers then need one or two
// passes.  The workgroup whose ticket is the last makes the plan.
constexpr int RANGE_BLOCK = 1024;       // few, large workgroups: each ends with device-wide atomics on shared words
template <typename T>
__global__ __launch_bounds__(RANGE_BLOCK) void sort_range_kernel(const T* __restrict__ keys, int64_t n, int64_t head, int64_t nvec, int rev,
                                                                 int first_source, SortCtl* ctl) {
    typedef typename SortKey<T>::U U;
    typedef unsigned long long W;
    constexpr int VEC = 16 / sizeof(T);
    constexpr bool RELATIVE = std::is_integral<T>::value;
    __shared__ W part[3][RANGE_BLOCK / WAVE];
    const U u0 = enc_bits<T>(__builtin_bit_cast(U, keys[0]), rev, (U)0);
    U mn = u0, mx = u0, var = 0;
    for_each_key<T>(keys, n, head, nvec, [&](const U (&k)[VEC], int cnt) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            if (j < cnt) {
                const U u = enc_bits<T>(k[j], rev, (U)0);
                if (RELATIVE) { mn = u < mn ? u : mn; mx = u > mx ? u : mx; }
                var |= (U)(u ^ u0);
            }
        }
    });
    W inv = wave_reduce((W)(U)~mn, OpMax()), top = wave_reduce((W)mx, OpMax()), dif = wave_reduce((W)var, OpOr());
    if (lane_id() == 0) { part[0][threadIdx.x / WAVE] = inv; part[1][threadIdx.x / WAVE] = top; part[2][threadIdx.x / WAVE] = dif; }
    __syncthreads();
    if (threadIdx.x >= WAVE) return;
    int finishes_last = 0;
    if (threadIdx.x == 0) {
        for (int w = 1; w < RANGE_BLOCK / WAVE; ++w) {
            inv = part[0][w] > inv ? part[0][w] : inv;
            top = part[1][w] > top ? part[1][w] : top;
            dif |= part[2][w];
        }
        if (RELATIVE) {
            if (inv != 0ull) atomicMax(&ctl->inv_min, inv);
            if (top != 0ull) atomicMax(&ctl->key_max, top);
        }
        if (dif != 0ull) atomicOr(&ctl->varying, dif);
        publish_barrier();
        finishes_last = atomicAdd(&ctl->range_ticket, 1u) == gridDim.x - 1u;
        if (!RELATIVE && finishes_last) ctl->inv_min = ~0ull;       // the smallest key is taken as 0
    }
    if (__builtin_amdgcn_readfirstlane(finishes_last) == 0) return;
    const U smallest = (U)~(U)load_agent(&ctl->inv_min);
    if (threadIdx.x == 0)
        sort_make_plan(ctl, (int)sizeof(T), RELATIVE, RELATIVE ? load_agent(&ctl->key_max) - (W)smallest : 0ull, load_agent(&ctl->varying), first_source);
}

// ---- digit counts of every tile -----------------------------------------------------------------------------------
// Same tiles as sort_pass_kernel, one per workgroup; the order of the keys inside the tile does not matter here, so
// aligned full tiles are read as 16-byte vectors.  One LDS atomic per key into one of SUB histograms per wave,
// chosen by the lane: skewed digits (exponent bytes, the high bytes of small integers) then queue up 16 deep on a
// counter instead of 64 deep, and no lane has to find out who else holds its digit.
// SEVERAL: tiles a workgroup, in turn.
template <typename T, int BLOCK, int ITEMS, int SUB, typename C, bool SEVERAL = false>
__global__ __launch_bounds__(BLOCK, 8) void sort_upsweep_kernel(const T* __restrict__ orig, const typename SortKey<T>::U* buf_a,
                                                                const typename SortKey<T>::U* buf_b, uint32_t n, int pass, int rev,
                                                                SortCtl* ctl, C* __restrict__ tile_count) {
    typedef typename SortKey<T>::U U;
    constexpr int TILE = BLOCK * ITEMS, NW = BLOCK / WAVE;
    static_assert(sizeof(C) == 4 || TILE < 65536, "a count fits the table's type");
    constexpr int VEC = 16 / (int)sizeof(T), NV = ITEMS / VEC;
    typedef typename VecOf<U, VEC>::type VU;
    __shared__ uint32_t cnt[NW * SUB][256];
    pass = sort_pass_index(ctl, pass);
    if (pass < 0) return;
    const SortStep step = sort_step(ctl, pass);
    if (step.skip != 0u) return;
    const bool first = (uint32_t)pass == step.first_pass;
    const U* in = first ? (const U*)orig : (step.src_b != 0u ? buf_b : buf_a);
    const U umin = (U)~step.inv_min;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
    for (uint32_t tile = blockIdx.x;;) {
        for (int i = tid; i < NW * SUB * 256; i += BLOCK) (&cnt[0][0])[i] = 0;
        const uint32_t e0 = tile * (uint32_t)TILE;
        const uint32_t woff = e0 + (uint32_t)wave * (WAVE * ITEMS) + lane;
        uint32_t* row = cnt[wave * SUB + (lane & (SUB - 1))];
        // When many lanes hold the same digit (judged on every fourth key) the two most frequent values -- as seen from the
        // first lane still in play -- are taken out with a ballot each and added by that lane alone; uniform floats have
        // 50% and 37% of their keys in two values of the exponent digit.
        bool skewed = false;
        auto count = [&](uint32_t d, bool valid, int i) {
            if ((i & 3) == 0) skewed = digits_skewed(d, valid);
            if (skewed) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const uint64_t active = __ballot(valid);
                    if (active != 0ull) {
                        const int head = __ffsll((unsigned long long)active) - 1;
                        const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, head);
                        const uint64_t same = __ballot(valid && d == d0);
                        if (lane == head) atomicAdd(&row[d0], (uint32_t)__popcll(same));
                        valid = valid && d != d0;
                    }
                }
            }
            if (valid) atomicAdd(&row[d], 1u);
        };
        // (the two read paths share no variables: merged into one key array they made the compiler shuffle it through
        // private memory)
        bool vectors = false;
        if constexpr (NV > 0) vectors = e0 + (uint32_t)TILE <= n && (((uintptr_t)(in + e0)) & 15) == 0;
        if (vectors) {
            const VU* vin = (const VU*)(in + e0);
            VU v[NV > 0 ? NV : 1];
#pragma unroll
            for (int r = 0; r < NV; ++r) v[r] = vin[r * BLOCK + tid];
            __syncthreads();
#pragma unroll
            for (int r = 0; r < NV; ++r) {
#pragma unroll
                for (int j = 0; j < VEC; ++j) {
                    U k = (U)v[r][j];
                    if (first) k = enc_bits<T>(k, rev, umin);
                    count(digit_of(k, pass), true, r * VEC + j);
                }
            }
        } else {
            U key[ITEMS];
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const uint32_t e = woff + i * WAVE;
                key[i] = (U)0;
                if (e < n) key[i] = in[e];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < ITEMS; ++i) {
                const U k = first ? enc_bits<T>(key[i], rev, umin) : key[i];
                count(digit_of(k, pass), woff + i * WAVE < n, i);
            }
        }
        __syncthreads();
        if (BLOCK == 256 || tid < 256) {
            uint32_t c = 0;
#pragma unroll
            for (int w = 0; w < NW * SUB; ++w) c += cnt[w][tid];
            tile_count[(uint64_t)tile * 256 + tid] = (C)c;
        }
        if (!SEVERAL) break;
        tile += gridDim.x;
        if (tile * (uint32_t)TILE >= n) break;
        __syncthreads();
    }
}

// ---- where every tile's keys go (large sorts) --------------------------------------------------------------------------
// Input: count[tile][digit].  Output, for sort_pass_kernel: count[tile][digit] becomes the number of keys of the digit in
// the earlier tiles of the same chunk of `chunk_rows` tiles; chunk_prefix[chunk][digit] the number in all earlier chunks;
// ctl->hist[pass][digit] the first output slot of the digit (exclusive scan of the digit totals).
// One workgroup of 1024 threads per chunk: 4 groups of rows x 256 digits.  The workgroup that stores its chunk totals
// last (a ticket) scans the totals of all chunks; nobody waits for anybody.  At most 256 chunks.
constexpr int TS_GROUPS = 4, TS_BLOCK = TS_GROUPS * 256, TS_UNROLL = 16, TS_MAX_CHUNKS = 256;

// Rows [first, first + rows) of column d of x (256 words a row), TS_UNROLL loads in flight: their sum; with WRITE,
// out[row][d] = start + the sum of the rows in front.
template <bool WRITE, bool COHERENT>
__device__ __forceinline__ uint32_t ts_rows(const uint32_t* x, uint32_t first, uint32_t rows, uint32_t d, uint32_t start, uint32_t* out) {
    uint32_t run = start;
    for (uint32_t r = 0; r < rows; r += TS_UNROLL) {
        uint32_t v[TS_UNROLL];
#pragma unroll
        for (int j = 0; j < TS_UNROLL; ++j) {
            v[j] = 0;
            if (r + j < rows) {
                const uint32_t* q = x + (uint64_t)(first + r + j) * 256 + d;
                v[j] = COHERENT ? load_agent(q) : *q;
            }
        }
#pragma unroll
        for (int j = 0; j < TS_UNROLL; ++j) {
            if (WRITE && r + j < rows) out[(uint64_t)(first + r + j) * 256 + d] = run;
            run += v[j];
        }
    }
    return run - start;
}

// Exclusive scan down rows [a, b) of column d, for the thread of row group g: out[row][d] = sum of the rows of the
// column in front, over all groups; returns the column total.  Up to MAXR rows a group stay in registers between the
// two steps (one round trip to memory); longer groups are read twice.
template <int MAXR, bool COHERENT>
__device__ __forceinline__ uint32_t ts_scan_groups(const uint32_t* x, uint32_t* out, uint32_t a, uint32_t b, uint32_t d, uint32_t g,
                                                   uint32_t (*gsum)[256]) {
    const uint32_t rows = b - a;
    const bool in_regs = __syncthreads_and(rows <= (uint32_t)MAXR) != 0;
    uint32_t v[MAXR];
    uint32_t mine = 0;
    if (in_regs) {
#pragma unroll
        for (int j = 0; j < MAXR; ++j) {
            v[j] = 0;
            if ((uint32_t)j < rows) {
                const uint32_t* q = x + (uint64_t)(a + j) * 256 + d;
                v[j] = COHERENT ? load_agent(q) : *q;
            }
        }
#pragma unroll
        for (int j = 0; j < MAXR; ++j) mine += v[j];
    } else {
        mine = ts_rows<false, COHERENT>(x, a, rows, d, 0u, nullptr);
    }
    gsum[g][d] = mine;
    __syncthreads();
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int k = 0; k < TS_GROUPS; ++k) {
        const uint32_t s = gsum[k][d];
        if ((uint32_t)k < g) before += s;
        total += s;
    }
    if (in_regs) {
        uint32_t run = before;
#pragma unroll
        for (int j = 0; j < MAXR; ++j) {
            if ((uint32_t)j < rows) out[(uint64_t)(a + j) * 256 + d] = run;
            run += v[j];
        }
    } else {
        ts_rows<true, COHERENT>(x, a, rows, d, before, out);
    }
    return total;
}

__global__ __launch_bounds__(TS_BLOCK) void sort_tilescan_kernel(SortCtl* ctl, int pass, uint32_t* count, uint32_t ntiles, uint32_t chunk_rows,
                                                                 uint32_t* chunk_total, uint32_t* chunk_prefix) {
    __shared__ uint32_t gsum[2][TS_GROUPS][256];
    __shared__ uint32_t wsum[256 / WAVE];
    __shared__ uint32_t lds_ticket;
    pass = sort_pass_index(ctl, pass);
    if (pass < 0 || ctl->skip[pass]) return;
    const uint32_t d = threadIdx.x & 255u, g = threadIdx.x >> 8, chunk = blockIdx.x, nchunks = gridDim.x;
    {
        const uint32_t r0 = chunk * chunk_rows, r1 = r0 + chunk_rows < ntiles ? r0 + chunk_rows : ntiles;
        const uint32_t per = (r1 - r0 + TS_GROUPS - 1) / TS_GROUPS;
        const uint32_t a = r0 + g * per < r1 ? r0 + g * per : r1, b = a + per < r1 ? a + per : r1;
        const uint32_t total = ts_scan_groups<16, false>(count, count, a, b, d, g, gsum[0]);
        if (g == 0) store_agent(chunk_total + (uint64_t)chunk * 256 + d, total);
    }
    publish_barrier();                       // this thread's total is visible device-wide ...
    __syncthreads();                         // ... and so is every other thread's of this workgroup
    if (threadIdx.x == 0) lds_ticket = atomicAdd(&ctl->scan_ticket[pass], 1u);
    __syncthreads();
    if (lds_ticket != nchunks - 1u) return;
    // the last one: exclusive scan of the chunk totals down the chunks, then of the digit totals across the digits
    const uint32_t per = (nchunks + TS_GROUPS - 1) / TS_GROUPS;
    const uint32_t a = g * per < nchunks ? g * per : nchunks, b = a + per < nchunks ? a + per : nchunks;
    const uint32_t total = ts_scan_groups<TS_MAX_CHUNKS / TS_GROUPS, true>(chunk_total, chunk_prefix, a, b, d, g, gsum[1]);
    const uint32_t inc = wave_scan_inclusive(total, OpAdd(), 0u);          // the same in all four groups
    if (g == 0 && d % WAVE == WAVE - 1) wsum[d / WAVE] = inc;
    __syncthreads();
    if (g == 0) {
        uint32_t start = inc - total;
        for (uint32_t w = 0; w < d / WAVE; ++w) start += wsum[w];
        ctl->hist[pass][d] = start;
    }
}

// ---- one pass ----------------------------------------------------------------------------------------------------
// Tile = BLOCK threads x ITEMS keys.  Wave w owns the w-th part of the tile; its item i of lane l is key
// i * 64 + l of that part (coalesced loads; the order (i, l) is memory order, which the ranking keeps).
// DIRECT (keys of 2 bytes): `counts` are the raw counts of every tile (uint16, a row of 256 a tile) and the workgroup sums the columns it
// needs itself; otherwise they are the exclusive counts of sort_tilescan_kernel.
// waves per SIMD the register allocation aims at: the kernel is bound by its vector instructions, and three or four
// waves hide the latencies (measured: 4 against 6 workgroups a CU differ by 4%)
template <typename T, bool PERM, bool DIRECT> constexpr int sort_pass_waves() { return (DIRECT || (!PERM && sizeof(T) <= 4)) ? 4 : 3; }

// SEVERAL: tiles a workgroup, in turn (as a loop, every pass takes 4 % longer).
template <typename T, int BLOCK, int ITEMS, bool PERM, bool DIRECT, bool SEVERAL = false>
__global__ __launch_bounds__(BLOCK, (sort_pass_waves<T, PERM, DIRECT>())) void sort_pass_kernel(const T* __restrict__ orig, typename SortKey<T>::U* buf_a,
                                                               typename SortKey<T>::U* buf_b, uint32_t* val_a, uint32_t* val_b,
                                                               int64_t* __restrict__ perm_out, uint32_t n, int pass, int rev, SortCtl* ctl,
                                                               const void* __restrict__ counts,
                                                               const uint32_t* __restrict__ chunk_prefix, uint32_t chunk_rows,
                                                               uint32_t ntiles, uint32_t xcd_chunk) {
    typedef typename SortKey<T>::U U;
    constexpr int TILE = BLOCK * ITEMS, NW = BLOCK / WAVE;
    constexpr int GROUPS = DIRECT ? BLOCK / 128 : 1;       // groups of rows of the table, 128 lanes (two counts each) a group
    __shared__ U lds_keys[TILE];
    __shared__ uint32_t lds_vals[PERM ? TILE : 1];
    __shared__ uint32_t cnt[NW][256];             // per wave and digit: count, then slot in the sorted tile of the wave's first key of the digit
    __shared__ uint32_t goff[256];                // global slot of the digit's first key of this tile, minus its slot in the sorted tile
    __shared__ uint32_t wsum[2][256 / WAVE];
    __shared__ uint2 part_before[GROUPS][DIRECT ? 128 : 1], part_all[GROUPS][DIRECT ? 128 : 1];

    const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
    const bool first_of_few = pass == -1;
    pass = sort_pass_index(ctl, pass);
    SortStep step{};
    if (pass >= 0) step = sort_step(ctl, pass);
    if (pass < 0 || step.skip != 0u) {
        // all keys equal: no pass ran, and the last one writes the identity permutation, or the copy of the keys
        if ((first_of_few || pass == (int)sizeof(T) - 1) && ctl->nexec == 0u && (PERM || (const void*)orig != (const void*)buf_a)) {
            const int64_t step = (int64_t)gridDim.x * BLOCK;
            for (int64_t i = (int64_t)blockIdx.x * BLOCK + tid; i < (int64_t)n; i += 4 * step) {
                T k[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (!PERM && i + u * step < (int64_t)n) k[u] = orig[i + u * step];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (i + u * step >= (int64_t)n) continue;
                    if (PERM) perm_out[i + u * step] = i + u * step + 1;
                    else ((T*)buf_a)[i + u * step] = k[u];
                }
            }
        }
        return;
    }
    const bool first = (uint32_t)pass == step.first_pass, last = (uint32_t)pass == step.last_pass;
    const U umin = (U)~step.inv_min;
    const bool src_b = step.src_b != 0u;
    const U* in = first ? (const U*)orig : (src_b ? buf_b : buf_a);
    U* dst = src_b ? buf_a : buf_b;
    const uint32_t* vsrc = src_b ? val_b : val_a;
    uint32_t* vdst = src_b ? val_a : val_b;
    for (uint32_t at = blockIdx.x;;) {
        for (int i = tid; i < NW * 256; i += BLOCK) (&cnt[0][0])[i] = 0;
        __syncthreads();
        const uint32_t tile = !DIRECT && xcd_chunk != 0u ? (at & 7u) * xcd_chunk + (at >> 3) : at;
        if (tile < ntiles) {
            const uint32_t e0 = tile * (uint32_t)TILE;
            const uint32_t woff = e0 + (uint32_t)wave * (WAVE * ITEMS) + lane;

            // Every tile but the last is full: its code carries no bounds checks (they cost an exec-mask save and a
            // branch per key and round).
            auto sort_tile = [&](auto full_tile) {
                constexpr bool FULL = decltype(full_tile)::value;
                // load (and map on the first pass)
                U key[ITEMS];
                uint32_t val[PERM ? ITEMS : 1];
                uint32_t rank[ITEMS];
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    const uint32_t e = woff + i * WAVE;
                    key[i] = (U)~(U)0;
                    if (FULL || e < n) key[i] = in[e];
                }
                if constexpr (PERM) {
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i) val[i] = woff + i * WAVE;              // first pass: the key's own index
                    if (!first) {
#pragma unroll
                        for (int i = 0; i < ITEMS; ++i)
                            if (FULL || woff + i * WAVE < n) val[i] = vsrc[woff + i * WAVE];
                    }
                }
                if constexpr (DIRECT) {
                    // columns of the table of counts: all rows, and the rows of the tiles in front.  At most 256 rows, 16 in flight.
                    const uint32_t c = (uint32_t)tid & 127u, g = (uint32_t)tid >> 7;
                    const uint32_t* col = (const uint32_t*)counts + c;
                    uint2 bef = {0u, 0u}, sum = {0u, 0u};
                    constexpr uint32_t UNR = 16;
                    for (uint32_t r0 = g; r0 < ntiles; r0 += GROUPS * UNR) {
                        uint32_t w[UNR];
#pragma unroll
                        for (uint32_t u = 0; u < UNR; ++u) {
                            const uint32_t r = r0 + u * GROUPS;
                            w[u] = col[(uint64_t)(r < ntiles ? r : ntiles - 1u) * 128];
                        }
#pragma unroll
                        for (uint32_t u = 0; u < UNR; ++u) {
                            const uint32_t r = r0 + u * GROUPS;
                            const uint32_t lo = r < ntiles ? w[u] & 0xffffu : 0u, hi = r < ntiles ? w[u] >> 16 : 0u;
                            sum.x += lo;
                            sum.y += hi;
                            bef.x += r < tile ? lo : 0u;
                            bef.y += r < tile ? hi : 0u;
                        }
                    }
                    part_before[g][c] = bef;
                    part_all[g][c] = sum;
                }
                if (first) {
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i) key[i] = enc_bits<T>(key[i], rev, umin);    // padding keys are never counted
                }
                // rank inside the wave: lanes with the same digit find each other with 8 ballots; every lane reads the
                // wave's counter of its digit -- the rank of the group's first key -- and then the lowest lane of the group
                // adds the size of the group to it.  LDS executes the instructions of one wave in order, so the read of
                // the next round sees this add, and the 16 rounds queue up back to back; a result is used two rounds later.
                uint32_t* wcnt = cnt[wave];
                constexpr int DEPTH = 2;                       // counter reads in flight before their result is used
                uint32_t pend_before[DEPTH], pend_below[DEPTH];
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    const bool valid = FULL || woff + i * WAVE < n;
                    const uint32_t d = digit_of(key[i], pass);
                    uint32_t same_lo, same_hi;
                    match_digit_halves(d, same_lo, same_hi);
                    if (!FULL) {
                        const uint64_t vm = __ballot(valid);
                        same_lo &= (uint32_t)vm;
                        same_hi &= (uint32_t)(vm >> 32);
                    }
                    const uint32_t below = __builtin_amdgcn_mbcnt_hi(same_hi, __builtin_amdgcn_mbcnt_lo(same_lo, 0u));
                    const uint32_t before = __hip_atomic_load(&wcnt[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    __builtin_amdgcn_wave_barrier();
                    if (valid && below == 0u) {
                        const uint32_t total = (uint32_t)__builtin_popcount(same_lo) + (uint32_t)__builtin_popcount(same_hi);
                        __hip_atomic_fetch_add(&wcnt[d], total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    }
                    if (i >= DEPTH) rank[i - DEPTH] = pend_before[i % DEPTH] + pend_below[i % DEPTH];
                    pend_before[i % DEPTH] = before;
                    pend_below[i % DEPTH] = below;
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int i = ITEMS; i < ITEMS + DEPTH; ++i) rank[i - DEPTH] = pend_before[i % DEPTH] + pend_below[i % DEPTH];
                __syncthreads();
                // digit d = tid (the first 256 threads): count of the tile and of each wave, first slot inside the sorted tile
                // (exclusive scan over the digits) and in the whole output
                uint32_t wave_count[NW];
                uint32_t count = 0, excl = 0, all = 0, inc = 0, inc_all = 0;
                const bool has_digit = BLOCK == 256 || tid < 256;
                if (has_digit) {
#pragma unroll
                    for (int w = 0; w < NW; ++w) {
                        wave_count[w] = cnt[w][tid];
                        count += wave_count[w];
                    }
                    if constexpr (DIRECT) {
#pragma unroll
                        for (int g = 0; g < GROUPS; ++g) {
                            const uint2 b = part_before[g][tid >> 1], a = part_all[g][tid >> 1];
                            excl += (tid & 1) ? b.y : b.x;
                            all += (tid & 1) ? a.y : a.x;
                        }
                        inc_all = wave_scan_inclusive(all, OpAdd(), 0u);
                        if (lane == WAVE - 1) wsum[1][wave] = inc_all;
                    } else {
                        excl = ((const uint32_t*)counts)[(uint64_t)tile * 256 + tid] + chunk_prefix[(uint64_t)(tile / chunk_rows) * 256 + tid];
                    }
                    inc = wave_scan_inclusive(count, OpAdd(), 0u);
                    if (lane == WAVE - 1) wsum[0][wave] = inc;
                }
                __syncthreads();
                if (has_digit) {
                    uint32_t start = inc - count, base = DIRECT ? inc_all - all : ctl->hist[pass][tid];
                    for (int w = 0; w < wave; ++w) {
                        start += wsum[0][w];
                        if (DIRECT) base += wsum[1][w];
                    }
                    goff[tid] = base + excl - start;
#pragma unroll
                    for (int w = 0; w < NW; ++w) {
                        cnt[w][tid] = start;
                        start += wave_count[w];
                    }
                }
                __syncthreads();
                // reorder the tile in LDS.  Reads first, writes after, so that the 16 table reads are in flight together.
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    uint32_t d = digit_of(key[i], pass);
                    asm volatile("" : "+v"(d));            // computed again here: 16 LDS addresses kept from the ranking cost a wave of occupancy
                    rank[i] += wcnt[d];
                }
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    if (FULL || woff + i * WAVE < n) {
                        lds_keys[rank[i]] = key[i];
                        if constexpr (PERM) lds_vals[rank[i]] = val[i];
                    }
                }
                __syncthreads();
                // write runs of equal digits: thread q takes the q-th key of the sorted tile.  Again all reads of a kind
                // together; `last` is decided once, not per key.
                const uint32_t valid_n = n - e0 < (uint32_t)TILE ? n - e0 : (uint32_t)TILE;
                U out_key[ITEMS];
                uint32_t slot[ITEMS];
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) {
                    const uint32_t q = (uint32_t)tid + i * BLOCK;
                    out_key[i] = (U)0;
                    if (FULL || q < valid_n) out_key[i] = lds_keys[q];
                }
#pragma unroll
                for (int i = 0; i < ITEMS; ++i) slot[i] = goff[digit_of(out_key[i], pass)] + (uint32_t)tid + i * BLOCK;
                auto writable = [&](int i) { return FULL || (uint32_t)tid + i * BLOCK < valid_n; };
                if constexpr (PERM) {
                    uint32_t out_val[ITEMS];
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i) {
                        out_val[i] = 0;
                        if (FULL || (uint32_t)tid + i * BLOCK < valid_n) out_val[i] = lds_vals[(uint32_t)tid + i * BLOCK];
                    }
                    if (last) {
#pragma unroll
                        for (int i = 0; i < ITEMS; ++i) if (writable(i)) perm_out[slot[i]] = (int64_t)out_val[i] + 1;
                    } else {
#pragma unroll
                        for (int i = 0; i < ITEMS; ++i) if (writable(i)) { dst[slot[i]] = out_key[i]; vdst[slot[i]] = out_val[i]; }
                    }
                } else if (last) {
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i) if (writable(i)) ((T*)dst)[slot[i]] = dec_bits<T>(out_key[i], rev, umin);
                } else {
#pragma unroll
                    for (int i = 0; i < ITEMS; ++i) if (writable(i)) dst[slot[i]] = out_key[i];
                }
            };
            if (e0 + (uint32_t)TILE <= n) sort_tile(std::true_type{}); else sort_tile(std::false_type{});
        }
        if (!SEVERAL) break;
        at += gridDim.x;
        if (at >= (xcd_chunk != 0u ? xcd_chunk * 8u : ntiles)) break;
        __syncthreads();
    }
}

// ---- finish ------------------------------------------------------------------------------------------------------
// sort!: after an odd number of passes the result sits in buffer B.
// most: passes that may have run; keys that would have taken more were sorted in another way.
template <typename W>
__global__ __launch_bounds__(256) void sort_finish_kernel(const SortCtl* ctl, W* a, const W* b, int64_t nwords, uint32_t most) {
    if (ctl->nexec > most || (ctl->nexec & 1u) == 0u) return;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nwords; i += (int64_t)gridDim.x * 256) a[i] = b[i];
}

}  // namespace rk

#include "rk_sort_buckets.hpp"
#include "rk_sort_split.hpp"
#include "rk_sort_quantiles.hpp"

namespace rk {

// ---- host --------------------------------------------------------------------------------------------------------
// keys per tile: 256 lanes x 16 (large sorts) or 1024 x 4.  (512 lanes x 16 for large sorts halve the table of counts, tile
// scan 17.8 -> 15.7 us a pass of Float32[2^26], but the pass itself takes 141 instead of 121 us.)
constexpr int64_t SORT_TILE = 4096;
constexpr int SORT_ITEMS = (int)SORT_TILE / SORT_BLOCK;
constexpr int DIRECT_BLOCK = 1024, DIRECT_ITEMS = (int)SORT_TILE / DIRECT_BLOCK;
// Up to here a pass (over 2-byte keys) sums the columns of the table of counts itself.  Every tile reads the counts of all tiles, so that
// traffic grows with their square: four passes over Float32 keys, which no longer come here, summed here / by the tile scan, 0.75 x 2^20
// keys 61.4 / 102 us, 2^20 64.6 / 112, 1.5 x 2^20 98 / 117, 2^21 112 / 131, 2^22 267 / 136.  256 tiles are a workgroup a compute unit.
constexpr uint32_t DIRECT_TILES = 256;

struct SortLayout {
    size_t count_off, chunk_total_off, chunk_prefix_off, keys_b_off, keys_a_off, val_a_off, val_b_off, total;
    size_t compact_off, spl_key_off, spl_pos_off, table_off;
    uint32_t ntiles, chunk_rows, nchunks, k;
    bool tiny, direct, buckets, quantiles, split;
    LsLayout ls;
    SqLayout sq;
};

static SortLayout sort_layout(size_t key_size, bool integers, int64_t n, bool perm) {
    SortLayout l{};
    l.ntiles = (uint32_t)((n + SORT_TILE - 1) / SORT_TILE);
    size_t off = (sizeof(SortCtl) + 255) & ~(size_t)255;
    l.tiny = n <= ST_MAX;
    l.direct = l.ntiles <= DIRECT_TILES;
    l.buckets = l.direct && !l.tiny && key_size >= 4;
    l.quantiles = key_size == 4 && !perm && n > (integers ? SQ_MIN_INTEGERS : LS_MAX_FLOATS) && n <= SQ_MAX_KEYS;
    l.split = !l.direct && !l.quantiles && (key_size == 8 ? n <= LS_MAX_KEYS : key_size == 4 && !integers && n <= LS_MAX_FLOATS);
    const size_t ctl_end = off;
    l.count_off = off;
    if (l.direct) {
        if (!l.buckets && !l.tiny) off += (size_t)l.ntiles * 256 * sizeof(uint16_t);
    } else {
        off += (size_t)l.ntiles * 256 * sizeof(uint32_t);
        l.chunk_rows = (l.ntiles + TS_MAX_CHUNKS - 1) / TS_MAX_CHUNKS;
        l.nchunks = (l.ntiles + l.chunk_rows - 1) / l.chunk_rows;
        l.chunk_total_off = off;  off += (size_t)TS_MAX_CHUNKS * 256 * sizeof(uint32_t);
        l.chunk_prefix_off = off; off += (size_t)TS_MAX_CHUNKS * 256 * sizeof(uint32_t);
    }
    if (l.split) {                                           // in the place of the counts: one of the two ways is taken
        l.ls = ls_layout(ctl_end, key_size, n);
        if (l.ls.total > off) off = l.ls.total;
    }
    if (l.quantiles) {                                       // (as above)
        l.sq = sq_layout(ctl_end, n);
        if (l.sq.total > off) off = l.sq.total;
    }
    const size_t kbytes = ((size_t)n * key_size + 255) & ~(size_t)255, vbytes = ((size_t)n * 4 + 255) & ~(size_t)255;
    l.keys_b_off = off; off += kbytes;
    if (perm) {
        l.keys_a_off = off; off += kbytes;
        l.val_a_off = off; off += vbytes;
        l.val_b_off = off; off += vbytes;
    }
    if (l.buckets) {
        l.k = sb_buckets(n);
        const auto take = [&](size_t bytes) { const size_t at = off; off += (bytes + 255) & ~(size_t)255; return at; };
        l.compact_off = take((size_t)l.k * SB_OVER * key_size);
        l.spl_key_off = take((size_t)l.k * key_size);
        l.spl_pos_off = take((size_t)l.k * 4);
        l.table_off = take((size_t)l.ntiles * l.k * 4);
    }
    l.total = off;
    return l;
}

// What a temporary needs that serves every sort of up to n keys of a size, floats and integers: a caller may keep the one of its
// largest sort.  A way's own need grows with the number of keys, but falls where another way, or larger tiles, take over.
static size_t sort_tmp_need(size_t key_size, int64_t n, bool perm) {
    const int64_t last[] = {ST_MAX, DIRECT_TILES * SORT_TILE, LS_SMALL_TILES, LS_MAX_FLOATS, SQ_MIN_INTEGERS, SQ_MAX_KEYS, LS_MAX_KEYS, n};     // of a way
    size_t need = 0;
    for (int64_t m : last)
        for (int integers = 0; integers < 2; ++integers) {
            const size_t total = sort_layout(key_size, integers != 0, m < n ? m : n, perm).total;
            need = total > need ? total : need;
        }
    return need;
}

// The kernels of rk_sort_buckets.hpp; the sorted tiles lie in buffer B.  A bucket that is too large for LDS is put together and
// sorted where its keys end up (sort!, sort) or in buffer A (sortperm).
template <typename T, bool PERM>
static int32_t sort_buckets(const SortLayout& l, const void* keys, void* sorted_out, int64_t* perm_out, int64_t n, int rev, char* base, hipStream_t stream) {
    typedef typename SortKey<T>::U U;
    static_assert(SB_TILE == SORT_TILE && SB_MAX_TILES == DIRECT_TILES, "ntiles counts both");
    SortCtl* ctl = (SortCtl*)base;
    U* spl_key = (U*)(base + l.spl_key_off);
    uint32_t* spl_pos = (uint32_t*)(base + l.spl_pos_off);
    uint32_t* table = (uint32_t*)(base + l.table_off);
    U* tile_key = (U*)(base + l.keys_b_off);
    uint16_t* tile_val = PERM ? (uint16_t*)(base + l.val_b_off) : nullptr;
    U* big_key = PERM ? (U*)(base + l.keys_a_off) : nullptr;
    uint32_t* big_val = PERM ? (uint32_t*)(base + l.val_a_off) : nullptr;
    const uint32_t samples = l.k * SB_OVER;
    if (samples <= SB_DIRECT_SAMPLES) {
        sort_splitters_kernel<T, true><<<samples / SB_SPL_EACH, SB_SPL_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, rev, ctl, l.k, nullptr, spl_key, spl_pos);
    } else {
        U* compact = (U*)(base + l.compact_off);
        sort_sample_kernel<T><<<samples / 256, 256, 0, stream>>>((const T*)keys, (uint32_t)n, rev, samples, compact);
        RK_LAUNCH_CHECK();
        sort_splitters_kernel<T, false><<<samples / SB_SPL_EACH, SB_SPL_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, rev, ctl, l.k, compact, spl_key, spl_pos);
    }
    RK_LAUNCH_CHECK();
    sort_tile_kernel<T, PERM><<<l.ntiles, SB_TILE_BLOCK, 0, stream>>>((const T*)keys, (uint32_t)n, rev, l.k, spl_key, spl_pos, table, tile_key, tile_val);
    RK_LAUNCH_CHECK();
    sort_bucket_kernel<T, PERM><<<l.k, SB_SORT_BLOCK, 0, stream>>>(l.k, l.ntiles, table, rev, tile_key, tile_val, big_key, big_val, (T*)sorted_out, perm_out);
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

// sorted_out: where sort! and sort leave the sorted keys (`keys` itself for sort!)
template <typename T, bool PERM>
static int32_t sort_typed(const void* keys, void* sorted_out, int64_t* perm_out, int64_t n, int rev, void* tmp, size_t tmp_bytes, hipStream_t stream) {
    typedef typename SortKey<T>::U U;
    constexpr int PASSES = (int)sizeof(T);
    const SortLayout l = sort_layout(sizeof(T), std::is_integral<T>::value, n, PERM);
    if (tmp == nullptr || !is_aligned(tmp, 256) || tmp_bytes < l.total) return RK_ERR_WORKSPACE;
    char* base = (char*)tmp;
    SortCtl* ctl = (SortCtl*)base;
    U* buf_b = (U*)(base + l.keys_b_off);
    U* buf_a = PERM ? (U*)(base + l.keys_a_off) : (U*)sorted_out;
    uint32_t* val_a = PERM ? (uint32_t*)(base + l.val_a_off) : nullptr;
    uint32_t* val_b = PERM ? (uint32_t*)(base + l.val_b_off) : nullptr;
    const int cus = device_info().cus;

    if (l.tiny) {
        sort_tiny_kernel<T, PERM><<<1, ST_BLOCK, 0, stream>>>((const T*)keys, (T*)sorted_out, perm_out, (uint32_t)n, rev, ctl);
        RK_LAUNCH_CHECK();
        return RK_SUCCESS;
    }
    constexpr bool FLOAT_KEYS = !std::is_integral<T>::value;
    if constexpr (sizeof(T) >= 4) {
        if (l.buckets) return sort_buckets<T, PERM>(l, keys, sorted_out, perm_out, n, rev, base, stream);
    }
    if constexpr (FLOAT_KEYS && sizeof(T) >= 4) {
        if (l.split) return sort_split<T, PERM>(l.ls, keys, sorted_out, perm_out, n, rev, base, ctl, buf_a, buf_b, val_a, val_b, stream);
    }
    const bool all_passes = FLOAT_KEYS && !l.direct;
    // sortperm: the first pass reads the caller's keys and writes buffer A.  sort: the last one writes the result, whatever their number
    // (a copy behind an odd number of them 85 us for 2^26 Float32); sort!: the keys lie where the result goes, so the first cannot.
    const int first_source = PERM ? SORT_B : keys != sorted_out ? SORT_ENDS_IN_A : SORT_A;
    if (!(all_passes && l.quantiles)) {                      // (of those sq_sample_kernel does it)
        sort_init_kernel<<<1, 256, 0, stream>>>(ctl, all_passes ? PASSES : 0, first_source);
        RK_LAUNCH_CHECK();
    }
    if (!all_passes) {
        constexpr int KVEC = 16 / (int)sizeof(T);
        int64_t head = (int64_t)(((16 - ((uintptr_t)keys & 15)) & 15) / sizeof(T));
        if (head > n) head = n;
        const int64_t nvec = (n - head) / KVEC;
        // 4 vectors a lane and few workgroups: each ends with device-wide atomics on shared words
        int64_t g = (nvec + RANGE_BLOCK * 4 - 1) / (RANGE_BLOCK * 4);
        if (g > cus * 2) g = cus * 2;
        if (g < 1) g = 1;
        sort_range_kernel<T><<<(unsigned)g, RANGE_BLOCK, 0, stream>>>((const T*)keys, n, head, nvec, rev, first_source, ctl);
        RK_LAUNCH_CHECK();
    }
    if constexpr (sizeof(T) == 4 && !PERM) {
        if (l.quantiles) {
            const int32_t rc = sort_quantiles<T>(l.sq, keys, sorted_out, n, rev, base, ctl, first_source, buf_b, stream);
            if (rc != RK_SUCCESS) return rc;
        }
    }
    // tunable, read once: XCD-contiguous tiles (RK_SORT_XCD=0: off).  Large sorts launch one workgroup per tile: the
    // hardware's dispatcher balances the load better than a fixed share of tiles per resident workgroup (2^26 Float32:
    // 866 against 986 us with 4 a CU), and each XCD takes a contiguous eighth of the tiles, so the runs that neighbouring
    // tiles write next to each other meet in one L2 (workgroups go to the XCDs round-robin by their index).
    static const int xcd_map = [] { const char* e = std::getenv("RK_SORT_XCD"); return e ? std::atoi(e) : 1; }();
    // Behind sort_quantiles, whose buckets nearly always fit, these kernels end at once, and sooner the fewer their workgroups.
    unsigned pgrid = (l.ntiles + 7u) & ~7u;
    if (l.quantiles && pgrid > (unsigned)cus * 16u) pgrid = (unsigned)cus * 16u;
    const unsigned ugrid = pgrid < l.ntiles ? pgrid : l.ntiles;
    const uint32_t xcd_chunk = xcd_map != 0 ? (l.ntiles + 7u) / 8u : 0u;
    if (l.direct) {
        if constexpr (sizeof(T) < 4) {
            uint16_t* counts = (uint16_t*)(base + l.count_off);
            for (int p = 0; p < PASSES; ++p) {
                sort_upsweep_kernel<T, DIRECT_BLOCK, DIRECT_ITEMS, 1, uint16_t><<<l.ntiles, DIRECT_BLOCK, 0, stream>>>((const T*)keys, buf_a, buf_b, (uint32_t)n, p, rev, ctl, counts);
                RK_LAUNCH_CHECK();
                sort_pass_kernel<T, DIRECT_BLOCK, DIRECT_ITEMS, PERM, true><<<l.ntiles, DIRECT_BLOCK, 0, stream>>>((const T*)keys, buf_a, buf_b, val_a, val_b, perm_out, (uint32_t)n, p, rev, ctl, counts, nullptr, 1u, l.ntiles, 0u);
                RK_LAUNCH_CHECK();
            }
        }
    } else {
        uint32_t* counts = (uint32_t*)(base + l.count_off);
        uint32_t* chunk_total = (uint32_t*)(base + l.chunk_total_off);
        uint32_t* chunk_prefix = (uint32_t*)(base + l.chunk_prefix_off);
        for (int i = 0; i < (l.split ? (int)SORT_FEW_PASSES : PASSES); ++i) {
            const int p = l.split ? -1 - i : i;
            const auto count = [&](auto several) {
                sort_upsweep_kernel<T, SORT_BLOCK, SORT_ITEMS, 4, uint32_t, decltype(several)::value><<<ugrid, SORT_BLOCK, 0, stream>>>((const T*)keys, buf_a, buf_b, (uint32_t)n, p, rev, ctl, counts);
            };
            const auto pass = [&](auto several) {
                sort_pass_kernel<T, SORT_BLOCK, SORT_ITEMS, PERM, false, decltype(several)::value><<<pgrid, SORT_BLOCK, 0, stream>>>((const T*)keys, buf_a, buf_b, val_a, val_b, perm_out, (uint32_t)n, p, rev, ctl, counts, chunk_prefix, l.chunk_rows, l.ntiles, xcd_chunk);
            };
            constexpr bool MAY = sizeof(T) == 4 && !PERM;    // (l.quantiles needs)
            if (MAY && l.quantiles) count(std::integral_constant<bool, MAY>{});
            else count(std::false_type{});
            RK_LAUNCH_CHECK();
            sort_tilescan_kernel<<<l.nchunks, TS_BLOCK, 0, stream>>>(ctl, p, counts, l.ntiles, l.chunk_rows, chunk_total, chunk_prefix);
            RK_LAUNCH_CHECK();
            if (MAY && l.quantiles) pass(std::integral_constant<bool, MAY>{});
            else pass(std::false_type{});
            RK_LAUNCH_CHECK();
        }
        if constexpr (sizeof(T) == 8) {
            if (l.split) {
                const int32_t rc = sort_split<T, PERM>(l.ls, keys, sorted_out, perm_out, n, rev, base, ctl, buf_a, buf_b, val_a, val_b, stream);
                if (rc != RK_SUCCESS) return rc;
            }
        }
    }
    if (!PERM && keys == sorted_out && (l.quantiles || !(all_passes && PASSES % 2 == 0))) {
        const uint32_t most = l.split ? SORT_FEW_PASSES : (uint32_t)PASSES;
        // whole 32-bit words: buffers are 256-byte padded, the caller's array is at least element-aligned; 16-bit keys
        // with an odd count copy one element more than n only inside buffer padding on the source side -- so copy by element there
        const int64_t nwords = sizeof(T) == 2 ? n : ((int64_t)n * (int64_t)sizeof(T) + 3) / 4;
        int64_t g = (nwords + 255) / 256;
        if (g > cus * 16) g = cus * 16;
        if (sizeof(T) == 2) sort_finish_kernel<uint16_t><<<(unsigned)g, 256, 0, stream>>>(ctl, (uint16_t*)buf_a, (const uint16_t*)buf_b, nwords, most);
        else sort_finish_kernel<uint32_t><<<(unsigned)g, 256, 0, stream>>>(ctl, (uint32_t*)buf_a, (const uint32_t*)buf_b, nwords, most);
        RK_LAUNCH_CHECK();
    }
    return RK_SUCCESS;
}

static bool sort_dtype_size(int dt, size_t* size) {
    switch (dt) {
        case RK_F32: case RK_I32: *size = 4; return true;
        case RK_F64: case RK_I64: *size = 8; return true;
        case RK_F16: case RK_I16: *size = 2; return true;
        default: return false;
    }
}

}  // namespace rk

using namespace rk;

extern "C" size_t rk_sort_tmp_bytes(rk_dtype dt, int64_t n, int32_t with_perm) {
    size_t ks = 0;
    if (!sort_dtype_size((int)dt, &ks) || n <= 0) return 256;
    return sort_tmp_need(ks, n, with_perm != 0);
}

template <bool PERM>
static int32_t sort_dispatch(rk_dtype dt, const void* keys, void* out, int64_t* perm_out, int64_t n, int32_t rev, void* tmp, size_t tmp_bytes, void* stream) {
    size_t ks = 0;
    if (!sort_dtype_size((int)dt, &ks)) return ((int)dt >= RK_F32 && (int)dt <= RK_I16) ? RK_ERR_UNSUPPORTED : RK_ERR_INVALID_ARGUMENT;
    if (n < 0) return RK_ERR_INVALID_ARGUMENT;
    if (n == 0) return RK_SUCCESS;
    if (keys == nullptr || !is_aligned(keys, ks)) return RK_ERR_INVALID_ARGUMENT;
    if (!PERM && (out == nullptr || !is_aligned(out, ks))) return RK_ERR_INVALID_ARGUMENT;
    if (n >= ((int64_t)1 << 31)) return RK_ERR_TOO_LARGE;
    hipStream_t st = (hipStream_t)stream;
    const int r = (rev ? SORT_REV : 0) | (PERM ? 0 : SORT_KEEP_NAN);
    switch ((int)dt) {
        case RK_F32: return sort_typed<float, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
        case RK_F64: return sort_typed<double, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
        case RK_I32: return sort_typed<int32_t, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
        case RK_I64: return sort_typed<int64_t, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
        case RK_F16: return sort_typed<half_bits, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
        default:     return sort_typed<int16_t, PERM>(keys, out, perm_out, n, r, tmp, tmp_bytes, st);
    }
}

// No kernel of the sort waits for another workgroup, so there is no give-up to report.
extern "C" int32_t rk_sort_status(const void* tmp, size_t tmp_bytes, void* stream) {
    if (tmp == nullptr) return RK_ERR_INVALID_ARGUMENT;
    if (!is_aligned(tmp, 256) || tmp_bytes < sizeof(SortCtl)) return RK_ERR_WORKSPACE;
    RK_HIP(hipStreamSynchronize((hipStream_t)stream));
    return RK_SUCCESS;
}

extern "C" int32_t rk_sort(rk_dtype dt, void* keys, int64_t n, int32_t rev, void* tmp, size_t tmp_bytes, void* stream) {
    return sort_dispatch<false>(dt, keys, keys, nullptr, n, rev, tmp, tmp_bytes, stream);
}

// The first pass that runs reads the caller's keys wherever they are, so a sorted copy needs no copy (sort(x) of Float32[2^26]
// 849 -> 753 us).
extern "C" int32_t rk_sort_to(rk_dtype dt, const void* keys, void* out, int64_t n, int32_t rev, void* tmp, size_t tmp_bytes, void* stream) {
    size_t ks = 0;
    if (n > 0 && keys != nullptr && out != nullptr && keys != out && sort_dtype_size((int)dt, &ks)) {
        const uintptr_t a = (uintptr_t)keys, b = (uintptr_t)out, bytes = (uintptr_t)n * ks;
        if (a < b + bytes && b < a + bytes) return RK_ERR_INVALID_ARGUMENT;          // the same array or none of it
    }
    return sort_dispatch<false>(dt, keys, out, nullptr, n, rev, tmp, tmp_bytes, stream);
}

extern "C" int32_t rk_sortperm(rk_dtype dt, const void* keys, int64_t* perm_out, int64_t n, int32_t rev, void* tmp, size_t tmp_bytes,
                               void* stream) {
    if (n > 0 && perm_out == nullptr) return RK_ERR_INVALID_ARGUMENT;
    return sort_dispatch<true>(dt, keys, nullptr, perm_out, n, rev, tmp, tmp_bytes, stream);
}
