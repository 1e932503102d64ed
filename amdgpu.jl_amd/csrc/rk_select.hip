// findall(::ROCArray{Bool}) in one pass over the mask: stream compaction with the chained look-back of the
// scan.  Replaces the cumsum + `_ker!` pair of src/kernels/indexing.jl:8-36 (9 bytes per element for the Int64
// cumsum, 9 more for the scatter) by 1 byte per element read plus the indices written.
#include <cstdlib>

#include "rk_common.hpp"
#include "rk_scan_impl.hpp"

namespace rk {

constexpr int SEL_CHUNK = WAVE * 16;                         // Bools one wave covers with one 16-byte load per lane

struct SelShape {
    int64_t s[RK_MAX_DIMS];
    int ndim;
};

// Writes the 1-based index of element `i` (0-based, column-major) as entry `pos` of ys.
template <bool LINEAR, bool SMALL>
__device__ __forceinline__ void emit_index(int64_t* __restrict__ ys, int64_t pos, int64_t i, const SelShape& shp) {
    if constexpr (LINEAR) {
        ys[pos] = i + 1;
    } else if constexpr (SMALL) {                            // every extent and the length fit 32 bits
        uint32_t rem = (uint32_t)i;
        for (int d = 0; d < shp.ndim; ++d) {
            const uint32_t e = (uint32_t)shp.s[d], q = rem / e;
            ys[pos * shp.ndim + d] = (int64_t)(rem - q * e) + 1;
            rem = q;
        }
    } else {
        int64_t rem = i;
        for (int d = 0; d < shp.ndim; ++d) {
            const int64_t q = rem / shp.s[d];
            ys[pos * shp.ndim + d] = rem - q * shp.s[d] + 1;
            rem = q;
        }
    }
}

// Persistent workgroups take tiles of SEL_NW * SEL_K * 1024 Bools in acquisition order (see scan_chain_kernel).
// A lane counts the set bytes of its SEL_K 16-byte loads, the counts are scanned across the wave (DPP) and the
// workgroup (LDS), the tile total is published and the tile's offset resolved by the two-level look-back.
// Output: per load, the lanes drop the in-chunk offsets of their set bytes into the wave's LDS strip at their
// scanned positions; the wave then reads the strip back in order and writes indices with coalesced stores (a
// lane writing its own run directly makes every store instruction touch 64 different lines: 4x slower at high
// density).  Only bit 0 of a byte is looked at (Julia's Bool).
// ORDERED: one workgroup per tile (its number from the launch order or, for grids beyond what is resident at once, from the
// counter: ordered_tile_id), the look-back and the end of the call as in scan_ordered_kernel
// (no tile counter, only the first tile of a group of 64 reads group descriptors, each on a line of its own).
// Set bytes of another tile, counted by the calling wave (the look-back's way out when that tile's workgroup is not
// there to publish its count: desc_lookback_alone).  Every tile in front of another is full.
template <int SEL_TILE> struct SelectTileCount {
    const uint8_t* bools;
    int aligned;
    __device__ __forceinline__ int64_t operator()(int64_t p) const {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const uint8_t* q = bools + p * (int64_t)SEL_TILE;
        int32_t c = 0;
        for (int i = lane_id() * 16; i < SEL_TILE; i += WAVE * 16) {
            if (aligned) {
                const u32x4 x = *(const u32x4*)(q + i) & 0x01010101u;
                c += __popc(x[0]) + __popc(x[1]) + __popc(x[2]) + __popc(x[3]);
            } else {
                for (int b = 0; b < 16; ++b) c += q[i + b] & 1;
            }
        }
        return (int64_t)wave_reduce(c, OpAdd());
    }
};

template <bool LINEAR, bool SMALL, int SEL_NW, int SEL_K, bool ORDERED>
__global__ __launch_bounds__(SEL_NW * WAVE) void findall_select_kernel(const uint8_t* __restrict__ bools, int64_t n, int64_t* __restrict__ ys,
                                                                       int64_t* __restrict__ count_out, SelShape shp, int aligned,
                                                                       unsigned long long* counter, uint32_t* tickets, int ticket_group,
                                                                       uint64_t* desc, int64_t ntiles, int64_t ngroups, int64_t desc_capacity,
                                                                       WaitCtl wc, WaitAlone wa, int dynamic_ids) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int SEL_TILE = SEL_NW * SEL_CHUNK * SEL_K;
    __shared__ uint16_t lds_strip[SEL_NW][SEL_CHUNK];
    __shared__ int32_t lds_wave[SEL_NW];
    __shared__ int64_t lds_prefix;
    __shared__ unsigned long long lds_id;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id();
    uint64_t* tile_desc = desc;                                          // [2 words][ntiles]
    uint64_t* group_desc = desc + (int64_t)Words<int64_t>::N * ntiles;   // [2 words][ngroups]; ORDERED: a line per group
    const OpAdd op;

    unsigned long long cur;
    if constexpr (ORDERED) {
        const OrderedId id = ordered_tile_id(counter, dynamic_ids, true);
        cur = ((unsigned long long)id.epoch << 32) | (unsigned long long)id.tile;
    } else {
        if (tid == 0) lds_id = __hip_atomic_fetch_add(counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        cur = lds_id;
    }
    while ((int64_t)(cur & 0xffffffffull) < ntiles) {
        const int64_t tile = (int64_t)(cur & 0xffffffffull);
        const uint32_t epoch = (uint32_t)(cur >> 32);
        wc.stamp = epoch;
        const int64_t e0 = tile * SEL_TILE;
        const int64_t left = n - e0;
        const int valid = left < SEL_TILE ? (int)left : SEL_TILE;
        const int woff = wave * (SEL_CHUNK * SEL_K) + lane * 16;
        // per 16-byte load: bit b of `hits` = byte b of the lane's 16 is set; `pk` packs the lane's first output
        // position inside the chunk (high half) with the hits (low half), so a tile costs one register per load
        uint32_t pk[SEL_K];
        int32_t ktot[SEL_K];                     // hits of the whole chunk (wave-uniform)
        int32_t carry = 0;
#pragma unroll
        for (int k0 = 0; k0 < SEL_K; k0 += 4) {
            u32x4 x[4];
            if (aligned && valid == SEL_TILE) {
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = load_nt((const u32x4*)(bools + e0 + woff + (k0 + k) * SEL_CHUNK));
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint32_t word = 0;
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            const int idx = woff + (k0 + k) * SEL_CHUNK + q * 4 + b;
                            if (idx < valid) word |= (uint32_t)bools[e0 + idx] << (8 * b);
                        }
                        x[k][q] = word;
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 4; k += 2) {
                // bit 0 of the 16 bytes -> a 16-bit mask in memory order: a dot product of the four bytes of a word with
                // (1, 2, 4, 8) or (16, 32, 64, 128) gathers four of them (a 32-bit multiply does too, at a quarter of
                // the rate).  The counts of two loads share one scan across the wave (a chunk holds at most 1024 hits).
                uint32_t hits[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const u32x4 b = x[k + h] & 0x01010101u;
                    const uint32_t lo = __builtin_amdgcn_udot4(b[1], 0x80402010u, __builtin_amdgcn_udot4(b[0], 0x08040201u, 0u, false), false);
                    const uint32_t hi = __builtin_amdgcn_udot4(b[3], 0x80402010u, __builtin_amdgcn_udot4(b[2], 0x08040201u, 0u, false), false);
                    hits[h] = lo | (hi << 8);
                }
                const int32_t c = (int32_t)(__popc(hits[0]) | ((uint32_t)__popc(hits[1]) << 16));
                const int32_t inc = wave_scan_inclusive(c, op, 0);
                const uint32_t exc = (uint32_t)(inc - c);
                pk[k0 + k] = (exc << 16) | hits[0];
                pk[k0 + k + 1] = (exc & 0xffff0000u) | hits[1];
                const uint32_t tot = (uint32_t)read_lane(inc, WAVE - 1);
                ktot[k0 + k] = (int32_t)(tot & 0xffffu);
                ktot[k0 + k + 1] = (int32_t)(tot >> 16);
                carry += ktot[k0 + k] + ktot[k0 + k + 1];
            }
        }
        if (lane == 0) lds_wave[wave] = carry;
        __syncthreads();
        int32_t wave_prefix = 0, tile_count = 0;
#pragma unroll
        for (int w = 0; w < SEL_NW; ++w) {
            const int32_t c = lds_wave[w];
            if (w < wave) wave_prefix += c;
            tile_count += c;
        }
        if (wave == 0) {
            int64_t tile_prefix = 0;
            if (lane == 0) desc_publish(tile_desc, ntiles, tile, (int64_t)tile_count, (epoch << 2) | DESC_A);
            if (tile > 0) {
                if constexpr (ORDERED) {
                    bool expired = false;
                    tile_prefix = desc_lookback_leader(tile_desc, ntiles, group_desc, tile, tile, tile >> 6, epoch, (int64_t)tile_count,
                                                       (int64_t)0, op, (int64_t)0, wc, wa, expired);
                    if (expired)
                        tile_prefix = desc_lookback_alone(tile_desc, ntiles, group_desc, tile, tile, tile >> 6, epoch, (int64_t)tile_count,
                                                          (int64_t)0, op, (int64_t)0, SelectTileCount<SEL_TILE>{bools, aligned}, wa.counter);
                } else
                    tile_prefix = desc_lookback2(tile_desc, ntiles, group_desc, ngroups, tile, tile, tile >> 6, epoch, (int64_t)tile_count,
                                                 (int64_t)0, op, (int64_t)0, wc);
            }
            if (lane == 0) {
                lds_prefix = tile_prefix;
                if (tile == ntiles - 1 && count_out != nullptr) *count_out = tile_prefix + tile_count;
            }
        }
        __syncthreads();
        int64_t base = lds_prefix + wave_prefix;
        // The hits of consecutive chunks share the strip while they fit (SEL_CHUNK entries; an entry is an offset from
        // the first chunk of the batch, < 16 * 1024): a sparse mask leaves in one round per wave instead of one per
        // chunk, each of which costs two LDS round trips.  fill, kbase: wave-uniform.
        uint16_t* strip = lds_strip[wave];
        int32_t fill = 0, kbase = 0;
        auto flush = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const int64_t i0 = e0 + wave * (SEL_CHUNK * SEL_K) + kbase * SEL_CHUNK;
            for (int i = lane; i < fill; i += WAVE) emit_index<LINEAR, SMALL>(ys, base + i, i0 + strip[i], shp);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();                              // the strip is reused by the next batch
            base += fill;
            fill = 0;
        };
#pragma unroll
        for (int k = 0; k < SEL_K; ++k) {
            if (ktot[k] == 0) continue;                                   // wave-uniform
            if (fill + ktot[k] > SEL_CHUNK) flush();
            if (fill == 0) kbase = k;
            int32_t p = fill + (int32_t)(pk[k] >> 16);
            const uint32_t rel = (uint32_t)((k - kbase) * SEL_CHUNK + lane * 16 - 1);
            for (uint32_t m = pk[k] & 0xffffu; m != 0u; m &= m - 1u) strip[p++] = (uint16_t)(rel + __ffs(m));
            fill += ktot[k];
        }
        if (fill > 0) flush();
        if constexpr (ORDERED) break;
        if (tid == 0) lds_id = __hip_atomic_fetch_add(counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        cur = lds_id;
    }
    if constexpr (ORDERED)
        ordered_finish((uint32_t)(cur >> 32), (int64_t)Words<int64_t>::N * ntiles + ngroups * GROUP_DESC_STRIDE, counter, tickets, ticket_group,
                       desc, desc_capacity);
    else
        chain_finish(cur, ntiles, (int64_t)Words<int64_t>::N * (ntiles + ngroups), counter, desc, desc_capacity);
}

__global__ void store_count_kernel(int64_t* p, int64_t v) { *p = v; }

// 16-byte loads per lane and tile (RK_SELECT_LOADS: 4, 8 or 16).  Measured on MI355X, 2^28 Bools, 1 % / 25 % / 100 %
// set, 8 waves in launch order: 4 loads 112 / 188 / 425 us, 8 loads 78 / 167 / 462 us, 16 loads 63 / 159 / 473 us: every
// tile costs about 10 ns whatever feeds it, so larger tiles win until the output dominates.
int tune_select_loads() {
    static const int v = [] { const char* s = std::getenv("RK_SELECT_LOADS"); const int x = s ? std::atoi(s) : 0; return (x == 4 || x == 8 || x == 16) ? x : 16; }();
    return v;
}
int tune_select_tile_ki() {
    static const int v = [] { const char* s = std::getenv("RK_SELECT_TILE_KI"); const int x = s ? std::atoi(s) : 0; return (x == 32 || x == 64 || x == 128) ? x : 0; }();
    return v;
}
int tune_select_blocks_per_cu() {
    static const int v = [] { const char* s = std::getenv("RK_SELECT_BLOCKS_PER_CU"); const int x = s ? std::atoi(s) : 0; return (x >= 1 && x <= 2) ? x : 2; }();
    return v;
}

// One workgroup of 8 waves per tile in launch order (1), or persistent workgroups of 16 waves fed by a tile counter (0).
// 2^26 / 2^28 Bools, 1 % / 25 % / 100 % set, 16 loads: ordered 22.7 / 39.4 / 122 us and 63 / 159 / 473 us, counter-fed
// 24.1 / 40.8 / 118 and 69 / 168 / 460 us (four workgroups a compute unit overlap their phases better than two; the
// look-back itself was not the limit: 16 waves in launch order measured 25 / 42 / 123 us).
int tune_select_ordered() {
    static const int v = [] { const char* s = std::getenv("RK_SELECT_ORDERED"); return s ? std::atoi(s) : 1; }();
    return v;
}

size_t findall_workspace_need(int64_t n) {
    const int64_t SEL_TILE = 8 * SEL_CHUNK * 4;                            // the smallest tile any configuration uses
    const int64_t ntiles = (n + SEL_TILE - 1) / SEL_TILE, ngroups = (ntiles + WAVE - 1) / WAVE;
    return ((size_t)ntiles * Words<int64_t>::N + (size_t)ngroups * GROUP_DESC_STRIDE) * sizeof(uint64_t);   // the ordered layout, the larger
}

}  // namespace rk

using namespace rk;

extern "C" int32_t rk_findall(const uint8_t* bools, int ndim, const int64_t* shape, int64_t* ys, int64_t* count_out, void* ws,
                              size_t ws_bytes, void* stream) {
    if (ndim < 0 || ndim > RK_MAX_DIMS || (ndim > 0 && shape == nullptr)) return RK_ERR_INVALID_ARGUMENT;
    SelShape shp{};
    shp.ndim = ndim;
    int64_t n = 1;
    bool small = true;
    for (int d = 0; d < RK_MAX_DIMS; ++d) {
        shp.s[d] = d < ndim ? shape[d] : 1;
        if (shp.s[d] < 0) return RK_ERR_INVALID_ARGUMENT;
        if (shp.s[d] != 0 && n > INT64_MAX / shp.s[d]) return RK_ERR_INVALID_ARGUMENT;
        n *= shp.s[d];
    }
    if (n == 0) {
        if (count_out != nullptr) {
            store_count_kernel<<<1, 1, 0, (hipStream_t)stream>>>(count_out, 0);
            RK_LAUNCH_CHECK();
        }
        return RK_SUCCESS;
    }
    if (bools == nullptr || ys == nullptr) return RK_ERR_INVALID_ARGUMENT;
    if (n > 0xffffffffll) small = false;
    const bool ordered = tune_select_ordered() != 0;
    int nw = 16, kl = tune_select_loads();
    if (ordered) {
        // Tiles of 32, 64 or 128 Ki Bools (RK_SELECT_TILE_KI forces one): a small mask in large tiles leaves most compute
        // units idle behind a chain of a few tiles.  25 % set, back to back: 2^21 Bools 9.6 / 12.1 / 16.5 us, 2^24
        // 17.0 / 17.7 / 22.7, 2^25 24.2 / 24.0 / 24.7, 2^26 43.7 / 44.1 / 39.2, 2^27 89.9 / 87.6 / 82.8 (16 Ki: no better)
        int ki = tune_select_tile_ki();
        if (ki == 0) ki = n <= ((int64_t)1 << 24) ? 32 : n <= ((int64_t)1 << 25) ? 64 : 128;
        nw = 8;
        kl = ki == 128 ? 16 : ki == 64 ? 8 : 4;
    }
    const int64_t SEL_TILE = (int64_t)nw * SEL_CHUNK * kl;
    const int64_t ntiles = (n + SEL_TILE - 1) / SEL_TILE, ngroups = (ntiles + WAVE - 1) / WAVE;
    if (ntiles > 0x3fffffff) return RK_ERR_TOO_LARGE;
    Workspace w{};
    if (!carve_workspace(ws, ws_bytes, findall_workspace_need(n), &w)) return RK_ERR_WORKSPACE;
    const int64_t cap = (int64_t)(w.desc_bytes / sizeof(uint64_t));
    int64_t grid = (int64_t)device_info().cus * tune_select_blocks_per_cu();
    if (grid > ntiles || ordered) grid = ntiles;
    const int tg = ordered_ticket_group(ntiles);
    unsigned long long* counter = (unsigned long long*)&w.hdr->scan_counter;
    const int aligned = is_aligned(bools, 16) ? 1 : 0;
    const WaitCtl wc = wait_ctl(w.hdr);
    const int dyn = ordered ? ordered_dynamic_ids(ntiles, nw * WAVE, true) : 0;
    hipStream_t st = (hipStream_t)stream;
#define RK_SELECT3(LIN, SM, NWW, KK, ORD)                                                                                        \
    findall_select_kernel<LIN, SM, NWW, KK, ORD><<<(unsigned)grid, NWW * WAVE, 0, st>>>(bools, n, ys, count_out, shp, aligned,      \
                                                                                        counter, w.tickets, tg, w.desc, ntiles,    \
                                                                                        ngroups, cap, wc, wait_alone(w.hdr), dyn)
#define RK_SELECT2(LIN, SM, KK)                                                                                                  \
    do {                                                                                                                         \
        if (!ordered) RK_SELECT3(LIN, SM, 16, KK, false);                                                                        \
        else RK_SELECT3(LIN, SM, 8, KK, true);                                                                                   \
    } while (0)
#define RK_SELECT(LIN, SM)                                                                                                       \
    do {                                                                                                                         \
        if (kl == 4) RK_SELECT2(LIN, SM, 4);                                                                                     \
        else if (kl == 8) RK_SELECT2(LIN, SM, 8);                                                                                \
        else RK_SELECT2(LIN, SM, 16);                                                                                            \
    } while (0)
    if (ndim <= 1) RK_SELECT(true, true);
    else if (small) RK_SELECT(false, true);
    else RK_SELECT(false, false);
#undef RK_SELECT
#undef RK_SELECT2
#undef RK_SELECT3
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

// ---- x[.., indices]: the gather behind logical indexing ------------------------------------------------------------
// y[i, j] = x[i, idx[j] - 1] for i < inner: `x[mask]`, `x[:, mask]`, `x[:, :, mask]` (test/hip_rocarray/indexing.jl:5-18)
// after Base.to_index has turned the mask into findall(mask) (src/kernels/indexing.jl:1).  Elements are opaque.
namespace rk {

template <typename E> struct GatherElem { typedef E type; };
struct Bytes16 { uint64_t lo, hi; };

template <typename E>
__global__ __launch_bounds__(256) void gather_slices_kernel(const E* __restrict__ x, const int64_t* __restrict__ idx, E* __restrict__ y,
                                                            int64_t inner, int64_t total, int64_t nsrc) {
    const int64_t f = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (f >= total) return;
    int64_t i = 0, j = f;
    if (inner != 1) { j = f / inner; i = f - j * inner; }
    const int64_t s = idx[j] - 1;
    if (s < 0 || s >= nsrc) return;          // an index outside x selects nothing (the caller checks bounds)
    y[f] = x[s * inner + i];
}

}  // namespace rk

extern "C" int32_t rk_gather_slices(const void* x, const int64_t* idx, void* y, size_t elsize, int64_t inner, int64_t nidx, int64_t nsrc,
                                    void* stream) {
    if (inner < 0 || nidx < 0 || nsrc < 0) return RK_ERR_INVALID_ARGUMENT;
    if (elsize != 1 && elsize != 2 && elsize != 4 && elsize != 8 && elsize != 16) return RK_ERR_UNSUPPORTED;
    if (inner == 0 || nidx == 0) return RK_SUCCESS;
    if (x == nullptr || idx == nullptr || y == nullptr) return RK_ERR_INVALID_ARGUMENT;
    const size_t align = elsize < 16 ? elsize : 8;
    if (!is_aligned(x, align) || !is_aligned(y, align)) return RK_ERR_INVALID_ARGUMENT;
    if (nidx > INT64_MAX / inner) return RK_ERR_TOO_LARGE;
    const int64_t total = inner * nidx, blocks = (total + 255) / 256;
    if (blocks > 0x7fffffff) return RK_ERR_TOO_LARGE;
    hipStream_t st = (hipStream_t)stream;
#define RK_GATHER(E) rk::gather_slices_kernel<E><<<(unsigned)blocks, 256, 0, st>>>((const E*)x, idx, (E*)y, inner, total, nsrc)
    switch (elsize) {
        case 1: RK_GATHER(uint8_t); break;
        case 2: RK_GATHER(uint16_t); break;
        case 4: RK_GATHER(uint32_t); break;
        case 8: RK_GATHER(uint64_t); break;
        default: RK_GATHER(rk::Bytes16); break;
    }
#undef RK_GATHER
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

// ---- x[mask] ------------------------------------------------------------------------------------------------------
// The length of the result has to be known before it can be allocated; what the count leaves behind makes the rest a plain
// streaming kernel, which does not read the mask again (rk_mask_count_bits, rk_mask_select_bits; the entry points with the smaller
// temporary read it twice):
//   mask_count_kernel    set bytes of every tile of 4096 Bools (one wave), as exclusive prefixes inside groups of tiles,
//                        the exclusive prefixes of the groups (the workgroup that finishes last scans them), and the mask, a bit a Bool
//   mask_select_kernel, mask_select_dense_kernel
//                        a wave per tile: its first output slot is two loads away, so there is no look-back, no barrier
//                        and nothing to wait for; selected elements go from x to y without an index in between
// Bound by memory: the mask, the lines of x that hold a selected element, and the result.  Before, this was a u8 -> Int64 reduction,
// the one-pass findall and a gather by its Int64 indices (16 bytes of index traffic per selected element): Float32[2^26], 25 %
// set, the whole call 193 -> 113 us.  Bits instead of the mask bytes for the second kernel, and a count whose loads do not stay in
// the caches (where they push out what the call before has written), us a call of 2^26 at 1, 25, 50 and 90 %:
//   bytes twice       Float32 53 95 105 130, Int64 54 149 184 250     (5 us of these the wait for the stream instead of the count)
//   bits              Float32 46 84  96 127, Int64 47 141 190 239
//   and so            Float32 42 84  95 111, Int64 43 140 162 240
namespace rk {

constexpr int MSK_TILE = 4096, MSK_LOADS = MSK_TILE / SEL_CHUNK;
constexpr int MSK_BLOCK = 1024, MSK_WAVES = MSK_BLOCK / WAVE;

// Tiles per group, i.e. per workgroup of the count: 16 (one a wave) keeps the chip busy down to short masks, 64 keeps the
// number of group totals that one workgroup scans at the end small.  Float32, 16 / 32 / 64, us a call at 25 %: 2^24 32.9 / 33.1 / 33.1,
// 2^25 58.1 / 56.0 / 57.2, 2^26 88.7 / 85.8 / 84.3.
inline int msk_group_shift(int64_t n) { return n <= ((int64_t)1 << 24) ? 4 : n <= ((int64_t)1 << 25) ? 5 : 6; }
struct MaskTmp {
    int64_t ntiles, ngroups;
    size_t tile_off, bits_off, bytes, bits_bytes;          // [group prefixes: Int64][tile prefixes: UInt32][a bit a Bool: 64 words of 64 a tile]
};
inline MaskTmp mask_tmp(int64_t n) {
    MaskTmp m;
    m.ntiles = (n + MSK_TILE - 1) / MSK_TILE;
    m.ngroups = (m.ntiles + (1 << msk_group_shift(n)) - 1) >> msk_group_shift(n);
    m.tile_off = ((size_t)m.ngroups * sizeof(int64_t) + 255) & ~(size_t)255;
    m.bits_off = m.tile_off + (((size_t)m.ntiles * sizeof(uint32_t) + 255) & ~(size_t)255);
    m.bytes = m.bits_off;                                               // (without the bits)
    m.bits_bytes = (size_t)m.ntiles * (MSK_TILE / 8);
    return m;
}

// 16 Bools at `i`, zeros beyond n.  A whole vector wherever one fits: only the vector that the array's end cuts (and every
// vector of a mask at an odd address) goes byte by byte, and then all of its loads are issued before the first is used.
typedef uint32_t mask_vec __attribute__((ext_vector_type(4)));
__device__ __forceinline__ mask_vec mask_load16(const uint8_t* __restrict__ mask, int64_t i, int64_t n, int aligned) {
    mask_vec v = {0u, 0u, 0u, 0u};
    if (aligned && i + 16 <= n) return *(const mask_vec*)(mask + i);
    if (i >= n) return v;
    uint32_t b[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) b[j] = mask[i + j < n ? i + j : n - 1];
#pragma unroll
    for (int j = 0; j < 16; ++j)
        if (i + j < n) v[j / 4] |= b[j] << (8 * (j % 4));
    return v;
}

// Bit 0 of 16 bytes, in order.
__device__ __forceinline__ uint32_t mask_bits16(const mask_vec& v) {
    const mask_vec b = v & 0x01010101u;
    const uint32_t lo = __builtin_amdgcn_udot4(b[1], 0x80402010u, __builtin_amdgcn_udot4(b[0], 0x08040201u, 0u, false), false);
    const uint32_t hi = __builtin_amdgcn_udot4(b[3], 0x80402010u, __builtin_amdgcn_udot4(b[2], 0x08040201u, 0u, false), false);
    return lo | (hi << 8);
}

// What lane l reads of a tile by its four loads, Bools k * 1024 + 16 l ... of the tile, 16 bits each: word l of the tile's bits.
__device__ __forceinline__ uint64_t mask_word(const mask_vec (&x)[MSK_LOADS]) {
    static_assert(MSK_LOADS == 4, "");
    return (uint64_t)(mask_bits16(x[2]) | mask_bits16(x[3]) << 16) << 32 | (mask_bits16(x[0]) | mask_bits16(x[1]) << 16);
}

// BITS: the words stay behind, and nothing reads the mask again.
template <int TPW, bool BITS>        // TPW: tiles per wave
__global__ __launch_bounds__(MSK_BLOCK) void mask_count_kernel(const uint8_t* __restrict__ mask, int64_t n, int aligned, int64_t ntiles,
                                                               uint32_t* __restrict__ tile_prefix, uint64_t* __restrict__ bits, int64_t* group_prefix,
                                                               int64_t* count_out, uint32_t* tickets, int ticket_group) {
    __shared__ uint32_t lds_count[MSK_WAVES * TPW];
    __shared__ int64_t lds_wave[MSK_WAVES];
    __shared__ int lds_last;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id();
    const OpAdd op;
    const int64_t first = (int64_t)blockIdx.x * (MSK_WAVES * TPW);
    uint32_t c[TPW];
    mask_vec x[TPW][MSK_LOADS];
    if (aligned && (first + MSK_WAVES * TPW) * MSK_TILE <= n) {
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int k = 0; k < MSK_LOADS; ++k)
            {
                const mask_vec* const from = (const mask_vec*)(mask + (first + wave * TPW + t) * MSK_TILE + k * SEL_CHUNK + lane * 16);
                x[t][k] = BITS ? load_nt(from) : *from;
            }
    } else {
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int k = 0; k < MSK_LOADS; ++k)
                x[t][k] = mask_load16(mask, (first + wave * TPW + t) * MSK_TILE + k * SEL_CHUNK + lane * 16, n, aligned);
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const uint64_t b = mask_word(x[t]);
        const int64_t tile = first + wave * TPW + t;
        c[t] = (uint32_t)__popcll(b);
        if (BITS && tile < ntiles) bits[tile * WAVE + lane] = b;
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const uint32_t s = wave_reduce(c[t], op);
        if (lane == 0) lds_count[wave * TPW + t] = s;
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t v = lane < MSK_WAVES * TPW ? lds_count[lane] : 0u;
        const uint32_t inc = wave_scan_inclusive(v, op, 0u);
        if (lane < MSK_WAVES * TPW && first + lane < ntiles) tile_prefix[first + lane] = inc - v;
        if (lane == WAVE - 1) {
            // two levels of completion tickets, as in the reductions: atomics on one address take 14 ns each
            store_agent(group_prefix + blockIdx.x, (int64_t)inc);
            publish_barrier();
            const int64_t nb = gridDim.x, ng = (nb + ticket_group - 1) / ticket_group, grp = blockIdx.x / ticket_group;
            const uint32_t gsize = (uint32_t)(grp == ng - 1 ? nb - grp * ticket_group : ticket_group);
            int last = 0;
            uint32_t* gt = tickets + grp * TICKET_STRIDE;
            if (__hip_atomic_fetch_add(gt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gsize - 1u) {
                *gt = 0;
                uint32_t* lt = tickets + ng * TICKET_STRIDE;
                if (__hip_atomic_fetch_add(lt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)ng - 1u) {
                    *lt = 0;
                    last = 1;
                }
            }
            lds_last = last;
        }
    }
    __syncthreads();
    if (!lds_last) return;
    // the last one: exclusive scan of the group totals, MSK_BLOCK at a time
    int64_t carry = 0;
    for (int64_t g0 = 0; g0 < (int64_t)gridDim.x; g0 += MSK_BLOCK) {
        const int64_t g = g0 + tid;
        const int64_t v = g < (int64_t)gridDim.x ? load_agent(group_prefix + g) : 0;
        const int64_t inc = wave_scan_inclusive(v, op, (int64_t)0);
        if (lane == WAVE - 1) lds_wave[wave] = inc;
        __syncthreads();
        int64_t before = carry;
        for (int w = 0; w < MSK_WAVES; ++w) {
            const int64_t t = lds_wave[w];
            if (w < wave) before += t;
            carry += t;
        }
        if (g < (int64_t)gridDim.x) group_prefix[g] = before + inc - v;
        __syncthreads();
    }
    if (tid == 0) *count_out = carry;
}

// The lane's word of a tile, from the bits of the count or from the mask.
template <bool BITS> __device__ __forceinline__ uint64_t mask_tile_word(const void* __restrict__ mask, int64_t n, int aligned, int64_t tile, int lane) {
    if constexpr (BITS) return ((const uint64_t*)mask)[tile * WAVE + lane];
    const uint8_t* const bytes = (const uint8_t*)mask;
    const int64_t e0 = tile * MSK_TILE + lane * 16;
    typedef uint32_t mask_vec_at4 __attribute__((ext_vector_type(4), aligned(4)));
    mask_vec m[MSK_LOADS];
    if (aligned && tile * MSK_TILE + MSK_TILE <= n) {       // (to 4 bytes)
#pragma unroll
        for (int k = 0; k < MSK_LOADS; ++k) m[k] = (mask_vec)__builtin_nontemporal_load((const mask_vec_at4*)(bytes + e0 + k * SEL_CHUNK));
    } else {
#pragma unroll
        for (int k = 0; k < MSK_LOADS; ++k) {
            const int64_t i = e0 + k * SEL_CHUNK;
            m[k] = aligned && i + 16 <= n ? (mask_vec)__builtin_nontemporal_load((const mask_vec_at4*)(bytes + i)) : mask_load16(bytes, i, n, 0);
        }
    }
    return mask_word(m);
}

// A wave per tile.  The set positions of the tile are listed in LDS (strip; the lanes' hits are ranked by one scan for every
// two loads), then every lane takes every 64th of them: loads of x walk forward over the tile, stores are whole lines.
// A list of the tile's hits and not a masked store per 64 elements: at 25 % set that is a quarter of the loads and stores.
template <typename E, bool BITS>
__global__ __launch_bounds__(256) void mask_select_kernel(const void* __restrict__ mask, int64_t n, int aligned, const E* __restrict__ x,
                                                          E* __restrict__ y, int64_t nsel, int64_t ntiles,
                                                          const uint32_t* __restrict__ tile_prefix, const int64_t* __restrict__ group_prefix,
                                                          int group_shift) {
    constexpr int STRIP = 2048, GATHER = 4;              // list entries a wave holds; elements a lane has in flight
    __shared__ uint16_t lds_strip[256 / WAVE][STRIP];
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const OpAdd op;
    const int64_t tile = (int64_t)blockIdx.x * (256 / WAVE) + wave;
    if (tile >= ntiles) return;
    const int64_t e0 = tile * MSK_TILE;
    const uint64_t m = mask_tile_word<BITS>(mask, n, aligned, tile, lane);
    int64_t base = group_prefix[tile >> group_shift] + (int64_t)tile_prefix[tile];
    const E* src = x + e0;
    uint16_t* strip = lds_strip[wave];
    int fill = 0;
    auto flush = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int i = lane; i < fill; i += GATHER * WAVE) {
            E v[GATHER];
#pragma unroll
            for (int u = 0; u < GATHER; ++u) {           // unconditional: past the end the last entry is read again
                const int j = i + u * WAVE;
                v[u] = src[strip[j < fill ? j : fill - 1]];
            }
#pragma unroll
            for (int u = 0; u < GATHER; ++u) {
                const int j = i + u * WAVE;
                if (j < fill && base + j < nsel) y[base + j] = v[u];      // nsel: a mask that changed since the count stays in bounds
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        base += fill;
        fill = 0;
    };
#pragma unroll
    for (int k0 = 0; k0 < MSK_LOADS; k0 += 2) {
        const uint32_t hits[2] = {(uint32_t)(m >> (16 * k0)) & 0xffffu, (uint32_t)(m >> (16 * k0 + 16)) & 0xffffu};
        const int32_t c = (int32_t)(__popc(hits[0]) | ((uint32_t)__popc(hits[1]) << 16));
        const int32_t inc = wave_scan_inclusive(c, op, 0);
        const uint32_t exc = (uint32_t)(inc - c), tot = (uint32_t)read_lane(inc, WAVE - 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int t = (int)(h == 0 ? tot & 0xffffu : tot >> 16);
            if (fill + t > STRIP) flush();
            int p = fill + (int)(h == 0 ? exc & 0xffffu : exc >> 16);
            const uint32_t rel = (uint32_t)((k0 + h) * SEL_CHUNK + lane * 16 - 1);
            for (uint32_t b = hits[h]; b != 0u; b &= b - 1u) strip[p++] = (uint16_t)(rel + __ffs(b));
            fill += t;
        }
    }
    if (fill > 0) flush();
}

// Where most lines of x hold a selected element anyway (4- and 8-byte elements): x is read 16 bytes a lane, where the bits of the
// same elements have a hit, so that no load waits for a list, and the selected ones are put together in LDS.  A step is four such
// loads; those of the next are issued before a step is worked on (two steps ahead: no faster).  The bits are read first, all of the tile's:
// where hits are clustered, most lines of x hold none.  Bound by memory.  (The result 16 bytes a lane instead of one element: Float32[2^26]
// 90 % 111.6 -> 108.9, else the same; nontemporal as well: 25 % 84.7 -> 89.2, 90 % 128.)
// The whole call, by list of hits -> so, both reading mask bytes instead of bits, us: Float32[2^26] 10 % 91 -> 88, 25 % 108.5 -> 95, 50 % 129 -> 105, 90 % 170 -> 131; Int64[2^26] 25 %
// 178 -> 149, 90 % 268 -> 250; every hit of Int64[2^26] in the first quarter 85.2 -> 84.3, in runs of 13 of 100 tiles 80.2 -> 75.5 (x read
// whole, beside its mask bytes: 150 and 145).  (Loads that stay in the caches instead of nontemporal ones: Float32[2^26] 25 % 106.5, 90 % 143.)
template <typename E, bool BITS>
__global__ __launch_bounds__(256) void mask_select_dense_kernel(const void* __restrict__ mask, int64_t n, const E* __restrict__ x, E* __restrict__ y,
                                                                int64_t nsel, int64_t ntiles, const uint32_t* __restrict__ tile_prefix,
                                                                const int64_t* __restrict__ group_prefix, int group_shift) {
    constexpr int V = 16 / (int)sizeof(E), LOADS = 4, STEP = LOADS * WAVE * V, STEPS = MSK_TILE / STEP;
    typedef E vec __attribute__((ext_vector_type(V)));
    struct Loaded { vec x[LOADS]; };
    __shared__ alignas(16) E lds_strip[256 / WAVE][STEP];
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const int64_t tile = (int64_t)blockIdx.x * (256 / WAVE) + wave;
    if (tile >= ntiles) return;
    const int64_t e0 = tile * MSK_TILE;
    E* const strip = lds_strip[wave];
    auto wave_sync = [] {                                   // what the lanes of the wave wrote to LDS is there for all of them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // Load k of a lane is elements (k * 64 + lane) * V ...: their bits are the lowest V of a 16 of one of the words that it takes.
    constexpr int WORDS = 16 / V;
    static_assert(WORDS * WAVE * V == SEL_CHUNK, "as many loads of x for the 1024 Bools of a load as words");
    uint64_t w[WORDS];
#pragma unroll
    for (int q = 0; q < WORDS; ++q) w[q] = BITS ? ((const uint64_t*)mask)[tile * WAVE + q * (WAVE / WORDS) + lane / WORDS] : 0ull;
    int64_t base = group_prefix[tile >> group_shift] + (int64_t)tile_prefix[tile];
    if constexpr (!BITS) {                                  // the words change lanes in the strip
        uint64_t* const words = (uint64_t*)strip;
        words[lane] = mask_tile_word<false>(mask, n, 1, tile, lane);
        wave_sync();
#pragma unroll
        for (int q = 0; q < WORDS; ++q) w[q] = words[q * (WAVE / WORDS) + lane / WORDS];
        wave_sync();
    }
#pragma unroll
    for (int q = 0; q < WORDS; ++q) w[q] >>= lane % WORDS * V;
    uint64_t any = 0u;
#pragma unroll
    for (int q = 0; q < WORDS; ++q) any |= w[q];
    any &= 0x0001000100010001ull * ((1u << V) - 1u);
    if (__ballot(any != 0u) == 0ull) return;
    auto m = [&](int k) { return (uint32_t)(w[k % WORDS] >> (k / WORDS * 16)) & ((1u << V) - 1u); };
    auto load = [&](Loaded& l, int s) {
#pragma unroll
        for (int g = 0; g < LOADS; ++g) {
            const int k = s * LOADS + g;
            const int64_t i = e0 + k * (WAVE * V) + lane * V;
            if (m(k) == 0u) continue;
            if (i + V <= n) {
                l.x[g] = load_nt((const vec*)(x + i));
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (i + j < n) l.x[g][j] = x[i + j];
            }
        }
    };
    Loaded cur;
    load(cur, 0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        Loaded next;
        if (s + 1 < STEPS) load(next, s + 1);
        // hits of a lane, a byte a load; of the lanes in front they are 252 at most, so the bytes of the sum do not meet
        uint32_t c = 0u;
#pragma unroll
        for (int g = 0; g < LOADS; ++g) c |= (uint32_t)__popc(m(s * LOADS + g)) << (8 * g);
        const uint32_t exc = wave_scan_inclusive(c, OpAdd(), 0u) - c;
        const uint32_t front = (uint32_t)read_lane((int32_t)exc, WAVE - 1), own = (uint32_t)read_lane((int32_t)c, WAVE - 1);
        uint32_t fill = 0u;
#pragma unroll
        for (int g = 0; g < LOADS; ++g) {
            uint32_t p = fill + ((exc >> (8 * g)) & 0xffu);
#pragma unroll
            for (int j = 0; j < V; ++j) {
                if ((m(s * LOADS + g) >> j) & 1u) strip[p++] = cur.x[g][j];
            }
            fill += ((front >> (8 * g)) & 0xffu) + ((own >> (8 * g)) & 0xffu);
        }
        wave_sync();
        for (uint32_t i = lane; i < fill; i += WAVE)
            if (base + i < nsel) y[base + i] = strip[i];    // nsel: a mask that changed since the count stays in bounds
        wave_sync();
        base += fill;
        if (s + 1 < STEPS) cur = next;
    }
}

}  // namespace rk

namespace rk {

template <bool BITS>
static int32_t mask_count(const uint8_t* mask, int64_t n, int64_t* count_out, void* tmp, size_t tmp_bytes, void* ws, size_t ws_bytes, hipStream_t st) {
    if (n < 0 || count_out == nullptr) return RK_ERR_INVALID_ARGUMENT;
    if (n == 0) {
        store_count_kernel<<<1, 1, 0, st>>>(count_out, 0);
        RK_LAUNCH_CHECK();
        return RK_SUCCESS;
    }
    if (mask == nullptr) return RK_ERR_INVALID_ARGUMENT;
    const MaskTmp t = mask_tmp(n);
    Workspace w{};
    if (tmp == nullptr || !is_aligned(tmp, 256) || tmp_bytes < t.bytes + (BITS ? t.bits_bytes : 0) || !carve_workspace(ws, ws_bytes, 0, &w)) return RK_ERR_WORKSPACE;
    const int tg = ordered_ticket_group(t.ngroups);
    if (t.ngroups > 0x7fffffff) return RK_ERR_TOO_LARGE;
    const int aligned = is_aligned(mask, 16) ? 1 : 0;
    int64_t* gp = (int64_t*)tmp;
    uint32_t* tp = (uint32_t*)((char*)tmp + t.tile_off);
    uint64_t* bits = (uint64_t*)((char*)tmp + t.bits_off);
#define RK_MCOUNT(TPW) mask_count_kernel<TPW, BITS><<<(unsigned)t.ngroups, MSK_BLOCK, 0, st>>>(mask, n, aligned, t.ntiles, tp, bits, gp, count_out, w.tickets, tg)
    switch (msk_group_shift(n)) {
        case 4: RK_MCOUNT(1); break;
        case 5: RK_MCOUNT(2); break;
        default: RK_MCOUNT(4); break;
    }
#undef RK_MCOUNT
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

template <bool BITS>
static int32_t mask_select(const uint8_t* mask, int64_t n, const void* x, void* y, size_t elsize, int64_t nsel, const void* tmp, size_t tmp_bytes, hipStream_t st) {
    if (n < 0 || nsel < 0) return RK_ERR_INVALID_ARGUMENT;
    if (elsize != 1 && elsize != 2 && elsize != 4 && elsize != 8 && elsize != 16) return RK_ERR_UNSUPPORTED;
    if (n == 0 || nsel == 0) return RK_SUCCESS;
    if ((!BITS && mask == nullptr) || x == nullptr || y == nullptr) return RK_ERR_INVALID_ARGUMENT;
    const size_t align = elsize < 16 ? elsize : 8;
    if (!is_aligned(x, align) || !is_aligned(y, align)) return RK_ERR_INVALID_ARGUMENT;
    const MaskTmp t = mask_tmp(n);
    if (tmp == nullptr || !is_aligned(tmp, 256) || tmp_bytes < t.bytes + (BITS ? t.bits_bytes : 0)) return RK_ERR_WORKSPACE;
    const int64_t blocks = (t.ntiles + 3) / 4;
    if (blocks > 0x7fffffff) return RK_ERR_TOO_LARGE;
    const int64_t* gp = (const int64_t*)tmp;
    const uint32_t* tp = (const uint32_t*)((const char*)tmp + t.tile_off);
    const void* from = BITS ? (const void*)((const char*)tmp + t.bits_off) : mask;
    const int aligned = is_aligned(mask, 4) ? 1 : 0;         // (of a mask that is read)
    const int shift = msk_group_shift(n);
    // The less of x comes from the Infinity Cache, the earlier reading it 16 bytes a lane pays.  By list of hits / so, us a call at 3, 6, 10, 25, 40
    // and 60 % at random, from bits: Float32[2^26] 62/61 76/71 83/78 96/85 107/91 123/99, Int64[2^26] 69/75 100/94 126/113 167/141 184/150 210/204;
    // 128 MiB: Float32[2^25] 35/39 46/44 49/48 55/51 58/54 64/58, Int64[2^24] 29/32 34/36 41/42 53/51 56/53 58/57; 64 MiB: Float32[2^24] 27/27 29/29
    // 30/32 33/34 35/35 44/38; Float32[2^22] and less the same until 40 %, at 90 % 33 and 29.
    // From mask bytes: Float32[2^24] 10 % 36.7 by list and 40.4, 25 % 39.0 and 41.3, 50 % 45.0 and 44.5; Int64[2^24] 43.9 and 52.7, 56.1 and 55.6,
    // 62.8 and 61.2; beyond 128 MiB an eighth is the line (7 %: Float32[2^26] 86.7 and 86.3, Int64[2^26] 118 and 136; 10 %: 91 and 88, 139 and 139).
    const uint64_t x_bytes = (uint64_t)n * elsize, mib128 = (uint64_t)1 << 27;
    const int64_t line = BITS ? (x_bytes > mib128 ? n / 16 : x_bytes > mib128 / 2 ? n / 8 : n / 2) : x_bytes > mib128 ? n / 8 : n / 4 * 3;
    if ((elsize == 4 || elsize == 8) && nsel >= line && is_aligned(x, 16) && (BITS || aligned)) {
        if (elsize == 4) mask_select_dense_kernel<uint32_t, BITS><<<(unsigned)blocks, 256, 0, st>>>(from, n, (const uint32_t*)x, (uint32_t*)y, nsel, t.ntiles, tp, gp, shift);
        else mask_select_dense_kernel<uint64_t, BITS><<<(unsigned)blocks, 256, 0, st>>>(from, n, (const uint64_t*)x, (uint64_t*)y, nsel, t.ntiles, tp, gp, shift);
        RK_LAUNCH_CHECK();
        return RK_SUCCESS;
    }
#define RK_MSEL(E) mask_select_kernel<E, BITS><<<(unsigned)blocks, 256, 0, st>>>(from, n, aligned, (const E*)x, (E*)y, nsel, t.ntiles, tp, gp, shift)
    switch (elsize) {
        case 1: RK_MSEL(uint8_t); break;
        case 2: RK_MSEL(uint16_t); break;
        case 4: RK_MSEL(uint32_t); break;
        case 8: RK_MSEL(uint64_t); break;
        default: RK_MSEL(Bytes16); break;
    }
#undef RK_MSEL
    RK_LAUNCH_CHECK();
    return RK_SUCCESS;
}

}  // namespace rk

extern "C" size_t rk_mask_tmp_bytes(int64_t n) { return n <= 0 ? 256 : mask_tmp(n).bytes; }

extern "C" int32_t rk_mask_count(const uint8_t* mask, int64_t n, int64_t* count_out, void* tmp, size_t tmp_bytes, void* ws, size_t ws_bytes,
                                 void* stream) {
    return mask_count<false>(mask, n, count_out, tmp, tmp_bytes, ws, ws_bytes, (hipStream_t)stream);
}

extern "C" int32_t rk_mask_select(const uint8_t* mask, int64_t n, const void* x, void* y, size_t elsize, int64_t nsel, const void* tmp,
                                  size_t tmp_bytes, void* stream) {
    return mask_select<false>(mask, n, x, y, elsize, nsel, tmp, tmp_bytes, (hipStream_t)stream);
}

extern "C" size_t rk_mask_bits_tmp_bytes(int64_t n) { return n <= 0 ? 256 : mask_tmp(n).bytes + mask_tmp(n).bits_bytes; }

extern "C" int32_t rk_mask_count_bits(const uint8_t* mask, int64_t n, int64_t* count_out, void* tmp, size_t tmp_bytes, void* ws, size_t ws_bytes,
                                      void* stream) {
    return mask_count<true>(mask, n, count_out, tmp, tmp_bytes, ws, ws_bytes, (hipStream_t)stream);
}

extern "C" int32_t rk_mask_select_bits(int64_t n, const void* x, void* y, size_t elsize, int64_t nsel, const void* tmp, size_t tmp_bytes,
                                       void* stream) {
    return mask_select<true>(nullptr, n, x, y, elsize, nsel, tmp, tmp_bytes, (hipStream_t)stream);
}
