// Stable LSD counting sort (radix 256) of 32-bit keys on gfx950, with the input positions as values.
//
// Each pass sorts by one 8-bit digit and keeps the previous order among equal digits, so
// the composition over ceil(bits/8) passes equals a stable sort by the whole key
// (std::stable_sort by key, bit for bit).  A pass:
//   hist     one workgroup per tile of keys: digit counts
//   scan     per digit, exclusive scan of its counts over the tiles (small sorts: in the scatter)
//   scatter  each tile re-ranks its keys in input order and writes key/value to its final slot
// A wave takes a run of consecutive keys, 64 at a time, and finds the lanes that share its digit by
// one ballot per digit bit, whatever the keys (a walk over the distinct digits costs one round each:
// keys in random order have up to 64 of them).  Its running counts per digit stay in its own LDS row,
// so the 64-key rounds need no barrier.
//
// Measured per pass, hist / scatter: 1,048,576 keys in random order 74 / 80 -> 8.0 / 16 us;
// 150,000 nearly sorted keys 15 / 20 -> 3.4 / 4.8 us, 19,600 9.2 / 12.4 -> 3.4 / 5.9 us (its scan included).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "mpm_internal.hpp"

namespace nclr_dev {

constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / 64;
// Keys per tile: 4096, or 1024 up to kSmallSort keys, where 4096 would leave most of the chip's CUs
// without a tile.
constexpr int kLargeItems = 16, kSmallItems = 4;
constexpr int64_t kSmallSort = int64_t(1) << 18;
// Up to this many tiles a scatter workgroup sums its digit offsets from the tiles' counts itself, which
// saves the scan's launch (64 counts a thread: 16 loads in flight, 4 rounds of L2 latency).
constexpr int64_t kFusedTiles = 64;

// Lanes of the current wave whose `d` equals this lane's, by its `bits` low bits (for valid lanes).
__device__ __forceinline__ uint64_t match_digit(uint32_t d, bool valid, int bits) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        if (b >= bits) break;  // uniform
        const bool one = (d >> b) & 1u;
        const uint64_t m = __ballot(one);
        peers &= one ? m : ~m;
    }
    return peers;
}

// A tile's keys: wave w, round r, lane l holds key base + (w ITEMS + r) 64 + l.
template <int ITEMS>
__device__ __forceinline__ int64_t tile_key(int r) {
    return (int64_t(blockIdx.x) * kSortWaves + (threadIdx.x >> 6)) * (ITEMS * 64) + r * 64 + (threadIdx.x & 63);
}

template <int ITEMS>
__device__ __forceinline__ void load_keys(uint32_t (&k)[ITEMS], const uint32_t* __restrict__ keys, int64_t n) {
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t idx = tile_key<ITEMS>(r);
        k[r] = idx < n ? keys[idx] : 0u;
    }
}

// FUSED: counts of tile b at hist[b][.], else of digit d at hist[d][.].
template <int ITEMS, bool FUSED>
__global__ __launch_bounds__(kSortThreads) void k_radix_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                             int bits, uint32_t* __restrict__ hist, int64_t tiles) {
    __shared__ uint32_t counts[256];
    const int t = threadIdx.x;
    counts[t] = 0;
    uint32_t k[ITEMS];
    load_keys<ITEMS>(k, keys, n);
    __syncthreads();
    const uint32_t dmask = (1u << bits) - 1u;
    const int lane = t & 63;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = tile_key<ITEMS>(r) < n;
        const uint32_t d = (k[r] >> shift) & dmask;
        const uint64_t peers = match_digit(d, valid, bits);
        // the lowest lane of each group adds the group's size
        if (valid && (peers & ((1ull << lane) - 1ull)) == 0ull) atomicAdd(&counts[d], uint32_t(__popcll(peers)));
    }
    __syncthreads();
    if (FUSED) hist[int64_t(blockIdx.x) * 256 + t] = counts[t];
    else hist[int64_t(t) * tiles + blockIdx.x] = counts[t];
}

// Inclusive scan of one value per thread over a workgroup of N threads (Hillis-Steele in LDS).
template <int N>
__device__ __forceinline__ uint32_t block_inclusive_scan(uint32_t v, uint32_t* part) {
    const int t = threadIdx.x;
    part[t] = v;
    __syncthreads();
#pragma unroll
    for (int off = 1; off < N; off <<= 1) {
        const uint32_t u = t >= off ? part[t - off] : 0u;
        __syncthreads();
        part[t] += u;
        __syncthreads();
    }
    return part[t];
}

// Per digit d (one workgroup each): exclusive scan of hist[d][0..tiles) in place, total to
// digit_total[d].  Coalesced rounds of 256 tiles.
__global__ __launch_bounds__(256) void k_radix_digit_scan(uint32_t* __restrict__ hist, int64_t tiles,
                                                          uint32_t* __restrict__ digit_total) {
    __shared__ uint32_t part[256];
    uint32_t* row = hist + int64_t(blockIdx.x) * tiles;
    uint32_t carry = 0;
    for (int64_t b = 0; b < tiles; b += 256) {
        const int64_t i = b + threadIdx.x;
        const uint32_t v = i < tiles ? row[i] : 0u;
        const uint32_t inc = block_inclusive_scan<256>(v, part);
        if (i < tiles) row[i] = carry + inc - v;
        carry += part[255];
        __syncthreads();
    }
    if (threadIdx.x == 0) digit_total[blockIdx.x] = carry;
}

// FIRST: the values are the input positions.
template <int ITEMS, bool FUSED, bool FIRST>
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(const uint32_t* __restrict__ keys_in,
                                                                const uint32_t* __restrict__ vals_in,
                                                                uint32_t* __restrict__ keys_out,
                                                                uint32_t* __restrict__ vals_out, int64_t n, int shift,
                                                                int bits, const uint32_t* __restrict__ hist,
                                                                const uint32_t* __restrict__ digit_total,
                                                                int64_t tiles) {
    __shared__ uint32_t wave_count[kSortWaves][256];  // then: where the wave's keys of a digit start
    __shared__ uint32_t part[256];
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    uint32_t k[ITEMS], v[ITEMS], rank[ITEMS];
    load_keys<ITEMS>(k, keys_in, n);
    if (!FIRST) load_keys<ITEMS>(v, vals_in, n);
    // start of digit t in this tile = keys with a smaller digit + keys with digit t in earlier tiles
    uint32_t total = 0, before = 0;
    if (FUSED) {
        for (int64_t b0 = 0; b0 < tiles; b0 += 16) {
            uint32_t c[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) c[u] = b0 + u < tiles ? hist[(b0 + u) * 256 + t] : 0u;
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                total += c[u];
                before += b0 + u < int64_t(blockIdx.x) ? c[u] : 0u;
            }
        }
    } else {
        total = digit_total[t];
        before = hist[int64_t(t) * tiles + blockIdx.x];
    }
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) wave_count[w][t] = 0;
    const uint32_t start = block_inclusive_scan<kSortThreads>(total, part) - total + before;  // has barriers
    const uint32_t dmask = (1u << bits) - 1u;
    // rank among the wave's keys of the same digit, in order: the group's lowest lane takes the
    // running count and adds the group's size
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = tile_key<ITEMS>(r) < n;
        const uint32_t d = (k[r] >> shift) & dmask;
        const uint64_t peers = match_digit(d, valid, bits);
        const int leader = __ffsll((unsigned long long)peers) - 1;
        uint32_t run = 0;
        if (valid && lane == leader) run = atomicAdd(&wave_count[wave][d], uint32_t(__popcll(peers)));
        rank[r] = __shfl(run, leader < 0 ? 0 : leader) + uint32_t(__popcll(peers & ((1ull << lane) - 1ull)));
    }
    __syncthreads();
    uint32_t at = start;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t c = wave_count[w][t];
        wave_count[w][t] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t idx = tile_key<ITEMS>(r);
        if (idx >= n) continue;
        const uint32_t pos = wave_count[wave][(k[r] >> shift) & dmask] + rank[r];
        keys_out[pos] = k[r];
        vals_out[pos] = FIRST ? uint32_t(idx) : v[r];
    }
}

}  // namespace nclr_dev

namespace nclr_host {

using namespace nclr_dev;

static int tile_keys(int64_t n) { return kSortThreads * (n <= kSmallSort ? kSmallItems : kLargeItems); }
int64_t sort_tiles(int64_t n) { return (n + tile_keys(n) - 1) / tile_keys(n); }

static int radix_passes(int bits) { return bits <= 0 ? 1 : (bits + 7) / 8; }
uint32_t* radix_keys_in(uint32_t* keys, uint32_t* keys_tmp, int bits) {
    return radix_passes(bits) % 2 ? keys_tmp : keys;
}

template <int ITEMS, bool FUSED, bool FIRST>
static void radix_pass(const uint32_t* kin, const uint32_t* vin, uint32_t* kout, uint32_t* vout, uint32_t* hist,
                       int64_t n, int64_t tiles, int shift, int bits, hipStream_t s) {
    uint32_t* digit_total = hist + 256 * tiles;
    k_radix_hist<ITEMS, FUSED><<<unsigned(tiles), kSortThreads, 0, s>>>(kin, n, shift, bits, hist, tiles);
    if (!FUSED) k_radix_digit_scan<<<256, 256, 0, s>>>(hist, tiles, digit_total);
    k_radix_scatter<ITEMS, FUSED, FIRST><<<unsigned(tiles), kSortThreads, 0, s>>>(kin, vin, kout, vout, n, shift, bits,
                                                                                 hist, digit_total, tiles);
}

// Stable sort of n keys (in radix_keys_in's buffer) by their low `bits` bits: the sorted keys in
// `keys`, the input positions in sorted order in `vals`.  keys_tmp / vals_tmp are scratch of n
// entries; hist holds 256 * sort_tiles(n) + 256 counters.
hipError_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t* hist,
                            int64_t n, int bits, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const int64_t tiles = sort_tiles(n);
    const int passes = radix_passes(bits);
    uint32_t *kin = radix_keys_in(keys, keys_tmp, bits), *vin = nullptr;
    for (int p = 0; p < passes; ++p) {
        const int shift = 8 * p;
        const int dbits = std::max(0, std::min(8, bits - shift));  // digits use only the requested low bits
        uint32_t* kout = kin == keys ? keys_tmp : keys;
        uint32_t* vout = kout == keys ? vals : vals_tmp;
        auto pass = [&](auto items, auto fused) {
            if (p == 0) radix_pass<items.value, fused.value, true>(kin, vin, kout, vout, hist, n, tiles, shift, dbits, s);
            else radix_pass<items.value, fused.value, false>(kin, vin, kout, vout, hist, n, tiles, shift, dbits, s);
        };
        using Small = std::integral_constant<int, kSmallItems>;
        if (tiles <= kFusedTiles && n <= kSmallSort) pass(Small{}, std::true_type{});
        else if (n <= kSmallSort) pass(Small{}, std::false_type{});
        else pass(std::integral_constant<int, kLargeItems>{}, std::false_type{});
        kin = kout;
        vin = vout;
    }
    return hipGetLastError();
}

}  // namespace nclr_host
