// Stable LSD radix sort of one workgroup's tile in LDS, with the keys (and values) of each thread in
// registers between the passes.
#pragma once

#include "common.hpp"

namespace lcpp_hip {

// A pass costs a rank chain of ITEMS dependent LDS round trips per wave, four barriers and one LDS
// exchange, whatever the digits are; digits that are the same in every key of the tile are skipped (a
// tile of 30-bit codes or of small 64-bit integers takes only the passes that can move anything).
//
// Item j of lane l of wave w is the tile's item w * 64 * ITEMS + 64 j + l (each wave holds a contiguous
// range, so ranking the waves in order keeps the sort stable).  `sort_bits(key)` gives the key's compared
// bits in the low `bits` bits of a word; items past `valid` stay behind the others (they take the largest
// digit of every pass and come last in the tile).
// SKIP_IDLE: waves without items sit the passes out (for tiles that often leave waves empty; where they do not, the
// branches cost more: 2,048 u32 pairs in one tile 8.9 -> 9.2 us per call).
template <typename U, typename V, bool PAIRS, int BLOCK, int ITEMS, bool SKIP_IDLE = false>
struct BlockSort {
    static constexpr int kWaves = BLOCK / kWave;
    static constexpr uint32_t kTile = static_cast<uint32_t>(BLOCK) * ITEMS;
    static constexpr uint32_t kBins = 256;
    static_assert(BLOCK >= static_cast<int>(kBins), "thread t scans digit t");

    struct Shared {
        U key[kTile];
        V value[PAIRS ? kTile : 1];
        uint32_t count[kWaves][kBins];
        uint32_t total[kBins / kWave];
        U vary[kWaves];
    };

    // Compared bits that differ between some two items of the tile.
    template <typename Bits>
    static __device__ __forceinline__ U varying_bits(const U (&k)[ITEMS], uint32_t valid, Bits sort_bits, Shared& s) {
        const uint32_t first = threadIdx.x / kWave * kWave * ITEMS + lane_id();
        // Against the wave's own first item, then across the waves' first items.
        U ref = sort_bits(k[0]);
        if constexpr (sizeof(U) == 4) ref = __builtin_amdgcn_readfirstlane(ref);
        else ref = wave_read_lane(ref, 0);
        U diff = 0;
#pragma unroll
        for (int j = 0; j < ITEMS; ++j)
            if (first + j * kWave < valid) diff |= sort_bits(k[j]) ^ ref;
        diff = wave_reduce(diff, OrBits{});
        const uint32_t wave = threadIdx.x / kWave;
        if (lane_id() == 0) {
            s.vary[wave] = diff;
            s.key[wave] = ref;
        }
        __syncthreads();
        const uint32_t waves = (valid + kWave * ITEMS - 1) / (kWave * ITEMS);  // waves that hold items
        U all = 0;
        const U ref0 = s.key[0];
        for (uint32_t w = 0; w < waves; ++w) all |= s.vary[w] | (s.key[w] ^ ref0);
        return all;
    }

    struct OrBits {
        template <typename T>
        __device__ __forceinline__ T operator()(T a, T b) const { return a | b; }
        template <typename T>
        __device__ __forceinline__ static constexpr T identity() { return T(0); }
    };

    // Sorts in registers: on return item j of lane l of wave w is the tile's item of that number in sorted
    // order.  Collective over the workgroup; `s` is free again after the caller's next barrier.
    template <typename Bits>
    static __device__ __forceinline__ void sort(U (&k)[ITEMS], V (&v)[PAIRS ? ITEMS : 1], uint32_t valid, uint32_t bits,
                                                Bits sort_bits, Shared& s) {
        const uint32_t tid = threadIdx.x;
        const uint32_t lane = lane_id();
        const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        const uint32_t first = wave * kWave * ITEMS + lane;
        const U vary = varying_bits(k, valid, sort_bits, s);
        const bool idle = SKIP_IDLE && wave * kWave * ITEMS >= valid;  // the wave's counters stay zero
        uint32_t* const cnt = s.count[wave];
        for (uint32_t shift = 0; shift < bits; shift += 8) {
            if ((static_cast<uint32_t>(vary >> shift) & 0xFFu) == 0) continue;  // the same in every item
#pragma unroll
            for (uint32_t i = 0; i < kBins / kWave; ++i) cnt[i * kWave + lane] = 0;
            wave_lds_order();
            uint32_t rank[ITEMS];  // digit << 16 | rank among the wave's items of that digit
            if (!idle) {
#pragma unroll
                for (int j = 0; j < ITEMS; ++j) {
                    uint32_t d = static_cast<uint32_t>(sort_bits(k[j]) >> shift) & 0xFFu;
                    if (first + j * kWave >= valid) d = 0xFFu;
                    const uint64_t peers = match_digit(d);
                    const uint32_t below = popc_lanes_below(peers);
                    const uint32_t base = cnt[d];
                    rank[j] = (d << 16) | (base + below);
                    if ((peers >> lane) == 1ull) cnt[d] = base + below + 1;
                    wave_lds_order();
                }
            }
            __syncthreads();
            uint32_t before[kWaves];  // the digit's items in the waves before each wave
            uint32_t sum = 0, incl = 0;
            if (tid < kBins) {
#pragma unroll
                for (int w = 0; w < kWaves; ++w) {
                    const uint32_t c = s.count[w][tid];
                    before[w] = sum;
                    sum += c;
                }
                incl = wave_inclusive_scan(sum, SumOp{});
                if (lane == kWave - 1) s.total[wave] = incl;
            }
            __syncthreads();
            if (tid < kBins) {
                uint32_t start = incl - sum;
                for (uint32_t w = 0; w < wave; ++w) start += s.total[w];
#pragma unroll
                for (int w = 0; w < kWaves; ++w) s.count[w][tid] = start + before[w];
            }
            __syncthreads();
            if (!idle) {
#pragma unroll
                for (int j = 0; j < ITEMS; ++j) {
                    const uint32_t pos = cnt[rank[j] >> 16] + (rank[j] & 0xFFFFu);
                    s.key[pos] = k[j];
                    if constexpr (PAIRS) s.value[pos] = v[j];
                }
            }
            __syncthreads();
            if (!idle) {
#pragma unroll
                for (int j = 0; j < ITEMS; ++j) {
                    k[j] = s.key[first + j * kWave];
                    if constexpr (PAIRS) v[j] = s.value[first + j * kWave];
                }
            }
        }
    }
};

}  // namespace lcpp_hip
