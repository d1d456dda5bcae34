// Segmented radix-order sort of every segment that fits LDS, for gfx950: a wave per small segment and a
// workgroup per medium one, in one launch.
//
// The other route (segsort.hip) sorts small segments jointly per 2,048-item tile, which costs a pass over their
// labels, a second sort of the segment that crosses the tile's end and two searches per tile, in a launch of its
// own; its chain of LDS round trips and barriers runs 4 items per lane and pass at 16 waves per CU (78 us at 4 M
// u32 + u32 pairs in 13,333 log-normal segments of mean 300, and 73 us more for the medium segments).  Here:
//   * A wave sorts up to 512 items with no barrier: digits are ranked by ballot matches against the wave's own
//     256 counters, four of which each lane scans, and the items move through the wave's own LDS.  Items per
//     lane follow the length (1, 2, 4 or 8), since a rank step costs the same whether its items are real.
//   * Tiny segments (up to 16 items) take a 16-lane row each, four at a time.
//   * Medium segments are collected by the workgroup's waves and sorted by all 512 threads, 2, 4 or 8 items per
//     thread (of narrow items in large inputs by segsort.hip's block kernel: medium_apart).
//   * Digits that are the same in a whole segment are skipped.
// The kinds of key differ by two mask words, so the code exists once per key and value size.
#include "block_sort.hpp"
#include "segsort_waves.hpp"

#include <algorithm>
#include <bit>

namespace lcpp_hip {
namespace {

constexpr int kSwBlock = 512;
constexpr int kSwWaves = kSwBlock / kWave;
constexpr uint32_t kSwTiny = 16;      // items that a 16-lane row sorts
constexpr uint32_t kSwSmall = 512;    // items that one wave sorts
// The workgroup sorts up to kSwMedium (segsort_waves.hpp).
constexpr uint32_t kSwPerWaveMost = 8;  // segments
constexpr uint32_t kSwPerWave = kSwMedium / kSwWaves;
static_assert(kSwSmall <= kSwPerWave, "a wave's share of the workgroup's arrays holds a small segment");

// Compared bits of a key, in the low bits of a word.
template <typename U>
struct SegmentBits {
    U float_mask, sign_mask, desc_mask, bit_mask;
    uint32_t begin;
    __device__ __forceinline__ U operator()(U x) const {
        const U all = static_cast<U>(static_cast<std::make_signed_t<U>>(x) >> (sizeof(U) * 8 - 1));
        return ((x ^ ((all & float_mask) | sign_mask) ^ desc_mask) >> begin) & bit_mask;
    }
};

// One wave's view of the workgroup's LDS.
template <typename U, typename V, bool PAIRS>
struct WaveLds {
    U* key;
    V* value;
    uint32_t* count;  // 256, 16-byte aligned
};

struct OrOp {
    template <typename T>
    __device__ __forceinline__ T operator()(T a, T b) const { return a | b; }
    template <typename T>
    __device__ __forceinline__ static constexpr T identity() { return T(0); }
};

// Stable sort of the segment [at, at + len), len <= 64 ITEMS, by one wave; every item is read before any is
// written.  Item j of lane l is item 64 j + l.
template <typename U, typename V, bool PAIRS, int ITEMS>
__device__ __forceinline__ void wave_sort(const U* keys_in, U* keys_out, const V* values_in, V* values_out, uint64_t at,
                                          uint32_t len, uint32_t bits, const SegmentBits<U>& sort_bits,
                                          const WaveLds<U, V, PAIRS>& s) {
    typedef uint32_t Four __attribute__((ext_vector_type(4)));
    const uint32_t lane = lane_id();
    U k[ITEMS];
    V v[PAIRS ? ITEMS : 1];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = j * kWave + lane;
        k[j] = i < len ? keys_in[at + i] : U(0);
        if constexpr (PAIRS) v[j] = i < len ? values_in[at + i] : V(0);
    }
    const U ref = wave_read_lane(sort_bits(k[0]), 0);
    U vary = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (j * kWave + lane < len) vary |= sort_bits(k[j]) ^ ref;
    vary = wave_reduce(vary, OrOp{});
    Four* const quads = reinterpret_cast<Four*>(s.count);
    for (uint32_t shift = 0; shift < bits; shift += 8) {
        if ((static_cast<uint32_t>(vary >> shift) & 0xFFu) == 0) continue;
        quads[lane] = Four{0u, 0u, 0u, 0u};
        wave_lds_order();
        uint32_t rank[ITEMS];  // digit << 16 | rank among the items of that digit
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            uint32_t d = static_cast<uint32_t>(sort_bits(k[j]) >> shift) & 0xFFu;
            if (j * kWave + lane >= len) d = 0xFFu;  // missing items rank last
            const uint64_t peers = match_digit(d);
            const uint32_t below = popc_lanes_below(peers);
            const uint32_t base = s.count[d];
            rank[j] = (d << 16) | (base + below);
            if ((peers >> lane) == 1ull) s.count[d] = base + below + 1;
            wave_lds_order();
        }
        Four c = quads[lane];
        const uint32_t sum = c[0] + c[1] + c[2] + c[3];
        uint32_t start = wave_inclusive_scan(sum, SumOp{}) - sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t n = c[i];
            c[i] = start;
            start += n;
        }
        quads[lane] = c;
        wave_lds_order();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            const uint32_t pos = s.count[rank[j] >> 16] + (rank[j] & 0xFFFFu);
            s.key[pos] = k[j];
            if constexpr (PAIRS) s.value[pos] = v[j];
        }
        wave_lds_order();
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) {
            k[j] = s.key[j * kWave + lane];
            if constexpr (PAIRS) v[j] = s.value[j * kWave + lane];
        }
        wave_lds_order();
    }
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = j * kWave + lane;
        if (i < len) {
            keys_out[at + i] = k[j];
            if constexpr (PAIRS) values_out[at + i] = v[j];
        }
    }
}

template <typename U, typename V, bool PAIRS, int ITEMS>
__device__ __forceinline__ void block_sort_segment(const U* keys_in, U* keys_out, const V* values_in, V* values_out,
                                                   uint64_t at, uint32_t len, uint32_t bits,
                                                   const SegmentBits<U>& sort_bits, unsigned char* lds) {
    using Sorter = BlockSort<U, V, PAIRS, kSwBlock, ITEMS, true>;
    const uint32_t first = threadIdx.x / kWave * kWave * ITEMS + lane_id();
    U k[ITEMS];
    V v[PAIRS ? ITEMS : 1];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = first + j * kWave;
        k[j] = i < len ? keys_in[at + i] : U(0);
        if constexpr (PAIRS) v[j] = i < len ? values_in[at + i] : V(0);
    }
    Sorter::sort(k, v, len, bits, sort_bits, *reinterpret_cast<typename Sorter::Shared*>(lds));
    __syncthreads();  // every item is read, and the LDS is free for the next segment
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = first + j * kWave;
        if (i < len) {
            keys_out[at + i] = k[j];
            if constexpr (PAIRS) values_out[at + i] = v[j];
        }
    }
}

// Number of items before lane i's `key` among the `len` items of its 16-lane row: every rotation of the row (S = 1 ..
// 15) brings another lane's key, with that lane's index.
template <typename U, int S = 1>
__device__ __forceinline__ uint32_t row_place(U key, uint32_t i, uint32_t len) {
    if constexpr (S == 16) {
        return 0;
    } else {
        constexpr int kRowRor = 0x120 + S;
        const U other = dpp_move<kRowRor>(key, key);
        const uint32_t j = dpp_move<kRowRor>(i, i);
        const bool first = j < len && (other < key || (other == key && j < i));
        return (first ? 1u : 0u) + row_place<U, S + 1>(key, i, len);
    }
}

// Stable sorts of the tiny segments that the lanes in `tiny` hold, four at a time, one in each 16-lane row: every item
// counts the items before it, which is its place.  About 80 instructions for four segments, without LDS; a wave sort of
// each costs as much as one of 64 items (2^26 u32 pairs, 15 % of them in segments of 10 and the rest in segments of
// 4,096, in random order: 1,184 -> 679 us per call).
template <typename U, typename V, bool PAIRS>
__device__ __forceinline__ void row_sorts(const U* keys_in, U* keys_out, const V* values_in, V* values_out, uint32_t b,
                                          uint32_t len, uint64_t tiny, const SegmentBits<U>& sort_bits) {
    const uint32_t lane = lane_id();
    const uint32_t i = lane % 16;
    while (tiny != 0) {
        uint32_t begin = 0, l = 0;
#pragma unroll
        for (uint32_t row = 0; row < 4; ++row) {
            if (tiny == 0) break;
            const int from = __builtin_ctzll(tiny);
            tiny &= tiny - 1;
            const uint32_t rb = wave_read_lane(b, from), rl = wave_read_lane(len, from);
            if (lane / 16 == row) {
                begin = rb;
                l = rl;
            }
        }
        const uint64_t at = begin;
        U k = 0;
        V v = 0;
        if (i < l) {
            k = keys_in[at + i];
            if constexpr (PAIRS) v = values_in[at + i];
        }
        const uint32_t place = row_place(sort_bits(k), i, l);
        if (i < l) {
            keys_out[at + place] = k;
            if constexpr (PAIRS) values_out[at + place] = v;
        }
    }
}

// Workgroup g takes the segments [g * per_group, (g + 1) * per_group), each wave per_wave (<= kSwPerWaveMost) of
// them, whose bounds its lanes read together.  The longest segment above kSwMedium goes to words[0] (a load first:
// atomics on one address serialise).
// 40 KB of LDS for four-byte pairs: three workgroups per CU, 24 waves, at most 80 VGPRs, for which the builds of u32 +
// u32 pairs and u64 keys spill two and four (with 82 and none, two workgroups run: 2^26 u32 pairs in segments of 64
// 658 -> 788 us per call).
// MEDIUM: with the medium segments; without, the caller has them, the tiny ones and `words` done elsewhere.
template <typename U, typename V, bool PAIRS, bool MEDIUM>
__global__ __launch_bounds__(kSwBlock, sizeof(U) + (PAIRS ? sizeof(V) : 0) <= 8 ? 6 : 4) void segsort_waves_kernel(
    const U* keys_in, U* keys_out, const V* values_in, V* values_out, const uint32_t* __restrict__ begins,
    const uint32_t* __restrict__ ends, uint32_t num_segments, uint32_t per_group, uint32_t per_wave, uint64_t n, uint32_t bits,
    SegmentBits<U> sort_bits, uint32_t* words) {
    using Sorter = BlockSort<U, V, PAIRS, kSwBlock, static_cast<int>(kSwMedium / kSwBlock), true>;
    constexpr uint32_t kWaveBytes = 1024 + kSwSmall * (sizeof(U) + (PAIRS ? sizeof(V) : 0));
    constexpr uint32_t kLdsBytes = MEDIUM ? sizeof(typename Sorter::Shared) : kSwWaves * kWaveBytes;
    __shared__ __attribute__((aligned(16))) unsigned char s_lds[kLdsBytes];
    static_assert(kWaveBytes <= sizeof(typename Sorter::Shared) / kSwWaves, "the waves' arrays fit the workgroup's");
    __shared__ uint16_t s_medium[kSwWaves * kSwPerWaveMost];  // segments of the group, by number
    __shared__ uint32_t s_mediums, s_long;
    const uint32_t lane = lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if constexpr (MEDIUM) {
        if (threadIdx.x == 0) {
            s_mediums = 0;
            s_long = 0;
        }
        __syncthreads();
    }
    unsigned char* const mine = s_lds + wave * kWaveBytes;
    const WaveLds<U, V, PAIRS> s{reinterpret_cast<U*>(mine + 1024), reinterpret_cast<V*>(mine + 1024 + kSwSmall * sizeof(U)),
                                 reinterpret_cast<uint32_t*>(mine)};
    const uint64_t group = static_cast<uint64_t>(blockIdx.x) * per_group;
    const uint32_t member = wave * per_wave + lane;
    const uint64_t x = group + member;
    uint32_t b = 0, len = 0;
    if (lane < per_wave && member < per_group && x < num_segments) {
        b = begins[x];
        const uint32_t e = ends[x];
        len = b < e && e <= n ? e - b : 0u;
    }
    if constexpr (MEDIUM) {
        if (len > kSwMedium) {
            atomicMax(&s_long, len);
        } else if (len > kSwSmall) {
            s_medium[atomicAdd(&s_mediums, 1u)] = static_cast<uint16_t>(member);
        } else if (len == 1) {
            keys_out[b] = keys_in[b];
            if constexpr (PAIRS) values_out[b] = values_in[b];
        }
    }
    // Where the tiny segments are sorted decides how the compiler lays out the sorts beside them: first costs
    // 512-item segments of u32 + u64 pairs 9 % (2^26 items: 527 -> 575 us), last 4,096-item ones of u64 + u64 pairs
    // 13 % (1,449 -> 1,640).
    constexpr bool kTinyFirst = MEDIUM && sizeof(U) == 8;
    if constexpr (kTinyFirst)
        row_sorts<U, V, PAIRS>(keys_in, keys_out, values_in, values_out, b, len, wave_ballot(len > 1 && len <= kSwTiny),
                               sort_bits);
    uint64_t small = wave_ballot(len > kSwTiny && len <= kSwSmall);
    while (small != 0) {
        const uint32_t from = static_cast<uint32_t>(__builtin_ctzll(small));
        small &= small - 1;
        // wave_read_lane keeps the unsigned type: the builtin's int would be sign-extended from 2^31 on.
        const uint64_t at = wave_read_lane(b, static_cast<int>(from));
        const uint32_t l = wave_read_lane(len, static_cast<int>(from));
        if (l <= 64) wave_sort<U, V, PAIRS, 1>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s);
        else if (l <= 128) wave_sort<U, V, PAIRS, 2>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s);
        else if (l <= 256) wave_sort<U, V, PAIRS, 4>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s);
        else wave_sort<U, V, PAIRS, 8>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s);
    }
    if constexpr (!MEDIUM) return;
    if constexpr (!kTinyFirst)
        row_sorts<U, V, PAIRS>(keys_in, keys_out, values_in, values_out, b, len, wave_ballot(len > 1 && len <= kSwTiny),
                               sort_bits);
    __syncthreads();  // the list is complete, and the waves are done with their LDS
    const uint32_t mediums = s_mediums;
    for (uint32_t i = 0; i < mediums; ++i) {
        const uint64_t y = group + s_medium[i];
        const uint64_t at = begins[y];
        const uint32_t l = ends[y] - static_cast<uint32_t>(at);
        if (l <= 1024) block_sort_segment<U, V, PAIRS, 2>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s_lds);
        else if (l <= 2048) block_sort_segment<U, V, PAIRS, 4>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s_lds);
        else block_sort_segment<U, V, PAIRS, 8>(keys_in, keys_out, values_in, values_out, at, l, bits, sort_bits, s_lds);
    }
    if (words && threadIdx.x == 0 && s_long &&
        __hip_atomic_load(&words[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < s_long)
        atomicMax(&words[0], s_long);
}

}  // namespace

template <typename U, typename V, bool PAIRS>
int segsort_waves(const U* keys_in, U* keys_out, const V* values_in, V* values_out, const uint32_t* begins,
                  const uint32_t* ends, uint64_t num_segments, uint64_t n, SegmentKeys kind, uint32_t begin_bit,
                  uint32_t end_bit, bool descending, uint32_t* words, bool medium, hipStream_t stream) {
    const uint32_t bits = end_bit - begin_bit;
    SegmentBits<U> sort_bits;
    sort_bits.float_mask = kind == SegmentKeys::kFloat ? static_cast<U>(~U(0)) : U(0);
    sort_bits.sign_mask = kind == SegmentKeys::kUnsigned ? U(0) : static_cast<U>(U(1) << (sizeof(U) * 8 - 1));
    sort_bits.desc_mask = descending ? static_cast<U>(~U(0)) : U(0);
    sort_bits.bit_mask = bits == 0 ? U(0) : static_cast<U>(static_cast<U>(~U(0)) >> (sizeof(U) * 8 - bits));
    sort_bits.begin = bits == 0 ? 0u : begin_bit;
    // Workgroups that the chip holds together (three per CU).  Segments of more than kSwSmall items on average, of
    // which a workgroup sorts one after the other: one per workgroup up to four rounds of workgroups, then two, four
    // and eight (powers of two: 2^22 u32 + u64 pairs in segments of 1,024 take 90.5 us in groups of three, 84 in
    // groups of two or four; 33 segments of mean 1,500, u32 pairs, took 105.8 us per call with eight and 58.5 with
    // one; 4,194,304 u64 + u32 pairs in segments of 700 200.5 us with seven and 180.7 with one).  Shorter ones: one
    // per workgroup while the workgroups do not fill the chip, then up to one per wave, and from four rounds of
    // workgroups on more, so that they cost a part of a workgroup's start; at most eight per wave, since where the
    // long ones stand together their workgroups run alone at the end (2^26 u32 pairs, 13,926 segments of 4,096 items
    // before 1,006,632 of 10: 4,602 us per call with 42 per wave, 1,351 with eight).
    const uint64_t resident = static_cast<uint64_t>(device_cu_count()) * 3;
    const bool mostly_medium = n / num_segments > kSwSmall;
    const uint64_t per_wave =
        mostly_medium ? 1 : std::clamp<uint64_t>(num_segments / (resident * kSwWaves * 4), 1, kSwPerWaveMost);
    const uint64_t per_group =
        per_wave > 1 || !medium ? per_wave * kSwWaves
        : mostly_medium        ? std::bit_floor(std::clamp<uint64_t>(num_segments / (resident * 4), 1, kSwWaves))
                               : std::clamp<uint64_t>(num_segments / resident, 1, kSwWaves);
    const uint64_t groups = ceil_div(num_segments, per_group);
    LaunchScope scope("segsort_waves", stream);
    const auto launch = [&](auto kernel) {
        kernel<<<static_cast<unsigned>(groups), kSwBlock, 0, stream>>>(
            keys_in, keys_out, values_in, values_out, begins, ends, static_cast<uint32_t>(num_segments),
            static_cast<uint32_t>(per_group), static_cast<uint32_t>(per_wave), n, bits, sort_bits, words);
    };
    if (medium) launch(segsort_waves_kernel<U, V, PAIRS, true>);
    else if constexpr (kSwApart<U, V, PAIRS>) launch(segsort_waves_kernel<U, V, PAIRS, false>);
    return check_hip(hipGetLastError(), "segsort waves launch");
}

#define LCPP_HIP_SEGSORT_WAVES(U, V, P)                                                                            \
    template int segsort_waves<U, V, P>(const U*, U*, const V*, V*, const uint32_t*, const uint32_t*, uint64_t,    \
                                        uint64_t, SegmentKeys, uint32_t, uint32_t, bool, uint32_t*, bool,              \
                                        hipStream_t);
LCPP_HIP_SEGSORT_WAVES(uint32_t, uint32_t, false)
LCPP_HIP_SEGSORT_WAVES(uint32_t, uint32_t, true)
LCPP_HIP_SEGSORT_WAVES(uint32_t, uint64_t, true)
LCPP_HIP_SEGSORT_WAVES(uint64_t, uint32_t, false)
LCPP_HIP_SEGSORT_WAVES(uint64_t, uint32_t, true)
LCPP_HIP_SEGSORT_WAVES(uint64_t, uint64_t, true)
#undef LCPP_HIP_SEGSORT_WAVES

}  // namespace lcpp_hip
