// Onesweep DeviceRadixSort of medium inputs for gfx950: the tiles of a pass resident together, one launch for
// the histogram and one per pass.
//
// The large-input passes (radix_sort.hip) are built for throughput: tiles of 14,336 or 18,432 keys leave most
// of the 256 CUs idle below a few million keys, and a tile's pass is a chain of 18 or 28 dependent rank
// rounds (18 us per pass at 1,000,003 pairs, 70 tiles), behind a fill and a bin scan of their own.  Here:
//   * Tiles are 1024 threads x 4 keys, two workgroups per CU, so that up to kMidSortMax keys the tiles of a
//     pass are resident together and a rank chain is 4 rounds.  Per call (u32 + u32 pairs, start of the range to
//     its end): 40,000 pairs 69.8 -> 33.4 us, 100,003 73.8 -> 38.2, 1,000,003 87.5 -> 60.0, 2,000,003 97.3 ->
//     79.7; u64 + u32 pairs 109 -> 69, 121 -> 78, 189 -> 122, 220 -> 165.  5, 6 or 8 keys per thread: 61.7, 64.0,
//     66.7 us at 1,000,003 pairs.  Above 2^21 keys the tiles no longer run together and the large-input passes
//     are faster (3,000,003 pairs: 116 us here, 105 there).  A tile of 8-byte keys with 8-byte values takes 85 KB
//     of LDS, one workgroup per CU: from 2^20 of them on a pass runs in two rounds, and a call takes about what
//     the large-input passes take (u64 + u64 pairs there and here: 1,000,003 196.7 and 131.0 us, 1,300,001 207.2
//     and 198.4, 2,097,152 236.1 and 232.1; all keys equal 224.4 and 230.5).
//   * Two workgroups per CU leave 64 registers: pairs of 12 bytes spill up to five (1 to 5, by key type and order).
//   * Histogram workgroups store their digit counts as rows (nothing to clear first); every workgroup of pass
//     0 adds up the rows of its own pass behind its key loads, and the first ones those of the later passes.
//   * The digit counts of the tiles before a tile are added up over two levels: groups of 16 tiles (of 32 up to
//     32 tiles, where the first level is all there is), whose last tile publishes the group's sum in its row (no
//     other tile reads that one's own counts).  A tile reads at most 15 (31) rows of its group and one row per
//     earlier group, in two steps of which each is one cross-XCD round trip.  (The chained look-back of the large
//     inputs reads up to one row per earlier tile here, where all tiles publish at the same time: the reads of
//     the same rows by hundreds of workgroups made a step cost 4 us, 97 us per call of 1,000,003 pairs.)
//   * The rows serve every pass: an entry carries the pass number, so the entries of the pass before read as
//     unpublished, and the histogram clears them once.
#include "radix_keys.hpp"

#include <algorithm>

namespace lcpp_hip {
namespace radix {
namespace {

constexpr uint32_t kDigits = 256;
constexpr int kBlock = 1024;
constexpr int kWaves = kBlock / kWave;
constexpr int kSplit = kBlock / static_cast<int>(kDigits);  // threads per digit
constexpr int kWindow = 8;                                  // rows in flight per thread

// Entry of a row: bit 31 published, 29:27 pass, 26:0 count.
constexpr uint32_t kPublished = 1u << 31;
constexpr uint32_t kCount = (1u << 27) - 1;
static_assert(kMidSortMax <= kCount, "counts fit an entry");
// The entry without its pass number, or 0 (unpublished) when it is of another pass.
__device__ __forceinline__ uint32_t entry_of(uint32_t raw, uint32_t pass) {
    return ((raw >> 27) & 7u) == pass ? raw & ~(7u << 27) : 0u;
}

constexpr int kHistBlock = 1024;
constexpr int kHistCopies = 8;  // a digit's counter copies, by lane: at most eight lanes meet in one

// rows[b][p][d] = number of keys of workgroup b's slice with digit d in pass p; clears the look-back region.
template <typename K, bool DESC>
__global__ __launch_bounds__(kHistBlock) void mid_histogram_kernel(const K* __restrict__ keys, uint32_t n,
                                                                   uint32_t per_block, uint32_t begin_bit,
                                                                   uint32_t bits, uint32_t passes,
                                                                   uint32_t* __restrict__ rows,
                                                                   uint32_t* __restrict__ lookback,
                                                                   uint32_t lookback_words) {
    using U = typename KeyTraits<K>::U;
    constexpr int KIND = KeyTraits<K>::kind;
    constexpr int PASSES_MAX = sizeof(U);
    __shared__ __attribute__((aligned(16))) uint32_t s_hist[PASSES_MAX * kDigits * kHistCopies];
    const uint32_t tid = threadIdx.x;
    const uint32_t first = blockIdx.x * per_block;
    const uint32_t last = min(n, first + per_block);
    const U* ukeys = reinterpret_cast<const U*>(keys);
    constexpr int kBatch = 8;
    U k[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) k[j] = first + tid + j * kHistBlock < last ? ukeys[first + tid + j * kHistBlock] : U(0);
    for (uint32_t i = blockIdx.x * kHistBlock + tid; i < lookback_words; i += gridDim.x * kHistBlock) lookback[i] = 0;
    for (uint32_t i = tid; i < passes * kDigits * kHistCopies; i += kHistBlock) s_hist[i] = 0;
    __syncthreads();
    const uint32_t copy = tid % kHistCopies;
    const SortBits<U, KIND> sort_bits{begin_bit, static_cast<U>(~U(0)) >> (sizeof(U) * 8 - bits)};
    for (uint32_t at = first + tid; at < last; at += kBatch * kHistBlock) {
        U next[kBatch];
        const uint32_t to = at + kBatch * kHistBlock;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) next[j] = to + j * kHistBlock < last ? ukeys[to + j * kHistBlock] : U(0);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (at + j * kHistBlock >= last) break;
            const U x = sort_bits(twiddle_in<U, KIND, DESC>(k[j]));
#pragma unroll
            for (int p = 0; p < PASSES_MAX; ++p) {
                if (static_cast<uint32_t>(p) >= passes) break;
                const uint32_t d = static_cast<uint32_t>(x >> (8 * p)) & 0xFFu;
                atomicAdd(&s_hist[(p * kDigits + d) * kHistCopies + copy], 1u);
            }
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) k[j] = next[j];
    }
    __syncthreads();
    for (uint32_t i = tid; i < passes * kDigits; i += kHistBlock) {
        uint32_t total = 0;
#pragma unroll
        for (int c = 0; c < kHistCopies; ++c) total += s_hist[i * kHistCopies + c];
        rows[blockIdx.x * passes * kDigits + i] = total;
    }
}

// Sum over the histogram rows of one pass's digit d.
__device__ __forceinline__ uint32_t sum_rows(const uint32_t* rows, uint32_t count, uint32_t stride, uint32_t at) {
    uint32_t total = 0;
    constexpr uint32_t kBatch = 16;
    for (uint32_t r = 0; r < count; r += kBatch) {
        uint32_t c[kBatch];
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) c[j] = r + j < count ? rows[(r + j) * stride + at] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) total += c[j];
    }
    return total;
}

// Adds up published rows of 256 digit counts, the whole workgroup together: thread t takes digit t % 256 and
// every kSplit-th row.
template <typename K, bool DESC>
struct Walk {
    using U = typename KeyTraits<K>::U;
    const K* keys;  // of the pass
    SortBits<U, KeyTraits<K>::kind> sort_bits;
    uint32_t shift, pass, tile_items, spin_limit;
    uint32_t (*s_part)[kDigits];
    uint32_t* s_count;
    uint32_t* s_row;

    __device__ __forceinline__ uint32_t digit(U key) const {
        return static_cast<uint32_t>(sort_bits(twiddle_in<U, KeyTraits<K>::kind, DESC>(key)) >> shift) & 0xFFu;
    }

    // The sum of this thread's digit over `count` rows, `stride` words apart; row r counts `tiles` tiles from
    // first_tile + r * tiles.  The workgroup polls until all are published; a row still unpublished after
    // `spin_limit` polls is counted from the keys and published by compare-and-swap, so progress does not depend on
    // the order of dispatch.  (The tiles before another are full.)
    __device__ __forceinline__ uint32_t sum(uint32_t* rows, uint32_t stride, uint32_t count, uint32_t first_tile,
                                            uint32_t tiles) const {
        const uint32_t part = threadIdx.x / kDigits;
        const uint32_t d = threadIdx.x % kDigits;
        uint32_t total = 0;
        for (uint32_t r0 = 0; r0 < count; r0 += kSplit * kWindow) {
            uint32_t v[kWindow];
#pragma unroll
            for (int w = 0; w < kWindow; ++w) {
                const uint32_t r = r0 + w * kSplit + part;
                v[w] = r < count ? entry_of(atomic_load_agent(&rows[r * stride + d]), pass) : kPublished;
            }
            uint32_t spins = 0;
            while (true) {
                int waiting = -1;
#pragma unroll
                for (int w = 0; w < kWindow; ++w)
                    if (v[w] == 0) waiting = w;
                if (!__syncthreads_or(waiting >= 0)) break;
                if (spins >= spin_limit) {
                    if (threadIdx.x == 0) *s_row = 0;
                    if (threadIdx.x < kDigits) s_count[threadIdx.x] = 0;
                    __syncthreads();
                    if (waiting >= 0) atomicMax(s_row, r0 + waiting * kSplit + part + 1u);
                    __syncthreads();
                    const uint32_t r = *s_row - 1u;
                    const U* theirs = reinterpret_cast<const U*>(keys) + (first_tile + r * tiles) * tile_items;
                    for (uint32_t i = threadIdx.x; i < tiles * tile_items; i += kBlock)
                        atomicAdd(&s_count[digit(theirs[i])], 1u);
                    __syncthreads();
#pragma unroll
                    for (int w = 0; w < kWindow; ++w) {
                        if (r != r0 + w * kSplit + part || v[w] != 0) continue;
                        uint32_t expected = atomic_load_agent(&rows[r * stride + d]);
                        const uint32_t desired = kPublished | (pass << 27) | s_count[d];
                        // One that loses to the owner's publication has the same count.
                        if (entry_of(expected, pass) == 0)
                            __hip_atomic_compare_exchange_strong(&rows[r * stride + d], &expected, desired, __ATOMIC_RELAXED,
                                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        v[w] = entry_of(desired, pass);
                    }
                    __syncthreads();  // s_row and s_count are set again by the next one
                    continue;
                }
                __builtin_amdgcn_s_sleep(1);
                ++spins;
#pragma unroll
                for (int w = 0; w < kWindow; ++w) {
                    const uint32_t r = r0 + w * kSplit + part;
                    if (v[w] == 0) v[w] = entry_of(atomic_load_agent(&rows[r * stride + d]), pass);
                }
            }
#pragma unroll
            for (int w = 0; w < kWindow; ++w) total += v[w] & kCount;
        }
        s_part[part][d] = total;
        __syncthreads();
        total = 0;
#pragma unroll
        for (int g = 0; g < kSplit; ++g) total += s_part[g][d];
        __syncthreads();
        return total;
    }
};

// One pass.  rows: the histogram rows in pass 0, whose first workgroups leave the later passes' digit totals in
// bins; nullptr in the later ones.
template <typename K, bool DESC, int VB>
// Two workgroups per CU: 64 VGPRs.
__global__ __launch_bounds__(kBlock, 8) void mid_onesweep_kernel(const K* __restrict__ keys_in, K* __restrict__ keys_out,
                                                              const void* __restrict__ values_in,
                                                              void* __restrict__ values_out, uint32_t n,
                                                              const uint32_t* rows, uint32_t row_count,
                                                              uint32_t* bins, uint32_t* lookback, uint32_t group_tiles,
                                                              uint32_t pass,
                                                              uint32_t passes, uint32_t begin_bit, uint32_t bits,
                                                              uint32_t spin_limit) {
    using U = typename KeyTraits<K>::U;
    using VW = typename ValueWord<VB>::type;
    constexpr int KIND = KeyTraits<K>::kind;
    constexpr int ITEMS = kMidItems;
    constexpr uint32_t TILE = kMidTile;
    static_assert(TILE == static_cast<uint32_t>(kBlock) * ITEMS);
    constexpr size_t kLds = TILE * (sizeof(U) + VB) + sizeof(uint32_t) * kDigits * (kWaves + 1 + kSplit) + 64;
    static_assert(sizeof(U) + VB > 12 || 2 * kLds <= (160u << 10), "two workgroups per CU for items of up to 12 bytes");
    __shared__ U s_key[TILE];
    __shared__ VW s_value[VB ? TILE : 1];
    __shared__ uint32_t s_count[kWaves][kDigits];
    __shared__ uint32_t s_base[kDigits];  // a digit's output position minus its position in the tile
    __shared__ uint32_t s_lb[kSplit][kDigits];
    __shared__ uint32_t s_total[2][kDigits / kWave];
    __shared__ uint32_t s_lb_tile;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t tile = blockIdx.x;
    const uint32_t tile_base = tile * TILE;
    const uint32_t valid = min(TILE, n - tile_base);
    const SortBits<U, KIND> sort_bits{begin_bit, static_cast<U>(~U(0)) >> (sizeof(U) * 8 - bits)};
    const uint32_t shift = 8 * pass;
    const U* ukeys = reinterpret_cast<const U*>(keys_in) + tile_base;
    const uint32_t first = wave * kWave * ITEMS + lane;
    U keys[ITEMS];
    VW vals[VB ? ITEMS : 1];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t i = first + k * kWave;
        keys[k] = i < valid ? ukeys[i] : U(0);
    }
    if constexpr (VB != 0) {
        const VW* uvals = reinterpret_cast<const VW*>(values_in) + tile_base;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t i = first + k * kWave;
            vals[k] = i < valid ? uvals[i] : VW(0);
        }
    }
    // The digit's total over all keys: the sum of the histogram rows, or what pass 0 left of it in bins.
    uint32_t digit_total = 0;
    if (tid < kDigits) {
        if (rows) {
            digit_total = sum_rows(rows, row_count, passes * kDigits, tid);
            for (uint32_t p = 1 + tile; p < passes; p += gridDim.x)
                bins[p * kDigits + tid] = sum_rows(rows, row_count, passes * kDigits, p * kDigits + tid);
        } else {
            digit_total = bins[pass * kDigits + tid];
        }
    }

    // Rank inside the wave (radix_sort.hip): ballot match, per-wave digit counters.
    uint32_t* const cnt = s_count[wave];
#pragma unroll
    for (uint32_t i = 0; i < kDigits / kWave; ++i) cnt[i * kWave + lane] = 0;
    wave_lds_order();
    uint32_t rank[ITEMS];  // digit << 16 | rank among the wave's keys of that digit
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        keys[k] = twiddle_in<U, KIND, DESC>(keys[k]);
        uint32_t d = static_cast<uint32_t>(sort_bits(keys[k]) >> shift) & 0xFFu;
        if (first + k * kWave >= valid) d = 0xFFu;  // missing keys rank last
        const uint64_t peers = match_digit(d);
        const uint32_t below = popc_lanes_below(peers);
        const uint32_t base = cnt[d];
        rank[k] = (d << 16) | (base + below);
        if ((peers >> lane) == 1ull) cnt[d] = base + below + 1;
        wave_lds_order();
    }
    __syncthreads();

    const uint32_t group = tile / group_tiles, member = tile - group * group_tiles;
    const bool ends_group = member == group_tiles - 1;
    uint32_t before[kWaves];
    uint32_t count = 0, local = 0, global = 0;
    if (tid < kDigits) {
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            before[w] = count;
            count += s_count[w][tid];
        }
        if (tid == kDigits - 1) count -= TILE - valid;  // missing keys are not counted
        if (!ends_group) atomic_store_agent(&lookback[tile * kDigits + tid], kPublished | (pass << 27) | count);
        local = wave_inclusive_scan(count, SumOp{});
        global = wave_inclusive_scan(digit_total, SumOp{});
        if (lane == kWave - 1) {
            s_total[0][wave] = local;
            s_total[1][wave] = global;
        }
        local -= count;
        global -= digit_total;
    }
    __syncthreads();
    if (tid < kDigits) {
        for (uint32_t w = 0; w < wave; ++w) {
            local += s_total[0][w];
            global += s_total[1][w];
        }
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s_count[w][tid] = local + before[w];
    }
    __syncthreads();
    // Reorder by digit in LDS before the walk.
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t pos = cnt[rank[k] >> 16] + (rank[k] & 0xFFFFu);
        s_key[pos] = keys[k];
        if constexpr (VB != 0) s_value[pos] = vals[k];
    }

    // Counts of the tiles before this one: first the earlier tiles of its group, then the groups before it.
    uint32_t excl = 0;
    if (tile > 0) {
        Walk<K, DESC> walk{keys_in, sort_bits, shift, pass, TILE, spin_limit, s_lb, s_base, &s_lb_tile};
        const uint32_t group_first = group * group_tiles;
        const uint32_t inside = walk.sum(lookback + group_first * kDigits, kDigits, member, group_first, 1u);
        if (ends_group && tid < kDigits)
            atomic_store_agent(&lookback[tile * kDigits + tid], kPublished | (pass << 27) | (inside + count));
        excl = inside + walk.sum(lookback + (group_tiles - 1) * kDigits, group_tiles * kDigits, group, 0u, group_tiles);
    }
    if (tid < kDigits) s_base[tid] = global + excl - local;
    __syncthreads();

    U* ukeys_out = reinterpret_cast<U*>(keys_out);
    VW* uvals_out = reinterpret_cast<VW*>(values_out);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = tid + j * kBlock;
        if (i < valid) {
            const U key = s_key[i];
            // Always below n for a correct sort.
            const uint32_t g = min(s_base[static_cast<uint32_t>(sort_bits(key) >> shift) & 0xFFu] + i, n - 1);
            ukeys_out[g] = twiddle_out<U, KIND, DESC>(key);
            if constexpr (VB != 0) uvals_out[g] = s_value[i];
        }
    }
}

template <typename K, int VB, bool DESC>
int launch_mid(const MidPlan& M, const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* keys_tmp,
               void* values_tmp, uint32_t n, uint32_t begin_bit, uint32_t bits, uint32_t spin_limit, hipStream_t stream) {
    if (M.tiles != ceil_div(n, kMidTile) || static_cast<uint64_t>(M.rows) * M.per_row < n)
        return set_error(kInvalidArgument, "DeviceRadixSort: the plan does not cover the keys");
    int st;
    {
        LaunchScope scope("radix_histogram", stream);
        mid_histogram_kernel<K, DESC><<<M.rows, kHistBlock, 0, stream>>>(keys_in, n, M.per_row, begin_bit, bits, M.passes,
                                                                        M.row_words, M.lookback, M.tiles * kDigits);
        st = check_hip(hipGetLastError(), "radix_histogram launch");
        if (st != kOk) return st;
    }
    for (uint32_t p = 0; p < M.passes; ++p) {
        const bool to_out = (M.passes - 1 - p) % 2 == 0;
        const K* src = p == 0 ? keys_in : to_out ? keys_tmp : keys_out;
        const void* vsrc = p == 0 ? values_in : to_out ? values_tmp : values_out;
        LaunchScope scope("radix_onesweep", stream);
        mid_onesweep_kernel<K, DESC, VB><<<M.tiles, kBlock, 0, stream>>>(
            src, to_out ? keys_out : keys_tmp, vsrc, to_out ? values_out : values_tmp, n, p == 0 ? M.row_words : nullptr,
            M.rows, M.bins, M.lookback, M.group, p, M.passes, begin_bit, bits, spin_limit);
        st = check_hip(hipGetLastError(), "radix_onesweep launch");
        if (st != kOk) return st;
    }
    return kOk;
}

}  // namespace

template <typename K, int VB>
int mid_sort(const MidPlan& M, const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* keys_tmp,
             void* values_tmp, uint32_t n, uint32_t begin_bit, uint32_t end_bit, bool descending, uint32_t spin_limit,
             hipStream_t stream) {
    const uint32_t bits = end_bit - begin_bit;
    return descending ? launch_mid<K, VB, true>(M, keys_in, keys_out, values_in, values_out, keys_tmp, values_tmp, n,
                                                begin_bit, bits, spin_limit, stream)
                      : launch_mid<K, VB, false>(M, keys_in, keys_out, values_in, values_out, keys_tmp, values_tmp, n,
                                                 begin_bit, bits, spin_limit, stream);
}

#define LCPP_HIP_MID_SORT_V(K, VB)                                                                                   \
    template int mid_sort<K, VB>(const MidPlan&, const K*, K*, const void*, void*, K*, void*, uint32_t, uint32_t,    \
                                 uint32_t, bool, uint32_t, hipStream_t);
#define LCPP_HIP_MID_SORT(K) LCPP_HIP_MID_SORT_V(K, 0) LCPP_HIP_MID_SORT_V(K, 4) LCPP_HIP_MID_SORT_V(K, 8)
LCPP_HIP_MID_SORT(uint32_t)
LCPP_HIP_MID_SORT(int32_t)
LCPP_HIP_MID_SORT(float)
LCPP_HIP_MID_SORT(uint64_t)
LCPP_HIP_MID_SORT(int64_t)
LCPP_HIP_MID_SORT(double)
#undef LCPP_HIP_MID_SORT
#undef LCPP_HIP_MID_SORT_V

}  // namespace radix
}  // namespace lcpp_hip
