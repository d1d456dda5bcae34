// DeviceRadixSort of small inputs for gfx950: one or two launches instead of a fill, a histogram, a bin scan
// and one onesweep pass per digit.
//
// The onesweep path of a few thousand keys spends its time on launches and on one tile's chain of dependent
// LDS round trips per pass (seven launches, 16-19 us per pass at 20,011 pairs), with all but one or two CUs
// idle: 83 us per call of 20,011 f32 + u32 pairs, 68 of 2,000 u32 + u32 pairs; here 16.5 and 8.4.  Every pass
// of a tile runs in LDS inside one launch:
//   * up to kSmallOneTile items: one workgroup sorts them all and writes the output.
//   * up to small_sort_max items: tiles of kRunItems items are sorted by one workgroup each into the scratch
//     buffer; then every item's output position is its index in its run plus, for every other run, the
//     number of that run's items that go before it (a binary search in LDS, which holds all the keys), and
//     the items are written there.  Items of earlier runs go before equal keys, so the sort is stable.
// The line at small_sort_max is where the keys fill the LDS (152 KB; 32,768 pairs take 18.9 us, 72 on the
// onesweep path).
#include "block_sort.hpp"
#include "radix_keys.hpp"

namespace lcpp_hip {
namespace radix {
namespace {

// 512 threads x 2 items: per call of 20,011 / 8,192 u32 + u32 pairs 15.1 / 11.4 us (8,192 u64 + u32: 17.4),
// against 15.4 / 12.9 (21.9) with 512 x 4 or 1024 x 2, 16.1 / 12.4 (19.1) with 256 x 4 and 17.5 / 15.0 (25.8)
// with 256 x 8: short rank chains on many CUs, for a few more searches per item.
constexpr int kRunBlock = 512;
constexpr int kRunItemsPerThread = 2;
constexpr uint32_t kRunItems = kRunBlock * kRunItemsPerThread;  // 1024
// One workgroup sorts up to kSmallOneTile items: one launch, 8.4 us per call of 2,000 pairs; 4,096 pairs in one
// workgroup (1024 x 4) take 12.2 us, more than two launches.
constexpr int kOneItemsPerThread = kSmallOneTile / kRunBlock;
constexpr int kMergeBlock = 256;

// Sorts tile blockIdx.x of BLOCK * ITEMS items in LDS.
template <typename K, bool DESC, int VB, int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void sort_tiles_kernel(const K* keys_in, K* keys_out, const void* values_in,
                                                           void* values_out, uint32_t n, uint32_t begin_bit,
                                                           uint32_t bits) {
    using U = typename KeyTraits<K>::U;
    using VW = typename ValueWord<VB>::type;
    constexpr int KIND = KeyTraits<K>::kind;
    using Sorter = BlockSort<U, VW, VB != 0, BLOCK, ITEMS>;
    __shared__ typename Sorter::Shared s;
    const uint32_t base = blockIdx.x * Sorter::kTile;
    const uint32_t valid = min(Sorter::kTile, n - base);
    const uint32_t first = threadIdx.x / kWave * kWave * ITEMS + lane_id();
    const U* kin = reinterpret_cast<const U*>(keys_in) + base;
    const VW* vin = reinterpret_cast<const VW*>(values_in) + base;
    U k[ITEMS];
    VW v[VB ? ITEMS : 1];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = first + j * kWave;
        k[j] = i < valid ? twiddle_in<U, KIND, DESC>(kin[i]) : U(~U(0));
        if constexpr (VB != 0) v[j] = i < valid ? vin[i] : VW(0);
    }
    const SortBits<U, KIND> sort_bits{begin_bit, static_cast<U>(~U(0)) >> (sizeof(U) * 8 - bits)};
    Sorter::sort(k, v, valid, bits, sort_bits, s);
    U* kout = reinterpret_cast<U*>(keys_out) + base;
    VW* vout = reinterpret_cast<VW*>(values_out) + base;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t i = first + j * kWave;
        if (i < valid) {
            kout[i] = twiddle_out<U, KIND, DESC>(k[j]);
            if constexpr (VB != 0) vout[i] = v[j];
        }
    }
}

// Adds to `place`, for every run of [first, last), the number of its items that go before `key`: those below
// it, and with TIES the equal ones too.  kAtOnce independent searches run side by side; a wave's 64
// neighbouring keys search neighbouring places, so the reads of a step are broadcasts or adjacent words.
template <bool TIES, typename U>
__device__ __forceinline__ uint32_t count_before(const U* s_key, U key, uint32_t first, uint32_t last) {
    constexpr int kAtOnce = 4;
    uint32_t place = 0;
    for (uint32_t r0 = first; r0 < last; r0 += kAtOnce) {
        const U* run[kAtOnce];
        uint32_t pos[kAtOnce];
#pragma unroll
        for (int a = 0; a < kAtOnce; ++a) {
            run[a] = s_key + min(r0 + a, last - 1) * kRunItems;
            pos[a] = 0;
        }
#pragma unroll
        for (uint32_t step = kRunItems / 2; step > 0; step >>= 1) {
#pragma unroll
            for (int a = 0; a < kAtOnce; ++a) {
                const U other = run[a][pos[a] + step - 1];
                if (TIES ? other <= key : other < key) pos[a] += step;
            }
        }
#pragma unroll
        for (int a = 0; a < kAtOnce; ++a) {  // the steps count all items but one
            const U other = run[a][pos[a]];
            if (TIES ? other <= key : other < key) ++pos[a];
            if (r0 + a < last) place += pos[a];
        }
    }
    return place;
}

// Scatters the items of the sorted runs of kRunItems items (the last one may be shorter) to their places.
// A workgroup's items belong to one run.
template <typename K, bool DESC, int VB>
__global__ __launch_bounds__(kMergeBlock) void merge_runs_kernel(const K* __restrict__ keys_in, K* __restrict__ keys_out,
                                                                 const void* __restrict__ values_in,
                                                                 void* __restrict__ values_out, uint32_t n,
                                                                 uint32_t begin_bit, uint32_t bits) {
    using U = typename KeyTraits<K>::U;
    using VW = typename ValueWord<VB>::type;
    constexpr int KIND = KeyTraits<K>::kind;
    static_assert(kRunItems % kMergeBlock == 0, "a workgroup's items belong to one run");
    __shared__ __attribute__((aligned(16))) U s_key[small_sort_max(sizeof(U))];
    const U* kin = reinterpret_cast<const U*>(keys_in);
    const SortBits<U, KIND> sort_bits{begin_bit, static_cast<U>(~U(0)) >> (sizeof(U) * 8 - bits)};
    const uint32_t i = blockIdx.x * kMergeBlock + threadIdx.x;
    U mine = 0;
    VW value = 0;
    if (i < n) {
        mine = kin[i];
        if constexpr (VB != 0) value = reinterpret_cast<const VW*>(values_in)[i];
    }
    // Stage every key, several vector loads in flight per thread (the runs are only known to be aligned to
    // their own size).
    constexpr uint32_t E = 16 / sizeof(U);
    constexpr int kBatch = 5;
    typedef U Vec __attribute__((ext_vector_type(E), aligned(sizeof(U))));
    typedef U LdsVec __attribute__((ext_vector_type(E)));
    const uint32_t vecs = n / E;
    for (uint32_t at = threadIdx.x; at < vecs; at += kBatch * kMergeBlock) {
        Vec x[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (at + j * kMergeBlock < vecs) x[j] = *reinterpret_cast<const Vec*>(kin + (at + j * kMergeBlock) * E);
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            if (at + j * kMergeBlock < vecs) {
                LdsVec y;
#pragma unroll
                for (uint32_t e = 0; e < E; ++e) y[e] = sort_bits(twiddle_in<U, KIND, DESC>(x[j][e]));
                *reinterpret_cast<LdsVec*>(s_key + (at + j * kMergeBlock) * E) = y;
            }
        }
    }
    // The rest of the last run is padded with the largest key.  Only items of earlier runs search it, and
    // those count smaller keys only, so a pad is never counted.
    const uint32_t runs = (n + kRunItems - 1) / kRunItems;
    for (uint32_t at = vecs * E + threadIdx.x; at < runs * kRunItems; at += kMergeBlock)
        s_key[at] = at < n ? sort_bits(twiddle_in<U, KIND, DESC>(kin[at])) : U(~U(0));
    __syncthreads();
    if (i >= n) return;
    const U key = s_key[i];
    const uint32_t own = blockIdx.x / (kRunItems / kMergeBlock);
    const uint32_t place = i - own * kRunItems + count_before<true>(s_key, key, 0u, own) +
                           count_before<false>(s_key, key, own + 1, runs);
    reinterpret_cast<U*>(keys_out)[place] = mine;
    if constexpr (VB != 0) reinterpret_cast<VW*>(values_out)[place] = value;
}

template <typename K, int VB, bool DESC>
int launch_small(const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* runs_keys, void* runs_values,
                 uint32_t n, uint32_t begin_bit, uint32_t bits, hipStream_t stream) {
    if (n <= kSmallOneTile) {
        LaunchScope scope("radix_small_sort", stream);
        if (n <= kRunItems)
            sort_tiles_kernel<K, DESC, VB, kRunBlock, kRunItemsPerThread>
                <<<1, kRunBlock, 0, stream>>>(keys_in, keys_out, values_in, values_out, n, begin_bit, bits);
        else
            sort_tiles_kernel<K, DESC, VB, kRunBlock, kOneItemsPerThread>
                <<<1, kRunBlock, 0, stream>>>(keys_in, keys_out, values_in, values_out, n, begin_bit, bits);
        return check_hip(hipGetLastError(), "radix_small_sort launch");
    }
    {
        LaunchScope scope("radix_small_sort", stream);
        sort_tiles_kernel<K, DESC, VB, kRunBlock, kRunItemsPerThread>
            <<<static_cast<unsigned>(ceil_div(n, kRunItems)), kRunBlock, 0, stream>>>(
                keys_in, runs_keys, values_in, runs_values, n, begin_bit, bits);
        const int st = check_hip(hipGetLastError(), "radix_small_sort launch");
        if (st != kOk) return st;
    }
    LaunchScope scope("radix_small_merge", stream);
    merge_runs_kernel<K, DESC, VB><<<static_cast<unsigned>(ceil_div(n, kMergeBlock)), kMergeBlock, 0, stream>>>(
        runs_keys, keys_out, runs_values, values_out, n, begin_bit, bits);
    return check_hip(hipGetLastError(), "radix_small_merge launch");
}

}  // namespace

template <typename K, int VB>
int small_sort(const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* runs_keys, void* runs_values,
               uint32_t n, uint32_t begin_bit, uint32_t end_bit, bool descending, hipStream_t stream) {
    const uint32_t bits = end_bit - begin_bit;
    return descending ? launch_small<K, VB, true>(keys_in, keys_out, values_in, values_out, runs_keys, runs_values, n,
                                                  begin_bit, bits, stream)
                      : launch_small<K, VB, false>(keys_in, keys_out, values_in, values_out, runs_keys, runs_values, n,
                                                   begin_bit, bits, stream);
}

#define LCPP_HIP_SMALL_SORT(K)                                                                                     \
    template int small_sort<K, 0>(const K*, K*, const void*, void*, K*, void*, uint32_t, uint32_t, uint32_t, bool, \
                                  hipStream_t);                                                                    \
    template int small_sort<K, 4>(const K*, K*, const void*, void*, K*, void*, uint32_t, uint32_t, uint32_t, bool, \
                                  hipStream_t);                                                                    \
    template int small_sort<K, 8>(const K*, K*, const void*, void*, K*, void*, uint32_t, uint32_t, uint32_t, bool, \
                                  hipStream_t);
LCPP_HIP_SMALL_SORT(uint32_t)
LCPP_HIP_SMALL_SORT(int32_t)
LCPP_HIP_SMALL_SORT(float)
LCPP_HIP_SMALL_SORT(uint64_t)
LCPP_HIP_SMALL_SORT(int64_t)
LCPP_HIP_SMALL_SORT(double)
#undef LCPP_HIP_SMALL_SORT

}  // namespace radix
}  // namespace lcpp_hip
