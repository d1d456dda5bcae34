// Key types of the radix sorts: storage words, the bit-ordered image of a key and its digits.
#pragma once

#include "common.hpp"

namespace lcpp_hip {
namespace radix {

enum KeyKind { kUnsigned = 0, kSigned = 1, kFloat = 2 };

template <typename K> struct KeyTraits;
template <> struct KeyTraits<uint32_t> { using U = uint32_t; static constexpr int kind = kUnsigned; };
template <> struct KeyTraits<int32_t> { using U = uint32_t; static constexpr int kind = kSigned; };
template <> struct KeyTraits<float> { using U = uint32_t; static constexpr int kind = kFloat; };
template <> struct KeyTraits<uint64_t> { using U = uint64_t; static constexpr int kind = kUnsigned; };
template <> struct KeyTraits<int64_t> { using U = uint64_t; static constexpr int kind = kSigned; };
template <> struct KeyTraits<double> { using U = uint64_t; static constexpr int kind = kFloat; };

template <int VB> struct ValueWord { using type = uint32_t; };
template <> struct ValueWord<8> { using type = uint64_t; };

// Bit-ordered transform (common/util_type.h:97-175 TwiddleIn/TwiddleOut; descending inverts,
// agent/radix_rank_sort_operations.h:123-155).
template <typename U, int KIND, bool DESC>
__device__ __forceinline__ U twiddle_in(U k) {
    constexpr U kHigh = U(1) << (sizeof(U) * 8 - 1);
    if constexpr (KIND == kSigned) k ^= kHigh;
    if constexpr (KIND == kFloat) k ^= (k & kHigh) ? U(~U(0)) : kHigh;
    if constexpr (DESC) k = ~k;
    return k;
}

template <typename U, int KIND, bool DESC>
__device__ __forceinline__ U twiddle_out(U k) {
    constexpr U kHigh = U(1) << (sizeof(U) * 8 - 1);
    if constexpr (DESC) k = ~k;
    if constexpr (KIND == kSigned) k ^= kHigh;
    if constexpr (KIND == kFloat) k ^= (k & kHigh) ? kHigh : U(~U(0));
    return k;
}

// Digit of a bit-ordered key.  For floats the ordered image of -0.0 is mapped to that of +0.0
// before extraction (ShiftDigitExtractor / ProcessFloatMinusZero,
// agent/radix_rank_sort_operations.h:31-62), so both zeros rank as equal keys.
template <typename U, int KIND>
__device__ __forceinline__ uint32_t digit_of(U ordered, uint32_t shift, uint32_t mask) {
    if constexpr (KIND == kFloat) {
        constexpr U kHigh = U(1) << (sizeof(U) * 8 - 1);
        if (ordered == U(~kHigh)) ordered = kHigh;
    }
    return static_cast<uint32_t>(ordered >> shift) & mask;
}

// The bits of an ordered key that a sort of bits [begin, end) compares, in the low bits of a word: two keys
// are equal for the sort exactly when these are.
template <typename U, int KIND>
struct SortBits {
    uint32_t begin;
    U mask;  // end - begin ones
    __device__ __forceinline__ U operator()(U ordered) const {
        if constexpr (KIND == kFloat) {
            constexpr U kHigh = U(1) << (sizeof(U) * 8 - 1);
            if (ordered == U(~kHigh)) ordered = kHigh;
        }
        return (ordered >> begin) & mask;
    }
};

// small_sort (radix_small.hip): sorts of up to small_sort_max(sizeof(K)) items without histogram or look-back.
// `runs_*` is a buffer of n keys (and values) other than the output, needed above kSmallOneTile items.
constexpr uint32_t kSmallOneTile = 2048;
constexpr uint32_t small_sort_max(size_t key_bytes) { return static_cast<uint32_t>((152u << 10) / key_bytes); }
template <typename K, int VB>
int small_sort(const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* runs_keys, void* runs_values,
               uint32_t n, uint32_t begin_bit, uint32_t end_bit, bool descending, hipStream_t stream);

// mid_sort (radix_mid.hip): onesweep passes over small tiles that run together, for up to kMidSortMax items.
constexpr uint32_t kMidSortMax = 1u << 21;
constexpr int kMidItems = 4;
constexpr uint32_t kMidTile = 1024 * kMidItems;
// Tiles per group of the two-level sums: one level up to 32 tiles (100,003 keys 35.1 us per call, 37.9 with groups
// of 16), then groups of 16 (262,144 keys 40.9 us, 46.1 with groups of 32).
constexpr uint32_t mid_group(uint32_t tiles) { return tiles <= 32 ? 32u : 16u; }
struct MidPlan {
    uint32_t passes;
    uint32_t tiles;    // of kMidTile keys
    uint32_t group;    // tiles per group
    uint32_t rows;     // histogram workgroups, per_row keys each
    uint32_t per_row;
    uint32_t* bins;       // passes x 256
    uint32_t* lookback;   // tiles x 256
    uint32_t* row_words;  // rows x passes x 256, in memory that pass 0 does not write
};
template <typename K, int VB>
int mid_sort(const MidPlan& plan, const K* keys_in, K* keys_out, const void* values_in, void* values_out, K* keys_tmp,
             void* values_tmp, uint32_t n, uint32_t begin_bit, uint32_t end_bit, bool descending, uint32_t spin_limit,
             hipStream_t stream);

}  // namespace radix
}  // namespace lcpp_hip
