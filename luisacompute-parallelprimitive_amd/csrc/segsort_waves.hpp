// segsort_waves (segsort_waves.hip): sorts every segment of up to kSwMedium items in radix order.
#pragma once

#include "common.hpp"

namespace lcpp_hip {

// Items of the longest segment sorted here; segsort.hip sorts longer ones in chunks.
constexpr uint32_t kSwMedium = 4096;

enum class SegmentKeys { kUnsigned, kSigned, kFloat };

// Types whose medium segments may be sorted apart (see segsort.hip).
template <typename U, typename V, bool PAIRS>
constexpr bool kSwApart = sizeof(U) + (PAIRS ? sizeof(V) : 0) <= 8;

// Stable; in place when the outputs are the inputs.  Segments above kSwMedium are left alone, and the length of the
// longest one is posted to words[0] when `words` is set.
// Without `medium` (types of kSwApart only) it sorts the segments of 17 to 512 items and nothing else.
template <typename U, typename V, bool PAIRS>
int segsort_waves(const U* keys_in, U* keys_out, const V* values_in, V* values_out, const uint32_t* begins,
                  const uint32_t* ends, uint64_t num_segments, uint64_t n, SegmentKeys kind, uint32_t begin_bit,
                  uint32_t end_bit, bool descending, uint32_t* words, bool medium, hipStream_t stream);

}  // namespace lcpp_hip
