// What the two kernels that walk down strips of output columns share: the
// layer's outputs (depthwise_columns.hip) and its weight deltas
// (depthwise_columns_deltas.hip).
#pragma once
#include "igemm_common.hpp"

#include <utility>

namespace mxk {

constexpr int kColThreads = 256;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

/// K x K taps at stride S over strips of STRIP output columns.
template <int K, int S, int STRIP> struct ColumnWalk {
  static constexpr int kColumns = S * (STRIP - 1) + K; // of input, in a strip
  static constexpr int kLive = (K + S - 1) / S; // output rows under way
  static constexpr int kPeriod = kLive * S; // input rows until they come round
};

/// Channel CH of two elements of a channel pair.
template <int CH>
__device__ __forceinline__ half2v pairOf(uint32_t first, uint32_t second) {
  return __builtin_bit_cast(
      half2v, __builtin_amdgcn_perm(second, first,
                                    CH == 0 ? 0x05040100u : 0x07060302u));
}

/// Calls each with 0, 1, ... until one answers false.
template <int... I, class F>
__device__ __forceinline__ bool whileEach(std::integer_sequence<int, I...>,
                                          F &&each) {
  return (each(std::integral_constant<int, I>{}) && ...);
}

/// Whether the layer reads input row `row`: one of rows lo .. hi - 1.
__device__ __forceinline__ bool rowIsRead(int row, uint32_t lo, uint32_t hi) {
  return uint32_t(row) - lo < hi - lo;
}

} // namespace mxk
