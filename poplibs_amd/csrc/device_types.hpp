// Device-side element conversions shared by the kernels.
#ifndef poplibs_amd_device_types_hpp
#define poplibs_amd_device_types_hpp
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mxk {

/// OCP 8-bit float -> fp32 in software.  E4M3FN: bias 7, S.1111.111 is NaN, no
/// infinities.  E5M2: bias 15, IEEE-like infinities / NaNs.  Every finite code
/// is exactly representable in fp32 (and in fp16).
__device__ __forceinline__ float decodeFp8(uint32_t code, int format) {
  const uint32_t sign = (code & 0x80u) << 24;
  uint32_t bits;
  if (format == 1) { // E4M3FN
    const uint32_t e = (code >> 3) & 0xfu, m = code & 7u;
    if (e == 0xfu && m == 7u)
      bits = 0x7fc00000u;
    else if (e == 0u)
      return __uint_as_float(sign | __float_as_uint(float(m) * 0x1p-9f));
    else
      bits = ((e + 120u) << 23) | (m << 20); // 127 - 7 = 120
  } else { // E5M2
    const uint32_t e = (code >> 2) & 0x1fu, m = code & 3u;
    if (e == 0x1fu)
      bits = m ? 0x7fc00000u : 0x7f800000u;
    else if (e == 0u)
      return __uint_as_float(sign | __float_as_uint(float(m) * 0x1p-16f));
    else
      bits = ((e + 112u) << 23) | (m << 21); // 127 - 15 = 112
  }
  return __uint_as_float(sign | bits);
}

template <class T> struct Load;
template <> struct Load<float> {
  static __device__ __forceinline__ float at(const float *p, size_t i, int) {
    return p[i];
  }
};
template <> struct Load<__half> {
  static __device__ __forceinline__ float at(const __half *p, size_t i, int) {
    return __half2float(p[i]);
  }
};
template <> struct Load<uint8_t> {
  static __device__ __forceinline__ float at(const uint8_t *p, size_t i,
                                             int format) {
    return decodeFp8(p[i], format);
  }
};

/// Two fp32 sums rounded to half, to nearest even, as fp32 values: the empty
/// asm keeps the compiler from folding the multiply-add that produced a sum
/// into the conversion (v_fma_mixlo_f16 rounds once, from the exact result),
/// which it does for some of a kernel's sums and not for others.  Every
/// vector-ALU kernel rounds through here, so that a layer's output does not
/// depend on which of them ran it - and is the fp32 partial cast to half that
/// the reference's partialsType float produces.
__device__ __forceinline__ __half2 roundPairToHalf(float a, float b) {
  asm("" : "+v"(a), "+v"(b));
  return __floats2half2_rn(a, b);
}

/// fp32 -> output element, round to nearest even.
__device__ __forceinline__ void storeOut(float *p, size_t i, float v) {
  p[i] = v;
}
__device__ __forceinline__ void storeOut(__half *p, size_t i, float v) {
  asm("" : "+v"(v)); // (as in roundPairToHalf)
  p[i] = __float2half_rn(v);
}

/// Division of a 31-bit number by a launch constant: one multiply-high and a
/// shift (round-up method: mul = ceil(2^(31 + s) / d), s = ceil(log2 d)).
struct FastDiv {
  uint32_t mul, shift, one; // one: all bits set when the divisor is 1
  __device__ __forceinline__ uint32_t operator()(uint32_t n) const {
    // a select written with bit operations: no branch, whatever the compiler
    // knows about `one`
    const uint32_t q = __umulhi(n, mul) >> shift;
    return q ^ ((q ^ n) & one);
  }
};

inline FastDiv makeFastDiv(uint32_t d) {
  if (d <= 1)
    return {0, 0, 0xffffffffu};
  uint32_t s = 0;
  while ((1ull << s) < d)
    ++s;
  const uint64_t m = ((1ull << (31 + s)) + d - 1) / d;
  return {uint32_t(m), s - 1, 0};
}

/// 16 bytes of neighbouring elements at any address: global memory takes such
/// accesses, at full speed where the address happens to be a multiple of 16.
typedef uint32_t AnyWords
    __attribute__((ext_vector_type(4), aligned(1), may_alias));
template <class T> union Piece {
  T e[16 / sizeof(T)];
  uint32_t w[4];
};
template <class T>
__device__ __forceinline__ Piece<T> loadPiece(const T *at) {
  const AnyWords v = *reinterpret_cast<const AnyWords *>(at);
  Piece<T> p;
  p.w[0] = v.x, p.w[1] = v.y, p.w[2] = v.z, p.w[3] = v.w;
  return p;
}
template <class T>
__device__ __forceinline__ void storePiece(T *at, const Piece<T> &p) {
  *reinterpret_cast<AnyWords *>(at) = AnyWords{p.w[0], p.w[1], p.w[2], p.w[3]};
}

/// The bias of E neighbouring channels, kept as it was loaded - in accesses of
/// up to 16 bytes, from any address - until it is wanted: it is on its way
/// meanwhile.  Zeros without a bias.
template <class OutT, int E> struct BiasVec {
  static constexpr int kWords = E * int(sizeof(OutT)) / 4;
  static_assert(kWords * 4 == E * int(sizeof(OutT)), "whole words");
  typedef uint32_t Words
      __attribute__((ext_vector_type(kWords), aligned(1), may_alias));
  uint32_t raw[kWords];
  __device__ __forceinline__ void load(const OutT *bias, uint32_t first) {
    Words words = {};
    if (bias)
      words = *reinterpret_cast<const Words *>(bias + first);
#pragma unroll
    for (int i = 0; i != kWords; ++i)
      raw[i] = words[i];
  }
  __device__ __forceinline__ float at(int e) const {
    if constexpr (sizeof(OutT) == 4)
      return __uint_as_float(raw[e]);
    else
      return __half2float(
          __ushort_as_half(uint16_t(raw[e / 2] >> (e % 2 * 16))));
  }
};

/// Four consecutive outputs as one vector store; p is aligned to the vector.
__device__ __forceinline__ void storeOut4(float *p, const float (&v)[4]) {
  *reinterpret_cast<float4 *>(p) = float4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ void storeOut4(__half *p, const float (&v)[4]) {
  union {
    __half2 h[2];
    uint2 u;
  } pack;
  pack.h[0] = roundPairToHalf(v[0], v[1]);
  pack.h[1] = roundPairToHalf(v[2], v[3]);
  *reinterpret_cast<uint2 *>(p) = pack.u;
}

/// Cache policy of a store that goes through the L2 to memory at once
/// (device scope) instead of leaving a dirty line there.  What a kernel leaves
/// dirty in the eight L2s is written back when it ends, before the next kernel
/// of the stream starts; for a kernel of a few microseconds whose output comes
/// all at its end that write-back is a measurable part (3x3 on 28x28, 128
/// channels: 9.1 -> 8.9 us).  Kernels that stream their output while they run
/// lose by it (1x1 on 56x56: 12.3 -> 15.5 us).
constexpr int kWriteThroughStore = 16;

typedef unsigned int ThroughWords4 __attribute__((ext_vector_type(4)));
typedef unsigned int ThroughWords2 __attribute__((ext_vector_type(2)));
/// 16 or 8 bytes into a buffer by that policy, at a multiple of their size (another
/// address gives the same bytes, more slowly: 22 MB in rows of 548 bytes took
/// 19.1 us, 12.8 by way of the L2).  A buffer store and no assembly: the compiler
/// has to see it, because a vector instruction may rewrite the registers of a
/// store of more than 8 bytes only after two wait states, and a store may read
/// an MFMA's result only after more, which it sees to.
__device__ __forceinline__ void storeThrough(__amdgpu_buffer_rsrc_t to,
                                             uint32_t byte, ThroughWords4 v) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_buffer_store_b128(v, to, byte, 0, kWriteThroughStore);
#endif
}
__device__ __forceinline__ void storeThrough(__amdgpu_buffer_rsrc_t to,
                                             uint32_t byte, ThroughWords2 v) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_buffer_store_b64(v, to, byte, 0, kWriteThroughStore);
#endif
}
/// Four consecutive outputs, the first of them element i of the buffer.
__device__ __forceinline__ void storeOut4Through(__amdgpu_buffer_rsrc_t to,
                                                 uint32_t i, const float *,
                                                 const float (&v)[4]) {
  storeThrough(to, i * 4,
               __builtin_bit_cast(ThroughWords4, float4{v[0], v[1], v[2], v[3]}));
}
__device__ __forceinline__ void storeOut4Through(__amdgpu_buffer_rsrc_t to,
                                                 uint32_t i, const __half *,
                                                 const float (&v)[4]) {
  const __half2 h[2] = {roundPairToHalf(v[0], v[1]),
                        roundPairToHalf(v[2], v[3])};
  ThroughWords2 u;
  __builtin_memcpy(&u, h, 8);
  storeThrough(to, i * 2, u);
}
/// What such a kernel is told of an output: its bytes, for the buffer's range, or 0
/// where they are more than a buffer's offset reaches.
constexpr uint32_t reachableBytes(uint64_t bytes) {
  return bytes < 0x80000000u ? uint32_t(bytes) : 0;
}

} // namespace mxk
#endif
