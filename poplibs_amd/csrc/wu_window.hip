// Weight deltas of a dense or grouped layer on the matrix cores, straight from
// the layer's own tensors and without LDS on the way in:
//   dW[g][co][ci][kh][kw] = sum over b, y, x of
//       deltas[b][y][x][g][co] *
//           acts[b][y strideH + kh - padH][x strideW + kw - padW][g][ci]
// (lib/poplin/Convolution.cpp:3437-3483 calculateWeightDeltas; wu_tap.hip has
// the same sum with a workgroup per tap and transposing LDS reads.)
//
// As a matrix product the pixels are K, and both tensors hold K outermost,
// while an MFMA lane wants eight consecutive k of one row.  Here the lane
// gathers them: lane (q, r) of a wave reads channels J r .. J r + J - 1 of
// eight neighbouring pixels of one output row (J = 2 or 4 halves, one load per
// pixel, 16 lanes a run of 16 J channels), and byte permutes pair the pixels
// up: operand j then holds channels J r + j, 8 k per lane - any assignment of
// channels to MFMA rows will do as long as the result is stored by it.  The
// eight pixels are in registers, so the taps of a kernel row are the same
// loads shifted: strideW 7 + kW columns serve them all, three taps of a unit
// stride in 10 loads instead of 24.  Nothing passes through LDS but the waves'
// sums at the end.
//
// Unit = eight columns of an output row (the last one of a row a partial one,
// its missing pixels zeroed in both operands by the permutes' selectors);
// k-step of a wave = four units, one per lane quarter; the waves of a workgroup
// take the k-steps of its chunk in turn, their sums meet in LDS.  Workgroup =
// (chunk of k-steps, tile of 16 JO output x 16 JI input channels, kernel row).
// A tile of a layer of narrow groups is as many whole groups as have room in
// it, of which the blocks on the diagonal are kept.
//
// What bounds it: a SIMD's vector ALU and matrix pipe take turns, and a k-step
// of 64 x 32 channels and three taps is 40 permutes and some 70 instructions
// of addressing beside its 24 MFMAs (960 cycles).  Wider tiles would share the
// permutes (64 x 64: 64 of them for 48 MFMAs) but leave a SIMD one wave, which
// took 2 000 cycles a k-step; narrow groups and few channels are where it
// gains most: nothing is multiplied but the tile's own blocks, against nine
// 128 x 128 tiles per group or a convolution of its own.  The pass, us, before
// and after: 32 groups of 8, 3 x 3, 31 x 32 x 32 80 -> 20; 32 of 4, 36 x 28 x 28
// 52 -> 15; 72 -> 72, 1 x 1, 21 x 9 x 9 8.9 -> 6.3; 256 -> 64, 1 x 1, 32 x 56 x 56
// 20 -> 17; over 3 500 random layers it halves the pass (geometric mean).
//
// Eight waves: their sums pass through LDS twice, 192 KB for a tile of 32 x 32 and
// three taps, which with sixteen was 1.5 us of a small layer's pass (7 x 15 x 15,
// 3 x 3 stride 2, 208 -> 64 9.7 -> 6.5 us; 21 x 39 x 39 stride 2, 32 groups of 16
// 22.4 -> 18.7; 8 x 54 x 54, 32 -> 64 13.2 -> 11.3; tiles and chunks fitted anew).
// Four are faster only where the tile is 32 x 32 and the chunk short (0.3 % over
// 330 layers), a quarter slower on long ones.  A wave's fp32 sums are twice as long
// for the same chunk, but the chunks are others: with fp32 results the deltas of 56
// layers were off by 0.97 times as much as before on average against 64-bit sums
// (0.77 to 1.21, at 0.6e-7 to 1.8e-7).
//
// With one chunk the deltas leave in weight order, one launch in all; with
// several, fp32 sums go to the workspace as [chunk][tap][g][co][ci] and
// wuWindowSumKernel adds them in order.
#include "igemm_common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mxk {
namespace {

constexpr uint32_t kWinInvalid = 0x40000000u;
constexpr uint32_t kWinUnit = 8;  // columns of a unit
constexpr uint32_t kWinUnits = 4; // units of a k-step

struct WuWindowArgs {
  WuTapDesc d;
  uint32_t units, unitsPerChunk, segs; // units of the layer, a chunk, a row
  uint32_t taps, coTiles, ciTiles, perTile;
  uint32_t tilesPerChunk;
  uint32_t resultCo, resultCi;
  uint32_t actPixelBytes, deltaPixelBytes, actRowBytes;
  uint32_t actBytes, deltaBytes;
  uint32_t strideF, strideTap; // of the result, in elements
  uint64_t chunkElems;
  uint32_t outThrough; // bytes of a chunk's, 0 where out of a buffer's reach
  FastDiv divSegs, divOutH, divTilesPerChunk, divKH, divCiTiles, divCoTiles;
  FastDiv divCo;
};

struct WinPlace {
  uint32_t chunk, g0, coTile, ciTile, kh;
};

/// Workgroup -> (chunk, groups, co tile, ci tile, kernel row), the row fastest;
/// an XCD gets whole chunks.
__device__ __forceinline__ WinPlace placeOfWorkgroup(const WuWindowArgs &a) {
  WinPlace w;
  const uint32_t block = xcdSwizzle(blockIdx.x, gridDim.x);
  w.chunk = a.divTilesPerChunk(block);
  uint32_t id = block - w.chunk * a.tilesPerChunk;
  uint32_t over = a.divKH(id);
  w.kh = id - over * a.d.kH;
  id = over, over = a.divCiTiles(id);
  w.ciTile = id - over * a.ciTiles;
  id = over, over = a.divCoTiles(id);
  w.coTile = id - over * a.coTiles;
  w.g0 = over * a.perTile;
  return w;
}

/// The waves' sums meet in LDS, a tap at a time, and leave.
template <int JO, int JI, int KW, int NW, class OutT>
__device__ __forceinline__ void
storeWindow(const WuWindowArgs &a, const WinPlace &w,
            const floatx4 (&acc)[KW][JO][JI], char *lds, OutT *out) {
  const WuTapDesc &d = a.d;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t q = (t & 63) >> 4, r = t & 15;
  // Lane (q, r) holds output channels JO r + i and the 4 JI input channels from
  // 4 JI q on (register n of block j is JI n + j of them): JI pieces of four,
  // the output channel's pieces JI q and up.  A piece's place within its 16
  // rotates, so that neither the writes nor the reads, which go along an output
  // channel, meet in a bank.
  constexpr int kPieces = 4 * JI; // of an output channel
  auto placeOf = [](uint32_t i, uint32_t p, uint32_t rr) {
    const uint32_t v = p % JI, qq = p / JI;
    return (i * JI + v) * 64 + qq * 16 +
           ((rr + p + (JI == 2 ? 8 * (i & 1) : 0)) & 15);
  };
  floatx4 *sums = reinterpret_cast<floatx4 *>(lds);
  constexpr int kVectors = JO * JI * 64; // of the tile
  const uint32_t tap0 = w.kh * KW;
#pragma unroll
  for (int k = 0; k != KW; ++k) {
    if (k != 0)
      __syncthreads();
#pragma unroll
    for (int i = 0; i != JO; ++i)
#pragma unroll
      for (int v = 0; v != JI; ++v) {
        floatx4 x;
#pragma unroll
        for (int n = 0; n != 4; ++n)
          x[n] = acc[k][i][(4 * v + n) % JI][(4 * v + n) / JI];
        sums[wave * kVectors + placeOf(i, q * JI + v, r)] = x;
      }
    __syncthreads();
    for (int e = t; e < kVectors; e += 64 * NW) {
      const uint32_t co = e / kPieces, p = e % kPieces;
      const uint32_t place = placeOf(co % JO, p, co / JO);
      floatx4 total = sums[place];
#pragma unroll
      for (int other = 1; other != NW; ++other)
        total += sums[other * kVectors + place];
      const uint32_t ci = p * 4;
      OutT *to = out + w.chunk * a.chunkElems + (tap0 + k) * a.strideTap;
      if (a.perTile == 1) {
        const uint32_t coIn = w.coTile * (16 * JO) + co,
                       ciIn = w.ciTile * (16 * JI) + ci;
        if (coIn >= a.resultCo || ciIn >= a.resultCi)
          continue;
        const size_t f =
            (size_t(w.g0) * a.resultCo + coIn) * a.resultCi + ciIn;
        if (a.strideF == 1 && a.resultCi % 4 == 0 && a.outThrough) {
          const float v[4] = {total[0], total[1], total[2], total[3]};
          storeOut4Through(bufferOf(to, a.outThrough), uint32_t(f), out, v);
        } else {
#pragma unroll
          for (uint32_t x = 0; x != 4; ++x)
            if (ciIn + x < a.resultCi)
              storeOut(to, (f + x) * a.strideF, total[x]);
        }
      } else {
        const uint32_t gl = a.divCo(co), coIn = co - gl * d.co;
        if (gl >= a.perTile || w.g0 + gl >= d.groups || coIn >= a.resultCo)
          continue;
        const size_t f = (size_t(w.g0 + gl) * a.resultCo + coIn) * a.resultCi;
#pragma unroll
        for (uint32_t x = 0; x != 4; ++x) {
          const uint32_t ciIn = ci + x - gl * d.ci;
          if (ciIn < a.resultCi)
            storeOut(to, (f + ciIn) * a.strideF, total[x]);
        }
      }
    }
  }
}

template <int J> struct WinLoad;
template <> struct WinLoad<2> {
  typedef uint32_t Words __attribute__((ext_vector_type(1)));
  static __device__ __forceinline__ Words at(__amdgpu_buffer_rsrc_t b,
                                             uint32_t off) {
    Words w;
    w[0] = __builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0);
    return w;
  }
};
template <> struct WinLoad<4> {
  typedef uint32_t Words __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ Words at(__amdgpu_buffer_rsrc_t b,
                                             uint32_t off) {
    return __builtin_bit_cast(
        Words, __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0));
  }
};

/// JO, JI: channels per lane of deltas and activations; KW: taps of a kernel
/// row; S: strideW; NW: waves.
template <int JO, int JI, int KW, int S, int NW, class OutT>
__global__ __launch_bounds__(64 * NW) void wuWindowKernel(
    const WuWindowArgs a, const char *__restrict__ acts,
    const char *__restrict__ deltas, OutT *__restrict__ out) {
  constexpr int NX = S * 7 + KW; // columns a unit's taps read
  extern __shared__ __align__(16) char lds[];
  const WuTapDesc &d = a.d;
  const int t = threadIdx.x;
  const int lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t q = lane >> 4, r = lane & 15;

  const WinPlace place = placeOfWorkgroup(a);
  const auto [chunk, g0, coTile, ciTile, kh] = place;
  const uint32_t u0 = chunk * a.unitsPerChunk;
  const uint32_t u1 =
      u0 + a.unitsPerChunk < a.units ? u0 + a.unitsPerChunk : a.units;

  const __amdgpu_buffer_rsrc_t actBuf = bufferOf(acts, a.actBytes);
  const __amdgpu_buffer_rsrc_t deltaBuf = bufferOf(deltas, a.deltaBytes);
  // (channels behind the group's last are a neighbour's: they end up in rows
  // and columns that are not stored)
  const uint32_t actLane = (g0 * d.ci + ciTile * (16 * JI) + JI * r) * 2;
  const uint32_t deltaLane = (g0 * d.co + coTile * (16 * JO) + JO * r) * 2;

  const uint32_t actFirst = actLane - uint32_t(d.padW) * a.actPixelBytes;

  using DeltaLoad = WinLoad<JO>;
  using ActLoad = WinLoad<JI>;
  struct Raw {
    typename DeltaLoad::Words delta[8];
    typename ActLoad::Words act[NX];
    uint32_t here; // pixels of the unit
  };
  auto load = [&](Raw &x, uint32_t first) {
    const uint32_t u = first + q;
    const uint32_t row = a.divSegs(u), seg = u - row * a.segs;
    const uint32_t b = a.divOutH(row), y = row - b * d.outH;
    const uint32_t x0 = seg * kWinUnit;
    const bool valid = u < u1;
    const uint32_t left = d.outW - x0;
    x.here = valid ? (left < kWinUnit ? left : kWinUnit) : 0u;
    // (24-bit products, four times as fast: wuWindowTakes sees to the ranges)
    uint32_t at =
        valid ? __umul24(__umul24(row, d.outW) + x0, a.deltaPixelBytes) +
                    deltaLane
              : kWinInvalid;
#pragma unroll
    for (int i = 0; i != 8; ++i)
      x.delta[i] = DeltaLoad::at(deltaBuf, at + i * a.deltaPixelBytes);
    const uint32_t iy = __umul24(y, d.strideH) + kh - uint32_t(d.padH);
    const uint32_t ix = x0 * S - uint32_t(d.padW);
    const bool rowIn = valid && iy - d.loH < d.hiH - d.loH;
    // (ix may be negative, the product of which is taken off afterwards; what
    // a row outside the input gives is not used)
    at = __umul24(__umul24(b, d.inH) + iy, a.actRowBytes) +
         __umul24(x0 * S, a.actPixelBytes) + actFirst;
    const uint32_t span = rowIn ? d.hiW - d.loW : 0u;
#pragma unroll
    for (int i = 0; i != NX; ++i)
      x.act[i] = ActLoad::at(actBuf, ix + i - d.loW < span
                                         ? at + i * a.actPixelBytes
                                         : kWinInvalid);
  };

  floatx4 acc[KW][JO][JI];
#pragma unroll
  for (int k = 0; k != KW; ++k)
#pragma unroll
    for (int i = 0; i != JO; ++i)
#pragma unroll
      for (int j = 0; j != JI; ++j)
        acc[k][i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

  auto multiply = [&](const Raw &x) {
    // Permute selectors per pair of pixels: both, the first alone, neither
    // (0x0c: a zero byte); for the even and the odd channel of a word.
    uint32_t even[4], odd[4];
#pragma unroll
    for (int m = 0; m != 4; ++m) {
      const bool two = x.here > 2u * m + 1, one = x.here > 2u * m;
      even[m] = two ? 0x05040100u : one ? 0x0c0c0100u : 0x0c0c0c0cu;
      odd[m] = two ? 0x07060302u : one ? 0x0c0c0302u : 0x0c0c0c0cu;
    }
    uintx4 rows[JO];
#pragma unroll
    for (int w = 0; w != JO / 2; ++w)
#pragma unroll
      for (int m = 0; m != 4; ++m) {
        const uint32_t lo = x.delta[2 * m][w], hi = x.delta[2 * m + 1][w];
        rows[2 * w][m] = __builtin_amdgcn_perm(hi, lo, even[m]);
        rows[2 * w + 1][m] = __builtin_amdgcn_perm(hi, lo, odd[m]);
      }
#pragma unroll
    for (int k = 0; k != KW; ++k) {
      uintx4 cols[JI];
#pragma unroll
      for (int w = 0; w != JI / 2; ++w)
#pragma unroll
        for (int m = 0; m != 4; ++m) {
          const uint32_t lo = x.act[S * 2 * m + k][w],
                         hi = x.act[S * (2 * m + 1) + k][w];
          cols[2 * w][m] = __builtin_amdgcn_perm(hi, lo, even[m]);
          cols[2 * w + 1][m] = __builtin_amdgcn_perm(hi, lo, odd[m]);
        }
      // The activations are the MFMA's row operand: a lane then has JI x 4
      // consecutive input channels of one output channel.
#pragma unroll
      for (int i = 0; i != JO; ++i)
#pragma unroll
        for (int j = 0; j != JI; ++j)
          acc[k][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(half8, cols[j]),
              __builtin_bit_cast(half8, rows[i]), acc[k][i][j], 0, 0, 0);
    }
  };

  // The loads of the wave's next k-step go out before this one's MFMAs.
  // (Pinned: left to itself the compiler issues them behind those.)  No k-step
  // beyond the wave's last is multiplied: an odd count rounded up cost 5 % of
  // the pass over 42 layers, up to 15 (10 x 31 x 31 stride 2, 56 -> 56 8.8 us,
  // 7.6; 5 x 30 x 30 stride 2, 160 -> 88 10.1, 8.8).  It is the loop that ends
  // early, not its body in the middle: with a way out between the two halves 446
  // layers are 3 % slower, those of long walks and 32 groups up to 10 (32 x 42 x 42,
  // 32 groups of 8 30.5 us, 26.8).  Loads a k-step further ahead
  // gain nothing, and neither do fewer instructions: 82 requests of 128 bytes
  // to the L2 per k-step of 64 x 32 channels, most of them for half a line or
  // two halves, keep the way from there busy.
  constexpr uint32_t kStride = NW * kWinUnits;
  uint32_t at = u0 + wave * kWinUnits;
  Raw even, odd;
  load(even, at);
  for (; at + kStride < u1; at += 2 * kStride) {
    load(odd, at + kStride);
    __builtin_amdgcn_sched_barrier(0);
    multiply(even);
    __builtin_amdgcn_sched_barrier(0);
    load(even, at + 2 * kStride);
    __builtin_amdgcn_sched_barrier(0);
    multiply(odd);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (at < u1)
    multiply(even);

  storeWindow<JO, JI, KW, NW>(a, place, acc, lds, out);
}

template <int J> struct WinFloats;
template <> struct WinFloats<1> {
  typedef float Words __attribute__((ext_vector_type(1)));
  static __device__ __forceinline__ Words at(__amdgpu_buffer_rsrc_t b,
                                             uint32_t off) {
    Words w;
    w[0] = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(b, off, 0, 0));
    return w;
  }
};
template <> struct WinFloats<2> {
  typedef float Words __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ Words at(__amdgpu_buffer_rsrc_t b,
                                             uint32_t off) {
    return __builtin_bit_cast(
        Words, __builtin_amdgcn_raw_buffer_load_b64(b, off, 0, 0));
  }
};
template <> struct WinFloats<3> {
  typedef float Words __attribute__((ext_vector_type(3)));
  static __device__ __forceinline__ Words at(__amdgpu_buffer_rsrc_t b,
                                             uint32_t off) {
    return __builtin_bit_cast(
        Words, __builtin_amdgcn_raw_buffer_load_b96(b, off, 0, 0));
  }
};

/// The same for fp32 tensors, with an MFMA for each of a unit's pixels: lane
/// (q, r) brings channels J r .. J r + J - 1 of pixel m of its unit, and k is
/// the lane quarter, so the loads are the operands as they are.  Nothing is
/// permuted; the matrix pipe (32 cycles for 16 x 16 x 4) is the bound, and
/// tiles of J = 1, 2 or 3 blocks both ways leave little of it to padding.  The
/// passes of these layers were convolutions of their own between two
/// rearrangements, four launches and more; us before and after, a pass in a
/// replayed graph: 48 -> 43 channels, 3 x 3, 15 x 9 x 9 28.2 -> 9.6; 312 -> 160,
/// 1 x 1 stride 2, 10 x 15 x 15 34.7 -> 5.8; 32 groups of 16, 3 x 3, 64 x 16 x 16
/// 224 -> 40; 128 -> 128, 3 x 3, 36 x 56 x 56 346 -> 275 (the matrix pipe's own
/// time 222).  Over 14 150 random layers of up to 512 channels and 10 GFLOP 3.8
/// times as fast (geometric mean).  Rows of few columns leave a unit of eight
/// half empty: wide layers of them are where it loses (floatWindowAsked in
/// Plan.cpp).
template <int J, int KW, int S, int NW, class OutT>
__global__ __launch_bounds__(64 * NW) void wuWindowFloatKernel(
    const WuWindowArgs a, const char *__restrict__ acts,
    const char *__restrict__ deltas, OutT *__restrict__ out) {
  constexpr int NX = S * 7 + KW; // columns a unit's taps read
  extern __shared__ __align__(16) char lds[];
  const WuTapDesc &d = a.d;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t q = (t & 63) >> 4, r = t & 15;
  const WinPlace place = placeOfWorkgroup(a);
  const auto [chunk, g0, coTile, ciTile, kh] = place;
  const uint32_t u0 = chunk * a.unitsPerChunk;
  const uint32_t u1 =
      u0 + a.unitsPerChunk < a.units ? u0 + a.unitsPerChunk : a.units;
  const __amdgpu_buffer_rsrc_t actBuf = bufferOf(acts, a.actBytes);
  const __amdgpu_buffer_rsrc_t deltaBuf = bufferOf(deltas, a.deltaBytes);
  const uint32_t actLane = (g0 * d.ci + ciTile * (16 * J) + J * r) * 4;
  const uint32_t deltaLane = (g0 * d.co + coTile * (16 * J) + J * r) * 4;
  const uint32_t actFirst = actLane - uint32_t(d.padW) * a.actPixelBytes;

  struct Raw {
    typename WinFloats<J>::Words delta[8], act[NX];
    uint32_t here; // pixels of the unit
  };
  auto load = [&](Raw &x, uint32_t first) {
    const uint32_t u = first + q;
    const uint32_t row = a.divSegs(u), seg = u - row * a.segs;
    const uint32_t b = a.divOutH(row), y = row - b * d.outH;
    const uint32_t x0 = seg * kWinUnit;
    const bool valid = u < u1;
    const uint32_t left = d.outW - x0;
    x.here = valid ? (left < kWinUnit ? left : kWinUnit) : 0u;
    uint32_t at = __umul24(__umul24(row, d.outW) + x0, a.deltaPixelBytes) +
                  deltaLane;
#pragma unroll
    for (uint32_t i = 0; i != 8; ++i)
      x.delta[i] = WinFloats<J>::at(
          deltaBuf, i < x.here ? at + i * a.deltaPixelBytes : kWinInvalid);
    const uint32_t iy = __umul24(y, d.strideH) + kh - uint32_t(d.padH);
    const uint32_t ix = x0 * S - uint32_t(d.padW);
    const bool rowIn = valid && iy - d.loH < d.hiH - d.loH;
    at = __umul24(__umul24(b, d.inH) + iy, a.actRowBytes) +
         __umul24(x0 * S, a.actPixelBytes) + actFirst;
    const uint32_t span = rowIn ? d.hiW - d.loW : 0u;
#pragma unroll
    for (int i = 0; i != NX; ++i)
      x.act[i] = WinFloats<J>::at(actBuf, ix + i - d.loW < span
                                              ? at + i * a.actPixelBytes
                                              : kWinInvalid);
  };

  floatx4 acc[KW][J][J];
#pragma unroll
  for (int k = 0; k != KW; ++k)
#pragma unroll
    for (int i = 0; i != J; ++i)
#pragma unroll
      for (int j = 0; j != J; ++j)
        acc[k][i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

  // (a partial unit's missing pixels are zero in both operands: an activation
  // that another tap's product has, and that is infinite, would else meet a
  // zero here)
  auto multiply = [&](const Raw &x, auto partial) {
#pragma unroll
    for (int m = 0; m != 8; ++m)
#pragma unroll
      for (int k = 0; k != KW; ++k)
#pragma unroll
        for (int j = 0; j != J; ++j) {
          float v = x.act[S * m + k][j];
          if constexpr (decltype(partial)::value)
            v = uint32_t(m) < x.here ? v : 0.0f;
#pragma unroll
          for (int i = 0; i != J; ++i)
            acc[k][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                v, x.delta[m][i], acc[k][i][j], 0, 0, 0);
        }
  };
  auto both = [&](const Raw &x) {
    if (__any(x.here != 8 && x.here != 0))
      multiply(x, std::true_type{});
    else
      multiply(x, std::false_type{});
  };
  constexpr uint32_t kStride = NW * kWinUnits;
  uint32_t at = u0 + wave * kWinUnits;
  Raw even, odd;
  load(even, at);
  for (; at + kStride < u1; at += 2 * kStride) {
    load(odd, at + kStride);
    __builtin_amdgcn_sched_barrier(0);
    both(even);
    __builtin_amdgcn_sched_barrier(0);
    load(even, at + 2 * kStride);
    __builtin_amdgcn_sched_barrier(0);
    both(odd);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (at < u1)
    both(even);
  storeWindow<J, J, KW, NW>(a, place, acc, lds, out);
}

/// out[f][tap] = sum over the chunks, in order, of partial[chunk][tap][f] for
/// f = (g, co, ci), a tap's sums filled up to whole vectors.  Workgroup = `per` runs of 64 f and all their taps
/// (kWinSlots slots at most): 16 lanes read 256 bytes of a tap, slot (run, tap,
/// part) the chunks part, part + parts, ..., four loads in flight; the parts
/// meet in LDS, whence the runs leave in weight order.
constexpr uint32_t kWinSlots = 64, kWinParts = 32;
struct WuWindowSumArgs {
  uint32_t chunks, taps, total, sums; // f, and as the workspace holds them
  uint32_t tapsHere, parts, per;
  FastDiv divParts, divTaps;
};
template <class OutT>
__global__ __launch_bounds__(1024) void wuWindowSumKernel(
    const float *__restrict__ partial, OutT *__restrict__ out,
    const WuWindowSumArgs a) {
  __shared__ floatx4 sums[kWinSlots * 16];
  const uint32_t f0 = blockIdx.x * a.per * 64;
  const uint32_t tap0 = blockIdx.y * a.tapsHere;
  const uint32_t left = a.taps - tap0;
  const uint32_t taps = left < a.tapsHere ? left : a.tapsHere;
  const uint32_t slot = threadIdx.x >> 4;
  const uint32_t sum = a.divParts(slot), part = slot - sum * a.parts;
  const uint32_t runHere = a.divTaps(sum), tapHere = sum - runHere * a.tapsHere;
  const uint32_t f = f0 + runHere * 64 + (threadIdx.x & 15) * 4;
  if (runHere < a.per && tapHere < taps && f < a.total) {
    const size_t stride = size_t(a.taps) * a.sums / 4;
    const floatx4 *src = reinterpret_cast<const floatx4 *>(partial) +
                         (size_t(tap0 + tapHere) * a.sums + f) / 4;
    floatx4 total = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t p = part;
    for (; p + 3 * a.parts < a.chunks; p += 4 * a.parts) {
      const floatx4 v0 = src[p * stride];
      const floatx4 v1 = src[(p + a.parts) * stride];
      const floatx4 v2 = src[(p + 2 * a.parts) * stride];
      const floatx4 v3 = src[(p + 3 * a.parts) * stride];
      total += (v0 + v1) + (v2 + v3);
    }
    for (; p < a.chunks; p += a.parts)
      total += src[p * stride];
    sums[threadIdx.x] = total;
  }
  __syncthreads();
  const float *flat = reinterpret_cast<const float *>(sums);
  const uint32_t run = 64 * a.per * a.tapsHere;
  for (uint32_t e = threadIdx.x; e < run; e += blockDim.x) {
    const uint32_t i = a.divTaps(e), tap = e - i * a.tapsHere;
    if (tap >= taps || f0 + i >= a.total)
      continue;
    float v = 0.0f;
    const uint32_t first = ((i >> 6) * a.tapsHere + tap) * a.parts;
    for (uint32_t p = 0; p != a.parts; ++p)
      v += flat[(first + p) * 64 + (i & 63)];
    storeOut(out, size_t(f0 + i) * a.taps + tap0 + tap, v);
  }
}

struct WinShape {
  uint32_t segs, units, perTile, coTiles, ciTiles, groupTiles, chunks;
  uint64_t tiles, elems;
  uint32_t sums; // of a tap in the workspace: whole vectors of four
};

WinShape winShape(const WuTapDesc &d) {
  WinShape s{};
  s.segs = (d.outW + kWinUnit - 1) / kWinUnit;
  s.units = d.batch * d.outH * s.segs;
  const uint32_t tile = std::min(d.windowCo, d.windowCi);
  s.perTile = std::max(
      1u, std::min(d.groups, tile / std::max(1u, std::max(d.co, d.ci))));
  s.groupTiles = (d.groups + s.perTile - 1) / s.perTile;
  s.coTiles = (s.perTile * d.co + d.windowCo - 1) / d.windowCo;
  s.ciTiles = (s.perTile * d.ci + d.windowCi - 1) / d.windowCi;
  s.tiles = uint64_t(s.groupTiles) * s.coTiles * s.ciTiles * d.kH;
  const uint32_t steps = (s.units + kWinUnits - 1) / kWinUnits;
  s.chunks = d.windowSteps ? (steps + d.windowSteps - 1) / d.windowSteps : 0;
  const uint32_t rco = d.resultCo ? d.resultCo : d.co,
                 rci = d.resultCi ? d.resultCi : d.ci;
  s.elems = uint64_t(d.groups) * rco * rci * d.kH * d.kW;
  s.sums = uint32_t((uint64_t(d.groups) * rco * rci + 3) / 4 * 4);
  return s;
}

} // namespace

bool wuWindowTakes(const WuTapDesc &d) {
  const uint64_t M = uint64_t(d.batch) * d.outH * d.outW;
  if (M == 0 || d.ci == 0 || d.co == 0 || d.groups == 0 || d.kH == 0)
    return false;
  if ((d.kW != 1 && d.kW != 3) || d.strideH == 0 ||
      (d.strideW != 1 && d.strideW != 2))
    return false;
  const bool floats = d.elemBytes == 4;
  if (d.elemBytes != 2 && !floats)
    return false;
  if (floats) {
    if (d.windowCo != d.windowCi || (d.windowCo != 16 && d.windowCo != 32 &&
                                     d.windowCo != 48))
      return false;
  } else if (((d.windowCo != 32 || d.windowCi != 32) &&
       (d.windowCo != 64 || d.windowCi != 32) &&
       (d.windowCo != 32 || d.windowCi != 64)))
    return false;
  if (d.windowSteps == 0)
    return false;
  // words of two channels at multiples of four bytes
  const uint64_t actPixel = uint64_t(d.groups) * d.ci * d.elemBytes,
                 deltaPixel = uint64_t(d.groups) * d.co * d.elemBytes;
  if (actPixel % 4 != 0 || deltaPixel % 4 != 0)
    return false;
  if (!floats && d.groups > 1 && (d.ci % 2 != 0 || d.co % 2 != 0))
    return false;
  if (d.resultCi > d.ci || d.resultCo > d.co)
    return false;
  // (a unit's columns beyond a row's end are addressed too: they stay below
  // kWinInvalid twice over)
  if (uint64_t(d.batch) * d.inH * d.inW * actPixel +
              64 * (actPixel + 256) >= kWinInvalid ||
      M * deltaPixel + 64 * (deltaPixel + 256) >= kWinInvalid)
    return false;
  // 24-bit products: rows, pixels, bytes of a pixel and of an input row
  const uint64_t k24 = 1u << 24;
  const WinShape s = winShape(d);
  if (uint64_t(d.batch) * d.outH * s.segs * kWinUnit >= k24 ||
      uint64_t(d.batch) * d.inH + d.kH >= k24 || M >= k24 ||
      (uint64_t(d.batch) * d.inH > 1 && d.inW * actPixel >= k24) ||
      actPixel >= k24 || deltaPixel >= k24 ||
      uint64_t(d.outH) * d.strideH >= k24 ||
      uint64_t(d.outW + kWinUnit) * d.strideW >= k24 ||
      d.padH < -(1 << 20) || d.padH > (1 << 20) || d.padW < -(1 << 20) ||
      d.padW > (1 << 20))
    return false;
  return s.chunks * s.tiles <= 0x7fffffffull && s.elems < (1ull << 31) &&
         wuWindowWorkspaceBytes(d) <= (1ull << 31);
}

uint64_t wuWindowWorkspaceBytes(const WuTapDesc &d) {
  const WinShape s = winShape(d);
  return s.chunks > 1 ? uint64_t(s.chunks) * d.kH * d.kW * s.sums * 4 : 0;
}

uint64_t wuWindowWorkgroups(const WuTapDesc &d) {
  const WinShape s = winShape(d);
  return s.chunks * s.tiles;
}

namespace {
/// The pass's time by tile, kernel columns and stride along a row: `call`, a
/// workgroup's k-steps at the pace of a wave (`wave` each of its own) or of the
/// CU (`step`), `round` + `roundStep` per k-step and round of workgroups beyond
/// the first, and the second launch with its partial sums or the one launch's
/// scattered results.  `places` rounds the workgroups of a CU up, to a whole one (1)
/// or a third (3): a fitted number, not the workgroups that a CU holds (by registers
/// two to three of every kernel here).  Fitted to 7 000 measurements on 330 layers
/// (4 to 64 images, fields of 7 to 64, 4 to 512 channels, up to 32 groups), within 5
/// to 9 %; the tile and chunks picked by it are on average 1.8 % behind the best of
/// those measured.  Larger layers go by it too: of 70 with up to 600 GFLOP the pass
/// is 1.06 times as fast on average as by the fit before, the slowest 0.88 (chunks of
/// a thousand k-steps cut into rounds: 224 x 42 x 42, 136 -> 120 274 us, 312 so).
struct WinFit {
  double call, wave, step, round, roundStep, second, partialMB, resultMB, places;
};
constexpr WinFit kWinFits[3][2][2] = {
    // 32 x 32: one column, three; stride 1, 2
    {{{3.00, 0.505, 0.080, 0.6, 0.090, 2.8, 0.66, 3.05, 1},
      {3.69, 0.372, 0.066, 1.0, 0.078, 2.5, 0.44, 1.45, 3}},
     {{5.29, 0.025, 0.088, 2.0, 0.071, 3.0, 0.40, 2.00, 1},
      {5.64, 0.593, 0.102, 3.4, 0.133, 2.8, 0.34, 1.29, 1}}},
    // 64 output x 32 input channels
    {{{3.51, 0.055, 0.105, 0.9, 0.125, 2.9, 0.55, 2.25, 1},
      {4.22, 0.153, 0.091, 1.1, 0.135, 2.4, 0.52, 0.58, 3}},
     {{6.48, 0.213, 0.110, 4.8, 0.107, 2.9, 0.47, 2.37, 1},
      {7.10, 0.233, 0.128, 4.8, 0.147, 2.5, 0.46, 2.28, 1}}},
    // 32 x 64
    {{{3.46, 0.143, 0.099, 0.9, 0.122, 2.9, 0.55, 0.60, 1},
      {4.12, 0.170, 0.085, 1.1, 0.143, 2.5, 0.49, 0.54, 3}},
     {{6.96, 0.099, 0.113, 5.0, 0.115, 2.8, 0.43, 2.12, 1},
      {7.76, 0.011, 0.154, 5.2, 0.174, 2.3, 0.44, 1.97, 1}}}};

/// fp32: tiles of 16, 32 and 48; one column, three (both strides).  Fitted to
/// 6 200 measurements on 340 layers, within 8 to 10 %; the pick 2 % behind the
/// best on average.
constexpr WinFit kWinFloatFits[3][2] = {
    {{4.63, 0.041, 0.077, 1.3, 0.113, 2.0, 3.15, 1.17, 2},
     {6.85, 0.011, 0.151, 4.2, 0.149, 2.5, 0.41, 0.78, 1}},
    {{4.99, 0.051, 0.178, 1.8, 0.186, 2.4, 0.85, 0.76, 2},
     {8.16, 0.018, 0.435, 6.5, 0.423, 3.3, 0.36, 1.48, 1}},
    {{5.72, 1.372, 0.311, 3.0, 0.340, 2.4, 0.54, 0.0, 2},
     {9.59, 3.941, 0.930, 10.5, 0.908, 4.1, 0.35, 1.29, 1}}};

uint32_t floatWaves(uint32_t tile) {
  return tile == 16 ? 16 : tile == 32 ? 8 : 4;
}

double winEstimateUs(const WuTapDesc &d, const WinShape &s,
                     uint32_t computeUnits) {
  const bool floats = d.elemBytes == 4;
  const int tile = floats                ? int(d.windowCo / 16) - 1
                   : d.windowCo == 64    ? 1
                   : d.windowCi == 64    ? 2
                                         : 0;
  const WinFit &f = floats ? kWinFloatFits[tile][d.kW == 1 ? 0 : 1]
                           : kWinFits[tile][d.kW == 1 ? 0 : 1][d.strideW - 1];
  const uint32_t waves = floats ? floatWaves(d.windowCo) : 8;
  const double steps = d.windowSteps;
  const double perCU = std::max(
      1.0, std::ceil(f.places * double(s.chunks * s.tiles) / computeUnits) /
               f.places);
  const double mb = double(s.elems) * 1e-6;
  return f.call + std::max(f.wave * std::ceil(steps / waves), f.step * steps) +
         (perCU - 1) * (f.round + f.roundStep * steps) +
         (s.chunks > 1 ? f.second + f.partialMB * 4 * mb * s.chunks
                       : f.resultMB * d.elemBytes * mb);
}
} // namespace

double wuWindowChoose(WuTapDesc &d, uint32_t computeUnits) {
  if ((d.kW != 1 && d.kW != 3) || (d.strideW != 1 && d.strideW != 2))
    return 1e30;
  // A 1 x 1 kernel that meets every pixel once: the field as one long row, so
  // that every unit is a whole one.
  if (d.kH == 1 && d.kW == 1 && d.strideH == 1 && d.strideW == 1 &&
      d.padH == 0 && d.padW == 0 && d.inH == d.outH && d.inW == d.outW &&
      d.loH == 0 && d.hiH == d.inH && d.loW == 0 && d.hiW == d.inW &&
      uint64_t(d.batch) * d.inH * d.inW < (1u << 23)) {
    d.inW = d.outW = d.hiW = d.batch * d.inH * d.inW;
    d.batch = d.inH = d.outH = d.hiH = 1;
  }
  double bestUs = 1e30;
  WuTapDesc best = d;
  for (uint32_t tile = 0; tile != 3; ++tile) {
    WuTapDesc t = d;
    t.windowCo = tile == 1 ? 64 : 32, t.windowCi = tile == 2 ? 64 : 32;
    if (d.elemBytes == 4)
      t.windowCo = t.windowCi = 16 * (tile + 1);
    t.windowSteps = 1;
    const WinShape one = winShape(t);
    if (one.tiles == 0 || (d.elemBytes == 2 && tile != 0 && one.perTile > 1))
      continue;
    const uint32_t steps = one.chunks;
    // (four workgroups for every CU at most: more lose to their own start)
    const uint64_t most =
        std::max<uint64_t>(1, 4ull * computeUnits / one.tiles);
    // (every count of chunks up to 16, then one in sixteen)
    for (uint32_t n = 1; n <= std::min<uint64_t>(steps, most);
         n += std::max(1u, n / 16)) {
      t.windowSteps = (steps + n - 1) / n;
      const WinShape s = winShape(t);
      const double us = winEstimateUs(t, s, computeUnits);
      if (us < bestUs && wuWindowTakes(t))
        bestUs = us, best = t;
    }
  }
  d = best;
  return bestUs;
}

namespace {
template <int JO, int JI, int KW, int S>
hipError_t launchWindow(const WuWindowArgs &a, uint32_t blocks, int outType,
                        const void *acts, const void *deltas, void *out,
                        hipStream_t stream) {
  constexpr int NW = 8, kLds = NW * JO * JI * 1024;
  static_assert(kLds <= 64 * 1024, "within the LDS of any launch");
  const dim3 grid(blocks), block(64 * NW);
  const char *x = static_cast<const char *>(acts);
  const char *dz = static_cast<const char *>(deltas);
  if (outType == kHalf)
    hipLaunchKernelGGL((wuWindowKernel<JO, JI, KW, S, NW, __half>), grid,
                       block, kLds, stream, a, x, dz,
                       static_cast<__half *>(out));
  else
    hipLaunchKernelGGL((wuWindowKernel<JO, JI, KW, S, NW, float>), grid, block,
                       kLds, stream, a, x, dz, static_cast<float *>(out));
  return hipGetLastError();
}

template <int J, int KW, int S>
hipError_t launchWindowFloat(const WuWindowArgs &a, uint32_t blocks,
                             int outType, const void *acts, const void *deltas,
                             void *out, hipStream_t stream) {
  constexpr int NW = J == 1 ? 16 : J == 2 ? 8 : 4; // (floatWaves)
  constexpr int kLds = NW * J * J * 1024;
  const dim3 grid(blocks), block(64 * NW);
  const char *x = static_cast<const char *>(acts);
  const char *dz = static_cast<const char *>(deltas);
  if (outType == kHalf)
    hipLaunchKernelGGL((wuWindowFloatKernel<J, KW, S, NW, __half>), grid, block,
                       kLds, stream, a, x, dz, static_cast<__half *>(out));
  else
    hipLaunchKernelGGL((wuWindowFloatKernel<J, KW, S, NW, float>), grid, block,
                       kLds, stream, a, x, dz, static_cast<float *>(out));
  return hipGetLastError();
}

template <int J>
hipError_t launchWindowFloats(const WuWindowArgs &a, uint32_t blocks,
                              int outType, const void *acts,
                              const void *deltas, void *out,
                              hipStream_t stream) {
  const auto go = a.d.kW == 1
                      ? a.d.strideW == 1 ? &launchWindowFloat<J, 1, 1>
                                         : &launchWindowFloat<J, 1, 2>
                      : a.d.strideW == 1 ? &launchWindowFloat<J, 3, 1>
                                         : &launchWindowFloat<J, 3, 2>;
  return go(a, blocks, outType, acts, deltas, out, stream);
}

template <int JO, int JI>
hipError_t launchWindowTaps(const WuWindowArgs &a, uint32_t blocks,
                            int outType, const void *acts, const void *deltas,
                            void *out, hipStream_t stream) {
  const auto go = a.d.kW == 1 ? a.d.strideW == 1 ? &launchWindow<JO, JI, 1, 1>
                                                 : &launchWindow<JO, JI, 1, 2>
                  : a.d.strideW == 1 ? &launchWindow<JO, JI, 3, 1>
                                     : &launchWindow<JO, JI, 3, 2>;
  return go(a, blocks, outType, acts, deltas, out, stream);
}
} // namespace

hipError_t launchWuWindow(const WuTapDesc &d, int outType, const void *acts,
                          const void *deltas, void *workspace, void *out,
                          hipStream_t stream) {
  if (!wuWindowTakes(d) || (outType != kHalf && outType != kFloat))
    return hipErrorInvalidValue;
  const WinShape s = winShape(d);
  const uint32_t taps = d.kH * d.kW;
  WuWindowArgs a{};
  a.d = d;
  a.units = s.units, a.unitsPerChunk = d.windowSteps * kWinUnits;
  a.segs = s.segs, a.taps = taps;
  a.coTiles = s.coTiles, a.ciTiles = s.ciTiles, a.perTile = s.perTile;
  a.tilesPerChunk = uint32_t(s.tiles);
  a.resultCo = d.resultCo ? d.resultCo : d.co;
  a.resultCi = d.resultCi ? d.resultCi : d.ci;
  a.actPixelBytes = d.groups * d.ci * d.elemBytes;
  a.deltaPixelBytes = d.groups * d.co * d.elemBytes;
  a.actRowBytes = d.inW * a.actPixelBytes;
  a.actBytes = d.batch * d.inH * a.actRowBytes;
  a.deltaBytes = d.batch * d.outH * d.outW * a.deltaPixelBytes;
  a.divSegs = makeFastDiv(s.segs), a.divOutH = makeFastDiv(d.outH);
  a.divTilesPerChunk = makeFastDiv(a.tilesPerChunk);
  a.divKH = makeFastDiv(d.kH), a.divCiTiles = makeFastDiv(s.ciTiles);
  a.divCoTiles = makeFastDiv(s.coTiles), a.divCo = makeFastDiv(d.co);
  const bool direct = s.chunks == 1;
  a.strideF = direct ? taps : 1, a.strideTap = direct ? 1 : s.sums;
  a.chunkElems = uint64_t(taps) * s.sums;
  const uint32_t blocks = uint32_t(s.chunks * s.tiles);
  void *to = direct ? out : workspace;
  const int toType = direct ? outType : int(kFloat);
  a.outThrough = reachableBytes(a.chunkElems * (toType == kFloat ? 4 : 2));
  hipError_t e;
  if (d.elemBytes == 4)
    e = d.windowCo == 16
            ? launchWindowFloats<1>(a, blocks, toType, acts, deltas, to, stream)
        : d.windowCo == 32
            ? launchWindowFloats<2>(a, blocks, toType, acts, deltas, to, stream)
            : launchWindowFloats<3>(a, blocks, toType, acts, deltas, to,
                                    stream);
  else if (d.windowCo == 64)
    e = launchWindowTaps<4, 2>(a, blocks, toType, acts, deltas, to, stream);
  else if (d.windowCi == 64)
    e = launchWindowTaps<2, 4>(a, blocks, toType, acts, deltas, to, stream);
  else
    e = launchWindowTaps<2, 2>(a, blocks, toType, acts, deltas, to, stream);
  if (e != hipSuccess || direct)
    return e;
  const uint32_t F = uint32_t(s.elems / taps);
  WuWindowSumArgs r{};
  r.chunks = s.chunks, r.taps = taps, r.total = F, r.sums = s.sums;
  r.tapsHere = std::min(taps, kWinSlots);
  r.parts = std::min({s.chunks, kWinSlots / r.tapsHere, kWinParts});
  const uint32_t runs = (F + 63) / 64;
  const uint32_t tapBlocks = (taps + r.tapsHere - 1) / r.tapsHere;
  r.per = std::max(1u, std::min(kWinSlots / (r.tapsHere * r.parts),
                                runs * tapBlocks / 2048));
  r.divParts = makeFastDiv(r.parts), r.divTaps = makeFastDiv(r.tapsHere);
  const dim3 grid((runs + r.per - 1) / r.per, tapBlocks);
  const dim3 block((r.per * r.tapsHere * r.parts * 16 + 63) / 64 * 64);
  if (outType == kHalf)
    hipLaunchKernelGGL(wuWindowSumKernel<__half>, grid, block, 0, stream,
                       static_cast<const float *>(workspace),
                       static_cast<__half *>(out), r);
  else
    hipLaunchKernelGGL(wuWindowSumKernel<float>, grid, block, 0, stream,
                       static_cast<const float *>(workspace),
                       static_cast<float *>(out), r);
  return hipGetLastError();
}

} // namespace mxk
