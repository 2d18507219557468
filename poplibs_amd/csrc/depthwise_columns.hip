// Depthwise convolution with 3 x 3, 5 x 5 or 7 x 7 taps at stride 1 or 2: a lane
// walks down a strip of output columns of two neighbouring channels.
//
// Twenty-five or forty-nine multiply-adds per output and channel make the
// vector ALU the bound, so the kernel is built around it: a lane holds its
// channels' taps, the sums of the output rows under way (as many as a kernel
// meets an input row in) and one input row of its strip, and every input
// element is read once per strip - not once per tap.  An input row of STRIP
// outputs is S (STRIP - 1) + K columns, one 4-byte load each, asked for a row
// ahead; with unit stride and 7 x 7 taps it feeds 7 output rows of 4 columns x
// 7 taps x 2 channels, 392 multiply-adds for 10 loads.  (A load instruction
// holds the address unit for some eight cycles whatever its width: one channel
// to a lane and strips twice as wide is 14 loads for them, and twice the
// stores; 5 to 20 % slower with 5 x 5 taps.)
//
// Taps and columns go into the sums in pairs (v_dot2_f32_f16: exact products,
// fp32 sums; 4.7 cycles a wave against 2.3 to 2.9 for each of two fmac, so no
// faster in itself, but half the registers of fp32 taps and no conversions: 7
// to 14 % over the same kernel on fp32 values); the odd last tap is a
// multiply-add on fp32 values, because a pair filled with a zero tap would turn
// an infinity beside the window into a NaN.  Against 64 bits the sums' error is
// 0.83 to 0.95 times a chain of fp32 multiply-adds (rms), and fp16 subnormals
// stay exact.
//
// Nothing goes through LDS.  Lanes are dealt (image, strip, channel pair),
// channels fastest, so that a load is a run of neighbouring channels; a band of
// output rows is a grid dimension.  Rows outside the input are left out,
// columns outside it read as zeros (out-of-range buffer offsets).
//
// Measured (N x H x W, channels; us; the LDS-tiled or row-ring kernel before):
// 7 x 7 taps 57 x 28 x 28, 240: 44.9 -> 19.8; 64 x 7 x 7, 768: 16.8 -> 9.7;
// stride 2, 13 x 106 x 106, 304: 191 -> 31.5 (its tensors' bytes take 21);
// 5 x 5 taps 32 x 28 x 28, 240: 15.8 -> 10.4; 8 x 90 x 90, 48: 13.2 -> 7.6;
// stride 2, 32 x 28 x 28, 240: 10.1 -> 6.5; 32 x 112 x 112, 96: 25.2 -> 20.4.
// 3 x 3 taps go here from the row ring where the two estimates say so (Plan.cpp):
// 43 x 26 x 26, 336 channels 14.4 -> 9.2, 47 x 19 x 19, 488 11.6 -> 8.8, 11 x 7 x 7
// stride 2, 688 3.1 -> 2.3; the small-workgroup kernel of up to 224 channels keeps
// its layers, which are within 10 % either way.
//
// The reference's role: depthwise layers go through
// lib/poplin/codelets/ConvPartialHorizontalMac.cpp there.
#include "depthwise_columns.hpp"

#include <algorithm>
#include <cmath>

namespace mxk {
namespace {

constexpr uint32_t kColInvalid = 0x40000000u;

struct ColumnsArgs {
  uint32_t items; // image x strip x pair of channels
  uint32_t pairs, strips, bands, bandRows, outH, outW;
  int32_t padH, padW;
  uint32_t loH, hiH, loW, hiW;
  uint32_t pixelBytes, rowBytes, imageBytes, inBytes; // of the input
  uint32_t outPixelBytes, outRowBytes, outImageBytes, outBytes;
  FastDiv divPairs, divStrips, divBands;
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int CH> __device__ __forceinline__ float channelOf(uint32_t two) {
  float v = float(__builtin_bit_cast(half2v, two)[CH]);
  // (a float from here on: a multiply-add that converts runs at half the rate)
  asm("" : "+v"(v));
  return v;
}

/// K x K taps, stride S; STRIP output columns per lane.
template <int K, int S, int STRIP, class OutT>
__global__ __launch_bounds__(kColThreads) void depthwiseColumnsKernel(
    const ColumnsArgs a, const char *__restrict__ in,
    const uint32_t *__restrict__ weights, const OutT *__restrict__ bias,
    char *__restrict__ out) {
  using Walk = ColumnWalk<K, S, STRIP>;
  constexpr int NX = Walk::kColumns, LIVE = Walk::kLive, PERIOD = Walk::kPeriod;
  const uint32_t block = xcdSwizzle(blockIdx.x, gridDim.x);
  const uint32_t itemBlock = a.divBands(block);
  const uint32_t band = block - itemBlock * a.bands;
  const uint32_t item = itemBlock * kColThreads + threadIdx.x;
  const bool here = item < a.items;
  const uint32_t id = here ? item : 0;
  const uint32_t over = a.divPairs(id), c = id - over * a.pairs;
  const uint32_t b = a.divStrips(over), x0 = (over - b * a.strips) * STRIP;
  const uint32_t y0 = band * a.bandRows;
  const uint32_t rowsOut = a.outH - y0 < a.bandRows ? a.outH - y0 : a.bandRows;
  const uint32_t rowsIn = (rowsOut - 1) * S + K;

  const __amdgpu_buffer_rsrc_t inBuf = bufferOf(in, a.inBytes);
  const __amdgpu_buffer_rsrc_t outBuf = bufferOf(out, a.outBytes);
  uint32_t offset[NX];
  {
    const uint32_t first = x0 * S - uint32_t(a.padW);
    const uint32_t at = b * a.imageBytes + c * 4;
#pragma unroll
    for (int i = 0; i != NX; ++i)
      offset[i] = here && first + i - a.loW < a.hiW - a.loW
                      ? at + (first + i) * a.pixelBytes
                      : kColInvalid;
  }
  // Row r of the band's input rows; the row's place travels in the scalar
  // offset.  (Rows outside the input are answered with one inside it and left
  // out of the sums, so that every load is unconditional.)
  const int firstRow = int(y0 * S) - a.padH;
  auto rowInside = [&](uint32_t r) {
    return rowIsRead(firstRow + int(r), a.loH, a.hiH);
  };
  uint32_t raw[NX];
  auto load = [&](uint32_t r) {
    const uint32_t at =
        (rowInside(r) ? uint32_t(firstRow + int(r)) : a.loH) * a.rowBytes;
#pragma unroll
    for (int i = 0; i != NX; ++i)
      raw[i] = __builtin_amdgcn_raw_buffer_load_b32(inBuf, offset[i], at, 0);
  };
  // (The bias is on its way before the rows.  Behind the weights it cost 0.2 to
  // 0.4 us: 16 x 56 x 56, 5 x 5 stride 2, 72 channels 4.8 us, now 4.4; 3 x 10 x
  // 10, 464 channels 3.3, now 3.0.)
  BiasVec<OutT, 2> biasRaw;
  biasRaw.load(bias, 2 * c);
  load(0);
  half2v pair[2][K][K / 2];
  float last[2][K];
  const uint32_t *w = weights + c;
#pragma unroll
  for (int kh = 0; kh != K; ++kh) {
#pragma unroll
    for (int kw = 0; kw != K / 2; ++kw) {
      const uint32_t first = w[(kh * K + 2 * kw) * a.pairs],
                     second = w[(kh * K + 2 * kw + 1) * a.pairs];
      pair[0][kh][kw] = pairOf<0>(first, second);
      pair[1][kh][kw] = pairOf<1>(first, second);
    }
    const uint32_t odd = w[(kh * K + K - 1) * a.pairs];
    last[0][kh] = channelOf<0>(odd), last[1][kh] = channelOf<1>(odd);
  }
  const float start[2] = {biasRaw.at(0), biasRaw.at(1)};
  float sum[2][LIVE][STRIP];
#pragma unroll
  for (int ch = 0; ch != 2; ++ch)
#pragma unroll
    for (int l = 0; l != LIVE; ++l)
#pragma unroll
      for (int j = 0; j != STRIP; ++j)
        sum[ch][l][j] = 0.0f;
  const uint32_t outAt =
      b * a.outImageBytes + x0 * a.outPixelBytes + c * 2 * uint32_t(sizeof(OutT));

  uint32_t base = 0;
  while (whileEach(std::make_integer_sequence<int, PERIOD>{}, [&](auto step) {
      constexpr int R = decltype(step)::value;
      const uint32_t r = base + R;
      if (r >= rowsIn)
        return false;
      half2v x[2][NX]; // columns i and i + 1
      float end[2][STRIP];
#pragma unroll
      for (int i = 0; i < NX - 1; i += S)
        x[0][i] = pairOf<0>(raw[i], raw[i + 1]),
        x[1][i] = pairOf<1>(raw[i], raw[i + 1]);
#pragma unroll
      for (int j = 0; j != STRIP; ++j)
        end[0][j] = channelOf<0>(raw[j * S + K - 1]),
        end[1][j] = channelOf<1>(raw[j * S + K - 1]);
      load(r + 1);
      auto add = [&](auto row) {
        constexpr int KH = decltype(row)::value;
        if constexpr ((R + PERIOD - KH) % S == 0) {
          constexpr int L = (R + PERIOD - KH) / S % LIVE;
#pragma unroll
          for (int kw = 0; kw != K / 2; ++kw)
#pragma unroll
            for (int j = 0; j != STRIP; ++j)
#pragma unroll
              for (int ch = 0; ch != 2; ++ch)
                sum[ch][L][j] = __builtin_amdgcn_fdot2(
                    pair[ch][KH][kw], x[ch][j * S + 2 * kw], sum[ch][L][j],
                    false);
#pragma unroll
          for (int j = 0; j != STRIP; ++j)
#pragma unroll
            for (int ch = 0; ch != 2; ++ch)
              sum[ch][L][j] = fmaf(last[ch][KH], end[ch][j], sum[ch][L][j]);
        }
      };
      if (rowInside(r)) {
        staticFor<0, K>([&](auto row) {
          // (rows above the band's first and below its last: nobody's)
          if (r - uint32_t(decltype(row)::value) <= (rowsOut - 1) * S)
            add(row);
        });
      }
      // the output row whose last input row this was
      if constexpr ((R + PERIOD - (K - 1)) % S == 0) {
        constexpr int L = (R + PERIOD - (K - 1)) / S % LIVE;
        if (r + 1 >= uint32_t(K)) {
          const uint32_t y = y0 + (r - (K - 1)) / S;
#pragma unroll
          for (int j = 0; j != STRIP; ++j) {
            const uint32_t at = here && x0 + j < a.outW
                                    ? outAt + j * a.outPixelBytes
                                    : kOutOfRange;
            float v[2];
#pragma unroll
            for (int ch = 0; ch != 2; ++ch) {
              v[ch] = sum[ch][L][j] + start[ch];
              asm("" : "+v"(v[ch])); // (rounded once, from the fp32 sum)
              sum[ch][L][j] = 0.0f;
            }
            if constexpr (sizeof(OutT) == 2)
              __builtin_amdgcn_raw_buffer_store_b32(
                  __builtin_bit_cast(uint32_t, __floats2half2_rn(v[0], v[1])),
                  outBuf, at, y * a.outRowBytes, 0);
            else
              __builtin_amdgcn_raw_buffer_store_b64(
                  u32x2{__builtin_bit_cast(uint32_t, v[0]),
                        __builtin_bit_cast(uint32_t, v[1])},
                  outBuf, at, y * a.outRowBytes, 0);
          }
        }
      }
      return true;
    }))
    base += PERIOD;
}

uint64_t columnItems(const DepthwiseDesc &d) {
  return uint64_t(d.batch) * ((d.outW + d.columns - 1) / d.columns) *
         (d.channels / 2);
}

} // namespace

bool depthwiseColumnsTakes(const DepthwiseDesc &d, int inType, int outType) {
  // (offsets are within a launch's tensors, which launchDepthwise keeps below
  // kColInvalid by splitting the batch: an image has to fit)
  const uint64_t inImage = uint64_t(d.inH) * d.inW * d.channels * 2;
  const uint64_t outImage = uint64_t(d.outH) * d.outW * d.channels *
                            (outType == kHalf ? 2 : 4);
  const int most = 1 << 20;
  return inType == kHalf && (outType == kHalf || outType == kFloat) &&
         d.elemBytes == 2 && d.kH == d.kW && (d.kH == 3 || d.kH == 5 || d.kH == 7) &&
         d.strideH == d.strideW && (d.strideH == 1 || d.strideH == 2) &&
         d.dilH == 1 && d.dilW == 1 && d.inDilH == 1 && d.inDilW == 1 &&
         d.loH < d.hiH && d.hiH <= d.inH && d.loW < d.hiW && d.hiW <= d.inW &&
         d.channels != 0 && d.channels % 2 == 0 && d.batch != 0 && d.outH != 0 && d.outW != 0 &&
         inImage < kColInvalid && outImage < kColInvalid && d.padH > -most &&
         d.padH < most && d.padW > -most && d.padW < most;
}

namespace {
// 3 x 3 taps: the same with their own figures, fitted to 6 100 timings of 500
// random layers (1 to 64 images of 7 to 112 squared, 32 to 960 channels) within 8
// to 9 %; the choice by it is 1 % behind the best.
double threeEstimateUs(const DepthwiseDesc &d) {
  struct Fit {
    double call, product, row, perRow, rate, start;
    int resident[2];
  };
  constexpr Fit fits[2] = {{1.62, 1.98, 11.7, 4.55, 4.78e6, 2.07, {8, 6}},
                           {1.78, 1.03, 6.47, 8.14, 5.53e6, 1.35, {8, 5}}};
  const uint32_t s = d.strideH, strip = d.columns;
  const Fit &f = fits[s - 1];
  const double rows = std::min(d.columnRows, d.outH);
  const double bands = std::ceil(d.outH / rows);
  const double blocks =
      std::ceil(double(columnItems(d)) / kColThreads) * bands;
  const double rowsIn = (rows - 1) * s + 3;
  const double columnsIn = s * (strip - 1) + 3;
  const double waveUs = (f.product * 12 * rows * strip +
                         f.row * rowsIn * (3 * columnsIn + f.perRow)) *
                        1e-3 / 2.4;
  const double resident = f.resident[strip / 2 - 1];
  const double perCu = blocks / 256;
  const double full = std::floor(perCu / resident);
  const double rest = std::ceil(perCu - full * resident);
  const double us = full * (resident + f.start) * waveUs +
                    (rest > 0 ? (rest + f.start) * waveUs : 0.0);
  const double bytes = 2.0 * d.batch * d.channels *
                       (double(d.inH) * d.inW + double(d.outH) * d.outW);
  return f.call + std::sqrt(std::hypot(us * us, std::pow(bytes / f.rate, 2)));
}
} // namespace

// What a strip and a band cost, fitted to 1700 timings of 130 random layers
// (the choice by it is within 2 % of the best on average): a wave issues its
// multiply-adds and, for each input row, three instructions a column and some
// twenty around them; the waves of a SIMD take turns, as if there were two
// thirds of one more (their waits), and the tensors pass at 5 TB/s beside it.
double depthwiseColumnsEstimateUs(const DepthwiseDesc &d) {
  if (d.kH == 3)
    return threeEstimateUs(d);
  const uint32_t k = d.kH, s = d.strideH, strip = d.columns;
  const double rows = std::min(d.columnRows, d.outH);
  const double bands = std::ceil(d.outH / rows);
  const double blocks =
      std::ceil(double(columnItems(d)) / kColThreads) * bands;
  const double rowsIn = (rows - 1) * s + k;
  const double columnsIn = s * (strip - 1) + k;
  const double waveUs = (4.34 * 2 * rows * strip * k * (k / 2 + 1) +
                         5.88 * rowsIn * (3 * columnsIn + 20)) *
                        1e-3 / 2.4;
  // (waves a SIMD holds, by the kernels' registers)
  const double resident =
      k == 5 ? (strip == 2 ? (s == 1 ? 5 : 6) : 4) : (strip == 2 ? 4 : 3);
  const double perCu = blocks / 256;
  const double full = std::floor(perCu / resident);
  const double rest = std::ceil(perCu - full * resident);
  const double us = full * (resident + 0.68) * waveUs +
                    (rest > 0 ? (rest + 0.68) * waveUs : 0.0);
  const double bytes = 2.0 * d.batch * d.channels *
                       (double(d.inH) * d.inW + double(d.outH) * d.outW);
  return 3.9 + std::sqrt(std::hypot(us * us, std::pow(bytes / 5.0e6, 2)));
}

void chooseDepthwiseColumns(DepthwiseDesc &d, uint32_t strip) {
  DepthwiseDesc t = d;
  double best = 0;
  d.columns = 0;
  for (t.columns = 2; t.columns <= 4; t.columns += 2) {
    if (strip != 0 && t.columns != strip)
      continue;
    for (uint32_t bands = 1; bands <= 32 && bands <= d.outH; ++bands) {
      t.columnRows = (d.outH + bands - 1) / bands;
      const double us = depthwiseColumnsEstimateUs(t);
      if (d.columns == 0 || us < best)
        best = us, d.columns = t.columns, d.columnRows = t.columnRows;
    }
  }
}

namespace {
template <int K, int S, int STRIP>
hipError_t launchColumns(const ColumnsArgs &a, uint32_t blocks, int outType,
                         const void *in, const void *weights, const void *bias,
                         void *out, hipStream_t stream) {
  if (outType == kHalf)
    hipLaunchKernelGGL((depthwiseColumnsKernel<K, S, STRIP, __half>),
                       dim3(blocks), dim3(kColThreads), 0, stream, a,
                       static_cast<const char *>(in),
                       static_cast<const uint32_t *>(weights),
                       static_cast<const __half *>(bias),
                       static_cast<char *>(out));
  else
    hipLaunchKernelGGL((depthwiseColumnsKernel<K, S, STRIP, float>),
                       dim3(blocks), dim3(kColThreads), 0, stream, a,
                       static_cast<const char *>(in),
                       static_cast<const uint32_t *>(weights),
                       static_cast<const float *>(bias),
                       static_cast<char *>(out));
  return hipGetLastError();
}
} // namespace

hipError_t launchDepthwiseColumns(const DepthwiseDesc &d, int inType,
                                  int outType, const void *in,
                                  const void *weightsPacked, const void *bias,
                                  void *out, hipStream_t stream) {
  if (!depthwiseColumnsTakes(d, inType, outType) ||
      (d.columns != 2 && d.columns != 4) || d.columnRows == 0)
    return hipErrorInvalidValue;
  ColumnsArgs a{};
  a.items = uint32_t(columnItems(d));
  a.pairs = d.channels / 2, a.strips = (d.outW + d.columns - 1) / d.columns;
  a.bandRows = std::min(d.columnRows, d.outH);
  a.bands = (d.outH + a.bandRows - 1) / a.bandRows;
  a.outH = d.outH, a.outW = d.outW;
  a.padH = d.padH, a.padW = d.padW;
  a.loH = d.loH, a.hiH = d.hiH, a.loW = d.loW, a.hiW = d.hiW;
  a.pixelBytes = d.channels * 2;
  a.rowBytes = d.inW * a.pixelBytes, a.imageBytes = d.inH * a.rowBytes;
  a.inBytes = d.batch * a.imageBytes;
  a.outPixelBytes = d.channels * (outType == kHalf ? 2 : 4);
  a.outRowBytes = d.outW * a.outPixelBytes;
  a.outImageBytes = d.outH * a.outRowBytes;
  a.outBytes = d.batch * a.outImageBytes;
  a.divPairs = makeFastDiv(a.pairs), a.divStrips = makeFastDiv(a.strips);
  a.divBands = makeFastDiv(a.bands);
  const uint64_t blocks =
      (columnItems(d) + kColThreads - 1) / kColThreads * a.bands;
  if (uint64_t(d.batch) * d.inH * a.rowBytes >= kColInvalid ||
      uint64_t(d.batch) * d.outH * a.outRowBytes >= kColInvalid ||
      blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  auto go = [&](auto k, auto s) {
    constexpr int K = decltype(k)::value, S = decltype(s)::value;
    return d.columns == 2
               ? launchColumns<K, S, 2>(a, uint32_t(blocks), outType, in, weightsPacked,
                                        bias, out, stream)
               : launchColumns<K, S, 4>(a, uint32_t(blocks), outType, in, weightsPacked,
                                        bias, out, stream);
  };
  using One = std::integral_constant<int, 1>;
  using Two = std::integral_constant<int, 2>;
  using Three = std::integral_constant<int, 3>;
  using Five = std::integral_constant<int, 5>;
  using Seven = std::integral_constant<int, 7>;
  if (d.kH == 3)
    return d.strideH == 1 ? go(Three{}, One{}) : go(Three{}, Two{});
  if (d.kH == 5)
    return d.strideH == 1 ? go(Five{}, One{}) : go(Five{}, Two{});
  return d.strideH == 1 ? go(Seven{}, One{}) : go(Seven{}, Two{});
}

} // namespace mxk
