// Weight deltas of a depthwise layer with 3 x 3, 5 x 5 or 7 x 7 taps at stride
// 1 or 2: dW[tap][c] = sum over images and output pixels of
// deltas[pixel][c] * acts[pixel under tap][c].
//
// A lane holds the K x K sums of two neighbouring channels and walks down
// strips of STRIP output columns: an input row of the strip is read once and
// meets the K / S rows of deltas under way, which stay in registers; columns go
// into the sums in pairs (v_dot2_f32_f16: exact products, fp32 sums).  The
// kernel that this one stands in for has a thread for each tap and vector of
// channels, so every tap reads both tensors again - from the caches, but 25 or
// 49 times.
//
// A workgroup takes up to 128 channels, a band of output rows and `rounds`
// strips for each of its slots (256 threads / channel pairs); the slots' sums
// meet in LDS and go to partial[slice][tap][c], which the caller adds in order.
//
// Bound by the vector ALU: 34 x 42 x 42, 480 channels, 5 x 5, 30 us of which
// the dot products take 11, pairing columns, row checks and halo rows the rest;
// its bytes take 22.  Loads two rows ahead: no difference.  The pass, with the
// kernel that adds the slices (N x H x W, channels; us, before -> now): 5 x 5
// taps 51 x 34 x 34, 664: 282 -> 52; 46 x 45 x 45, 304: 135 -> 42; 53 x 18 x 18,
// 240: 27.7 -> 16.7; stride 2, 31 x 45 x 45, 584: 84 -> 38; 7 x 7 taps 40 x 69 x
// 69, 80: 132 -> 35; 3 x 3 taps 38 x 14 x 14, 1080: 34.7 -> 15.9.
//
// Rows outside the input are left out, columns outside it and deltas outside
// the strip read as zeros.  A zero opposite an infinity would make a NaN where
// the product is not part of the sum: a wave whose sums are not all finite
// forms them again, one product at a time.
//
// The reference's role: the weight update passes of depthwise layers go
// through lib/poplin/codelets/ConvPartialHorizontalMac.cpp there.
#include "depthwise_columns.hpp"

#include <algorithm>
#include <cmath>

namespace mxk {
namespace {

struct ColumnDeltasArgs {
  uint32_t pairs, perBlock, blocksC, slots; // (of channel pairs)
  uint32_t strips, items, rounds; // image x strip; of them, per slot
  uint32_t bands, bandRows, outH, outW;
  int32_t padH, padW;
  uint32_t loH, hiH, loW, hiW;
  uint32_t pixelBytes, rowBytes, imageBytes, inBytes;
  uint32_t outRowBytes, outImageBytes, outBytes;
  FastDiv divPerBlock, divStrips, divBlocksC, divBands;
};

template <int K, int S, int STRIP>
__global__ __launch_bounds__(kColThreads) void depthwiseColumnDeltasKernel(
    const ColumnDeltasArgs a, const char *__restrict__ acts,
    const char *__restrict__ deltas, float *__restrict__ partial) {
  using Walk = ColumnWalk<K, S, STRIP>;
  constexpr int NX = Walk::kColumns, LIVE = Walk::kLive, PERIOD = Walk::kPeriod;
  __shared__ float meet[K * K][kColThreads];
  const uint32_t block = xcdSwizzle(blockIdx.x, gridDim.x);
  const uint32_t rest = a.divBlocksC(block);
  const uint32_t chunk = a.divBands(rest), band = rest - chunk * a.bands;
  const uint32_t slot = a.divPerBlock(threadIdx.x);
  const uint32_t lane = threadIdx.x - slot * a.perBlock;
  const uint32_t c = (block - rest * a.blocksC) * a.perBlock + lane;
  const bool active = slot < a.slots && c < a.pairs;
  const uint32_t y0 = band * a.bandRows;
  const uint32_t rowsOut = a.outH - y0 < a.bandRows ? a.outH - y0 : a.bandRows;
  const uint32_t rowsIn = (rowsOut - 1) * S + K;
  const int firstRow = int(y0 * S) - a.padH;
  const __amdgpu_buffer_rsrc_t inBuf = bufferOf(acts, a.inBytes);
  const __amdgpu_buffer_rsrc_t outBuf = bufferOf(deltas, a.outBytes);
  auto rowInside = [&](uint32_t r) {
    return rowIsRead(firstRow + int(r), a.loH, a.hiH);
  };

  float sum[2][K][K];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i != 2 * K * K; ++i)
      sum[i / (K * K)][i / K % K][i % K] = 0.0f;
  };
  clear();

  for (uint32_t round = 0; round != a.rounds; ++round) {
    const uint32_t item = (chunk * a.rounds + round) * a.slots + slot;
    const bool here = active && item < a.items;
    const uint32_t image = a.divStrips(here ? item : 0);
    const uint32_t x0 = ((here ? item : 0) - image * a.strips) * STRIP;
    uint32_t offset[NX], outOffset[STRIP];
    {
      const uint32_t first = x0 * S - uint32_t(a.padW);
      const uint32_t at = image * a.imageBytes + c * 4;
#pragma unroll
      for (int i = 0; i != NX; ++i)
        offset[i] = here && first + i - a.loW < a.hiW - a.loW
                        ? at + (first + i) * a.pixelBytes
                        : kOutOfRange;
      const uint32_t outAt = image * a.outImageBytes + c * 4;
#pragma unroll
      for (int j = 0; j != STRIP; ++j)
        outOffset[j] = here && x0 + j < a.outW
                           ? outAt + (x0 + j) * a.pixelBytes
                           : kOutOfRange;
    }
    // (rows outside are answered with one inside and left out of the sums, so
    // that every load is unconditional)
    uint32_t raw[NX], rawOut[STRIP];
    auto load = [&](uint32_t r) {
      const uint32_t at =
          (rowInside(r) ? uint32_t(firstRow + int(r)) : a.loH) * a.rowBytes;
#pragma unroll
      for (int i = 0; i != NX; ++i)
        raw[i] = __builtin_amdgcn_raw_buffer_load_b32(inBuf, offset[i], at, 0);
    };
    auto loadOut = [&](uint32_t y) {
      const uint32_t at =
          (y0 + (y < rowsOut ? y : rowsOut - 1)) * a.outRowBytes;
#pragma unroll
      for (int j = 0; j != STRIP; ++j)
        rawOut[j] =
            __builtin_amdgcn_raw_buffer_load_b32(outBuf, outOffset[j], at, 0);
    };
    loadOut(0);
    load(0);
    half2v delta[2][LIVE][STRIP / 2];
#pragma unroll
    for (int l = 0; l != LIVE; ++l)
#pragma unroll
      for (int j = 0; j != STRIP / 2; ++j)
        delta[0][l][j] = delta[1][l][j] = half2v{0, 0};
    uint32_t base = 0;
    while (whileEach(
        std::make_integer_sequence<int, PERIOD>{}, [&](auto step) {
          constexpr int R = decltype(step)::value;
          const uint32_t r = base + R;
          if (r >= rowsIn)
            return false;
          if constexpr (R % S == 0) {
#pragma unroll
            for (int j = 0; j != STRIP / 2; ++j)
              delta[0][R / S % LIVE][j] =
                  pairOf<0>(rawOut[2 * j], rawOut[2 * j + 1]),
              delta[1][R / S % LIVE][j] =
                  pairOf<1>(rawOut[2 * j], rawOut[2 * j + 1]);
            loadOut(r / S + 1);
          }
          half2v x[2][NX]; // columns i and i + S
          const bool inside = rowInside(r);
          if (inside) {
#pragma unroll
            for (int i = 0; i < NX - S; ++i)
              x[0][i] = pairOf<0>(raw[i], raw[i + S]),
              x[1][i] = pairOf<1>(raw[i], raw[i + S]);
          }
          load(r + 1);
          if (inside)
            staticFor<0, K>([&](auto row) {
              constexpr int KH = decltype(row)::value;
              if constexpr ((R + PERIOD - KH) % S == 0) {
                constexpr int L = (R + PERIOD - KH) / S % LIVE;
                // (rows above the band's first and below its last: nobody's)
                if (r - uint32_t(KH) <= (rowsOut - 1) * S) {
#pragma unroll
                  for (int j = 0; j != STRIP / 2; ++j)
#pragma unroll
                    for (int kw = 0; kw != K; ++kw)
#pragma unroll
                      for (int ch = 0; ch != 2; ++ch)
                        sum[ch][KH][kw] = __builtin_amdgcn_fdot2(
                            delta[ch][L][j], x[ch][2 * j * S + kw],
                            sum[ch][KH][kw], false);
                }
              }
            });
          return true;
        }))
      base += PERIOD;
  }

  float probe = 0.0f;
#pragma unroll
  for (int i = 0; i != 2 * K * K; ++i)
    probe = fmaf(sum[i / (K * K)][i / K % K][i % K], 0.0f, probe);
  if (__any(probe != 0.0f)) {
    // (an infinity or a NaN somewhere: only products of the sums)
    clear();
    for (uint32_t round = 0; round != a.rounds; ++round) {
      const uint32_t item = (chunk * a.rounds + round) * a.slots + slot;
      if (!active || item >= a.items)
        continue;
      const uint32_t image = a.divStrips(item);
      const uint32_t x0 = (item - image * a.strips) * STRIP;
      for (uint32_t y = y0; y != y0 + rowsOut; ++y)
        for (uint32_t x = x0; x < x0 + STRIP && x < a.outW; ++x) {
          const half2v z = *reinterpret_cast<const half2v *>(
              deltas + image * a.outImageBytes + y * a.outRowBytes +
              x * a.pixelBytes + c * 4);
#pragma unroll
          for (int kh = 0; kh != K; ++kh)
#pragma unroll
            for (int kw = 0; kw != K; ++kw) {
              const uint32_t row = y * S + kh - uint32_t(a.padH);
              const uint32_t col = x * S + kw - uint32_t(a.padW);
              if (row - a.loH < a.hiH - a.loH && col - a.loW < a.hiW - a.loW) {
                const half2v v = *reinterpret_cast<const half2v *>(
                    acts + image * a.imageBytes + row * a.rowBytes +
                    col * a.pixelBytes + c * 4);
#pragma unroll
                for (int ch = 0; ch != 2; ++ch)
                  sum[ch][kh][kw] =
                      fmaf(float(z[ch]), float(v[ch]), sum[ch][kh][kw]);
              }
            }
        }
    }
  }

  // The slots' sums meet, one channel of the pairs after the other: a thread
  // adds some of the taps of one pair, four at once (a walk over the slots is a
  // chain of LDS reads).
  float *dst = partial + (size_t(rest) * (K * K) * a.pairs + c) * 2;
#pragma unroll
  for (int ch = 0; ch != 2; ++ch) {
    if (ch != 0)
      __syncthreads();
#pragma unroll
    for (int i = 0; i != K * K; ++i)
      meet[i][threadIdx.x] = sum[ch][i / K][i % K];
    __syncthreads();
    if (active)
      for (uint32_t first = slot; first < K * K; first += 4 * a.slots) {
        const float *from[4];
        float total[4];
#pragma unroll
        for (uint32_t t = 0; t != 4; ++t) {
          const uint32_t tap = first + t * a.slots;
          from[t] = meet[tap < K * K ? tap : first] + lane;
          total[t] = 0.0f;
        }
#pragma unroll 4
        for (uint32_t s = 0; s != a.slots; ++s)
#pragma unroll
          for (int t = 0; t != 4; ++t)
            total[t] += from[t][s * a.perBlock];
#pragma unroll
        for (uint32_t t = 0; t != 4; ++t)
          if (first + t * a.slots < K * K)
            dst[size_t(first + t * a.slots) * a.pairs * 2 + ch] = total[t];
      }
  }
}

struct ColumnDeltasShape {
  uint32_t blocksC, perBlock, slots, strips, items, bands, bandRows, rounds,
      chunks;
};

ColumnDeltasShape shapeOf(const DepthwiseDesc &d) {
  ColumnDeltasShape h;
  const uint32_t pairs = d.channels / 2;
  h.blocksC = (pairs + 63) / 64;
  h.perBlock = (pairs + h.blocksC - 1) / h.blocksC;
  h.slots = kColThreads / h.perBlock;
  h.strips = (d.outW + d.columns - 1) / d.columns;
  h.items = d.batch * h.strips;
  h.bandRows = std::min(d.columnRows, d.outH);
  h.bands = (d.outH + h.bandRows - 1) / h.bandRows;
  h.rounds = d.columnRounds;
  h.chunks = uint32_t((uint64_t(h.items) + uint64_t(h.slots) * h.rounds - 1) /
                      (uint64_t(h.slots) * h.rounds));
  return h;
}

} // namespace

bool depthwiseColumnDeltasTakes(const DepthwiseDesc &d) {
  const uint64_t inBytes = uint64_t(d.batch) * d.inH * d.inW * d.channels * 2;
  const uint64_t outBytes =
      uint64_t(d.batch) * d.outH * d.outW * d.channels * 2;
  const int most = 1 << 20;
  return d.elemBytes == 2 && d.kH == d.kW &&
         (d.kH == 3 || d.kH == 5 || d.kH == 7) && d.strideH == d.strideW &&
         (d.strideH == 1 || d.strideH == 2) && d.dilH == 1 && d.dilW == 1 &&
         d.inDilH == 1 && d.inDilW == 1 && d.loH < d.hiH && d.hiH <= d.inH &&
         d.loW < d.hiW && d.hiW <= d.inW && d.channels != 0 && d.channels % 2 == 0 && d.batch != 0 &&
         d.outH != 0 && d.outW != 0 && inBytes < kOutOfRange &&
         outBytes < kOutOfRange && d.padH > -most && d.padH < most &&
         d.padW > -most && d.padW < most;
}

uint32_t depthwiseColumnDeltasSlices(const DepthwiseDesc &d) {
  const ColumnDeltasShape h = shapeOf(d);
  return h.bands * h.chunks;
}

// The pass (both kernels), by taps and stride fitted to 5 400 timings of 420 random
// layers over several sets of buffers (4 to 64 images of 7 to 112 squared, 32 to
// 960 channels), within 5 to 7 % (3 x 3 at stride 2 10 %); the choice by it is 0.8
// to 1.5 % behind the best on average.  A walk's instructions, as in
// depthwiseColumnsEstimateUs, by the workgroups that a CU holds (by strips of two
// and four) and their start (`start` walks), against the bytes; then the slices'
// sum and the slots' meeting.
double depthwiseColumnDeltasEstimateUs(const DepthwiseDesc &d) {
  struct Fit {
    double product, row, perRow, taps, start, call, rate, partial, slice, slot;
    int resident[2];
  };
  constexpr Fit fits[3][2] = {
      {{0.0, 4.96, 20.5, 0.0126, 2.12, 5.60, 5.94e6, 1.08e-6, 0.0037, 0.106, {8, 7}},
       {0.0, 6.03, 22.2, 0.0007, 1.48, 5.83, 6.60e6, 1.21e-6, 0.0037, 0.075, {8, 6}}},
      {{1.54, 5.12, 19.6, 0.0, 1.19, 7.89, 5.14e6, 0.86e-6, 0.0035, 0.012, {4, 4}},
       {0.10, 5.84, 19.9, 0.0, 1.40, 7.16, 5.34e6, 1.12e-6, 0.0023, 0.001, {4, 4}}},
      {{2.51, 5.14, 19.6, 0.0, 0.65, 10.18, 4.14e6, 0.73e-6, 0.0047, 0.0, {3, 2}},
       {0.0, 6.10, 19.9, 0.0057, 1.44, 8.08, 3.82e6, 0.66e-6, 0.0028, 0.0, {3, 2}}}};
  const ColumnDeltasShape h = shapeOf(d);
  const uint32_t k = d.kH, s = d.strideH, strip = d.columns;
  const Fit &f = fits[k / 2 - 1][s - 1];
  const double rowsIn = (h.bandRows - 1.0) * s + k;
  const double columnsIn = s * (strip - 1) + k;
  const double perRow = double(h.bandRows) * strip;
  const double waveUs =
      h.rounds *
          (f.product * perRow * k * k +
           f.row * (rowsIn * (3 * columnsIn + f.perRow) + 3 * perRow)) *
          1e-3 / 2.4 +
      f.taps * k * k;
  const double resident = f.resident[strip / 2 - 1];
  const double slices = double(h.bands) * h.chunks;
  const double perCu = slices * h.blocksC / 256;
  const double full = std::floor(perCu / resident);
  const double rest = std::ceil(perCu - full * resident);
  const double us = full * (resident + f.start) * waveUs +
                    (rest > 0 ? (rest + f.start) * waveUs : 0.0);
  const double bytes = 2.0 * d.batch * d.channels *
                       (double(d.inH) * d.inW + double(d.outH) * d.outW);
  return f.call +
         std::sqrt(std::hypot(us * us, std::pow(bytes / f.rate, 2))) +
         f.partial * slices * k * k * d.channels * 4 + f.slice * slices +
         f.slot * h.slots;
}

void chooseDepthwiseColumnDeltas(DepthwiseDesc &d, uint32_t strip) {
  DepthwiseDesc t = d;
  double best = 0;
  d.columns = 0;
  for (t.columns = 2; t.columns <= 4; t.columns += 2) {
    if (strip != 0 && t.columns != strip)
      continue;
    for (uint32_t bands = 1; bands <= 32 && bands <= d.outH; ++bands) {
      t.columnRows = (d.outH + bands - 1) / bands;
      t.columnRounds = 1;
      // (2 048 workgroups at most: beyond that their tiles cost more than the
      // shorter walks give)
      const ColumnDeltasShape h = shapeOf(t);
      const uint64_t most = 2048;
      const uint64_t blocks = uint64_t(h.blocksC) * h.bands * h.chunks;
      t.columnRounds = uint32_t((blocks + most - 1) / most);
      const double us = depthwiseColumnDeltasEstimateUs(t);
      if (d.columns == 0 || us < best)
        best = us, d.columns = t.columns, d.columnRows = t.columnRows,
        d.columnRounds = t.columnRounds;
    }
  }
}

namespace {
template <int K, int S>
hipError_t launchColumnDeltas(const ColumnDeltasArgs &a, uint32_t strip,
                              uint32_t blocks, const void *acts,
                              const void *deltas, float *partial,
                              hipStream_t stream) {
  if (strip == 2)
    hipLaunchKernelGGL((depthwiseColumnDeltasKernel<K, S, 2>), dim3(blocks),
                       dim3(kColThreads), 0, stream, a,
                       static_cast<const char *>(acts),
                       static_cast<const char *>(deltas), partial);
  else
    hipLaunchKernelGGL((depthwiseColumnDeltasKernel<K, S, 4>), dim3(blocks),
                       dim3(kColThreads), 0, stream, a,
                       static_cast<const char *>(acts),
                       static_cast<const char *>(deltas), partial);
  return hipGetLastError();
}
} // namespace

hipError_t launchDepthwiseColumnDeltas(const DepthwiseDesc &d,
                                       const void *acts, const void *deltas,
                                       float *partial, hipStream_t stream) {
  if (!depthwiseColumnDeltasTakes(d) || (d.columns != 2 && d.columns != 4) ||
      d.columnRows == 0 || d.columnRounds == 0)
    return hipErrorInvalidValue;
  const ColumnDeltasShape h = shapeOf(d);
  const uint64_t blocks = uint64_t(h.blocksC) * h.bands * h.chunks;
  if (blocks > 0x7fffffffull)
    return hipErrorInvalidConfiguration;
  ColumnDeltasArgs a{};
  a.pairs = d.channels / 2, a.perBlock = h.perBlock, a.blocksC = h.blocksC;
  a.slots = h.slots, a.strips = h.strips, a.items = h.items;
  a.rounds = h.rounds, a.bands = h.bands, a.bandRows = h.bandRows;
  a.outH = d.outH, a.outW = d.outW, a.padH = d.padH, a.padW = d.padW;
  a.loH = d.loH, a.hiH = d.hiH, a.loW = d.loW, a.hiW = d.hiW;
  a.pixelBytes = d.channels * 2;
  a.rowBytes = d.inW * a.pixelBytes, a.imageBytes = d.inH * a.rowBytes;
  a.inBytes = d.batch * a.imageBytes;
  a.outRowBytes = d.outW * a.pixelBytes;
  a.outImageBytes = d.outH * a.outRowBytes;
  a.outBytes = d.batch * a.outImageBytes;
  a.divPerBlock = makeFastDiv(a.perBlock);
  a.divStrips = makeFastDiv(a.strips);
  a.divBlocksC = makeFastDiv(a.blocksC), a.divBands = makeFastDiv(a.bands);
  auto go = [&](auto k) {
    constexpr int K = decltype(k)::value;
    return d.strideH == 1
               ? launchColumnDeltas<K, 1>(a, d.columns, uint32_t(blocks), acts,
                                          deltas, partial, stream)
               : launchColumnDeltas<K, 2>(a, d.columns, uint32_t(blocks), acts,
                                          deltas, partial, stream);
  };
  return d.kH == 3   ? go(std::integral_constant<int, 3>{})
         : d.kH == 5 ? go(std::integral_constant<int, 5>{})
                     : go(std::integral_constant<int, 7>{});
}

} // namespace mxk
