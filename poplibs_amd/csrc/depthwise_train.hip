// Depthwise kernels for the training passes of a depthwise layer (one input
// and one output channel per group, channels-last, fp16 data, fp32 sums):
//
//   depthwiseDirectKernel      a forward convolution that also takes a
//                              dilated (zero-stuffed) input, which is what
//                              the backward pass of a strided depthwise layer
//                              is; one thread per output pixel and vector of
//                              8 channels, taps that fall between input
//                              elements skipped.
//   depthwiseWeightDeltaKernel the gradient with respect to the weights,
//                              dW[tap][c] = sum over batch and output pixels
//                              of deltas[pixel][c] * acts[pixel under tap][c];
//                              one thread per (tap, vector of 8 channels),
//                              walking a slice of the pixels; the per-slice
//                              sums go to a workspace and a second kernel
//                              adds the slices in order.
//
// Both are bound by memory: they read each operand from HBM once (re-reads
// of neighbouring taps hit the caches) and have no matrix-core work.  They
// take the role of PopLibs' HorizontalMac vertices in the backward and weight
// update passes (lib/poplin/codelets/ConvPartialHorizontalMac.cpp:34-133).
#include "device_types.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace mxk {
namespace {

union Vec8 {
  uint4 raw;
  __half2 h2[4];
};

__device__ __forceinline__ void fma8(float (&acc)[8], const Vec8 &x,
                                     const Vec8 &k) {
#pragma unroll
  for (int i = 0; i != 4; ++i) {
    const float2 xf = __half22float2(x.h2[i]);
    const float2 kf = __half22float2(k.h2[i]);
    acc[2 * i] = fmaf(xf.x, kf.x, acc[2 * i]);
    acc[2 * i + 1] = fmaf(xf.y, kf.y, acc[2 * i + 1]);
  }
}

__device__ __forceinline__ void store8(__half *p, const float (&v)[8]) {
  Vec8 o;
#pragma unroll
  for (int i = 0; i != 4; ++i)
    o.h2[i] = roundPairToHalf(v[2 * i], v[2 * i + 1]);
  *reinterpret_cast<uint4 *>(p) = o.raw;
}
__device__ __forceinline__ void store8(float *p, const float (&v)[8]) {
  *reinterpret_cast<float4 *>(p) = float4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<float4 *>(p + 4) = float4{v[4], v[5], v[6], v[7]};
}

// The same for fp32 inputs: a 16-byte vector holds four channels.
__device__ __forceinline__ void fma4(float (&acc)[4], const uint4 &x,
                                     const uint4 &k) {
  acc[0] = fmaf(__uint_as_float(x.x), __uint_as_float(k.x), acc[0]);
  acc[1] = fmaf(__uint_as_float(x.y), __uint_as_float(k.y), acc[1]);
  acc[2] = fmaf(__uint_as_float(x.z), __uint_as_float(k.z), acc[2]);
  acc[3] = fmaf(__uint_as_float(x.w), __uint_as_float(k.w), acc[3]);
}
__device__ __forceinline__ void store4(float *p, const float (&v)[4]) {
  *reinterpret_cast<float4 *>(p) = float4{v[0], v[1], v[2], v[3]};
}
__device__ __forceinline__ void store4(__half *p, const float (&v)[4]) {
  const __half2 lo = roundPairToHalf(v[0], v[1]),
                hi = roundPairToHalf(v[2], v[3]);
  *reinterpret_cast<uint2 *>(p) = uint2{__builtin_bit_cast(uint32_t, lo),
                                        __builtin_bit_cast(uint32_t, hi)};
}

struct DirectArgs {
  DepthwiseDesc d;
  FastDiv divVecs, divOutW, divOutH, divInDilH, divInDilW;
  uint32_t vecs;
  uint64_t items; // batch * outH * outW * vecs
};

/// InT: __half (vectors of 8 channels) or float (of 4).
template <class OutT, class InT = __half>
__global__ __launch_bounds__(256) void depthwiseDirectKernel(
    DirectArgs a, const InT *__restrict__ in, const InT *__restrict__ w,
    const OutT *__restrict__ bias, OutT *__restrict__ out) {
  constexpr int E = 16 / int(sizeof(InT));
  const DepthwiseDesc &d = a.d;
  const uint64_t item = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (item >= a.items)
    return;
  // item = ((b * outH + oh) * outW + ow) * vecs + v
  const uint32_t pixel = a.divVecs(uint32_t(item));
  const uint32_t v = uint32_t(item) - pixel * a.vecs;
  const uint32_t row = a.divOutW(pixel);
  const uint32_t ow = pixel - row * d.outW;
  const uint32_t b = a.divOutH(row);
  const uint32_t oh = row - b * d.outH;
  const uint32_t c = v * E;
  float acc[E];
#pragma unroll
  for (int i = 0; i != E; ++i)
    acc[i] = bias ? Load<OutT>::at(bias, c + i, 0) : 0.0f;
  const int ihBase = int(oh * d.strideH) - d.padH;
  const int iwBase = int(ow * d.strideW) - d.padW;
  const InT *image = in + size_t(b) * d.inH * d.inW * d.channels + c;
  // Validity is separable: the kernel columns that read an input element
  // are worked out once (a bit each - up to 32 columns at a time), then for
  // every valid kernel row only those columns are visited.
  for (uint32_t kw0 = 0; kw0 < d.kW; kw0 += 32) {
    uint32_t columns = 0;
    const uint32_t kwEnd = min(d.kW - kw0, 32u);
    for (uint32_t j = 0; j != kwEnd; ++j) {
      const int iwD = iwBase + int((kw0 + j) * d.dilW);
      const uint32_t iw = a.divInDilW(uint32_t(iwD));
      if (iwD >= 0 && iw * d.inDilW == uint32_t(iwD) && iw >= d.loW &&
          iw < d.hiW)
        columns |= 1u << j;
    }
    if (columns == 0)
      continue;
    for (uint32_t kh = 0; kh != d.kH; ++kh) {
      const int ihD = ihBase + int(kh * d.dilH);
      const uint32_t ih = a.divInDilH(uint32_t(ihD));
      if (ihD < 0 || ih * d.inDilH != uint32_t(ihD) || ih < d.loH ||
          ih >= d.hiH)
        continue;
      const InT *row = image + size_t(ih) * d.inW * d.channels;
      const InT *taps = w + size_t(kh * d.kW + kw0) * d.channels + c;
      for (uint32_t rest = columns; rest != 0; rest &= rest - 1) {
        const uint32_t j = uint32_t(__ffs(int(rest))) - 1;
        const uint32_t iw =
            a.divInDilW(uint32_t(iwBase + int((kw0 + j) * d.dilW)));
        Vec8 x, k;
        x.raw = *reinterpret_cast<const uint4 *>(row + size_t(iw) * d.channels);
        k.raw = *reinterpret_cast<const uint4 *>(taps + size_t(j) * d.channels);
        if constexpr (E == 8)
          fma8(acc, x, k);
        else
          fma4(acc, x.raw, k.raw);
      }
    }
  }
  if constexpr (E == 8)
    store8(out + size_t(pixel) * d.channels + c, acc);
  else
    store4(out + size_t(pixel) * d.channels + c, acc);
}

struct BlockArgs {
  DepthwiseDesc d;
  FastDiv divVecs, divBlocksW, divStrips;
  uint32_t vecs, blocksW, strips;
  int32_t firstBlockH, firstBlockW;
  uint64_t items; // batch * strips * blocksW * vecs
};

/// The same convolution for an input dilated by S in both dimensions with
/// unit stride and unit kernel dilation (the backward pass of a layer of
/// stride S), K x K taps.  With oh - padH = S q + r (0 <= r < S) the taps
/// that read an input element are those with (r + kh) % S == 0, and they read
/// row q + (r + kh) / S: the same for every output of phase r.  So a thread
/// takes S x S blocks of outputs (one output of every phase), R blocks below
/// each other, for one vector of 8 channels: it loads the (R + ND - 1) x ND
/// input vectors they need (ND = (K + S - 2) / S + 1) and all K x K taps
/// once, and every output then takes exactly its own taps - no tests, no
/// divergence between neighbouring outputs, each input vector loaded once per
/// thread.
/// What bounds it is a wave's chain of instructions, 1 200 with two blocks of 5 x 5
/// taps: with one block to a thread instead of two (5 x 5) or four (3 x 3), and no
/// load under a condition of its own, 17 x 44 x 44, 400 channels, 5 x 5 17.8 -> 13.2
/// us, 19 x 25 x 25, 40, 3 x 3 4.4 -> 2.8; 70 layers 1.32 times as fast.  607 with
/// three calls' tensors in turn 1.28 times, 3 x 3 layers of more than 100 MB 1.02
/// (28; 15 x 71 x 71, 800 channels 35.3 -> 37.7, 26 x 78 x 78, 440 45.6 -> 41.7).
template <int S, int K, int R, class OutT>
__global__ __launch_bounds__(256, K == 5 ? 2 : 4) void
depthwiseDilatedBlockKernel(
    BlockArgs a, const __half *__restrict__ in, const __half *__restrict__ w,
    const OutT *__restrict__ bias, OutT *__restrict__ out) {
  const DepthwiseDesc &d = a.d;
  const uint64_t item = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (item >= a.items)
    return;
  // item = ((b * strips + strip) * blocksW + block column) * vecs + v
  const uint32_t col = a.divVecs(uint32_t(item));
  const uint32_t v = uint32_t(item) - col * a.vecs;
  const uint32_t t = a.divBlocksW(col);
  const uint32_t bw = col - t * a.blocksW;
  const uint32_t b = a.divStrips(t);
  const uint32_t strip = t - b * a.strips;
  const int qw = a.firstBlockW + int(bw);
  const int qh0 = a.firstBlockH + int(strip) * R;
  const uint32_t c = v * 8;
  constexpr int ND = (K + S - 2) / S + 1;
  constexpr int ROWS = R + ND - 1;

  const __half *image = in + size_t(b) * d.inH * d.inW * d.channels + c;
  Vec8 x[ROWS][ND];
#pragma unroll
  for (int i = 0; i != ROWS; ++i)
#pragma unroll
    for (int j = 0; j != ND; ++j) {
      // (an element outside is answered with one inside and put to zero below:
      // every load is unconditional)
      const int ih = min(max(qh0 + i, int(d.loH)), int(d.hiH) - 1);
      const int iw = min(max(qw + j, int(d.loW)), int(d.hiW) - 1);
      x[i][j].raw = *reinterpret_cast<const uint4 *>(
          image + (size_t(ih) * d.inW + size_t(iw)) * d.channels);
    }
  Vec8 k[K * K];
#pragma unroll
  for (int tap = 0; tap != K * K; ++tap)
    k[tap].raw =
        *reinterpret_cast<const uint4 *>(w + size_t(tap) * d.channels + c);
  BiasVec<OutT, 8> biasRaw;
  biasRaw.load(bias, c);
  float biasV[8];
#pragma unroll
  for (int i = 0; i != 8; ++i)
    biasV[i] = biasRaw.at(i);
#pragma unroll
  for (int i = 0; i != ROWS; ++i)
#pragma unroll
    for (int j = 0; j != ND; ++j) {
      const bool inside =
          uint32_t(qh0 + i) - d.loH < d.hiH - d.loH &&
          uint32_t(qw + j) - d.loW < d.hiW - d.loW;
      x[i][j].raw = inside ? x[i][j].raw : uint4{0, 0, 0, 0};
    }

  OutT *outImage = out + size_t(b) * d.outH * d.outW * d.channels + c;
#pragma unroll
  for (int i = 0; i != R; ++i)
#pragma unroll
    for (int rh = 0; rh != S; ++rh) {
      const int oh = S * (qh0 + i) + rh + d.padH;
      if (oh < 0 || oh >= int(d.outH))
        continue;
#pragma unroll
      for (int rw = 0; rw != S; ++rw) {
        const int ow = S * qw + rw + d.padW;
        if (ow < 0 || ow >= int(d.outW))
          continue;
        float acc[8];
#pragma unroll
        for (int e = 0; e != 8; ++e)
          acc[e] = biasV[e];
#pragma unroll
        for (int kh = 0; kh != K; ++kh)
#pragma unroll
          for (int kw = 0; kw != K; ++kw)
            if ((rh + kh) % S == 0 && (rw + kw) % S == 0)
              fma8(acc, x[i + (rh + kh) / S][(rw + kw) / S], k[kh * K + kw]);
        store8(outImage + (size_t(oh) * d.outW + size_t(ow)) * d.channels,
               acc);
      }
    }
}

/// Blocks of 3 x 3 taps up to which a thread takes one, not two: a short chain of
/// instructions counts where the chip is not filled, the taps' loads shared by two
/// beyond (9 x 58 x 58, 256 channels, 259 000 blocks 6.6 and 6.0 us; 10 x 42 x 42,
/// 192, 116 000 3.9 and 4.0; 25 x 9 x 9, 72, 8 100 2.8 and 3.1 - with four 4.3).
constexpr uint64_t kFewBlocks = 120000;

inline int floorDiv(int n, int d) { return n >= 0 ? n / d : -((-n + d - 1) / d); }

/// Launches depthwiseDilatedBlockKernel<S, K, R> on a shape it is built for.
template <int S, int K, int R>
hipError_t launchDilatedBlock(const DepthwiseDesc &d, int outType,
                              const void *in, const void *w, const void *bias,
                              void *out, hipStream_t stream) {
  BlockArgs a;
  a.d = d;
  a.vecs = d.channels / 8;
  a.firstBlockH = floorDiv(-d.padH, S);
  a.firstBlockW = floorDiv(-d.padW, S);
  const uint32_t blocksH =
      uint32_t(floorDiv(int(d.outH) - 1 - d.padH, S) - a.firstBlockH + 1);
  a.blocksW =
      uint32_t(floorDiv(int(d.outW) - 1 - d.padW, S) - a.firstBlockW + 1);
  a.strips = (blocksH + R - 1) / R;
  a.items = uint64_t(d.batch) * a.strips * a.blocksW * a.vecs;
  if (a.items >= (1ull << 31))
    return hipErrorInvalidConfiguration;
  a.divVecs = makeFastDiv(a.vecs);
  a.divBlocksW = makeFastDiv(a.blocksW);
  a.divStrips = makeFastDiv(a.strips);
  const dim3 grid{uint32_t((a.items + 255) / 256)}, block{256};
  if (outType == kHalf)
    hipLaunchKernelGGL((depthwiseDilatedBlockKernel<S, K, R, __half>), grid,
                       block, 0, stream, a, static_cast<const __half *>(in),
                       static_cast<const __half *>(w),
                       static_cast<const __half *>(bias),
                       static_cast<__half *>(out));
  else
    hipLaunchKernelGGL((depthwiseDilatedBlockKernel<S, K, R, float>), grid,
                       block, 0, stream, a, static_cast<const __half *>(in),
                       static_cast<const __half *>(w),
                       static_cast<const float *>(bias),
                       static_cast<float *>(out));
  return hipGetLastError();
}

struct DeltaArgs {
  DepthwiseDesc d;     // the FORWARD convolution
  FastDiv divVecs, divOutW, divOutH;
  uint32_t vecs, taps;
  uint32_t items;      // taps * vecs
  uint32_t itemsPerBlock, slots; // itemsPerBlock * slots <= 256 threads
  uint32_t pixels;     // batch * outH * outW
  uint32_t pixelsPerSlice, pixelsPerSlot, slices;
};

/// partial[slice][tap][c] = sum over the slice's output pixels.  A workgroup
/// takes itemsPerBlock (tap, channel vector) items and one slice of the
/// pixels; when there are few items, `slots` groups of threads walk a part of
/// the slice each and their sums meet in LDS.
/// InT: __half (vectors of 8 channels) or float (of 4).
template <class InT>
__global__ __launch_bounds__(256) void depthwiseWeightDeltaKernel(
    DeltaArgs a, const InT *__restrict__ acts, const InT *__restrict__ deltas,
    float *__restrict__ partial) {
  constexpr int E = 16 / int(sizeof(InT));
  __shared__ float meet[256][9]; // 8 sums per thread, padded
  const DepthwiseDesc &d = a.d;
  const uint32_t slot = threadIdx.x / a.itemsPerBlock;
  const uint32_t itemLocal = threadIdx.x - slot * a.itemsPerBlock;
  const uint32_t item = blockIdx.x * a.itemsPerBlock + itemLocal;
  const bool active = slot < a.slots && item < a.items;
  // item = tap * vecs + v: neighbouring threads read neighbouring channels
  const uint32_t tap = a.divVecs(active ? item : 0);
  const uint32_t c = ((active ? item : 0) - tap * a.vecs) * E;
  const uint32_t kh = tap / d.kW, kw = tap - kh * d.kW;
  const uint32_t slice = blockIdx.y;
  const uint32_t sliceEnd =
      min((slice + 1) * a.pixelsPerSlice, a.pixels);
  const uint32_t first =
      min(slice * a.pixelsPerSlice + slot * a.pixelsPerSlot, sliceEnd);
  const uint32_t last = active ? min(first + a.pixelsPerSlot, sliceEnd) : first;
  // (b, oh, ow) of the first pixel; they advance without dividing
  uint32_t row = a.divOutW(first);
  uint32_t ow = first - row * d.outW;
  uint32_t b = a.divOutH(row);
  uint32_t oh = row - b * d.outH;
  const int khd = int(kh * d.dilH) - d.padH, kwd = int(kw * d.dilW) - d.padW;
  float acc[E] = {};
  // Four pixels a round: their loads are issued together, so that a wave has
  // eight of them in flight (the walk is bound by load latency, not by
  // arithmetic).
  constexpr int kUnroll = 4;
  for (uint32_t p = first; p < last; p += kUnroll) {
    Vec8 x[kUnroll], z[kUnroll];
#pragma unroll
    for (int u = 0; u != kUnroll; ++u) {
      const int ih = int(oh * d.strideH) + khd, iw = int(ow * d.strideW) + kwd;
      const bool ok = p + u < last && ih >= int(d.loH) && ih < int(d.hiH) &&
                      iw >= int(d.loW) && iw < int(d.hiW);
      x[u].raw = uint4{0, 0, 0, 0};
      z[u].raw = uint4{0, 0, 0, 0};
      if (ok) {
        x[u].raw = *reinterpret_cast<const uint4 *>(
            acts +
            ((size_t(b) * d.inH + uint32_t(ih)) * d.inW + uint32_t(iw)) *
                d.channels +
            c);
        z[u].raw = *reinterpret_cast<const uint4 *>(
            deltas + size_t(p + u) * d.channels + c);
      }
      if (++ow == d.outW) {
        ow = 0;
        if (++oh == d.outH) {
          oh = 0;
          ++b;
        }
      }
    }
#pragma unroll
    for (int u = 0; u != kUnroll; ++u) {
      if constexpr (E == 8)
        fma8(acc, x[u], z[u]);
      else
        fma4(acc, x[u].raw, z[u].raw);
    }
  }
  if (a.slots > 1) {
#pragma unroll
    for (int i = 0; i != E; ++i)
      meet[threadIdx.x][i] = acc[i];
    __syncthreads();
    if (slot == 0)
      for (uint32_t s2 = 1; s2 != a.slots; ++s2)
#pragma unroll
        for (int i = 0; i != E; ++i)
          acc[i] += meet[s2 * a.itemsPerBlock + itemLocal][i];
  }
  if (!active || slot != 0)
    return;
  float *dst = partial + (size_t(slice) * a.taps + tap) * d.channels + c;
#pragma unroll
  for (int i = 0; i != E; i += 4)
    *reinterpret_cast<float4 *>(dst + i) =
        float4{acc[i], acc[i + 1], acc[i + 2], acc[i + 3]};
}

// The sum has eight parts where the outputs (taps x channels) outnumber this.
constexpr uint32_t kManyOutputs = 3500, kManyOutputsPerSlice = 25;

/// out[c][tap] = sum over slices of partial[slice][tap][c], in a fixed order:
/// a workgroup takes COLUMNS outputs and deals the slices to PARTS parts in turn,
/// COLUMNS lanes (contiguous in a slice) to each; a lane adds up its part's with
/// four loads in flight, then the sums of an output meet in steps of eight, each in
/// order (one thread adding all 64 is a chain of 64 LDS reads at the kernel's end).
///
/// What it costs is the chain of instructions of a wave: 32-bit offsets into a
/// buffer, beyond whose end zeros arrive, take one or two to a load, where slices
/// in runs with the loads' addresses and conditions worked out took ten and more (16
/// parts of 16 loads 1.5 us longer than 64 of four; the pass over 120 layers 1.014
/// times as fast with the offsets, 12 x 19 x 19, 5 x 5 stride 2 10.5 -> 9.6 us).  64
/// parts of 16 outputs make it short, but launch a wave for every output: with many
/// of those, eight parts of 32 take a quarter of the time (5 x 5 taps, 960 channels,
/// 16 slices: 8.0 -> 3.2 us).  Their chain is eight times as long, which shows right
/// behind the kernel that writes the slices: the line below is where both were level
/// over 70 passes.
/// WIDE: offsets beyond 31 bits, which take 13 million outputs: those are one or
/// two slices.
template <class OutT, int PARTS, int COLUMNS, bool WIDE>
__global__ __launch_bounds__(PARTS *COLUMNS) void depthwiseDeltaSumKernel(
    const float *__restrict__ partial, uint32_t slices, uint32_t taps,
    uint32_t channels, OutT *__restrict__ out) {
  static_assert(PARTS == 8 || PARTS == 64);
  __shared__ float meet[PARTS][COLUMNS];
  const uint32_t column = threadIdx.x % COLUMNS, part = threadIdx.x / COLUMNS;
  const uint32_t outputs = taps * channels;
  const uint32_t i = blockIdx.x * COLUMNS + column; // tap * C + c
  float sum = 0.0f;
  if constexpr (WIDE) {
    if (i < outputs)
      for (uint32_t s = part; s < slices; s += PARTS)
        sum += partial[size_t(s) * outputs + i];
  } else {
    const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(partial), short(0), int(slices * outputs * 4),
        0x00020000);
    const uint32_t step = PARTS * outputs * 4;
    uint32_t at = i < outputs ? (part * outputs + i) * 4 : 0x80000000u;
    constexpr int kInFlight = 4;
    for (uint32_t s = 0; s < slices; s += kInFlight * PARTS) {
      float v[kInFlight];
#pragma unroll
      for (uint32_t u = 0; u != kInFlight; ++u)
        v[u] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(buffer, at + u * step,
                                                        0, 0));
      at += kInFlight * step;
      sum += (v[0] + v[1]) + (v[2] + v[3]);
    }
  }
  meet[part][column] = sum;
  __syncthreads();
  if constexpr (PARTS == 64) {
    float eight = 0.0f;
    if (part < 8) {
      eight = meet[part * 8][column];
#pragma unroll
      for (int w = 1; w != 8; ++w)
        eight += meet[part * 8 + w][column];
    }
    __syncthreads();
    if (part < 8)
      meet[part][column] = eight;
    __syncthreads();
  }
  if (part != 0 || i >= outputs)
    return;
  float total = meet[0][column];
#pragma unroll
  for (int w = 1; w != 8; ++w)
    total += meet[w][column];
  const uint32_t tap = i / channels, c = i - tap * channels;
  storeOut(out, size_t(c) * taps + tap, total);
}

template <class OutT, int PARTS, int COLUMNS>
void launchDeltaSumIn(const float *partial, uint32_t slices, uint32_t taps,
                      uint32_t channels, void *out, hipStream_t stream) {
  const uint32_t outputs = taps * channels;
  // (offsets up to four rounds of parts beyond the slices)
  const bool wide = (uint64_t(slices) + 5 * PARTS) * outputs * 4 >= (1ull << 31);
  const auto kernel = wide
                          ? &depthwiseDeltaSumKernel<OutT, PARTS, COLUMNS, true>
                          : &depthwiseDeltaSumKernel<OutT, PARTS, COLUMNS, false>;
  hipLaunchKernelGGL(kernel, dim3((outputs + COLUMNS - 1) / COLUMNS),
                     dim3(PARTS * COLUMNS), 0, stream, partial, slices, taps,
                     channels, static_cast<OutT *>(out));
}

template <class OutT>
void launchDeltaSum(const float *partial, uint32_t slices, uint32_t taps,
                    uint32_t channels, void *out, hipStream_t stream) {
  if (taps * channels < kManyOutputs + uint64_t(kManyOutputsPerSlice) * slices)
    launchDeltaSumIn<OutT, 64, 16>(partial, slices, taps, channels, out,
                                   stream);
  else
    launchDeltaSumIn<OutT, 8, 32>(partial, slices, taps, channels, out, stream);
}

/// Threads of a workgroup: itemsPerBlock items by `slots` parts of a slice.
void deltaBlockShape(const DepthwiseDesc &d, uint32_t &itemsPerBlock,
                     uint32_t &slots) {
  const uint64_t items =
      uint64_t(d.kH) * d.kW * (uint64_t(d.channels) * d.elemBytes / 16);
  itemsPerBlock = uint32_t(std::min<uint64_t>(std::max<uint64_t>(items, 1), 256));
  slots = 256 / itemsPerBlock;
}

uint32_t deltaSlices(const DepthwiseDesc &d) {
  // About 4 workgroups per CU in all; a slot walks at least 16 pixels, or 8 or 4
  // where that leaves no more slices than the sum's 64 parts have in one round of
  // loads, and sums of 2 MB.  (The walk is a chain of latencies: 13 x 12 x 12, 40
  // channels, 3 x 3 6.7 us with 16, 5.2 with 4; but 46 x 13 x 13, 40 6.2 with 195
  // slices, 7.5 with 389, and 11 x 12 x 12 stride 2, 808, 5 x 5 8.5 with 2 MB, 9.9
  // with 4.)
  uint32_t itemsPerBlock, slots;
  deltaBlockShape(d, itemsPerBlock, slots);
  const uint64_t pixels = uint64_t(d.batch) * d.outH * d.outW;
  const uint64_t items =
      uint64_t(d.kH) * d.kW * (uint64_t(d.channels) * d.elemBytes / 16);
  const uint64_t itemBlocks = (items + itemsPerBlock - 1) / itemsPerBlock;
  const uint64_t most =
      (1024 + itemBlocks - 1) / std::max<uint64_t>(itemBlocks, 1);
  uint64_t slices = 1;
  for (uint32_t walk : {4u, 8u, 16u}) {
    slices = std::min<uint64_t>(most, (pixels + walk * slots - 1) /
                                          (walk * slots));
    if (slices <= 256 &&
        slices * d.kH * d.kW * d.channels * sizeof(float) <= 2000000)
      break;
  }
  slices = std::min<uint64_t>(std::max<uint64_t>(slices, 1), 65535);
  return uint32_t(slices);
}

} // namespace

bool depthwiseDirectInBlocks(const DepthwiseDesc &d) {
  return d.inDilH == 2 && d.inDilW == 2 && d.strideH == 1 && d.strideW == 1 &&
         d.dilH == 1 && d.dilW == 1 && d.kH == d.kW &&
         (d.kH == 3 || d.kH == 5) && d.outH < (1u << 30) &&
         d.outW < (1u << 30) && d.loH < d.hiH && d.loW < d.hiW;
}

hipError_t launchDepthwiseDirect(const DepthwiseDesc &d, int inType,
                                 int outType, const void *in,
                                 const void *weightsPacked, const void *bias,
                                 void *out, hipStream_t stream) {
  const uint32_t perVec = inType == kFloat ? 4 : 8;
  if ((inType != kHalf && inType != kFloat) ||
      d.elemBytes != (inType == kFloat ? 4u : 2u) ||
      d.channels % perVec != 0 || d.inDilH == 0 || d.inDilW == 0)
    return hipErrorInvalidValue;
  DirectArgs a;
  a.d = d;
  a.vecs = d.channels / perVec;
  a.items = uint64_t(d.batch) * d.outH * d.outW * a.vecs;
  if (a.items == 0)
    return hipSuccess;
  // item numbers are divided with 31-bit arithmetic
  if (a.items >= (1ull << 31))
    return hipErrorInvalidConfiguration;
  if (inType == kHalf && (outType == kHalf || outType == kFloat) &&
      depthwiseDirectInBlocks(d)) {
    const uint64_t blocks =
        uint64_t(d.batch) * (d.outH / 2 + 1) * (d.outW / 2 + 1) * a.vecs;
    const auto go = d.kH == 5                ? &launchDilatedBlock<2, 5, 1>
                    : blocks <= kFewBlocks ? &launchDilatedBlock<2, 3, 1>
                                             : &launchDilatedBlock<2, 3, 2>;
    return go(d, outType, in, weightsPacked, bias, out, stream);
  }
  a.divVecs = makeFastDiv(a.vecs);
  a.divOutW = makeFastDiv(d.outW);
  a.divOutH = makeFastDiv(d.outH);
  a.divInDilH = makeFastDiv(d.inDilH);
  a.divInDilW = makeFastDiv(d.inDilW);
  const dim3 grid{uint32_t((a.items + 255) / 256)}, block{256};
  if (inType == kFloat && outType == kFloat)
    hipLaunchKernelGGL((depthwiseDirectKernel<float, float>), grid, block, 0,
                       stream, a, static_cast<const float *>(in),
                       static_cast<const float *>(weightsPacked),
                       static_cast<const float *>(bias),
                       static_cast<float *>(out));
  else if (inType == kFloat && outType == kHalf)
    hipLaunchKernelGGL((depthwiseDirectKernel<__half, float>), grid, block, 0,
                       stream, a, static_cast<const float *>(in),
                       static_cast<const float *>(weightsPacked),
                       static_cast<const __half *>(bias),
                       static_cast<__half *>(out));
  else if (outType == kHalf)
    hipLaunchKernelGGL(depthwiseDirectKernel<__half>, grid, block, 0, stream, a,
                       static_cast<const __half *>(in),
                       static_cast<const __half *>(weightsPacked),
                       static_cast<const __half *>(bias),
                       static_cast<__half *>(out));
  else if (outType == kFloat)
    hipLaunchKernelGGL(depthwiseDirectKernel<float>, grid, block, 0, stream, a,
                       static_cast<const __half *>(in),
                       static_cast<const __half *>(weightsPacked),
                       static_cast<const float *>(bias),
                       static_cast<float *>(out));
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

size_t depthwiseWeightDeltaWorkspaceBytes(const DepthwiseDesc &d) {
  if (d.dense3x3 == 2)
    return depthwiseRowsDeltaWorkspaceBytes(d);
  if (d.columns)
    return size_t(depthwiseColumnDeltasSlices(d)) * d.kH * d.kW * d.channels *
           sizeof(float);
  return size_t(deltaSlices(d)) * d.kH * d.kW * d.channels * sizeof(float);
}

hipError_t launchDepthwiseWeightDeltas(const DepthwiseDesc &d, int outType,
                                       const void *acts, const void *deltas,
                                       void *workspace, void *weightDeltas,
                                       hipStream_t stream) {
  // half tensors, or fp32 ones (the slices' walk only)
  const uint32_t perVec = 16 / d.elemBytes;
  if ((d.elemBytes != 2 && d.elemBytes != 4) || d.channels % perVec != 0 ||
      d.inDilH != 1 || d.inDilW != 1 || (d.elemBytes == 4 && d.dense3x3 == 2))
    return hipErrorInvalidValue;
  DeltaArgs a;
  a.d = d;
  a.vecs = d.channels / perVec;
  a.taps = d.kH * d.kW;
  const uint64_t items = uint64_t(a.taps) * a.vecs;
  const uint64_t pixels = uint64_t(d.batch) * d.outH * d.outW;
  if (items == 0)
    return hipSuccess;
  if (items >= (1ull << 31) || pixels >= (1ull << 31) || !workspace)
    return hipErrorInvalidConfiguration;
  a.items = uint32_t(items);
  a.pixels = uint32_t(pixels);
  float *partial = static_cast<float *>(workspace);
  if (d.dense3x3 == 2) {
    // persistent workgroups with the rows in LDS rings: one tile each
    const hipError_t e = launchDepthwiseRowsDeltas(d, acts, deltas, partial,
                                                   &a.slices, stream);
    if (e != hipSuccess)
      return e;
  } else if (d.columns) {
    a.slices = depthwiseColumnDeltasSlices(d);
    const hipError_t e =
        launchDepthwiseColumnDeltas(d, acts, deltas, partial, stream);
    if (e != hipSuccess)
      return e;
  } else {
    a.slices = deltaSlices(d);
    deltaBlockShape(d, a.itemsPerBlock, a.slots);
    a.pixelsPerSlice = uint32_t((pixels + a.slices - 1) / a.slices);
    a.pixelsPerSlot = (a.pixelsPerSlice + a.slots - 1) / a.slots;
    a.divVecs = makeFastDiv(a.vecs);
    a.divOutW = makeFastDiv(d.outW);
    a.divOutH = makeFastDiv(d.outH);
    const dim3 grid{uint32_t((items + a.itemsPerBlock - 1) / a.itemsPerBlock),
                    a.slices},
        block{256};
    if (d.elemBytes == 4)
      hipLaunchKernelGGL(depthwiseWeightDeltaKernel<float>, grid, block, 0,
                         stream, a, static_cast<const float *>(acts),
                         static_cast<const float *>(deltas), partial);
    else
      hipLaunchKernelGGL(depthwiseWeightDeltaKernel<__half>, grid, block, 0,
                         stream, a, static_cast<const __half *>(acts),
                         static_cast<const __half *>(deltas), partial);
  }
  if (outType == kHalf)
    launchDeltaSum<__half>(partial, a.slices, a.taps, d.channels, weightDeltas,
                           stream);
  else if (outType == kFloat)
    launchDeltaSum<float>(partial, a.slices, a.taps, d.channels, weightDeltas,
                          stream);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

} // namespace mxk
